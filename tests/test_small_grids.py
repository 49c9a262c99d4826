"""Small and ragged grids against the oracle, bit for bit: launches cut into
chunks of one cell or plane, and the ghost cells that the passes of an x-y
run store beside their sources (whole arrays, corners included)."""
import numpy as np
import pytest

from tests.parity_util import assert_bitwise, random_state

# components that change sign across a wall of each axis
SIGNS = tuple(tuple(-1 if f in (1 + a, 4 + a) else 1 for f in range(9)) for a in range(3))


def _both(ctx, sizes, periodic, nsteps, use_run):
    from miso_amd import mhd
    from oracle import oracle as O
    og = O.make_grid(sizes, 2, dtype=np.float64)
    op = O.Params(cfl_number=0.4, periodic=periodic, sym_sign=SIGNS)
    g = mhd.Grid(*sizes, 2, dtype=np.float64, device="cuda:0")
    ref = random_state((g.i_total, g.j_total, g.k_total), 3, amp=0.05)
    O.ghost_fill(og, op, ref)
    q0 = ref.copy()
    ref_dts = O.run(og, op, ref, nsteps)
    O.ghost_fill(og, op, ref)
    m = mhd.MHD(mhd.Config({"mhd": {"cfl_number": 0.4}}), g, ctx, gm=5.0 / 3.0)
    bc = mhd.BoundaryCondition(periodic, SIGNS)
    m.apply_initial_condition(q0, bc)
    if use_run:
        dts = m.integrator.run(bc, m.qq, nsteps)
    else:
        dts = [m.integrator.step(bc, m.qq) for _ in range(nsteps)]
    return m.qq.to_host(ctx), ref, np.array(dts), ref_dts


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(2, 2, 1), (3, 5, 1), (64, 4, 1), (7, 61, 1), (129, 66, 1)])
@pytest.mark.parametrize("periodic", [(1, 1, 1), (0, 1, 1), (1, 0, 1), (0, 0, 1)])
@pytest.mark.parametrize("use_run", [False, True])
def test_xy_runs_with_their_ghost_cells(ctx, sizes, periodic, use_run):
    out, ref, dts, ref_dts = _both(ctx, sizes, periodic, 3, use_run)
    assert np.array_equal(dts, ref_dts), (dts, ref_dts)
    assert_bitwise(out, ref, f"{sizes} {periodic}")


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(4, 3, 2), (65, 2, 3), (61, 9, 1 + 64), (6, 131, 5)])
@pytest.mark.parametrize("periodic", [(1, 1, 1), (0, 0, 0), (1, 0, 1)])
def test_3d_runs_in_the_shortest_chunks(ctx, sizes, periodic):
    out, ref, dts, ref_dts = _both(ctx, sizes, periodic, 3, True)
    assert np.array_equal(dts, ref_dts), (dts, ref_dts)
    sl = (slice(None),) + (slice(2, -2),) * 3  # the oracle's 3D edges keep what was there
    assert_bitwise(out[sl], ref[sl], f"{sizes} {periodic}")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("sizes", [(61, 32790, 1), (61, 32700, 1)])
def test_long_strips_on_both_sides_of_the_y_walk(ctx, dtype, sizes):
    """A strip of 61 cells in x, long enough in y for the walking RK stage (4100
    waves) and just not (4088): the bits of the one-plane kernel."""
    from miso_amd import mhd
    from miso_amd.autotune import get_tiles, set_tiles
    t0 = get_tiles(ctx)
    default = (t0.rk_pencil_bx, t0.rk_pencil_by, t0.sweep_chunk, t0.rk_variant, t0.rk_zchunk,
               t0.av_fuse_xy, t0.av_xy_chunk)
    g = mhd.Grid(*sizes, 2, dtype=dtype, device="cuda:0")
    q0 = random_state((g.i_total, g.j_total, g.k_total), 4, dtype, amp=0.05)
    bc = mhd.BoundaryCondition((1, 0, 1), SIGNS)
    out = []
    for variant in (0, 5):
        set_tiles(ctx, 2, 8, 256, variant, 256, 1, 64)
        try:
            m = mhd.MHD(mhd.Config({"mhd": {"cfl_number": 0.4}}), g, ctx, gm=5.0 / 3.0)
            m.apply_initial_condition(q0, bc)
            dts = m.integrator.run(bc, m.qq, 2)
            out.append((list(dts), m.qq.to_host(ctx)))
        finally:
            set_tiles(ctx, *default)
    assert out[0][0] == out[1][0]
    assert_bitwise(out[1][1], out[0][1], str(sizes))


def _fills(ctx, fn):
    """Ghost fills launched by fn()."""
    import ctypes as C

    from miso_amd import hip
    hip.call("misohip_profile_enable", ctx.handle, 1)
    try:
        fn()
        ms, n = (C.c_double * 8)(), (C.c_int * 8)()
        hip.call("misohip_profile_read", ctx.handle, ms, n, 8)
    finally:
        hip.call("misohip_profile_enable", ctx.handle, 0)
    return n[4]


# the passes store the ghost cells up to a number of rows, by type and by the RK
# stage's kernel: beyond, that costs more than the fills
@pytest.mark.gpu
@pytest.mark.parametrize("dtype,sizes,fills", [
    (np.float64, (5, 6144, 1), 0), (np.float64, (5, 6145, 1), 12),
    (np.float32, (5, 20480, 1), 0), (np.float32, (5, 20481, 1), 12),
    (np.float64, (2000, 1920, 1), 0), (np.float64, (2000, 1936, 1), 12),
    (np.float32, (1300, 3072, 1), 0), (np.float32, (1300, 3073, 1), 12),
])
def test_ghost_fills_where_images_cost_more(ctx, dtype, sizes, fills):
    import torch
    from miso_amd import mhd
    g = mhd.Grid(*sizes, 2, dtype=dtype, device="cuda:0")
    m = mhd.MHD(mhd.Config({"mhd": {"cfl_number": 0.4}}), g, ctx, gm=5.0 / 3.0)
    bc = mhd.BoundaryCondition((1, 0, 1), SIGNS)
    m.apply_initial_condition(random_state((g.i_total, g.j_total, g.k_total), 4, dtype, amp=0.05),
                              bc)
    assert _fills(ctx, lambda: m.integrator.run(bc, m.qq, 2)) == fills
    q = m.qq.data.clone()
    m.integrator.apply_boundary_condition(bc, m.qq)
    assert torch.isfinite(q).all() and torch.equal(q, m.qq.data)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(5, 6144, 1), (5, 6145, 1)])
def test_strips_on_both_sides_of_the_images(ctx, sizes):
    out, ref, dts, ref_dts = _both(ctx, sizes, (1, 0, 1), 2, True)
    assert np.array_equal(dts, ref_dts), (dts, ref_dts)
    assert_bitwise(out, ref, str(sizes))
