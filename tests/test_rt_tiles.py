"""The patched RT sweep (rt_sweep_tile_kernel in miso_amd/csrc/rt.hip).

On the CPU, its patches emulated with a stand-in node function: 64 columns x
32 rows, P planes per launch, the upwind P columns and rows of a neighbouring
patch computed again.  Every swept node is stored once, no address lies
outside the ray's field, and the values are those of the plane-by-plane
sweep -- so the stale edge of a patch never reaches a node that it stores.
On the GPU: every intensity, the iterations, the last change and Q_rad equal
the one-plane-per-launch sweep's bit for bit, at sizes around a patch's edges.
"""
import itertools

import numpy as np
import pytest

from tests.test_rt_cone import _node, _plane_sweep, _ray

COLS, ROWS = 64, 32


def _patches(n, size, P):
    return 1 if n < size else 1 + -(-(n - (size - 1)) // (size - P))


def _first(a, size, P):
    return -1 if a == 0 else size - 1 + (a - 1) * (size - P) - P


def _patched_sweep(R, I, K, S, P, n):
    nb, nc = R["nb"], R["nc"]
    for p0 in range(0, R["nplanes"], P):
        start, writes = I.copy(), {}
        for a, b in itertools.product(range(_patches(nb, COLS, P)), range(_patches(nc, ROWS, P))):
            u0, v0 = _first(a, COLS, P), _first(b, ROWS, P)
            u, v = u0 + np.arange(COLS), v0 + np.arange(ROWS)[:, None]
            uown, vown = (u0 + P if a else 0), (v0 + P if b else 0)
            own = (u >= uown) & (u < nb) & (v >= vown) & (v < nc)
            bound = (u < 0) | (v < 0)

            def index(uu, vv, p):
                uu, vv = np.minimum(uu, nb - 1), np.clip(vv, -1, nc - 1)
                col = (uu + 1 if R["sb"] > 0 else nb - uu) * R["db"]
                assert (col >= 0).all() and (8 * col < 2 ** 32).all()
                row = R["start"] - R["db"] + (vv if R["sc"] > 0 else nc - 1 - vv) * R["dc"]
                c = row + col + p * R["da"]
                assert (c >= 0).all() and (c < n).all()
                return c

            c = index(u, v, p0 - 1)
            pi, pk, ps = start[c], K[c], S[c]
            for p in range(p0, min(p0 + P, R["nplanes"])):
                c = index(u, v, p)
                before = start[index(np.maximum(u, uown if a and b else -1),
                                     np.maximum(v, vown if a and b else -1), p)]

                def up(f):  # a lane's and a row's upwind neighbours; stale ones at the edge
                    f10 = np.concatenate([np.full((ROWS, 1), np.nan), f[:, :-1]], 1)
                    f01 = np.concatenate([f[:1], f[:-1]])
                    f11 = np.concatenate([f10[:1], f10[:-1]])
                    return f, f10, f01, f11

                now = _node(*up(pi), *up(ps), *up(pk), K[c], S[c])
                for cc, x in zip(c[own], now[own]):
                    assert cc not in writes
                    writes[int(cc)] = x
                pi, pk, ps = np.where(bound, before, now), K[c], S[c]
        for cc, x in writes.items():
            I[cc] = x


@pytest.mark.parametrize("dims", [(8, 8, 8), (68, 6, 36), (70, 38, 12), (36, 70, 21)])
@pytest.mark.parametrize("P", [2, 5, 16])
def test_patches_give_the_plane_sweep(dims, P):
    rng = np.random.default_rng(1)
    n = dims[0] * dims[1] * dims[2]
    K, S, I0 = rng.random(n), rng.random(n), rng.random(n)
    for dom, t, tr in ((0, (1, -1, 1), True), (0, (-1, 1, 1), False), (1, (-1, 1, -1), False),
                       (2, (1, 1, -1), False), (2, (-1, -1, 1), False)):
        R = _ray(dims, 2, dom, t, tr)
        want, got = I0.copy(), I0.copy()
        _plane_sweep(R, want, K, S)
        _patched_sweep(R, got, K, S, P, n)
        assert np.array_equal(want, got)


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,planes", [
    ((2, 2, 2), 2), ((16, 31, 16), 16), ((63, 32, 33), 16), ((64, 33, 15), 7),
    ((65, 127, 34), 4), ((130, 18, 60), 5), ((31, 64, 128), 3),
])
def test_patches_equal_the_plane_sweep_on_the_gpu(ctx, sizes, planes):
    import torch

    from miso_amd import mhd
    from miso_amd.rt import RT
    g = mhd.Grid(*sizes, 2, bounds=((0, 1), (0, 1), (0, 1)), device="cuda:0")
    rng = np.random.default_rng(3)
    shp = (g.k_total, g.j_total, g.i_total)
    kap = torch.from_numpy(20.0 * rng.random(shp) ** 3).to("cuda:0")
    S = torch.from_numpy(1 + 0.3 * rng.random(shp)).to("cuda:0")
    out = []
    for pl, yf in ((0, True), (planes, True), (planes, False)):
        rt = RT(g, 24)
        rt.abs_coeff.copy_(kap)
        rt.src_func.copy_(S)
        kw = dict(periodic=(True, True, False), face_kind=(0, 0, 0, 0, 1, 2), tolerance=1e-9,
                  max_iters=12, sweep_planes=pl, x_rays_yfast=yf)
        res = rt.solve(ctx, **kw)
        q = rt.qrad(ctx, **kw).cpu()
        out.append((res, rt.intensities().cpu(), q))
    for res, I, q in out[1:]:
        assert res == out[0][0]
        assert torch.equal(I, out[0][1])
        assert torch.equal(q, out[0][2])


# the two heights of a patch with the planes each takes per launch; sixteen
# planes only where a short patch holds a ray's whole c axis
@pytest.mark.parametrize("dims", [(8, 8, 8), (68, 6, 36), (70, 38, 12), (36, 70, 21), (22, 150, 9)])
@pytest.mark.parametrize("rows,P", [(32, 8), (20, 8), (20, 16)])
def test_patch_heights_give_the_plane_sweep(monkeypatch, dims, rows, P):
    import sys
    monkeypatch.setattr(sys.modules[__name__], "ROWS", rows)
    rng = np.random.default_rng(2)
    n = dims[0] * dims[1] * dims[2]
    K, S, I0 = rng.random(n), rng.random(n), rng.random(n)
    cases = 0
    for dom, t, tr in ((0, (1, -1, 1), True), (1, (-1, 1, -1), False), (2, (1, 1, -1), False)):
        R = _ray(dims, 2, dom, t, tr)
        if P > 8 and R["nc"] >= rows:
            continue
        want, got = I0.copy(), I0.copy()
        _plane_sweep(R, want, K, S)
        _patched_sweep(R, got, K, S, P, n)
        assert np.array_equal(want, got)
        cases += 1
    assert cases > 0


def _equal_to_plane_sweep(ctx, sizes, rays, kinds, max_iters):
    import torch

    from miso_amd import mhd
    from miso_amd.rt import RT
    g = mhd.Grid(*sizes, 2, bounds=((0, 1), (0, 1), (0, 1)), device="cuda:0")
    gen = torch.Generator(device="cuda:0").manual_seed(7)
    shp = (g.k_total, g.j_total, g.i_total)
    kap, S = (torch.rand(shp, generator=gen, device="cuda:0", dtype=torch.float64)
              for _ in range(2))
    out = []
    for pl, yf in ((0, True),) + kinds:
        rt = RT(g, rays)
        rt.abs_coeff.copy_(20.0 * kap ** 3)
        rt.src_func.copy_(1 + 0.3 * S)
        kw = dict(periodic=(True, True, False), face_kind=(0, 0, 0, 0, 1, 2), tolerance=1e-9,
                  max_iters=max_iters, sweep_planes=pl, x_rays_yfast=yf)
        res = rt.solve(ctx, **kw)
        q = rt.qrad(ctx, **kw).clone()
        out.append((res, rt.intensities().clone(), q))
        del rt
    for res, I, q in out[1:]:
        assert res == out[0][0]
        assert torch.equal(I, out[0][1])
        assert torch.equal(q, out[0][2])


# boxes of few nodes along one axis: sixteen planes a launch, in patches wider
# and narrower than the box, and of one ray
@pytest.mark.gpu
@pytest.mark.parametrize("sizes,rays", [((300, 40, 2), 24), ((131, 70, 19), 24), ((131, 70, 18), 24),
                                        ((70, 16, 16), 24), ((16, 150, 12), 24), ((90, 2, 35), 1),
                                        ((1100, 900, 3), 24)])
def test_thin_boxes_equal_the_plane_sweep(ctx, sizes, rays):
    _equal_to_plane_sweep(ctx, sizes, rays, ((16, True), (2, True)), 6)


# every ray x-fastest: x rays in cones (up to 32 nodes along z, planes of one and
# of several workgroups), by planes and in patches
@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(70, 31, 32), (73, 32, 31), (170, 70, 3), (20, 33, 33),
                                   (20, 20, 20), (70, 75, 72), (110, 112, 115)])
def test_one_layout_equals_the_plane_sweep(ctx, sizes):
    _equal_to_plane_sweep(ctx, sizes, 24, ((16, False), (4, False), (0, False)), 4)


# axes of at least 128 workgroups: patches of 32 rows, an axis' rays in launches
# and on a stream of their own; boxes with all, two and one of the axes so
@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [(128, 128, 128), (150, 131, 187), (70, 260, 250), (384, 384, 27)])
def test_full_launches_equal_the_plane_sweep(ctx, sizes):
    _equal_to_plane_sweep(ctx, sizes, 24, ((16, True),), 3)
