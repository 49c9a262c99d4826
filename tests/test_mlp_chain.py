"""The network in one launch (forward, and forward with the way back), the
weight gradients of all layers in one launch and the update with its packed
weight copies, at the sizes where their tiles end: against the float64
oracle, with its bf16 rounding points."""
import ctypes as C

import numpy as np
import pytest

from oracle import mlp_oracle as MO
from tests.test_mlp import GpuMLP, _bf16_dev, _params


def _ptr(t):
    return C.c_void_p(t.data_ptr())


def _net(ctx, sizes, max_batch, seed):
    Ws, bs = _params(sizes, seed)
    Ws = [w.astype(np.float32).astype(np.float64) for w in Ws]
    bs = [b.astype(np.float32).astype(np.float64) for b in bs]
    net = GpuMLP(ctx, sizes, max_batch)
    net.set(Ws, bs)
    return net, Ws, bs


def _grad(net, ctx, Xd, Td):
    loss = C.c_double()
    net.hip.call("misohip_mlp_grad", ctx.handle, net.h, _ptr(Xd), _ptr(Td), Xd.shape[0],
                 C.byref(loss))
    return loss.value


def _check_grads(net, Ws, bs, X, T, loss):
    lref, gW, gb = MO.loss_and_grads([MO.to_bf16(w) for w in Ws], bs, X, T)
    assert abs(loss - lref) <= 1e-3 * lref
    for l in range(len(Ws)):
        for which, ref in ((2, gW[l]), (3, gb[l])):
            g = net.get(l, which)
            assert np.linalg.norm(g - ref) <= 2e-2 * np.linalg.norm(ref), (l, which)


# one k-step and one tile of everything; odd numbers of tiles and k-steps; more
# outputs than one pass of 16 waves; X in two chunks; activations in global
# memory; a batch of many folds of the gradients' sums
@pytest.mark.gpu
@pytest.mark.parametrize("sizes,batch", [
    ([32, 32, 32], 32), ([96, 160, 96], 96), ([160, 96, 96, 224], 160),
    ([64, 288, 544], 64), ([2080, 64, 64], 32), ([64, 1600, 1600, 32], 64),
    ([1536, 256, 256, 256, 384], 1024), ([64, 64, 32], 8192)])
def test_gradients_and_update_at_tile_edges(ctx, sizes, batch):
    import torch
    net, Ws, bs = _net(ctx, sizes, batch, 11)
    rng = np.random.default_rng(12)
    X = MO.to_bf16(rng.standard_normal((batch, sizes[0])))
    T = rng.standard_normal((batch, sizes[-1])).astype(np.float32).astype(np.float64)
    Xd, Td = _bf16_dev(X), torch.from_numpy(T.astype(np.float32)).to("cuda:0")
    _check_grads(net, Ws, bs, X, T, _grad(net, ctx, Xd, Td))
    # the update, by the gradients just read, and both packed copies after it
    g = [net.get(l, w) for w in (2, 3) for l in range(len(Ws))]
    net.hip.call("misohip_mlp_adam", ctx.handle, net.h, C.c_float(1e-2), C.c_float(0.9),
                 C.c_float(0.999), C.c_float(1e-8), C.c_float(0.0))
    p = [w.copy() for w in Ws] + [b.copy() for b in bs]
    MO.adam_step(p, g, {}, 1e-2)
    new = [net.get(l, w) for w in (0, 1) for l in range(len(Ws))]
    for a, b in zip(new, p):  # fp32 against float64: the step itself is 1e-2
        assert np.abs(a - b).max() <= 1e-6 * max(1.0, np.abs(b).max())
    n = len(Ws)
    _check_grads(net, new[:n], new[n:], X, T, _grad(net, ctx, Xd, Td))
    net.close()


# single columns and partial tiles of 16; from 8192 columns on, tiles of 64
@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[32, 32, 32], [96, 160, 96], [224, 256, 256, 288],
                                   [64, 608, 64], [64, 640, 64], [64, 32, 1600]])
@pytest.mark.parametrize("batch", [1, 17, 8192, 8255])
def test_forward_at_tile_edges(ctx, sizes, batch):
    import torch
    net, Ws, bs = _net(ctx, sizes, 8256, 13)
    X = MO.to_bf16(np.random.default_rng(14).standard_normal((batch, sizes[0])))
    Y = torch.full((batch + 1, sizes[-1]), 7.0, dtype=torch.float32, device="cuda:0")
    net.hip.call("misohip_mlp_forward", ctx.handle, net.h, _ptr(_bf16_dev(X)), batch, _ptr(Y))
    torch.cuda.synchronize()
    ref, _, _ = MO.forward([MO.to_bf16(w) for w in Ws], bs, X)
    got = Y.cpu().numpy()
    assert np.abs(got[:batch] - ref).max() <= 2e-3 * np.abs(ref).max()
    assert (got[batch] == 7.0).all()  # nothing past the batch
    net.close()


@pytest.mark.gpu
@pytest.mark.parametrize("ni,nj,nz,n_hidden", [(9, 7, 32, 64), (97, 85, 32, 64),
                                               (40, 33, 1600, 32)])
def test_qrad_field_is_the_scaled_output(ctx, ni, nj, nz, n_hidden):
    """Q_rad of every column from Y, mu, sd, with and without the correction,
    flagged columns from q_rt; ghosts untouched; in batches where the
    activations' global buffers hold fewer columns than the box."""
    import torch
    from miso_amd import hip, mhd
    grid = mhd.Grid(ni, nj, nz, 2, dtype=np.float64, device="cuda:0")
    nc = ni * nj
    net, _, _ = _net(ctx, [3 * nz, n_hidden, nz], 64, 15)
    rng = np.random.default_rng(16)
    mu, sd = (rng.standard_normal(nz).astype(np.float32) for _ in range(2))
    z = np.zeros(3 * nz, np.float32)
    hip.call("misohip_mlp_set_norm", ctx.handle, net.h,
             *(a.ctypes.data_as(C.POINTER(C.c_float)) for a in (z, z + 1, mu, sd)))
    gen = torch.Generator(device="cuda:0").manual_seed(17)
    X = torch.randn((nc, 3 * nz), generator=gen, device="cuda:0").to(torch.bfloat16)
    Y = torch.empty((nc, nz), dtype=torch.float32, device="cuda:0")
    shape = (nz + 4, nj + 4, ni + 4)
    q_rt, corr = (torch.randn(shape, generator=gen, device="cuda:0", dtype=torch.float64)
                  for _ in range(2))
    flags = (torch.rand(nc, generator=gen, device="cuda:0") < 0.3).int()
    inner = (slice(2, -2),) * 3
    for c, f in ((None, None), (corr, flags)):
        q = torch.full(shape, 5.0, dtype=torch.float64, device="cuda:0")
        hip.call("misohip_mlp_qrad", ctx.handle, net.h, C.byref(grid.c_struct()), _ptr(X), _ptr(Y),
                 _ptr(f) if f is not None else None, _ptr(q_rt),
                 _ptr(c) if c is not None else None, _ptr(q))
        torch.cuda.synchronize()
        ref = (Y * torch.from_numpy(sd).cuda() + torch.from_numpy(mu).cuda()).double()
        ref = ref.reshape(nj, ni, nz).permute(2, 0, 1)
        if c is not None:
            ref = ref + c[inner]
            ref = torch.where(f.reshape(nj, ni).bool(), q_rt[inner], ref)
        want = torch.full(shape, 5.0, dtype=torch.float64, device="cuda:0")
        want[inner] = ref
        assert torch.equal(q, want)
    net.close()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "float64"])
@pytest.mark.parametrize("n,width,chosen", [(1, 4, 1), (7, 60, 3), (300, 64, 257), (5, 1536, 2),
                                            (4100, 132, 4097)])
def test_training_data_moments_and_scaling(dtype, n, width, chosen):
    """Column moments of chosen rows and the scaled columns against torch in
    64 bits; the scaled values are the same bits."""
    import torch
    from miso_amd import surrogate
    g = torch.Generator().manual_seed(n)
    x = (torch.randn((n, width), generator=g, dtype=torch.float64) * 0.1 - 1.0).to("cuda:0")
    x = x.to(getattr(torch, dtype))
    rows = torch.randperm(n, generator=g)[:chosen].to("cuda:0")
    mean, sd, mean_abs = surrogate._moments(x, rows)
    ref = x[rows].double()
    eps = 2.0 ** -52 * chosen  # a sum's rounding, of values of magnitude one
    assert (mean - ref.mean(0)).abs().max() <= eps
    assert (mean_abs - ref.abs().mean(0)).abs().max() <= eps
    if chosen > 1:
        assert ((sd - ref.std(0)).abs() <= 1e3 * eps * ref.std(0)).all()
    else:
        assert torch.isnan(sd).all()
    sd = sd.nan_to_num(nan=0.1).clamp_min(1e-12)
    want = (x.double() - mean) / sd
    assert torch.equal(surrogate._normalized(x, mean, sd, torch.bfloat16), want.to(torch.bfloat16))
    assert torch.equal(surrogate._normalized(x, mean, sd, torch.float32), want.float())
    odd = torch.cat([x[:1], x])[1:]  # rows from an odd offset on
    assert torch.equal(surrogate._normalized(odd, mean, sd, torch.float32), want.float())


@pytest.mark.gpu
def test_training_data_with_the_features_as_an_axis(ctx):
    """Raw features as (N, features, nz): each row's values in the order of
    (N, features nz), and the same weights."""
    import torch
    from miso_amd import surrogate
    nz, n = 32, 160
    g = torch.Generator().manual_seed(3)
    feats = (torch.randn((n, 4, nz), generator=g) * 0.1 + 1).to("cuda:0")
    targets = torch.randn((n, nz), generator=g, dtype=torch.float64).to("cuda:0")
    got = []
    for f in (feats.reshape(n, 4 * nz), feats):
        s = surrogate.ColumnSurrogate(ctx, nz, hidden=32, features=4, max_batch=64, seed=5)
        last, val = s.fit(f, targets, epochs=2, batch=32)
        w = []
        for layer, (i, o) in enumerate(zip(s.sizes[:-1], s.sizes[1:])):
            a = np.zeros((o, i), np.float32)
            from miso_amd import hip
            hip.call("misohip_mlp_get_layer", ctx.handle, s.h, layer, 0, a.ctypes.data_as(C.c_void_p))
            w.append(a)
        got.append((last, val, w, [a.ravel() for a in s.norm]))
        s.close()
    assert got[0][:2] == got[1][:2] and np.isfinite(got[0][1])
    for k in (2, 3):
        for a, b in zip(got[0][k], got[1][k]):
            assert np.array_equal(a, b)


@pytest.mark.gpu
def test_fit_of_no_rows(ctx):
    """No training data: NaN moments, no step, the weights as they were."""
    import torch
    from miso_amd import hip, surrogate
    nz = 32
    s = surrogate.ColumnSurrogate(ctx, nz, hidden=32, max_batch=64, seed=5)

    def weights():
        a = np.zeros((32, 3 * nz), np.float32)
        hip.call("misohip_mlp_get_layer", ctx.handle, s.h, 0, 0, a.ctypes.data_as(C.c_void_p))
        return a
    before = weights()
    assert s.fit(torch.empty((0, 3 * nz), device="cuda:0"),
                 torch.empty((0, nz), dtype=torch.float64, device="cuda:0"), epochs=2,
                 batch=32) == (0.0, None)
    assert len(s.history) == 2 and all(np.isnan(a).all() for a in s.norm)
    assert np.array_equal(weights(), before)
    s.close()


@pytest.mark.parametrize("feats,targets,error", [
    (dict(size=(100, 96)), dict(size=(99, 32)), IndexError),
    (dict(size=(100, 96)), dict(size=(0, 32)), IndexError),
    (dict(size=(100, 96)), dict(size=(100, 32), device="meta"), RuntimeError),
])
def test_fit_refuses_targets_it_would_read_past(feats, targets, error):
    """Fewer targets than feature rows, or targets elsewhere: refused before any
    kernel gets their pointers."""
    import torch
    from miso_amd.surrogate import ColumnSurrogate
    s = ColumnSurrogate.__new__(ColumnSurrogate)
    s.h = None
    with pytest.raises(error, match="target"):
        s.fit(torch.zeros(**feats), torch.zeros(**targets))


# hidden layers above 1024 in inference, and above what LDS holds in training: a
# launch per layer, 16 or 64 columns to a workgroup by their number, one or more
# rows of workgroups over the outputs; inputs in two chunks
@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [[64, 1056, 1056, 96], [32, 1600, 1600, 32], [2080, 2112, 160]])
@pytest.mark.parametrize("batch", [1, 17, 1100, 2081])
def test_forward_by_layers(ctx, sizes, batch):
    import torch
    net, Ws, bs = _net(ctx, sizes, 2112, 13)
    X = MO.to_bf16(np.random.default_rng(14).standard_normal((batch, sizes[0])))
    Y = torch.full((batch + 1, sizes[-1]), 7.0, dtype=torch.float32, device="cuda:0")
    net.hip.call("misohip_mlp_forward", ctx.handle, net.h, _ptr(_bf16_dev(X)), batch, _ptr(Y))
    torch.cuda.synchronize()
    ref, _, _ = MO.forward([MO.to_bf16(w) for w in Ws], bs, X)
    got = Y.cpu().numpy()
    assert np.abs(got[:batch] - ref).max() <= 2e-3 * np.abs(ref).max()
    assert (got[batch] == 7.0).all()
    net.close()


@pytest.mark.gpu
@pytest.mark.parametrize("sizes,batch", [([32, 1600, 32], 32), ([2080, 2112, 2112, 96], 96),
                                         ([32, 64, 2080], 64)])
def test_gradients_by_layers(ctx, sizes, batch):
    import torch
    net, Ws, bs = _net(ctx, sizes, batch, 11)
    rng = np.random.default_rng(12)
    X = MO.to_bf16(rng.standard_normal((batch, sizes[0])))
    T = rng.standard_normal((batch, sizes[-1])).astype(np.float32).astype(np.float64)
    _check_grads(net, Ws, bs, X, T,
                 _grad(net, ctx, _bf16_dev(X), torch.from_numpy(T.astype(np.float32)).to("cuda:0")))
    net.close()
