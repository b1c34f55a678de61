"""GPU: the surrogate network's forward pass and gradients (bec_fno_*, BF16 MFMA
GEMMs with FP32 accumulation) against the FP64 numpy oracle at a small size,
determinism of the gradients, and an optimiser smoke test."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CFG = dict(nz=32, ny=8, nx=8, mz=8, my=8, mx=8, width=8, layers=2, c_in=5, c_out=2, hidden=16, max_batch=3)


def _setup(seed=0):
    from bec_amd import fno as F
    from oracle import fno_oracle as FO
    net = F.FNO(seed=seed, **CFG)
    ocfg = FO.Config.from_struct(net.cfg)
    assert net.n_params == FO.param_count(ocfg)
    rng = np.random.default_rng(seed)
    cells = CFG["nz"] * CFG["ny"] * CFG["nx"]
    x = rng.normal(size=(3, cells, CFG["c_in"])).astype(np.float32)
    t = rng.normal(size=(3, cells, CFG["c_out"])).astype(np.float32)
    return F, FO, net, ocfg, x, t


def _grid(a, cfg):
    return a.reshape(a.shape[0], cfg.nz, cfg.ny, cfg.nx, a.shape[-1]).astype(np.float64)


def _blocks(cfg):
    W, H = cfg.width, cfg.hidden
    modes = cfg.mz * cfg.my * cfg.mx
    names = ["P", "p"]
    sizes = [cfg.c_in * W, W]
    for l in range(cfg.layers):
        names += [f"W{l}", f"b{l}", f"R{l}"]
        sizes += [W * W, W, modes * W * W * 2]
    names += ["Q1", "q1", "Q2", "q2"]
    sizes += [W * H, H, H * cfg.c_out, cfg.c_out]
    o = 0
    for n, s in zip(names, sizes):
        yield n, slice(o, o + s)
        o += s


def test_forward_and_gradients_match_oracle(bec):
    F, FO, net, ocfg, x, t = _setup()
    flat = net.get_params().astype(np.float64)
    y_gpu = net.predict(x)
    y_ref = FO.forward(ocfg, flat, _grid(x, ocfg)).reshape(y_gpu.shape)
    err = np.linalg.norm(y_gpu - y_ref) / np.linalg.norm(y_ref)
    print("forward rel L2 vs FP64 oracle:", err)
    assert err < 2e-2
    dx = F.DeviceArray(x.shape, np.float32, x)
    dt = F.DeviceArray(t.shape, np.float32, t)
    loss = net.loss_backward(dx, dt, 3)
    g_gpu = net.get_grads().astype(np.float64)
    loss_ref, g_ref = FO.loss_and_grads(ocfg, flat, _grid(x, ocfg), _grid(t, ocfg))
    assert loss == pytest.approx(loss_ref, rel=2e-2)
    report = {}
    for name, sl in _blocks(ocfg):
        a, b = g_gpu[sl], g_ref[sl]
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        cos = float(a @ b / (np.linalg.norm(a) * np.linalg.norm(b) + 1e-30))
        report[name] = (round(rel, 5), round(cos, 6))
        assert rel < 5e-2 and cos > 0.998, (name, rel, cos)
    print("gradient blocks (rel L2, cosine) vs FP64 oracle:", report)


def test_gradients_are_deterministic(bec):
    F, FO, net, ocfg, x, t = _setup(1)
    dx = F.DeviceArray(x.shape, np.float32, x)
    dt = F.DeviceArray(t.shape, np.float32, t)
    l1 = net.loss_backward(dx, dt, 3)
    g1 = net.get_grads()
    l2 = net.loss_backward(dx, dt, 3)
    g2 = net.get_grads()
    assert l1 == l2 and np.array_equal(g1, g2)


def test_adam_reduces_the_loss(bec):
    F, FO, net, ocfg, x, t = _setup(2)
    t = 0.3 * np.tanh(x[..., :2])            # a learnable per-cell target
    dx = F.DeviceArray(x.shape, np.float32, x)
    dt = F.DeviceArray(t.shape, np.float32, t)
    losses = []
    for _ in range(60):
        losses.append(net.loss_backward(dx, dt, 3))
        net.adam_step(3e-3)
    print("loss", losses[0], "->", losses[-1])
    assert losses[-1] < 0.2 * losses[0]


def test_production_size_forward_matches_oracle(bec):
    """The production network at batch 1 (the per-mode channel mixing on its one-row
    kernel, the plane transforms split in K) and at batch 2 (the mixing on the GEMM):
    the forward pass equals the FP64 oracle to the BF16 bar."""
    from bec_amd import fno as F
    from bec_amd import surrogate as S
    from oracle import fno_oracle as FO
    net = F.FNO(seed=5, max_batch=16, **S.NET)
    ocfg = FO.Config.from_struct(net.cfg)
    flat = net.get_params().astype(np.float64)
    th = S.sample_params(2, seed=9)
    x = np.stack([S.features(S.calc_for(t), t) for t in th])
    for b in (1, 2):
        y = net.predict(x[:b])
        ref = FO.forward(ocfg, flat, _grid(x[:b], ocfg)).reshape(y.shape)
        err = np.linalg.norm(y - ref) / np.linalg.norm(ref)
        print(f"batch {b}: forward rel L2 vs FP64 oracle {err:.2e}")
        assert np.abs(ref).max() > 0 and err < 1e-2


@pytest.mark.parametrize(
    "nz,n,mz,m,width,layers,c_in,hidden,batch",
    [
        (32, 8, 8, 8, 16, 2, 16, 32, 3),      # width 16: both parts of a mode in one K tile
        (64, 8, 6, 4, 32, 2, 16, 64, 1),      # one sample, fewer plane modes than points
        (128, 8, 16, 4, 32, 3, 16, 32, 2),
        (32, 4, 8, 4, 32, 1, 32, 16, 33),     # more samples than one K tile, 16 in the last rows
        (32, 8, 8, 8, 64, 1, 16, 16, 2),      # the widest network
        (48, 6, 8, 4, 32, 2, 5, 24, 2),       # shapes that some of the fused kernels do not cover
    ],
)
def test_network_shapes_match_oracle(bec, nz, n, mz, m, width, layers, c_in, hidden, batch):
    """The fused kernels at the edges of the shapes they cover.  The bars are those of
    the small network above: BF16 operands round at 2^-9, a dozen products deep."""
    from bec_amd import fno as F
    from oracle import fno_oracle as FO
    net = F.FNO(seed=3, nz=nz, ny=n, nx=n, mz=mz, my=m, mx=m, width=width, layers=layers, c_in=c_in, c_out=2,
                hidden=hidden, max_batch=batch)
    ocfg = FO.Config.from_struct(net.cfg)
    rng = np.random.default_rng(3)
    x = rng.normal(size=(batch, nz * n * n, c_in)).astype(np.float32)
    t = rng.normal(size=(batch, nz * n * n, 2)).astype(np.float32)
    flat = net.get_params().astype(np.float64)
    y = net.predict(x)
    ref = FO.forward(ocfg, flat, _grid(x, ocfg)).reshape(y.shape)
    assert np.linalg.norm(y - ref) < 2e-2 * np.linalg.norm(ref)
    net.loss_backward(F.DeviceArray(x.shape, np.float32, x), F.DeviceArray(t.shape, np.float32, t), batch)
    g = net.get_grads().astype(np.float64)
    _, g_ref = FO.loss_and_grads(ocfg, flat, _grid(x, ocfg), _grid(t, ocfg))
    for name, sl in _blocks(ocfg):
        a, b = g[sl], g_ref[sl]
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        assert rel < 5e-2 and a @ b > 0.998 * np.linalg.norm(a) * np.linalg.norm(b), (name, rel)


def test_more_planes_than_a_grid_dimension_holds(bec):
    """batch * mz = 65,536 kz planes in one launch of the plane transforms (a network that create accepts).  A
    sample's output does not depend on the batch it is in, so the oracle checks the first, the 2047th and the
    last (BF16 bar as above); the gradient of the whole batch is the mean of its halves' (the same products;
    sums of 2^20 FP32 terms in 256 ranges of 128 tiles: below 400 roundings of 6e-8 in a row)."""
    from bec_amd import fno as F
    from oracle import fno_oracle as FO
    B, cells = 2048, 32 * 16
    net = F.FNO(seed=4, nz=32, ny=4, nx=4, mz=32, my=4, mx=4, width=16, layers=1, c_in=8, c_out=2, hidden=16, max_batch=B)
    ocfg = FO.Config.from_struct(net.cfg)
    rng = np.random.default_rng(4)
    x = rng.normal(size=(B, cells, 8)).astype(np.float32)
    t = rng.normal(size=(B, cells, 2)).astype(np.float32)
    y = net.predict(x)
    some = [0, 2046, 2047]
    ref = FO.forward(ocfg, net.get_params().astype(np.float64), _grid(x[some], ocfg)).reshape(3, cells, 2)
    assert np.linalg.norm(y[some] - ref) < 2e-2 * np.linalg.norm(ref)
    g = []
    for at in (slice(0, B), slice(0, B // 2), slice(B // 2, B)):
        xs, ts = np.ascontiguousarray(x[at]), np.ascontiguousarray(t[at])
        net.loss_backward(F.DeviceArray(xs.shape, np.float32, xs), F.DeviceArray(ts.shape, np.float32, ts), len(xs))
        g.append(net.get_grads().astype(np.float64))
    for name, sl in _blocks(ocfg):
        mean = (g[1][sl] + g[2][sl]) / 2
        assert np.linalg.norm(g[0][sl] - mean) < 400 * 6e-8 * np.linalg.norm(mean), name


def test_output_anywhere_the_copy_takes_it(bec):
    """The output in device memory (stored by the last kernel), in pinned host memory and over the end of the
    input (both copied): the same bits."""
    from bec_amd import fno as F
    batch, cells = 3, 32 * 64
    net = F.FNO(seed=6, nz=32, ny=8, nx=8, mz=8, my=8, mx=8, width=16, layers=2, c_in=16, c_out=2, hidden=32, max_batch=batch)
    x = np.random.default_rng(6).normal(size=(batch, cells, 16)).astype(np.float32)
    y = net.predict(x)
    assert np.isfinite(y).all() and np.abs(y).max() > 0
    # pinned host memory
    hip = F.flib()
    pinned = F.C.c_void_p()
    assert hip.hipHostMalloc(F.C.byref(pinned), F.C.c_size_t(y.nbytes), F.C.c_uint(0)) == 0
    try:
        host = np.frombuffer((F.C.c_char * y.nbytes).from_address(pinned.value), dtype=np.float32)
        host[:] = 0
        net.forward(F.DeviceArray(x.shape, np.float32, x), F.DeviceView(_Pinned(pinned, y.nbytes), 0), batch)
        F.device_synchronize()
        assert np.array_equal(host.reshape(y.shape), y)
    finally:
        hip.hipHostFree(pinned)
    # over the last 16 values of the input and beyond it
    both = F.DeviceArray((x.size + y.size,), np.float32, np.concatenate([x.ravel(), np.zeros(y.size, np.float32)]))
    at = x.size - 16
    net.forward(both, F.DeviceView(both, 4 * at), batch)
    F.device_synchronize()
    assert np.array_equal(both.download()[at:at + y.size].reshape(y.shape), y)


class _Pinned:
    """Pinned host memory, as a view's base."""

    def __init__(self, ptr, nbytes):
        self.ptr, self.nbytes = ptr, nbytes


@pytest.mark.parametrize(
    "ny,nx,width,batch,wide",
    [
        (16, 16, 16, 32, True),    # 64 rows per wavefront, forward and adjoint, at every width
        (16, 16, 32, 32, True),
        (16, 16, 64, 32, True),    # 66,560 bytes of staged columns
        (16, 32, 32, 1, False),    # 66,048
        (16, 32, 64, 2, False),    # 132,096: the longest plane at the largest width
    ],
)
def test_plane_transform_forms_match_oracle(bec, ny, nx, width, batch, wide):
    """The plane transforms that take 64 rows of the DFT matrix per wavefront (a thousand workgroups and more)
    and those that stage more than 64 KiB, at the bars of the network shapes above."""
    from bec_amd import fno as F
    from oracle import fno_oracle as FO
    nz, mz, m = 32, 16, 8
    planes, rows = batch * mz, (2 * m * m, 2 * ny * nx)   # of the two directions
    assert all((r % 64 == 0 and planes * (r // 64) >= 1024) == wide for r in rows)
    cells = nz * ny * nx
    net = F.FNO(seed=8, nz=nz, ny=ny, nx=nx, mz=mz, my=m, mx=m, width=width, layers=1, c_in=8, c_out=2, hidden=16, max_batch=batch)
    ocfg = FO.Config.from_struct(net.cfg)
    rng = np.random.default_rng(8)
    x = rng.normal(size=(batch, cells, 8)).astype(np.float32)
    t = rng.normal(size=(batch, cells, 2)).astype(np.float32)
    flat = net.get_params().astype(np.float64)
    y = net.predict(x)
    ref = FO.forward(ocfg, flat, _grid(x, ocfg)).reshape(y.shape)
    assert np.linalg.norm(y - ref) < 2e-2 * np.linalg.norm(ref)
    net.loss_backward(F.DeviceArray(x.shape, np.float32, x), F.DeviceArray(t.shape, np.float32, t), batch)
    g = net.get_grads().astype(np.float64)
    _, g_ref = FO.loss_and_grads(ocfg, flat, _grid(x, ocfg), _grid(t, ocfg))
    for name, sl in _blocks(ocfg):
        a, b = g[sl], g_ref[sl]
        rel = np.linalg.norm(a - b) / max(np.linalg.norm(b), 1e-30)
        assert rel < 5e-2 and a @ b > 0.998 * np.linalg.norm(a) * np.linalg.norm(b), (name, rel)
