"""GPU parity of single GEMVs on every route of their dispatch: each activation
kind aligned (its own prologue; strided up to its unit limit, vector past it)
and one element off (the general one), strip mode and stream-K, int8 rows
through the GEMM kernels with device and host scales and, for the GEMV-only
outputs, through the strip kernel.  Accumulators and fp32 outputs bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

# strided at 5 and 16 units, vector past 16 and 32, ragged K (general), stream-K (20000 tiles)
SHAPES = [(1168, 100), (4096, 64), (4112, 48), (8208, 32), (1003, 68), (2048, 40000)]


def dev(a, shift=0):
    import torch
    t = torch.from_numpy(np.ascontiguousarray(a))
    buf = torch.zeros(t.numel() + 32, dtype=t.dtype, device="cuda")
    v = buf[shift:shift + t.numel()]
    v.copy_(t)
    return v


def quantized(kind, x, up, g):
    if kind == "f32" or kind == "f16":
        return O.quant_int8(x.astype(np.float32))
    if kind in ("f32rms", "f16rms"):
        return O.rmsnorm_quant(x, g, 1e-5)[:2]
    if kind == "relu2":
        return O.relu2_rmsnorm_quant(x, up, g, 1e-5)[:2]
    return O.silu_mul_quant(x, up)[:2]


@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "one_off"])
@pytest.mark.parametrize("kind", ["f32", "f16", "f32rms", "f16rms", "relu2", "silu"])
@pytest.mark.parametrize("K,N", SHAPES)
def test_gemv_single_kinds(cuda, K, N, kind, shift):
    import torch
    import ter_amd as T
    x = O.rand_normal_f32(K + N, K)
    x = x if kind in ("f32", "f32rms") else x.astype(np.float16)
    up = O.rand_normal_f32(K + 1, K).astype(np.float16)
    g = (0.5 + np.abs(O.rand_normal_f32(K + 2, K))).astype(np.float16)
    v11 = O.v11_pack(O.rand_trits(K + N, K, N, 0.4))
    W = T.PackedTrits.from_v11(v11, K, N, 0.037)
    kw = {}
    if kind in ("relu2", "silu"):
        kw["up"] = dev(up, shift)
    if kind in ("f32rms", "f16rms", "relu2"):
        kw["gamma"] = dev(g, shift)
    q, s = quantized(kind, x, up, g)
    y = torch.empty(N, dtype=torch.float32, device="cuda")
    acc = torch.empty(N, dtype=torch.int32, device="cuda")
    qo = torch.zeros(K, dtype=torch.int8, device="cuda")
    so = torch.zeros(1, dtype=torch.float32, device="cuda")
    T.gemv(W, dev(x, shift), y=y, acc=acc, q_out=qo, scale_out=so, **kw)
    ra, ry = O.gemv_v11(q, float(np.asarray(s).reshape(-1)[0]), v11, 0.037, K, N)
    assert (qo.cpu().numpy() == q).all()
    assert (acc.cpu().numpy() == ra).all()
    assert (y.cpu().numpy().view(np.uint32) == ry.view(np.uint32)).all()


@pytest.mark.parametrize("scale", ["device", "host"])
@pytest.mark.parametrize("shift", [0, 3])
@pytest.mark.parametrize("K,N", SHAPES + [(1, 4), (15, 8)])
def test_gemv_single_int8(cuda, K, N, shift, scale):
    import torch
    import ter_amd as T
    X = O.rand_int8(K, K)
    v11 = O.v11_pack(O.rand_trits(K + N, K, N, 0.4))
    W = T.PackedTrits.from_v11(v11, K, N, 0.037)
    x = dev(X, shift)
    kw = dict(x_scale=0.0123) if scale == "host" else dict(x_scale_dev=torch.full((1,), 0.0123, device="cuda"))
    ra, ry = O.gemv_v11(X, np.float32(0.0123), v11, 0.037, K, N)
    h = ry.astype(np.float16)
    acc = torch.empty(N, dtype=torch.int32, device="cuda")
    y16, r16 = (torch.ones(N, dtype=torch.float16, device="cuda") for _ in range(2))
    r = torch.ones(N, dtype=torch.float32, device="cuda")
    y, _ = T.gemv(W, x, **kw)
    T.gemv(W, x, acc=acc, y16=y16, resid=r, **kw)
    T.gemv(W, x, resid16=r16, **kw)
    assert (y.cpu().numpy().view(np.uint32) == ry.view(np.uint32)).all()
    assert (acc.cpu().numpy() == ra).all()
    assert (y16.cpu().numpy().view(np.uint16) == h.view(np.uint16)).all()
    one = np.float32(1)
    assert (r.cpu().numpy() == one + h.astype(np.float32)).all()
    assert (r16.cpu().numpy() == (one + h.astype(np.float32)).astype(np.float16)).all()


# both sides of the lines between the GEMM kernels, strip mode and stream-K (256 CUs)
ROUTES = [(1024, 4096), (1024, 4112), (1040, 64), (8192, 8192), (12288, 8208), (12304, 8208), (512, 16400),
          (528, 16400), (3088, 16400), (2064, 32768), (2064, 32784), (2816, 40960), (3583, 8192), (3585, 64), (1025, 8208)]


@pytest.mark.parametrize("scale", ["device", "host"])
@pytest.mark.parametrize("K,N", ROUTES)
def test_gemv_int8_routes(cuda, K, N, scale):
    test_gemv_single_int8(cuda, K, N, 0, scale)
