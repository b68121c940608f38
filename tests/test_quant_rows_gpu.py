"""GPU parity of the per-row quantizers at the edges of their launch shapes:
K around every change of the thread count and the chunks per thread (2048,
4096, 8192, 16384, 32768), around 8 and the strided partials' 256 and 1024,
rows at odd addresses, and rows of zeros, infinities and NaN.  int8 codes and
scales bit for bit against the oracle, which keeps the reference's order."""
import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu

SIZES = [1, 7, 8, 255, 256, 257, 1003, 1024, 2048, 2049, 2056, 4096, 4097, 8192, 8200, 16384, 16385, 32760, 32768]


def same(q, s, rq, rs):
    assert (q.cpu().numpy() == rq).all()
    assert (s.cpu().numpy().view(np.uint32) == np.asarray(rs, np.float32).view(np.uint32)).all()


def shifted(a, shift):
    """`a` on the GPU, `shift` elements past an allocation's start."""
    import torch
    t = torch.from_numpy(a)
    buf = torch.zeros(t.numel() + 64, dtype=t.dtype, device="cuda")
    v = buf[shift:shift + t.numel()].view(t.shape)
    v.copy_(t)
    return v


@pytest.mark.parametrize("shift", [0, 1], ids=["aligned", "one_off"])
@pytest.mark.parametrize("K", SIZES)
def test_quant_rows_edges(cuda, K, shift):
    import ter_amd as T
    M = 3
    x = O.rand_normal_f32(K, M * K).reshape(M, K)
    x[1] *= 300.0
    x[2] = 0.0
    g = (0.5 + np.abs(O.rand_normal_f32(K + 1, K))).astype(np.float16)
    h, u = x.astype(np.float16), O.rand_normal_f32(K + 2, M * K).reshape(M, K).astype(np.float16)
    xd, hd, ud, gd = (shifted(a, shift) for a in (x, h, u, g))
    same(*T.quant_int8(xd), *O.quant_int8_rows(x))
    for dv, hv in ((xd, x), (hd, h)):
        q, s = T.rmsnorm_quant(dv, gd, 1e-5)
        ref = [O.rmsnorm_quant(hv[m], g, 1e-5) for m in range(M)]
        same(q, s, np.stack([r[0] for r in ref]), [r[1] for r in ref])
    q, s = T.relu2_rmsnorm_quant(hd, ud, gd, 1e-5)
    ref = [O.relu2_rmsnorm_quant(h[m], u[m], g, 1e-5) for m in range(M)]
    same(q, s, np.stack([r[0] for r in ref]), [r[1] for r in ref])


def test_quant_rows_not_finite(cuda):
    """A row with an infinity or a NaN leaves the rows beside it alone."""
    import torch
    import ter_amd as T
    x = O.rand_normal_f32(9, 4 * 2560).reshape(4, 2560)
    ref = O.quant_int8_rows(x[[0, 3]])
    x[1, 77], x[2, 2559] = np.inf, np.nan
    q, s = T.quant_int8(torch.from_numpy(x).cuda())
    same(q[[0, 3]], s[[0, 3]], *ref)
