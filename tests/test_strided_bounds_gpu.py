"""GPU parity of the strided GEMV prologue at the edges of its K bounds: each
activation kind at the last unit count of one compiled bound and the first of
the next, with the last unit partial, as a single GEMV, as a list whose other
GEMV is shorter (units past the short K's range are staged nowhere), and as a
list that reads one activation vector, its weights apart and back to back (the
shared launch form).  Bit for bit."""
import numpy as np
import pytest

from oracle import oracle as O
from ter_amd._lib import PLAN_SHARED, PLAN_STRIDED

pytestmark = pytest.mark.gpu

UNITS = {"f32rms": (1, 8, 9, 10, 11, 16), "f16rms": (1, 8, 9, 10, 11, 16), "relu2": (1, 16, 17, 28, 29, 32),
         "f16": (1, 8, 9, 16), "silu": (1, 16, 17, 32), "smul": (1, 16, 17, 32)}


def dev(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def problem(kind, K, seed):
    x = O.rand_normal_f32(seed, K)
    if kind not in ("f32rms", "smul"):
        x = x.astype(np.float16)
    up = O.rand_normal_f32(seed + 1, K).astype(np.float16)
    g = (0.5 + np.abs(O.rand_normal_f32(seed + 2, K))).astype(np.float16)
    kw = {}
    if kind in ("relu2", "silu", "smul"):
        kw["up"] = dev(up)
    if kind in ("f32rms", "f16rms", "relu2"):
        kw["gamma"] = dev(g)
    if kind == "f16":
        q, s = O.quant_int8(x.astype(np.float32))
    elif kind in ("f32rms", "f16rms"):
        q, s = O.rmsnorm_quant(x, g, 1e-5)[:2]
    elif kind == "relu2":
        q, s = O.relu2_rmsnorm_quant(x, up, g, 1e-5)[:2]
    elif kind == "silu":
        q, s = O.silu_mul_quant(x, up)[:2]
    else:
        q, s = O.smul_quant(x, up)[:2]
    return dict(x=dev(x), **kw), q, float(np.asarray(s).reshape(-1)[0])


def weights(K, N, seed):
    import ter_amd as T
    v11 = O.v11_pack(O.rand_trits(seed, K, N, 0.4))
    return T.PackedTrits.from_v11(v11, K, N, 0.037), v11


CASES = [(k, u) for k, us in UNITS.items() for u in us]


@pytest.mark.parametrize("kind,units", CASES, ids=[f"{k}-{u}" for k, u in CASES])
def test_strided_bounds(cuda, kind, units):
    import torch
    import ter_amd as T
    K = units * 256 - (240 if units % 2 else 0)  # odd counts end in a unit of 16 rows
    act, q, s = problem(kind, K, 11 * K)
    short, qs, ss = problem(kind, 272, 5 * K)

    def check(items, refs, shared=False):
        plan = T.Plan(items)
        assert plan.mode & PLAN_STRIDED and bool(plan.mode & PLAN_SHARED) == shared
        for _ in range(2):
            for it in items:
                it["y"].fill_(-3)
            plan.launch()
            torch.cuda.synchronize()
            for it, ry in zip(items, refs):
                assert (it["y"].cpu().numpy().view(np.uint32) == ry.view(np.uint32)).all()
        plan.close()

    items, refs = [], []
    for i, N in enumerate((68, 32, 20)):
        W, v11 = weights(K, N, K + i)
        y = torch.empty(N, dtype=torch.float32, device="cuda")
        items.append(dict(w=W, y=y, **act))
        refs.append(O.gemv_v11(q, s, v11, 0.037, K, N)[1])
        if kind != "smul":
            T.gemv(W, y=y, **act)
            assert (y.cpu().numpy().view(np.uint32) == refs[-1].view(np.uint32)).all()
    check(items, refs)
    for it, W in zip(items, T.group_contiguous([it["w"] for it in items])):
        it["w"] = W
    check(items, refs, shared=True)
    W, v11 = weights(272, 40, K + 9)
    check([dict(w=W, y=torch.empty(40, dtype=torch.float32, device="cuda"), **short), items[0]],
          [O.gemv_v11(qs, ss, v11, 0.037, 272, 40)[1], refs[0]])
