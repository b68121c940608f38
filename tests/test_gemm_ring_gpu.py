"""GPU parity of the LDS-ring GEMM kernel in each of its row-block forms (16, 32,
64, 128 rows, pieces past 128): row counts that fill their blocks and not, N a
multiple of 4 and not, payloads of magnitude 1 and 9841, every output form, as
single GEMMs and in lists.

Integers must match exactly; fp32 and fp16 outputs bit for bit (one rounding of
the exact integer times one rounded product of scales).
"""
import numpy as np
import pytest

from gemm_shapes import RING_LIST, RING_SINGLE
from oracle import oracle as O

pytestmark = pytest.mark.gpu

FORMS = [("y",), ("y", "acc"), ("acc", "y16"), ("y16", "resid"), ("y", "acc", "y16", "resid")]


def bits(t):
    a = t.cpu().numpy()
    return a.view({2: np.uint16, 4: np.uint32}[a.dtype.itemsize])


class Problem:
    """One product X [M][K] times {-m, 0, m} weights, with its reference."""

    def __init__(self, M, K, N, mag):
        import torch
        import ter_amd as T
        trits = O.rand_trits(M * 7 + K + N, K, N, 0.4)
        X = O.rand_int8(M + 3 * K + N, M * K).reshape(M, K)
        X[0, :] = -128
        xs = (0.0007 * (np.arange(M) + 3)).astype(np.float32)
        ws = np.float32(0.043 / mag)
        if N % 4 == 0 and mag == 1:
            self.w = T.PackedTrits.from_v11(O.v11_pack(trits), K, N, float(ws))
        else:
            self.w = T.PackedTrits.from_payload(trits.astype(np.int32) * mag, float(ws))
        self.M, self.N = M, N
        self.x, self.xs = torch.from_numpy(X).cuda(), torch.from_numpy(xs).cuda()
        # (sums of at most 128 K: exact in float64)
        acc = (X.astype(np.float64) @ trits.astype(np.float64)).astype(np.int64)
        y = (acc * mag).astype(np.float32) * (xs * ws).astype(np.float32)[:, None]
        h = y.astype(np.float16)
        self.r0 = O.rand_normal_f32(M + N, M * N).reshape(M, N)
        self.want = dict(y=y, acc=acc.astype(np.int32), y16=h, resid=(self.r0 + h.astype(np.float32)).astype(np.float32))

    def buffers(self, form):
        import torch
        dt = dict(y=torch.float32, acc=torch.int32, y16=torch.float16)
        return {f: torch.from_numpy(self.r0).cuda() if f == "resid" else
                torch.full((self.M, self.N), 77, dtype=dt[f], device="cuda") for f in form}

    def check(self, out):
        for f, t in out.items():
            assert (bits(t) == self.want[f].view({2: np.uint16, 4: np.uint32}[self.want[f].dtype.itemsize])).all(), f


@pytest.mark.parametrize("mag", [1, 9841])
@pytest.mark.parametrize("M,K,N", RING_SINGLE)
def test_gemm_ring_single(cuda, M, K, N, mag):
    import ter_amd as T
    p = Problem(M, K, N, mag)
    for form in FORMS:
        out = p.buffers(form)
        T.mm_batched(p.w, p.x, x_scale_dev=p.xs, **out)
        p.check(out)


@pytest.mark.parametrize("mag", [1, 9841])
@pytest.mark.parametrize("name", RING_LIST)
def test_gemm_ring_list(cuda, name, mag):
    """Every GEMM of the list in another output form, launched twice."""
    import ter_amd as T
    specs = RING_LIST[name]
    problems = {s: Problem(*s, mag) for s in set(specs)}
    outs = [problems[s].buffers(FORMS[i % len(FORMS)]) for i, s in enumerate(specs)]
    plan = T.GemmPlan([dict(w=problems[s].w, x=problems[s].x, x_scale_dev=problems[s].xs, **o)
                       for s, o in zip(specs, outs)])
    for _ in range(2):
        for s, o in zip(specs, outs):
            for f, t in o.items():
                if f != "resid":
                    t.fill_(77)
                else:
                    import torch
                    t.copy_(torch.from_numpy(problems[s].r0))
        plan.launch()
        for s, o in zip(specs, outs):
            problems[s].check(o)
    plan.close()
