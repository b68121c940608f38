"""GPU parity of the split GEMM kernel at the edges of its tiles: every tile
(rows x strips, short and long K), row remainders around 16, 32 and 64, K
around the 128-row step, rows at any byte address, X shorter than one 16-byte
load, ragged N, and every output form; as single GEMMs and in lists.

Integers must match the oracle exactly; fp32 and fp16 outputs bit for bit (one
rounding of the exact integer times one rounded product of scales).
"""
import numpy as np
import pytest

from gemm_shapes import SPLIT_TAIL, SPLIT_TILES
from oracle import oracle as O

pytestmark = pytest.mark.gpu

# (M, K, N): with 256 CUs the tile is 64x8, 64x4, 32x4, 32x2, 16x2, 16x1, then the long-K forms of the last three
TILES = [(256, 130, 6912), (255, 129, 2560), (64, 128, 6912), (64, 127, 2560), (48, 640, 2560), (16, 2560, 640),
         (64, 5377, 2560), (33, 5121, 2560), (9, 8192, 260)]
EDGES = [(1, 1, 4), (3, 5, 8), (2, 8, 20), (15, 1, 36), (17, 63, 48), (31, 64, 16), (32, 65, 4), (65, 255, 132),
         (129, 257, 68), (200, 1003, 500), (256, 16, 12), (77, 1003, 1236)]


def bits(t):
    a = t.cpu().numpy()
    return a.view({2: np.uint16, 4: np.uint32}[a.dtype.itemsize])


def operands(M, K, N, shift):
    import torch
    import ter_amd as T
    trits = O.rand_trits(M * 7 + K + N, K, N, 0.4)
    X = O.rand_int8(M + 3 * K + N, M * K).reshape(M, K)
    X[0, :] = -128
    xs = (0.001 * (np.arange(M) + 1)).astype(np.float32)
    W = T.PackedTrits.from_v11(O.v11_pack(trits), K, N, 0.043)
    # X at `shift` bytes into an allocation filled with 127 on both sides
    buf = torch.full((M * K + 64,), 127, dtype=torch.int8, device="cuda")
    x = buf[shift:shift + M * K].view(M, K)
    x.copy_(torch.from_numpy(X))
    return W, X, x, xs, torch.from_numpy(xs).cuda(), O.v11_pack(trits)


def check(M, N, ra, ry, r0, out):
    assert (out["acc"].cpu().numpy() == ra).all()
    assert (bits(out["y"]) == ry.view(np.uint32)).all()
    h = ry.astype(np.float16)
    assert (bits(out["y16"]) == h.view(np.uint16)).all()
    want = (r0 + h.astype(np.float32)).astype(np.float32)
    assert (bits(out["resid"]) == want.view(np.uint32)).all()


def buffers(M, N, seed):
    import torch
    r0 = O.rand_normal_f32(seed, M * N).reshape(M, N)
    e = lambda dt: torch.full((M, N), 77, dtype=dt, device="cuda")
    return r0, dict(y=e(torch.float32), acc=e(torch.int32), y16=e(torch.float16), resid=torch.from_numpy(r0).cuda())


@pytest.mark.parametrize("shift", [0, 3], ids=["aligned", "unaligned"])
@pytest.mark.parametrize("M,K,N", TILES + EDGES)
def test_gemm_split_single(cuda, M, K, N, shift):
    import ter_amd as T
    W, X, x, xs, xsd, v11 = operands(M, K, N, shift)
    ra, ry = O.gemm_v11(X, xs, v11, 0.043, K, N)
    r0, out = buffers(M, N, M + K)
    T.mm_batched(W, x, x_scale_dev=xsd, **out)
    check(M, N, ra, ry, r0, out)


@pytest.mark.parametrize("specs,shift", [
    ([(256, 130, 2560), (256, 384, 640), (7, 33, 16)], 0), ([(64, 127, 640), (17, 257, 2560), (64, 6912, 128)], 0),
    ([(33, 200, 512), (2, 9, 64)], 1), ([(3, 5, 8), (40, 100, 24)], 0), ([(16, 2560, 640), (16, 6912, 2560)], 0),
], ids=["64_rows", "mixed_k", "unaligned", "short_x", "m16"])
def test_gemm_split_list(cuda, specs, shift):
    import ter_amd as T
    items, refs = [], []
    for M, K, N in specs:
        W, X, x, xs, xsd, v11 = operands(M, K, N, shift)
        r0, out = buffers(M, N, M + N)
        items.append(dict(w=W, x=x, x_scale_dev=xsd, **out))
        refs.append((M, N, *O.gemm_v11(X, xs, v11, 0.043, K, N), r0, out))
    T.GemmPlan(items).launch()
    for r in refs:
        check(*r)


def test_gemm_split_ragged_columns(cuda):
    """N not a multiple of 4 (payload weights): outputs element by element."""
    import torch
    import ter_amd as T
    M, K, N = 33, 200, 37
    w = O.rand_trits(5, K, N, 0.4).astype(np.int32)
    X = O.rand_int8(6, M * K).reshape(M, K)
    xs = (0.01 * (np.arange(M) + 1)).astype(np.float32)
    W = T.PackedTrits.from_payload(w, 0.02)
    y, acc = (torch.empty((M, N), dtype=dt, device="cuda") for dt in (torch.float32, torch.int32))
    T.mm_batched(W, torch.from_numpy(X).cuda(), y=y, acc=acc, x_scale_dev=torch.from_numpy(xs).cuda())
    ra = X.astype(np.int64) @ w
    assert (acc.cpu().numpy() == ra).all()
    want = ra.astype(np.float32) * (xs * np.float32(0.02)).astype(np.float32)[:, None]
    assert (bits(y) == want.view(np.uint32)).all()


# every tile with 16-byte loads, and at any address
VEC = [(t, d) for t in SPLIT_TILES for d in (0, 1)]
VEC_IDS = ["%dx%dx%d-%s" % (*t, "any" if d else "vec") for t, d in VEC]


@pytest.mark.parametrize("tile,odd", VEC, ids=VEC_IDS)
def test_gemm_split_tile_single(cuda, tile, odd):
    M, K, N = SPLIT_TILES[tile][0]
    test_gemm_split_single(cuda, M, K + odd, N, 0)


@pytest.mark.parametrize("tile,odd", VEC, ids=VEC_IDS)
def test_gemm_split_tile_list(cuda, tile, odd):
    specs = [SPLIT_TILES[tile][1], SPLIT_TAIL]
    test_gemm_split_list(cuda, [(M, K + odd, N) for M, K, N in specs], 0)
