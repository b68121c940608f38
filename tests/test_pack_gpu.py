"""GPU parity of the format conversions at the edges of their 16-byte pieces:
K around 16, 128 and 256, N around a strip, source and target at odd byte
addresses.  Bytes exactly the oracle's; fix-up slots left zero."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as O

pytestmark = pytest.mark.gpu


def at(a, shift):
    import torch
    buf = torch.full((a.size + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    v = buf[shift:shift + a.size]
    v.copy_(torch.from_numpy(a))
    return v


def export(W, K, N, shift):
    """to_v11 into an odd address; the bytes around the target keep theirs."""
    import torch
    from ter_amd import _lib as L
    n = (N // 4) * K
    buf = torch.full((n + 64,), 0xA5, dtype=torch.uint8, device="cuda")
    L.check(L.lib().ter_hip_unpack_v11(C.byref(W.wpk), buf.data_ptr() + shift,
                                       torch.cuda.current_stream().cuda_stream), "ter_hip_unpack_v11")
    b = buf.cpu().numpy()
    assert (b[:shift] == 0xA5).all() and (b[shift + n:] == 0xA5).all()
    return b[shift:shift + n]


@pytest.mark.parametrize("shift", [0, 1, 7])
@pytest.mark.parametrize("K,N", [(1, 4), (15, 8), (16, 16), (17, 20), (255, 4), (256, 64), (257, 36), (1000, 12),
                                 (2560, 68)])
def test_pack_v11_edges(cuda, K, N, shift):
    import torch
    import ter_amd as T
    t = O.rand_trits(K * 31 + N, K, N, 0.4)
    v11 = O.v11_pack(t).reshape(-1)
    src = v11.copy()
    src[::3] |= np.where((src[::3] & 3) == 0, 3, 0).astype(np.uint8)  # code 11 reads as 0
    W = T.PackedTrits.from_v11(at(src, shift), K, N, 0.5)
    assert (export(W, K, N, shift) == v11).all()
    assert not W.buf[-8 * N:].any()
    X = O.rand_int8(K, 2 * K).reshape(2, K)
    acc = torch.empty((2, N), dtype=torch.int32, device="cuda")
    T.mm_batched(W, torch.from_numpy(X).cuda(), acc=acc, x_scale_dev=torch.ones(2, device="cuda"))
    assert (acc.cpu().numpy() == X.astype(np.int64) @ t).all()


@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("K,N", [(4, 32), (16, 8), (20, 32), (128, 4), (132, 32), (256, 20), (272, 8), (1000, 16),
                                 (2560, 36)])
def test_pack_i2s_edges(cuda, K, N, shift):
    import ter_amd as T
    raw = np.random.default_rng(K + N).integers(0, 256, N * K // 4, dtype=np.uint8)  # code 3 too
    W = T.PackedTrits.from_i2s(at(raw, shift), K, N, 0.5)
    assert (export(W, K, N, shift) == O.i2s_to_v11(raw, K, N).reshape(-1)).all()
    assert not W.buf[-8 * N:].any()
