"""The library's host code on the CPU, over a HIP runtime that runs no kernels
(tests/c/fake_hip.cpp): what a call launches, copies and waits for."""
import os
import shutil
import subprocess
import sys
import textwrap

import pytest

from gemm_shapes import RING_LIST, RING_SINGLE, SPLIT_TAIL, SPLIT_TILES

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PRELUDE = """
import ctypes as C, sys
fake = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
fake.fake_log.restype = C.c_char_p
fake.fake_fail.argtypes = [C.c_char_p]
from ter_amd import _lib as L
lib = C.CDLL(L.LIB_PATH)
for name, res, args in L.SIGNATURES:
    f = getattr(lib, name)
    f.restype, f.argtypes = res, args
keep = []
def buf(n):
    b = C.create_string_buffer(n + 4096)
    keep.append(b)
    return (C.addressof(b) + 4095) // 4096 * 4096
def log():
    lines = fake.fake_log().decode().splitlines()
    fake.fake_reset()
    return lines
def weight(K, N):
    w = L.WPK()
    nb = lib.ter_hip_wpk_bytes(K, N)
    assert lib.ter_hip_wpk_init(C.byref(w), buf(nb), nb, K, N, 0.5) == 0, lib.ter_hip_last_error()
    keep.append(w)
    return w
def gemm(M, K, N):  # the kernels one GEMM on int8 rows launches
    a = L.Act()
    a.data, a.kind, a.scale_dev = buf(M * K), L.X_I8, buf(4 * M)
    W = weight(K, N)
    log()
    assert lib.ter_hip_gemm(C.byref(W), C.byref(a), M, buf(64), None, None) == 0, lib.ter_hip_last_error()
    return [l for l in log() if l.startswith("launch")]
def gemm_list(items, wg_per_cu=0):  # the kernel a list of GEMMs (M, K, N) launches, and the plan's workgroups
    arr = (L.GemmItem * len(items))()
    for it, (M, K, N) in zip(arr, items):
        it.w, it.x, it.x_scale_dev, it.M, it.y = C.pointer(weight(K, N)), buf(M * K), buf(4 * M), M, buf(64)
    p, n = C.c_void_p(), C.c_int32()
    assert lib.ter_hip_gemm_plan_create(C.byref(p), arr, len(items), wg_per_cu) == 0, lib.ter_hip_last_error()
    b, m = C.c_uint64(), C.c_uint64()
    assert lib.ter_hip_plan_stats(p, C.byref(b), C.byref(m), C.byref(n)) == 0
    log()
    assert lib.ter_hip_plan_launch(p, None) == 0
    ran = [l for l in log() if l.startswith("launch")]
    assert len(ran) == 1, ran
    return ran[0], n.value
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    """The fake runtime, built; returns a function that runs a body over it in a fresh process."""
    gxx = shutil.which("g++")
    if gxx is None:
        pytest.skip("g++ not installed")
    so = str(tmp_path_factory.mktemp("fake") / "libfakehip.so")
    src = os.path.join(ROOT, "tests", "c", "fake_hip.cpp")
    subprocess.run([gxx, "-std=c++17", "-O1", "-shared", "-fPIC", "-Wall", src, "-o", so], check=True)

    def run(body):
        r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), so], cwd=ROOT, text=True,
                           stdout=subprocess.PIPE, stderr=subprocess.STDOUT, timeout=120)
        assert r.returncode == 0, r.stdout
        return r.stdout

    return run


@pytest.mark.parametrize("xmax", [100, 9000], ids=["int8", "int16"])
@pytest.mark.parametrize("kernel", ["done_kernel", "gem"], ids=["number", "product"])
def test_mm_row_waits_before_a_launch_error(fake, kernel, xmax):
    """A launch that fails leaves the row's upload (and the product) in flight
    on the buffers that the next call takes over: the call waits for the
    stream before it gives them up."""
    fake(f"""
    K, N = 512, 64
    W = weight(K, N)
    X = (C.c_int32 * K)(*[{xmax}] * K)
    out, xs, ys = (C.c_float * N)(), buf(2 * K), buf(4 * N)
    call = lambda: lib.ter_hip_mm_row(C.addressof(X), 0, K, 0.01, C.byref(W), N, C.addressof(out), xs, ys, None)
    assert call() == 0
    ran = log()
    assert "done_kernel" in ran[-1] and not any(l.startswith("sync") for l in ran), ran
    fake.fake_fail(b"{kernel}")
    assert call() == L.ERR_HIP
    ran = log()
    assert ran[-2].startswith("failed") and ran[-1].startswith("sync"), ran
    """)


@pytest.mark.parametrize("call,kernel", [
    ("lib.ter_hip_rmsnorm_quant(x, L.X_F32_RMS, x, 1e-5, 8, 16384, q, s, None)", "quant_rows_kernel"),
    ("lib.ter_hip_gemm(C.byref(W), C.byref(a), 256, y, None, None)", "gemm_split_kernel"),
    ("lib.ter_hip_gemm(C.byref(WL), C.byref(a), 64, y, None, None)", "gemm_lds_kernel"),
], ids=["rms_rows", "split", "ring"])
def test_large_lds_is_allowed_on_each_device(fake, call, kernel):
    """Kernels of more than 64 KiB of LDS: the limit is raised on the device of
    the call, once for each, and before the first launch there."""
    fake(f"""
    W, WL = weight(256, 6912), weight(256, 65536)
    x, q, s = buf(8 * 16384 * 4), buf(8 * 16384), buf(4096)
    a = L.Act()
    a.data, a.kind, a.scale_dev = buf(256 * 256), L.X_I8, s
    y = buf(64)
    for dev in (0, 1, 0, 1):
        fake.fake_device(dev)
        assert {call} == 0, lib.ter_hip_last_error()
    ran = log()
    launches = [l.split(" ", 5) for l in ran if l.startswith("launch") and "{kernel}" in l]
    assert [l[1] for l in launches] == ["0", "1", "0", "1"], ran
    for dev in "01":
        _, _, _, _, lds, fn = launches[int(dev)]
        at = [i for i, l in enumerate(ran) if l == f"attribute {{dev}} {{lds}} {{fn}}"]
        assert int(lds) > 65536 and len(at) == 1, ran
        assert at[0] < ran.index("launch " + " ".join(launches[int(dev)][1:])), ran
    """)


VEC_STRIP, STRIP = "gemv_strip_kernel<false, 0,", "gemv_strip_kernel<false, -1,"
VEC_STREAM, STREAM, SPLIT, RING = "gemv_t16_kernel<false, 0>", "gemv_t16_kernel<false, -1>", "gemm_split", "gemm_lds"


@pytest.mark.parametrize("K,N,shift,dev_scale,kernel", [
    # 16-byte aligned rows: the GEMM kernels for the shortest, strip mode, stream-K past 48 units and two strips per CU
    (1024, 4096, 0, 1, SPLIT), (1024, 4096, 0, 0, SPLIT), (1024, 4112, 0, 1, VEC_STRIP), (1040, 64, 0, 1, VEC_STRIP),
    (2560, 640, 0, 1, VEC_STRIP), (2560, 640, 0, 0, VEC_STRIP), (32768, 8192, 0, 1, VEC_STRIP),
    (12288, 8208, 0, 1, VEC_STRIP), (12304, 8208, 0, 1, VEC_STREAM), (12288, 40960, 0, 0, VEC_STRIP),
    # from four, eight and ten strips per CU on
    (512, 16400, 0, 1, RING), (512, 16400, 0, 0, VEC_STRIP), (528, 16400, 0, 1, VEC_STRIP), (4096, 40960, 0, 1, VEC_STRIP),
    (2560, 32768, 0, 1, VEC_STRIP), (2560, 32784, 0, 1, RING), (12304, 32768, 0, 1, VEC_STREAM), (12304, 32784, 0, 1, RING),
    (4096, 40976, 0, 1, RING), (4096, 40976, 0, 0, VEC_STREAM), (8192, 65536, 0, 1, RING),
    # other rows
    (3583, 8192, 0, 1, SPLIT), (3585, 64, 0, 1, STRIP), (3584, 8192, 1, 0, SPLIT), (3600, 64, 1, 1, STRIP),
    (1023, 16384, 0, 1, SPLIT), (1025, 8208, 0, 1, STRIP), (1023, 16400, 0, 1, STREAM), (15, 8, 0, 1, SPLIT),
])
def test_int8_gemv_route(fake, K, N, shift, dev_scale, kernel):
    """Where a single int8 GEMV runs, on both sides of each line of its rule (256 CUs)."""
    fake(f"""
    W = weight({K}, {N})
    a = L.Act()
    a.data, a.kind, a.scale = buf({K} + 64) + {shift}, L.X_I8, 0.5
    if {dev_scale}:
        a.scale_dev = buf(4)
    assert lib.ter_hip_gemv(C.byref(W), C.byref(a), buf({N} * 4), None, None) == 0, lib.ter_hip_last_error()
    ran = [l for l in log() if l.startswith("launch")]
    assert len(ran) == 1 and "{kernel}" in ran[0], ran
    """)


def layers(n, M, H, F, q, kv):
    return [(M, H, q), (M, H, kv), (M, H, kv), (M, q, H), (M, H, F), (M, H, F), (M, F, H)] * n


@pytest.mark.parametrize("M,K,N,kernel", [
    (32, 768, 65536, RING), (16, 4096, 32768, RING), (128, 2048, 32768, RING), (64, 2048, 65536, RING),
    (16, 2048, 16384, SPLIT), (64, 2560, 6912, SPLIT), (128, 8192, 8192, SPLIT), (256, 2560, 6912, SPLIT),
    (256, 2048, 16384, SPLIT),
])
def test_gemm_route(fake, M, K, N, kernel):
    """The kernel of a single GEMM (256 CUs): the faster one over weights from HBM."""
    fake(f"""
    ran = gemm({M}, {K}, {N})
    assert ran and all("{kernel}" in l for l in ran), ran
    """)


@pytest.mark.parametrize("items,kernel", [
    (layers(8, 128, 2560, 6912, 2560, 640), RING), (layers(4, 64, 2560, 6912, 2560, 640), RING),
    (layers(3, 8, 2560, 6912, 2560, 640), RING), (layers(1, 32, 2560, 6912, 2560, 640), SPLIT),
    (layers(4, 32, 2560, 6912, 2560, 640), SPLIT), (layers(2, 8, 2048, 8192, 2048, 512), SPLIT),
], ids=["bitnet_x8_m128", "bitnet_x4_m64", "bitnet_x3_m8", "bitnet_x1_m32", "bitnet_x4_m32", "llama_x2_m8"])
def test_gemm_list_route(fake, items, kernel):
    """The same for lists."""
    fake(f"""
    ran, _ = gemm_list({items})
    assert "{kernel}" in ran, ran
    """)


@pytest.mark.parametrize("M,K,N,groups", [(8, 3072, 640, 4), (8, 3088, 640, 8), (8, 5121, 640, 8), (8, 5119, 640, 4)])
def test_gemm_split_long_k(fake, M, K, N, groups):
    """The K groups of the 16 x 1 tile on both sides of its lines (aligned rows at 12 units of K, others at 20)."""
    fake(f"""
    ran = gemm({M}, {K}, {N})
    assert len(ran) == 1 and "gemm_split" in ran[0] and "SCfg<1, 1, 1, {groups}, 2>" in ran[0], ran
    """)


@pytest.mark.parametrize("odd", [0, 1], ids=["vec", "any"])
def test_gemm_split_tiles_reached(fake, odd):
    """The shapes of the GPU tests run every tile of the split kernel, in both load forms."""
    fake(f"""
    for (rows, strips, groups), (one, first) in {SPLIT_TILES}.items():
        want = "gemm_split_kernel<terhip::(anonymous namespace)::SCfg<%d, 1, %d, %d, 2>, {2 - odd}, %s>"
        M, K, N = one
        ran = gemm(M, K + {odd}, N)
        assert len(ran) == 1 and want % (rows // 16, strips, groups, "false") in ran[0], ran
        ran, _ = gemm_list([(M, K + {odd}, N) for M, K, N in (first, {SPLIT_TAIL})])
        assert want % (rows // 16, strips, groups, "true") in ran, ran
        keep.clear()
    """)


def test_gemm_ring_reached(fake):
    """Those of its tests run the ring kernel, with every count of row blocks."""
    fake(f"""
    import re
    blocks = lambda l: int(re.search(r"gemm_lds_kernel<terhip::.anonymous namespace.::LCfg<(\\d+)", l)[1])
    for M, K, N in {RING_SINGLE}:
        ran = gemm(M, K, N)
        assert len(ran) == -(-M // 128) and {{blocks(l) for l in ran}} == {{1 if M <= 16 else 2 if M <= 32 else 4 if M <= 64 else 8}}
        keep.clear()
    for name, items in {RING_LIST}.items():
        assert blocks(gemm_list(items)[0]) == (8 if name == "pieces" else int(name))
        keep.clear()
    """)
