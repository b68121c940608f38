// gemm_split.hip -- batched packed-trit GEMM for short launches on gfx950
// MFMA: one GEMM, or a list too short to give the CUs a block each of the
// LDS-ring kernel (gemm_lds.hip), whose blocks each walk all of K alone; and
// every GEMM whose X rows are not 16-byte aligned; short single int8 GEMVs as M
// = 1 (int8_gemv_route in abi.hip).
//
// Same semantics as gemm_lds.hip (cuda/ter_cuda_addonly_batched.cu:117-123):
// acc[m][j] = sum_k X[m][k] w[k][j] in exact int32, y = float(mag * acc) * (xs[m] * w_scale).
//
// Work.  A workgroup owns R = 16 MBW rows x BS column strips and all of K.
// Its waves form KG groups that split K (steps of 128 rows of K) and, within
// a group, SG strip groups of S strips that share the group's staged X.  At
// the end the KG partial tiles meet in LDS and the workgroup writes the
// outputs.  No workspace, no atomics, and any split gives the same integers.
//
// What bounds it.  A projection of a decode or prefill batch has 10-54 blocks
// of the ring kernel for 256 CUs, and each walks K serially: at M = 64, K =
// 6912, N = 2560 ten workgroups took 25 us.  With a tile per CU and K split
// over 4 to 16 waves the launch is a round of loads, a few steps per wave and
// one LDS exchange; what is left is the launch (about 3 us with its first
// loads) and each CU's read of its X rows and weights from L2, at 15-28 bytes
// per clock and CU by the L2's request counters, with the matrix cores busy
// 7-20% of the time.  Measured in graphs, weights from HBM / cached, the
// kernels that ran before in parentheses: M = 8, 2560 x 2560 4.9 / 3.3 us (8.6 /
// 8.1); M = 64, 2560 x 6912 7.3 / 5.9 (13.2 / 12.6) and 6912 x 2560 9.7 / 7.4 (25.7 /
// 25.3); M = 256, 2560 x 6912 11.8 / 10.9 (39 / 38, two launches); M = 256, 8192 x
// 8192 25.7 / 24.6 (90 / 89); M = 77, 1003 x 1236 (rows at any address), HIP
// events, 3.8 us (57).
//
// Loads.  X goes through registers to LDS: a load instruction covers 8 rows x
// 128 bytes, whole cache lines.  (Loading the MFMA A operand straight from
// memory covers 16 rows x 64 bytes: 10.8 against 7.3 us at M = 64, K = 6912.)  The weights are gathered
// into the MFMA B operand layout by dword loads (lane = column j + 16 * k
// group g; one dword = 16 trits), one line per column quad and step.  D steps
// are in flight in registers; step i + 1 is written to LDS while step i is
// multiplied.  With one strip group the staged X is the wave's own (LDS
// operations of a wave run in order: no barrier in the loop), else two LDS
// buffers and one LDS-only barrier per step.
//
// Operands.  Row r of a staged step holds its eight 16-byte chunks at
// positions c ^ (r / 2 % 8), so the 16 rows of an A operand read hit distinct
// banks.  The trits become signed int8 (a byte table indexed by u = w + 1);
// columns and K padding hold w = 0, so whatever X holds past its row's end
// counts nothing.
#include "common.h"

namespace terhip {
namespace {

typedef int i32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

// How the rows of X are read: 16-byte chunks through a range-checked buffer
// resource (16-byte aligned rows), 16-byte chunks at any byte address, or
// byte by byte (all of X shorter than one chunk).
enum XMode { kXBytes = 0, kXAny = 1, kXVec = 2 };

// Signed int8 weights of 16 trits (one T16 dword) in MFMA B operand order:
// byte b of word f is the trit of row 4 f + b; u = w + 1 -> w by table lookup.
__device__ __forceinline__ i32x4 unpack_signed(unsigned dw) {
    const unsigned kM = 0x03030303u, kT = 0x000100FFu;  // bytes: u=0 -> -1, 1 -> 0, 2 -> +1, 3 -> 0
    return i32x4{(int)__builtin_amdgcn_perm(0u, kT, dw & kM), (int)__builtin_amdgcn_perm(0u, kT, (dw >> 2) & kM),
                 (int)__builtin_amdgcn_perm(0u, kT, (dw >> 4) & kM), (int)__builtin_amdgcn_perm(0u, kT, (dw >> 6) & kM)};
}

// v >> 8 t bits, t in 0 .. 15 (16 and more: any value).
__device__ __forceinline__ u32x4 shift_bytes(u32x4 v, int t) {
    unsigned w[8] = {v.x, v.y, v.z, v.w, 0u, 0u, 0u, 0u};
    if (t & 8) {
#pragma unroll
        for (int i = 0; i < 6; ++i) w[i] = w[i + 2];
    }
    if (t & 4) {
#pragma unroll
        for (int i = 0; i < 5; ++i) w[i] = w[i + 1];
    }
    u32x4 r;
#pragma unroll
    for (int i = 0; i < 4; ++i) r[i] = __builtin_amdgcn_alignbyte(w[i + 1], w[i], t & 3);
    return r;
}

// Workgroup barrier for LDS alone: the global loads in flight stay in flight.
__device__ __forceinline__ void lds_barrier() {
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
}

// MBW row blocks of 16 rows per workgroup; S strips per wave, SG strip groups
// and KG groups of waves that split K; D steps of loads in registers.
template <int MBW_, int S_, int SG_, int KG_, int D_>
struct SCfg {
    static constexpr int MBW = MBW_, S = S_, SG = SG_, KG = KG_, D = D_;
    static constexpr int W = SG * KG, THREADS = 64 * W, R = 16 * MBW, BS = S * SG;
    static constexpr int XB = R * 128;                // bytes of a staged step of X
    static constexpr int NB = SG > 1 ? 2 : 1;         // staged steps per K group
    static constexpr int P = 16 * BS + 4;             // ints per row of a K group's partial tile
    static constexpr int XLDS = KG * NB * XB, PLDS = KG * R * P * 4;
    static constexpr int LDS = XLDS > PLDS ? XLDS : PLDS;
};
constexpr int kStepK = 128;

template <class C, int kX, bool kList>
__global__ __launch_bounds__(C::THREADS) void gemm_split_kernel(GemmDesc single, const GemmDesc* __restrict__ list,
                                                                const GemmBlock* __restrict__ blocks, int n_sb,
                                                                int pieces) {
#pragma clang fp contract(off)
    extern __shared__ __align__(16) unsigned char lds[];
    constexpr int MBW = C::MBW, S = C::S, D = C::D, R = C::R, P = C::P;
    GemmDesc d;
    int st0;
    if constexpr (kList) {
        const GemmBlock b = blocks[blockIdx.x];
        d = list[b.desc];
        st0 = b.strip0;
    } else {
        // blocks b, b + 8, .. (one XCD) take the row pieces of one strip block
        const int r = (int)blockIdx.x >> 3, q = r / pieces, p = r - q * pieces;
        const int sb = q * 8 + ((int)blockIdx.x & 7);
        if (sb >= n_sb) return;
        d = single;
        st0 = sb * C::BS;
        const int r0 = p * R;
        d.M -= r0;
        d.x += (long long)r0 * d.ldx;
        if (d.xs) d.xs += r0;
        const long long o = (long long)r0 * d.N;
        if (d.y) d.y += o;
        if (d.acc) d.acc += o;
        if (d.y16) d.y16 += o;
        if (d.resid) d.resid += o;
    }
    const int M = d.M < R ? d.M : R;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int kg = wave / C::SG, sg = wave % C::SG;
    const int j = lane & 15, g = lane >> 4;
    const int n_step = (d.K + kStepK - 1) / kStepK;
    const int t0 = n_step * kg / C::KG;
    const int n = n_step * (kg + 1) / C::KG - t0;                       // this K group's steps of 128 rows of K
    const int n_all = C::SG > 1 ? (n_step + C::KG - 1) / C::KG : n;     // the barriers every wave meets

    const int stw = st0 + sg * S;                                       // this wave's strips
    const int ns = max(0, min(S, d.n_strips - stw));
    const __amdgpu_buffer_rsrc_t wr = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(d.w + (long long)(ns ? stw : 0) * d.Ku * kTileBytes), 0, ns * d.Ku * kTileBytes, 0x00020000);
    const int total = M * d.ldx;
    const __amdgpu_buffer_rsrc_t xr = __builtin_amdgcn_make_buffer_rsrc((void*)d.x, 0, total, 0x00020000);
    const TER_GLOBAL char* xb = (const TER_GLOBAL char*)gptr(d.x);
    const int woff = (j >> 2) * 256 + g * 16 + (j & 3) * 4;
    // X load q of a step: rows 8 q .. 8 q + 7, whole 128-byte lines; lane l
    // row 8 q + l / 8, stored at 16-byte position l % 8 of the row: chunk
    // (l % 8) ^ (row / 2 % 8).  The strip groups share the loads of a step.
    constexpr int XL = 2 * MBW / C::SG;
    static_assert(2 * MBW % C::SG == 0, "X loads per wave");
    int xoff[XL];
#pragma unroll
    for (int q = 0; q < XL; ++q) {
        const int row = 8 * (q * C::SG + sg) + (lane >> 3);
        xoff[q] = row * d.ldx + (((lane & 7) ^ ((row >> 1) & 7)) * 16);
    }
    unsigned char* xl = lds + kg * C::NB * C::XB;

    u32x4 X[D][XL];
    unsigned B[D][S][2];
    // X and the weights of step t0 + i into register stage k; past the group's
    // end offsets beyond the resources (no memory traffic; never multiplied)
    auto load_x = [&](int k, int i) {
        const int t = t0 + i;
        if constexpr (kX == kXVec) {
            const int xo = i < n ? t * kStepK : 0x40000000;
#pragma unroll
            for (int q = 0; q < XL; ++q) X[k][q] = __builtin_amdgcn_raw_buffer_load_b128(xr, xoff[q] + xo, 0, 0);
        } else if constexpr (kX == kXAny) {
#pragma unroll
            for (int q = 0; q < XL; ++q) {
                const int o = min(xoff[q] + (i < n ? t : t0) * kStepK, total - 16);
                __builtin_memcpy(&X[k][q], (const TER_GLOBAL void*)(xb + o), 16);
            }
        }
    };
    auto load_w = [&](int k, int i) {
        const int t = t0 + i;
        const int wo = i < n ? (t >> 1) * kTileBytes + (t & 1) * 128 : 0x40000000;
#pragma unroll
        for (int s = 0; s < S; ++s)
#pragma unroll
            for (int h = 0; h < 2; ++h)
                B[k][s][h] = __builtin_amdgcn_raw_buffer_load_b32(wr, woff + wo + s * d.Ku * kTileBytes + h * 64, 0, 0);
    };
    // step i's X from register stage k to LDS
    auto stage = [&](int k, int i) {
        unsigned char* xd = xl + (C::NB > 1 ? (i & 1) * C::XB : 0);
        const int xo = (t0 + i) * kStepK;
#pragma unroll
        for (int q = 0; q < XL; ++q) {
            u32x4 a = X[k][q];
            if constexpr (kX == kXAny) {
                // a chunk past the end of X was read from its last 16 bytes
                const int t = xoff[q] + xo - (total - 16);
                if (__builtin_amdgcn_ballot_w64(t > 0)) a = t > 0 ? shift_bytes(a, t) : a;
            } else if constexpr (kX == kXBytes) {
                unsigned wd[4] = {0, 0, 0, 0};
                for (int e = 0; e < 16; ++e) {
                    const int o = xoff[q] + xo + e;
                    if (o < total) wd[e >> 2] |= (unsigned)(uint8_t)xb[o] << (8 * (e & 3));
                }
                a = u32x4{wd[0], wd[1], wd[2], wd[3]};
            }
            *reinterpret_cast<u32x4*>(xd + (q * C::SG + sg) * 1024 + lane * 16) = a;
        }
    };
    // the hand-over of a staged step between lanes (of one wave: no wait, the
    // order alone)
    auto stage_fence = [] {
        if constexpr (C::SG > 1)
            lds_barrier();
        else
            __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    };
    i32x4 acc[S][MBW];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int mb = 0; mb < MBW; ++mb) acc[s][mb] = i32x4{0, 0, 0, 0};
#pragma unroll
    for (int k = 0; k < D; ++k) {
        load_x(k, k);
        load_w(k, k);
    }
    // the output quads of this thread: row, 4 columns (all R x 4 BS quads over the workgroup)
    constexpr int Q = R * 4 * C::BS, NQ = (Q + C::THREADS - 1) / C::THREADS;
    float xs[NQ];
#pragma unroll
    for (int i = 0; i < NQ; ++i) xs[i] = d.xs ? gptr(d.xs)[min((tid + i * C::THREADS) / (4 * C::BS), M - 1)] : d.x_scale;

    if (n > 0) stage(0, 0);
    load_x(0, D);
    for (int i0 = 0; i0 < n_all; i0 += D) {
#pragma unroll
        for (int k = 0; k < D; ++k) {
            const int i = i0 + k;
            if (i < n_all) {
                stage_fence();
                const unsigned char* xd = xl + (C::NB > 1 ? (i & 1) * C::XB : 0);
                i32x4 A[2][MBW];
#pragma unroll
                for (int h = 0; h < 2; ++h)
#pragma unroll
                    for (int mb = 0; mb < MBW; ++mb)
                        A[h][mb] = *reinterpret_cast<const i32x4*>(xd + (16 * mb + j) * kStepK +
                                                                   (((4 * h + g) ^ ((j >> 1) & 7)) * 16));
                if constexpr (C::NB == 1) stage_fence();
                if (i + 1 < n) stage((k + 1) % D, i + 1);
                __builtin_amdgcn_sched_barrier(0);
                if (i < n) {
#pragma unroll
                    for (int h = 0; h < 2; ++h)
#pragma unroll
                        for (int s = 0; s < S; ++s) {
                            const i32x4 b = unpack_signed(B[k][s][h]);
#pragma unroll
                            for (int mb = 0; mb < MBW; ++mb)
                                acc[s][mb] = __builtin_amdgcn_mfma_i32_16x16x64_i8(A[h][mb], b, acc[s][mb], 0, 0, 0);
                        }
                }
            }
            load_x((k + 1) % D, i + 1 + D);
            load_w(k, i + D);
        }
    }
    lds_barrier();  // every wave is done with the staged X
    int* part = reinterpret_cast<int*>(lds);
    int* pw = part + kg * R * P + sg * S * 16;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
        for (int mb = 0; mb < MBW; ++mb)
#pragma unroll
            for (int e = 0; e < 4; ++e) pw[(16 * mb + 4 * g + e) * P + 16 * s + j] = acc[s][mb][e];
    lds_barrier();

    const bool vec = (d.N & 3) == 0 && ((reinterpret_cast<uintptr_t>(d.y) | reinterpret_cast<uintptr_t>(d.acc) |
                                         reinterpret_cast<uintptr_t>(d.resid)) & 15) == 0 &&
                     (reinterpret_cast<uintptr_t>(d.y16) & 7) == 0;
#pragma unroll
    for (int i = 0; i < NQ; ++i) {
        const int q = tid + i * C::THREADS, row = q / (4 * C::BS), c = (q % (4 * C::BS)) * 4;
        const int col = st0 * kStripCols + c;
        if (q >= Q || row >= M || col >= d.N) continue;
        i32x4 v = i32x4{0, 0, 0, 0};
#pragma unroll
        for (int w = 0; w < C::KG; ++w) v += *reinterpret_cast<const i32x4*>(part + (w * R + row) * P + c);
        const float sc = xs[i] * d.w_scale;
        const long long o = (long long)row * d.N + col;
        if (vec) {
            f32x4 y;
#pragma unroll
            for (int e = 0; e < 4; ++e) y[e] = acc_to_float(v[e], d.w_mag) * sc;
            if (d.acc) *reinterpret_cast<TER_GLOBAL i32x4*>(gptr(d.acc) + o) = v;
            if (d.y) *reinterpret_cast<TER_GLOBAL f32x4*>(gptr(d.y) + o) = y;
            if (d.y16 || d.resid) {
                uint16_t h[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    const float ye = y[e];
                    h[e] = float_to_half_bits(ye);
                }
                if (d.y16)
                    *reinterpret_cast<TER_GLOBAL unsigned long long*>(gptr(d.y16) + o) =
                        (unsigned long long)h[0] | (unsigned long long)h[1] << 16 | (unsigned long long)h[2] << 32 |
                        (unsigned long long)h[3] << 48;
                if (d.resid) {
                    TER_GLOBAL f32x4* rp = reinterpret_cast<TER_GLOBAL f32x4*>(gptr(d.resid) + o);
                    f32x4 rv = *rp;
#pragma unroll
                    for (int e = 0; e < 4; ++e) rv[e] = rv[e] + half_bits_to_float(h[e]);
                    *rp = rv;
                }
            }
        } else {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                if (col + e < d.N) emit_out(d, o + e, v[e], sc);
        }
    }
}

template <class C, int kX, bool kList>
hipError_t launch_as(const GemmDesc& single, const GemmDesc* list, const GemmBlock* blocks, int n_blocks,
                     hipStream_t st) {
    static LdsLimit limit;
    const hipError_t e = limit.allow(C::LDS, {reinterpret_cast<const void*>(&gemm_split_kernel<C, kX, kList>)});
    if (e != hipSuccess) return e;
    const int n_sb = (single.n_strips + C::BS - 1) / C::BS, pieces = (single.M + C::R - 1) / C::R;
    const int grid = kList ? n_blocks : 8 * ((n_sb + 7) / 8) * pieces;
    hipLaunchKernelGGL((gemm_split_kernel<C, kX, kList>), dim3(grid), dim3(C::THREADS), C::LDS, st, single, list,
                       blocks, n_sb, pieces);
    return hipGetLastError();
}

template <class C>
hipError_t launch_cfg(const GemmDesc& single, const GemmDesc* list, const GemmBlock* blocks, int n_blocks, bool vec,
                      hipStream_t st) {
    if (list)
        return vec ? launch_as<C, kXVec, true>(single, list, blocks, n_blocks, st)
                   : launch_as<C, kXAny, true>(single, list, blocks, n_blocks, st);
    return vec ? launch_as<C, kXVec, false>(single, list, blocks, n_blocks, st)
               : launch_as<C, kXAny, false>(single, list, blocks, n_blocks, st);
}

// The tiles, largest first; the small ones also for long K (L: more K groups,
// fewer steps per wave; gemm_split_long).
using T64x8 = SCfg<4, 1, 8, 2, 2>;
using T64x4 = SCfg<4, 1, 4, 4, 2>;
using T32x4 = SCfg<2, 1, 4, 4, 2>;
using T32x2 = SCfg<2, 1, 2, 4, 2>;
using T32x2L = SCfg<2, 1, 2, 8, 2>;
using T16x2 = SCfg<1, 1, 2, 4, 2>;
using T16x2L = SCfg<1, 1, 2, 8, 2>;
using T16x1 = SCfg<1, 1, 1, 4, 2>;
using T16x1L = SCfg<1, 1, 1, 8, 2>;
constexpr int kTiles = 6;
struct TileShape {
    int rows, strips;
    float unit_us;  // gemm_split_tile_us
};
constexpr TileShape kTile[kTiles] = {{64, 8, 0.60f}, {64, 4, 0.38f}, {32, 4, 0.23f},
                                     {32, 2, 0.16f}, {16, 2, 0.12f}, {16, 1, 0.062f}};

}  // namespace

int gemm_split_tiles() { return kTiles; }
int gemm_split_bytes_tile() { return kTiles - 1; }  // T16x1
int gemm_split_rows(int tile) { return kTile[tile].rows; }
int gemm_split_strips(int tile) { return kTile[tile].strips; }

// Time a tile over Ku 256-row units of K takes its CU beyond a launch's fixed
// part, for the choice of the kernel and tile (pick_gemm in abi.hip): fitted
// to HIP-event times of single GEMMs over cached weights (3 us fixed; tiles
// beyond the CU count take turns), which it gives within about 16% for M =
// 2-256, K = 256-8192, N = 640-16384.  E.g. M = 64, 6912 x 2560: 7.6 (measured
// 7.25) as 32 x 2 tiles, 9.7 (9.0) as 32 x 4; M = 256, 2560 x 6912: 10.2 (9.8) as
// 64 x 8, 12.1 (10.8) as 64 x 4; M = 8, 2560 x 16384: 5.9 (5.1) as 16 x 2, 6.0
// (5.9) as 16 x 1.
float gemm_split_tile_us(int tile, int Ku) { return kTile[tile].unit_us * (float)(Ku + 2); }

// Whether a launch of this tile and largest Ku takes the long-K form.  Short
// against long, weights from HBM (cached): one GEMM of 16 x 1 tiles at M = 8,
// 2560 x 2560 4.9, 4.7 us (3.3, 3.4), 3328 x 4096 5.6, 5.1 (3.7, 3.6), 5120 x 4096
// 6.7, 5.7 (4.1, 3.9); of 16 x 2 tiles 5120 x 8192 7.4, 7.0 (5.1, 5.2); of 32 x 2
// at M = 64, 5120 x 2560 7.9, 8.6 (6.3, 6.4), 6144 x 2560 8.6, 8.7 (7.0, 6.6); rows
// at any address, M = 16, 5001 x 2048 7.3, 7.8 (5.2, 5.8).  In a list the short
// items pay for the long ones: K = 1024 and 4096, M = 8 6.9, 7.8 (5.0, 5.9).
bool gemm_split_long(int tile, int Ku, bool single_vec) { return Ku > (single_vec && tile == kTiles - 1 ? 12 : 20); }

hipError_t launch_gemm_split(const GemmDesc& single, const GemmDesc* list_dev, const GemmBlock* blocks_dev,
                             int n_blocks, int tile, bool longk, bool vec, bool bytes, hipStream_t st) {
    if (bytes)
        return list_dev ? launch_as<T16x1, kXBytes, true>(single, list_dev, blocks_dev, n_blocks, st)
                        : launch_as<T16x1, kXBytes, false>(single, list_dev, blocks_dev, n_blocks, st);
    switch (2 * tile + (longk ? 1 : 0)) {
        case 0:
        case 1: return launch_cfg<T64x8>(single, list_dev, blocks_dev, n_blocks, vec, st);
        case 2:
        case 3: return launch_cfg<T64x4>(single, list_dev, blocks_dev, n_blocks, vec, st);
        case 4:
        case 5: return launch_cfg<T32x4>(single, list_dev, blocks_dev, n_blocks, vec, st);
        case 6: return launch_cfg<T32x2>(single, list_dev, blocks_dev, n_blocks, vec, st);
        case 7: return launch_cfg<T32x2L>(single, list_dev, blocks_dev, n_blocks, vec, st);
        case 8: return launch_cfg<T16x2>(single, list_dev, blocks_dev, n_blocks, vec, st);
        case 9: return launch_cfg<T16x2L>(single, list_dev, blocks_dev, n_blocks, vec, st);
        case 10: return launch_cfg<T16x1>(single, list_dev, blocks_dev, n_blocks, vec, st);
        case 11: return launch_cfg<T16x1L>(single, list_dev, blocks_dev, n_blocks, vec, st);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace terhip
