// pack.hip -- device repack between the reference v11 layout and T16, the
// synthetic-data generators used by the benchmark, and the per-row int8
// activation quantizer of the batched path.
//
// v11 (reference wire format, tools/convert_llama_to_packed.py:128-140 and
// the decoder in cuda/ter_cuda_forward_packed.cu:355-374): byte
// W_col[j_byte * K + k] holds columns 4 j_byte + s at bits 2s..2s+1 with the
// code map of include/ter/pack.hpp:8-21 (00 = 0, 01 = +1, 10 = -1, 11 = 0).
// T16 is described in common.h.
#include "common.h"

namespace terhip {
namespace {

typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_any __attribute__((aligned(1)));         // at any byte address
typedef unsigned int u32_any __attribute__((aligned(1)));

// Format conversion.  What bounds it: HBM, packed bytes in and packed bytes
// out.  A thread makes one lane's 16 bytes of a T16 tile (4 columns x 16 rows
// of K) from whole 16-byte pieces of the file format: v11 holds those 64
// trits in 16 consecutive bytes of one column quad, i2_s in 16 consecutive
// bytes of each column, and in both the four trits of a T16 field group come
// out of one dword with a shift and a mask.  Measured at 6912 x 2560 (4.4 MB in
// and out): i2_s 13.3 -> 4.3 us, v11 in 11.3 -> 3.5 us, v11 out 14.1 -> 3.6 us, against one byte load per
// trit and one byte store per four.

// Four 2-bit v11 codes, one per byte, -> u = w + 1 (00 -> 1, 01 -> 2, 10 -> 0, 11 -> 1).
__device__ __forceinline__ unsigned codes_to_u(unsigned c) {
    const unsigned k1 = 0x01010101u, b0 = c & k1, b1 = (c >> 1) & k1;
    return ((b0 & ~b1) << 1) | (b0 ^ b1 ^ k1);
}

// Four T16 fields u, one per byte, -> v11 codes (0 -> 10, 1 -> 00, 2 -> 01, 3 -> 00).
__device__ __forceinline__ unsigned u_to_codes(unsigned u) {
    const unsigned k1 = 0x01010101u, b0 = u & k1, b1 = (u >> 1) & k1;
    return ((~(b0 | b1) & k1) << 1) | (b1 & ~b0);
}

// This thread's lane slot: tile (strip s, unit u), columns n0 .. n0 + 3 and
// rows k0 .. k0 + 15 of K.
struct LaneSlot {
    int n0, k0, u, q;
    __device__ LaneSlot(long long i, int Ku) {
        const int lane = (int)(i & 63);
        const long long tile = i >> 6;
        const int s = (int)(tile / Ku);
        u = (int)(tile - (long long)s * Ku);
        q = lane & 15;
        n0 = s * kStripCols + (lane >> 4) * 4;
        k0 = u * kUnitK + q * 16;
    }
};

// The fix-up slots of a strip's columns, zero at rest: written by its first
// unit's threads (a fill inside the launch, where a memset would be a second
// one and a memset node of a captured graph).
__device__ __forceinline__ void clear_fix(const LaneSlot& l, unsigned long long* fix, int N) {
    if (l.u == 0 && l.q < 4 && l.n0 + l.q < N) gptr(fix)[l.n0 + l.q] = 0ull;
}

__global__ __launch_bounds__(256) void pack_v11_kernel(const uint8_t* __restrict__ v11, u32x4* __restrict__ t16,
                                                       unsigned long long* __restrict__ fix, int K, int N, int Ku,
                                                       long long n_slots) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n_slots) return;
    const LaneSlot l(i, Ku);
    clear_fix(l, fix, N);
    u32x4 raw = {0u, 0u, 0u, 0u};  // (code 00 is w = 0, the padding)
    if (l.n0 < N && l.k0 < K) {
        const TER_GLOBAL uint8_t* p = gptr(v11) + (long long)(l.n0 >> 2) * K + l.k0;
        if (l.k0 + 16 <= K) {
            raw = *reinterpret_cast<const TER_GLOBAL u32x4_any*>(p);
        } else {
            for (int e = 0; e < K - l.k0; ++e) raw[e >> 2] |= (unsigned)p[e] << (8 * (e & 3));
        }
    }
    u32x4 out;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        unsigned d = 0;
#pragma unroll
        for (int f = 0; f < 4; ++f) d |= codes_to_u((raw[f] >> (2 * j)) & 0x03030303u) << (2 * f);
        out[j] = d;
    }
    t16[i] = out;
}

// From microsoft/BitNet i2_s bytes (tools/convert_bitnet_to_packed.py:85-157,
// vendor/ntransformer/core/dequant.cpp:114-145): the (N, K) tensor row-major
// (element e = n K + k) in blocks of 128 elements per 32 bytes; byte p of a
// block holds positions p, p+32, p+64, p+96 at shifts 6, 4, 2, 0; codes 0 -> -1,
// 1 -> 0, 2 -> +1, 3 -> 0, i.e. u = w + 1 = {0, 1, 2, 1}.  K is a multiple of 4,
// so four rows of K lie in one dword of the codes at one shift; with K a
// multiple of 16 (k16) a thread's 16 rows lie in 16 consecutive bytes.
template <bool k16>
__global__ __launch_bounds__(256) void pack_i2s_kernel(const uint8_t* __restrict__ raw, u32x4* __restrict__ t16,
                                                       unsigned long long* __restrict__ fix, int K, int N, int Ku,
                                                       long long n_slots) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n_slots) return;
    const LaneSlot l(i, Ku);
    clear_fix(l, fix, N);
    const unsigned kM = 0x03030303u, k1 = 0x01010101u;
    u32x4 out;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        out[j] = 0x55555555u;  // u = 1: w = 0
        if (l.n0 + j >= N || l.k0 >= K) continue;
        const long long el = (long long)(l.n0 + j) * K + l.k0;
        u32x4 w;
        if constexpr (k16)
            w = *reinterpret_cast<const TER_GLOBAL u32x4_any*>(gptr(raw) + (el >> 7) * 32 + (el & 31));
        unsigned d = 0;
#pragma unroll
        for (int f = 0; f < 4; ++f) {
            const long long ef = el + 4 * f;
            unsigned c = 0;
            if constexpr (k16) {
                c = w[f];
            } else if (l.k0 + 4 * f < K) {
                c = *reinterpret_cast<const TER_GLOBAL u32_any*>(gptr(raw) + (ef >> 7) * 32 + (ef & 31));
            } else {
                c = 0x55555555u;  // code 1
            }
            c = (c >> (6 - 2 * (int)((ef & 127) >> 5))) & kM;
            c ^= (c & (c >> 1) & k1) << 1;  // code 3 -> 1
            d |= c << (2 * f);
        }
        out[j] = d;
    }
    t16[i] = out;
}

__global__ __launch_bounds__(256) void unpack_v11_kernel(const u32x4* __restrict__ t16, uint8_t* __restrict__ v11,
                                                         int K, int N, int Ku, long long n_slots) {
    const long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i >= n_slots) return;
    const LaneSlot l(i, Ku);
    if (l.n0 >= N || l.k0 >= K) return;
    const u32x4 w = t16[i];
    u32x4 out;
#pragma unroll
    for (int f = 0; f < 4; ++f) {
        unsigned d = 0;
#pragma unroll
        for (int j = 0; j < 4; ++j) d |= u_to_codes((w[j] >> (2 * f)) & 0x03030303u) << (2 * j);
        out[f] = d;
    }
    TER_GLOBAL uint8_t* p = gptr(v11) + (long long)(l.n0 >> 2) * K + l.k0;
    if (l.k0 + 16 <= K) {
        *reinterpret_cast<TER_GLOBAL u32x4_any*>(p) = out;
    } else {
        for (int e = 0; e < K - l.k0; ++e) p[e] = (uint8_t)(out[e >> 2] >> (8 * (e & 3)));
    }
}

__device__ __forceinline__ uint64_t splitmix(uint64_t seed, uint64_t idx) {
    uint64_t z = seed + (idx + 1) * 0x9E3779B97F4A7C15ull;
    z = (z ^ (z >> 30)) * 0xBF58476D1CE4E5B9ull;
    z = (z ^ (z >> 27)) * 0x94D049BB133111EBull;
    return z ^ (z >> 31);
}

// One thread per v11 byte: 4 trits of columns 4 jb .. 4 jb + 3 at row k.
__global__ void synth_v11_kernel(uint8_t* __restrict__ v11, int K, int N, uint64_t seed, uint32_t t0,
                                 uint32_t t1) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    const long long total = (long long)(N / 4) * K;
    if (i >= total) return;
    const int jb = (int)(i / K);
    const int k = (int)(i - (long long)jb * K);
    unsigned byte = 0;
#pragma unroll
    for (int sub = 0; sub < 4; ++sub) {
        const uint64_t idx = (uint64_t)k * (uint64_t)N + (uint64_t)(jb * 4 + sub);
        const uint32_t uu = (uint32_t)(splitmix(seed, idx) >> 32);
        const unsigned code = uu < t0 ? 0u : (uu < t1 ? 1u : 2u);
        byte |= code << (2 * sub);
    }
    v11[i] = (uint8_t)byte;
}

__global__ void synth_i8_kernel(int8_t* __restrict__ x, long long n, uint64_t seed, int lo, int hi) {
    const long long i = (long long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const uint64_t uu = splitmix(seed, (uint64_t)i) >> 32;
    const uint64_t span = (uint64_t)(hi - lo + 1);
    x[i] = (int8_t)(lo + (int)((uu * span) >> 32));
}

// Per-row quantizers, one workgroup per row: quant_int8_k
// (cuda/ter_cuda_forward_packed.cu:40-62) alone (kind X_F32), or behind the
// fused RMSNorm (rmsnorm_quant_f32_in_k / rmsnorm_quant_fp16_in_k,
// cuda/ter_cuda_forward_bitnet.cu:64-146) or relu^2(gate) * up and RMSNorm
// (relu2_mul_rmsnorm_quant_k, ibid.:258-309).  The sums of squares keep the
// reference's order: 256 (relu^2: 1024) strided partials with fused
// multiply-adds (the reference build contracts `local_sum += v * v`), then the
// halving tree; rms_inv = 1 / sqrt(ss / K + eps) correctly rounded (the
// reference's rsqrtf is an approximation); n = (x * rms_inv) * gamma.
//
// What bounds them: latency, with a workgroup per row and a row of a few KB.
// A thread loads its NC chunks of 8 elements at once (16-byte loads where x,
// up and gamma rows are 16-byte aligned with K a multiple of 8, else one load
// per element), keeps them in registers through both passes, and the row is
// read once.  For the norm's order the values also go to LDS as fp32, from
// where the partials' threads read their strided elements; every wave then
// forms the tree from the partials in LDS, so the sum needs two barriers and
// the absmax one.  1024 threads past K = 4096 (a chunk or two each).  Before,
// three passes of one-element loads: relu^2 at 64
// rows of 6912 21.9 -> 3.9 us, fp32 RMSNorm at 64 rows of 2560 7.0 -> 3.0,
// absmax at 256 rows of 2560 4.4 -> 2.6 (launches in a graph).
template <int T, int NC, int KIND, bool kVec>
__global__ __launch_bounds__(T) void quant_rows_kernel(const void* __restrict__ x, const uint16_t* __restrict__ up,
                                                       const uint16_t* __restrict__ gamma, float eps, int K,
                                                       int8_t* __restrict__ q, float* __restrict__ scale_out) {
#pragma clang fp contract(off)
    constexpr bool kRms = KIND != TER_HIP_X_F32;
    constexpr bool kF32 = KIND == TER_HIP_X_F32 || KIND == TER_HIP_X_F32_RMS;
    constexpr int NP = KIND == TER_HIP_X_RELU2_RMS ? 1024 : 256;  // strided partial sums of squares
    constexpr int EL = kF32 ? 4 : 2;
    extern __shared__ __align__(16) float lds[];                  // kRms: the row's values [8 T NC], then partials [NP]
    __shared__ float wmax[T / 64];
    const int m = blockIdx.x, t = threadIdx.x, lane = t & 63;
    const long long row0 = (long long)m * K;
    auto rsrc = [](const void* p, int bytes) { return __builtin_amdgcn_make_buffer_rsrc((void*)p, 0, bytes, 0x00020000); };
    const __amdgpu_buffer_rsrc_t xr = rsrc(static_cast<const char*>(x) + row0 * EL, K * EL);
    const __amdgpu_buffer_rsrc_t ur = rsrc(up + row0, KIND == TER_HIP_X_RELU2_RMS ? 2 * K : 0);
    const __amdgpu_buffer_rsrc_t gr = rsrc(gamma, kRms ? 2 * K : 0);

    // element i of this thread's chunk c: 8 consecutive ones, or (one load per
    // element) those a workgroup apart, so that a wave's loads stay contiguous
    auto at = [t](int c, int i) { return kVec ? 8 * (t + T * c) + i : t + T * (8 * c + i); };
    // raw values of every chunk (past K zeros), all loads issued first
    auto load8 = [&](__amdgpu_buffer_rsrc_t r, int c, unsigned (&w)[4]) {  // 8 halves
        if constexpr (kVec) {
            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(r, 2 * at(c, 0), 0, 0);
            w[0] = v.x; w[1] = v.y; w[2] = v.z; w[3] = v.w;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i)
                w[i] = (unsigned)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, 2 * at(c, 2 * i), 0, 0) |
                       (unsigned)(uint16_t)__builtin_amdgcn_raw_buffer_load_b16(r, 2 * at(c, 2 * i + 1), 0, 0) << 16;
        }
    };
    unsigned xw[NC][kF32 ? 8 : 4], uw[NC][4], gw[NC][4];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if constexpr (kF32) {
            if constexpr (kVec) {
#pragma unroll
                for (int h = 0; h < 2; ++h) {
                    const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(xr, 4 * at(c, 4 * h), 0, 0);
                    xw[c][4 * h] = v.x; xw[c][4 * h + 1] = v.y; xw[c][4 * h + 2] = v.z; xw[c][4 * h + 3] = v.w;
                }
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) xw[c][i] = __builtin_amdgcn_raw_buffer_load_b32(xr, 4 * at(c, i), 0, 0);
            }
        } else {
            load8(xr, c, xw[c]);
        }
        if constexpr (KIND == TER_HIP_X_RELU2_RMS) load8(ur, c, uw[c]);
        if constexpr (kRms) load8(gr, c, gw[c]);
    }
    auto half_of = [](const unsigned (&w)[4], int i) { return half_bits_to_float((uint16_t)(w[i >> 1] >> (16 * (i & 1)))); };
    float v[NC][8];
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            if constexpr (kF32)
                v[c][i] = __builtin_bit_cast(float, xw[c][i]);
            else if constexpr (KIND == TER_HIP_X_F16_RMS)
                v[c][i] = half_of(xw[c], i);
            else
                v[c][i] = relu2_mul(half_of(xw[c], i), half_of(uw[c], i));
        }
    if constexpr (kRms) {
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            if constexpr (kVec) {
#pragma unroll
                for (int h = 0; h < 2; ++h)
                    *reinterpret_cast<float4*>(lds + at(c, 4 * h)) =
                        float4{v[c][4 * h], v[c][4 * h + 1], v[c][4 * h + 2], v[c][4 * h + 3]};
            } else {
#pragma unroll
                for (int i = 0; i < 8; ++i) lds[at(c, i)] = v[c][i];
            }
        }
        __syncthreads();
        // partial p: elements p, p + NP, .. in order (threads past NP idle; with
        // fewer threads than partials each takes several)
        float* part = lds + 8 * T * NC;
        for (int p = t; p < NP; p += T) {
            // (values past K are zeros: exact no-ops)
            float s = 0.f;
#pragma unroll 16
            for (int i = 0; i < 8 * T * NC / NP; ++i) s = __builtin_fmaf(lds[p + NP * i], lds[p + NP * i], s);
            part[p] = s;
        }
        __syncthreads();
        // the tree's levels down to 64 per lane, then the wave's
        auto p256 = [&](int i) {
            if constexpr (NP == 1024)
                return (part[i] + part[i + 512]) + (part[i + 256] + part[i + 768]);
            else
                return part[i];
        };
        const float ss = tree_down64((p256(lane) + p256(lane + 128)) + (p256(lane + 64) + p256(lane + 192)));
        const float rms_inv = 1.0f / __builtin_sqrtf(ss / (float)K + eps);
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int i = 0; i < 8; ++i) v[c][i] = (v[c][i] * rms_inv) * half_of(gw[c], i);
    }
    float mx = 0.f;
#pragma unroll
    for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int i = 0; i < 8; ++i)
            if (at(c, i) < K) mx = fmaxf(mx, fabsf(v[c][i]));
    mx = fmaxf(mx, dpp_move_f<0xB1>(mx));   // lanes 1 and 2 apart (quad permutations), then the
    mx = fmaxf(mx, dpp_move_f<0x4E>(mx));   // half-row and row mirrors, then across rows
    mx = fmaxf(mx, dpp_move_f<0x141>(mx));
    mx = fmaxf(mx, dpp_move_f<0x140>(mx));
    mx = fmaxf(mx, lane_xor16(mx));
    mx = fmaxf(mx, lane_xor32(mx));
    if (lane == 0) wmax[t >> 6] = mx;
    __syncthreads();
#pragma unroll
    for (int w = 0; w < T / 64; ++w) mx = fmaxf(mx, wmax[w]);
    const float amax = mx + 1e-9f;
    const float scale = 127.0f / amax;
    if (t == 0) scale_out[m] = 1.0f / scale;
    int8_t* qr = q + row0;
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        if (at(c, 0) >= K) continue;
        unsigned w[2] = {0u, 0u};
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            int qi = (int)__builtin_rintf(v[c][i] * scale);
            qi = qi > 127 ? 127 : (qi < -128 ? -128 : qi);
            w[i >> 2] |= (unsigned)(uint8_t)qi << (8 * (i & 3));
        }
        if constexpr (kVec) {
            *reinterpret_cast<TER_GLOBAL unsigned long long*>(gptr(qr) + at(c, 0)) =
                (unsigned long long)w[0] | (unsigned long long)w[1] << 32;
        } else {
#pragma unroll
            for (int i = 0; i < 8; ++i)
                if (at(c, i) < K) gptr(qr)[at(c, i)] = (int8_t)(w[i >> 2] >> (8 * (i & 3)));
        }
    }
}

template <int T, int NC, int KIND>
hipError_t launch_quant_as(const void* x, const uint16_t* up, const uint16_t* gamma, float eps, int M, int K, int8_t* q,
                           float* s, hipStream_t st) {
    const int lds = KIND == TER_HIP_X_F32 ? 0 : (8 * T * NC + (KIND == TER_HIP_X_RELU2_RMS ? 1024 : 256)) * 4;
    auto a16 = [](const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; };
    const bool vec = K % 8 == 0 && a16(x) && a16(up) && a16(gamma) && (reinterpret_cast<uintptr_t>(q) & 7u) == 0;
    static LdsLimit limit;
    const hipError_t e = limit.allow(lds, {reinterpret_cast<const void*>(&quant_rows_kernel<T, NC, KIND, true>),
                                           reinterpret_cast<const void*>(&quant_rows_kernel<T, NC, KIND, false>)});
    if (e != hipSuccess) return e;
    if (vec)
        hipLaunchKernelGGL((quant_rows_kernel<T, NC, KIND, true>), dim3(M), dim3(T), lds, st, x, up, gamma, eps, K, q, s);
    else
        hipLaunchKernelGGL((quant_rows_kernel<T, NC, KIND, false>), dim3(M), dim3(T), lds, st, x, up, gamma, eps, K, q, s);
    return hipGetLastError();
}

// Threads and chunks by K (at most 32768).
template <int KIND>
hipError_t launch_quant_kind(const void* x, const uint16_t* up, const uint16_t* gamma, float eps, int M, int K,
                             int8_t* q, float* s, hipStream_t st) {
    if (K <= 2048) return launch_quant_as<256, 1, KIND>(x, up, gamma, eps, M, K, q, s, st);
    if (K <= 4096) return launch_quant_as<512, 1, KIND>(x, up, gamma, eps, M, K, q, s, st);
    if (K <= 8192) return launch_quant_as<1024, 1, KIND>(x, up, gamma, eps, M, K, q, s, st);
    if (K <= 16384) return launch_quant_as<1024, 2, KIND>(x, up, gamma, eps, M, K, q, s, st);
    if (K <= 32768) return launch_quant_as<1024, 4, KIND>(x, up, gamma, eps, M, K, q, s, st);
    return hipErrorInvalidValue;
}

inline unsigned grid_of(long long n, int block) { return (unsigned)((n + block - 1) / block); }

}  // namespace

hipError_t launch_pack_v11(const uint8_t* v11, uint8_t* t16, uint64_t* fix, int K, int N, hipStream_t st) {
    const int Ku = units_of(K);
    const long long n = (long long)strips_of(N) * Ku * 64;
    hipLaunchKernelGGL(pack_v11_kernel, dim3(grid_of(n, 256)), dim3(256), 0, st, v11, reinterpret_cast<u32x4*>(t16),
                       reinterpret_cast<unsigned long long*>(fix), K, N, Ku, n);
    return hipGetLastError();
}

hipError_t launch_pack_i2s(const uint8_t* raw, uint8_t* t16, uint64_t* fix, int K, int N, hipStream_t st) {
    const int Ku = units_of(K);
    const long long n = (long long)strips_of(N) * Ku * 64;
    auto* f = reinterpret_cast<unsigned long long*>(fix);
    if (K % 16 == 0)
        hipLaunchKernelGGL(pack_i2s_kernel<true>, dim3(grid_of(n, 256)), dim3(256), 0, st, raw,
                           reinterpret_cast<u32x4*>(t16), f, K, N, Ku, n);
    else
        hipLaunchKernelGGL(pack_i2s_kernel<false>, dim3(grid_of(n, 256)), dim3(256), 0, st, raw,
                           reinterpret_cast<u32x4*>(t16), f, K, N, Ku, n);
    return hipGetLastError();
}

hipError_t launch_unpack_v11(const uint8_t* t16, uint8_t* v11, int K, int N, hipStream_t st) {
    const int Ku = units_of(K);
    const long long n = (long long)strips_of(N) * Ku * 64;
    hipLaunchKernelGGL(unpack_v11_kernel, dim3(grid_of(n, 256)), dim3(256), 0, st,
                       reinterpret_cast<const u32x4*>(t16), v11, K, N, Ku, n);
    return hipGetLastError();
}

hipError_t launch_synth_v11(uint8_t* v11, int K, int N, uint64_t seed, uint32_t t0, uint32_t t1,
                            hipStream_t st) {
    const long long total = (long long)(N / 4) * K;
    hipLaunchKernelGGL(synth_v11_kernel, dim3(grid_of(total, 256)), dim3(256), 0, st, v11, K, N, seed,
                       t0, t1);
    return hipGetLastError();
}

hipError_t launch_synth_i8(int8_t* x, long long n, uint64_t seed, int lo, int hi, hipStream_t st) {
    hipLaunchKernelGGL(synth_i8_kernel, dim3(grid_of(n, 256)), dim3(256), 0, st, x, n, seed, lo, hi);
    return hipGetLastError();
}

hipError_t launch_rmsnorm_quant_rows(const void* x, const uint16_t* up, int kind, const uint16_t* gamma, float eps,
                                     int M, int K, int8_t* q, float* s, hipStream_t st) {
    if (kind == TER_HIP_X_F32_RMS) return launch_quant_kind<TER_HIP_X_F32_RMS>(x, nullptr, gamma, eps, M, K, q, s, st);
    if (kind == TER_HIP_X_F16_RMS) return launch_quant_kind<TER_HIP_X_F16_RMS>(x, nullptr, gamma, eps, M, K, q, s, st);
    return launch_quant_kind<TER_HIP_X_RELU2_RMS>(x, up, gamma, eps, M, K, q, s, st);
}

hipError_t launch_quant_rows(const float* x, int M, int K, int8_t* q, float* s, hipStream_t st) {
    return launch_quant_kind<TER_HIP_X_F32>(x, nullptr, nullptr, 0.f, M, K, q, s, st);
}

}  // namespace terhip
