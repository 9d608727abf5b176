// project.hip — the QKV projection of a decode step on gfx950: attention RMSNorm of the
// residual rows and the fused [Wq | Wk | Wv] product, one HBM-streaming launch.
//
// Reference: CudaModel::body runs k_rmsnorm (x -> h) and linear(h, L.qkv, qkv, B, QKV, E), a
// GEMV per weight segment for B == 1 (src/cuda/model_cuda.cu:1797-1799, GEMV :300-320); the CPU
// path runs rmsnorm then matvec with wq, wk, wv (src/model.cpp:176-179, src/ops.cpp:126-160).
// The rows come out raw, in the [Q | K | V] layout the decode step reads: the per-head QK-norm,
// RoPE and the cache append that the reference launches next (three more kernels) are the
// epilogue that ei_decode_step / ei_decode_step_paged apply inside the attention launch.
//
// A decode step's projection streams the weights once per launch (E x (H + 2 HKV) x 128 weights:
// 63 MB in fp32, 31 MB in fp16, 9-17 MB in blocks at Qwen3-4B).  One workgroup per CU keeps to a
// contiguous range of output rows.  A row's E weights are spread over the lanes of a row group (L lanes,
// 8 to 32 weights each; 1 to 8 groups to a workgroup work on different rows), so the normed activations
// that a lane multiplies by are the same for every row: they are loaded, normed and kept in registers
// once, and nothing but weights moves after that.  (Read from LDS for every pair of rows they bound the
// kernel with several activation rows: each wave reads rows x E x 4 bytes for two weight rows and waits for
// every read by itself.)  A lane keeps RB rows of weights in flight:
// each row's registers are loaded again, with the row RB further on, as soon as they are used, so the
// stream runs on under the arithmetic.  The partial sums of RB rows x NB activation rows are added over
// 32 lanes by one transposing butterfly and over the half-waves of the group through LDS.
//
// Measured, graph-timed per launch, activations read from LDS -> this layout (us; a plain read of the weights takes 6.2
// at 31.5 MB, 8.7 at 50 MB): F16 at E 2560, 6144 outputs, 2 rows 12.3 -> 8.1, 4 rows 24.1 -> 9.6; E 4096, 4 rows 39.0 ->
// 12.4; E 5120, 7168 outputs, 4 rows 74.8 -> 16.8; F32 there 66.5 -> 25.9; Q8_0 40.7 -> 16.6; Q4_K 40.1 -> 15.4; Q6_K
// 48.0 -> 17.1; one row of Q6_K at 5120 18.1 -> 15.5; Q4_K at E 1024, 4096 outputs, 4 rows 5.9 -> 4.4.  Several rows cost
// little more than one: the stream bounds them, and what is left over it is the launch's start, the norm
// and the last batch's sums.  Tried and not kept: the sums in LDS-read order with four or eight waves a
// workgroup (F16, E 2560, 4 rows: 14.2), activations loaded lane by lane from memory (16 values a lane, 64
// bytes apart: Q4_K one row 7.3 against 6.4), two workgroups a CU (8.9), 15 waves (7.8), branches around the
// reloads (vmcnt waits for everything behind them; F32 one row 15.0 against 11.6).
//
// Quantised weights (Q8_0, Q4_K, Q6_K: the block formats the reference computes with,
// src/quant.h:21-39) stay in their GGUF block layout.  Each lane decodes items of 16
// consecutive values (half a Q8_0 block, half a 32-value Q4_K sub-block, a 16-value Q6_K group)
// straight from registers, with the reference's values (src/quant.cpp:7-60), so every
// weight is the float the CPU path's convert_row gives, before the same FMA dot as the float
// kernels.
#include <hip/hip_fp16.h>

#include <type_traits>

#include "common.h"
#include "launch.h"

namespace ei {

constexpr int kProjMaxLdsFloats = 24576;  // rows per launch at hidden size E: at most this over E
typedef unsigned u32x4_t __attribute__((ext_vector_type(4)));

__device__ __forceinline__ void f16x8(const u32x4_t u, float* f) {
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const __half2 h = *reinterpret_cast<const __half2*>(&w[i]);
        f[2 * i] = __low2float(h);
        f[2 * i + 1] = __high2float(h);
    }
}

// ------------------------------------------------------------------ quantised weights
template <int T>
struct QFormat;
template <>
struct QFormat<8> {  // Q8_0
    static constexpr int kValues = 32, kBytes = 34;
};
template <>
struct QFormat<12> {  // Q4_K
    static constexpr int kValues = 256, kBytes = 144;
};
template <>
struct QFormat<14> {  // Q6_K
    static constexpr int kValues = 256, kBytes = 210;
};

__device__ __forceinline__ float f16_bits(uint32_t h) {
    return __half2float(__ushort_as_half((unsigned short)(h & 0xFFFFu)));
}
// 16 bytes from an address that may be only 2-byte aligned (Q8_0 and Q6_K blocks are 34 and 210
// bytes; gfx950 global loads need no natural alignment)
__device__ __forceinline__ u32x4_t load16(const uint8_t* p) {
    typedef u32x4_t __attribute__((aligned(2))) u32x4_u;
    return __builtin_nontemporal_load(reinterpret_cast<const u32x4_u*>(p));
}
// byte k of a word as a float (one v_cvt_f32_ubyte)
__device__ __forceinline__ float ubyte_f(uint32_t u, int k) { return (float)((u >> (8 * k)) & 0xFFu); }
// the word as computed, hidden from the optimizer: otherwise it folds a per-word mask into
// every byte's extraction (a bit-field extract per value before the byte conversion; Q4_K
// measured 4% faster with the mask kept, Q8_0 and Q6_K no faster)
__device__ __forceinline__ uint32_t opaque(uint32_t u) {
    asm volatile("" : "+v"(u));
    return u;
}

// One row's weights of a lane, as loaded: load() from the row's first byte, values() their floats.
// lane_in_row 0 .. L-1; F32 and F16 lanes take the 16-byte pieces c * L + lane_in_row (whole 1 KB per
// instruction), quantised lanes item lane_in_row (values 16 lane_in_row .. + 15).
template <int T, int E>
struct RowShape {
    static constexpr int kPer = T == 0 ? 4 : T == 1 ? 8 : 16;  // values per piece or item
    // 8 values a lane (F32, F16) while a row then takes at most 512 lanes, else 16 or 32
    static constexpr int kVals = T > 1 ? 16 : E / 8 <= 512 ? 8 : E / 16 <= 512 ? 16 : 32;
    static constexpr int kLanes = E / kVals;  // lanes of a row group
    static constexpr int kPieces = kVals / kPer;
    // row groups of a workgroup: 8 waves, or 10 where a row takes 160 or 320 lanes
    static constexpr int kGroups = kLanes == 160 ? 4 : kLanes == 320 ? 2 : 512 / kLanes;
    static constexpr int kThreads = kLanes * kGroups;
    static_assert(kLanes * kVals == E && kLanes % 32 == 0 && kThreads % 64 == 0 && kThreads <= 640, "hidden size");
    // where 4 values from value e on sit in a normed activation row in LDS: the first quarters of all
    // pieces, then the second ones, ..., so that a wave reads contiguous 16-byte parts, the rows of
    // quarters offset against each other so that its stores spread over the banks too
    static constexpr int kQuarters = kPer / 4, kQRow = E / kPer + (kQuarters == 4 ? 2 : kQuarters == 2 ? 4 : 0);
    static constexpr int kHRow = 4 * kQuarters * kQRow;  // floats of a row
    static __device__ __forceinline__ int h_at(int e) { return 4 * ((e / 4) % kQuarters * kQRow + e / kPer); }
    // first value of piece c of a lane
    static __device__ __forceinline__ int first(int c, int li) { return (c * kLanes + li) * kPer; }
};
template <int T, int E>
struct Weights {
    using S = RowShape<T, E>;
    static constexpr size_t kRowBytes = (size_t)E * (T == 0 ? 4 : 2);
    u32x4_t p[S::kPieces];
    __device__ __forceinline__ void load(const uint8_t* row, int li) {
#pragma unroll
        for (int c = 0; c < S::kPieces; ++c)
            p[c] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(row) + c * S::kLanes + li);
    }
    __device__ __forceinline__ void values(int, float* f) const {
#pragma unroll
        for (int c = 0; c < S::kPieces; ++c) {
            if constexpr (T == 1) {
                f16x8(p[c], f + 8 * c);
            } else {
                f[4 * c] = __uint_as_float(p[c].x), f[4 * c + 1] = __uint_as_float(p[c].y);
                f[4 * c + 2] = __uint_as_float(p[c].z), f[4 * c + 3] = __uint_as_float(p[c].w);
            }
        }
    }
};

template <int E>
struct Weights<8, E> {  // Q8_0: y = q * d (src/quant.cpp:7-13); item: half a block
    static constexpr size_t kRowBytes = (size_t)E / QFormat<8>::kValues * QFormat<8>::kBytes;
    u32x4_t q;
    uint32_t d16;
    __device__ __forceinline__ void load(const uint8_t* row, int li) {
        const uint8_t* blk = row + 34 * (li >> 1);
        q = load16(blk + 2 + 16 * (li & 1));
        d16 = *reinterpret_cast<const uint16_t*>(blk);
    }
    __device__ __forceinline__ void values(int, float* wv) const {
#pragma clang fp contract(off)
        const float d = f16_bits(d16);
        const float off = -128.f * d;  // exact (a power-of-two scaling)
        const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t u = qw[i] ^ 0x80808080u;  // int8 q + 128 per byte
            // (q + 128) d - 128 d in one rounding: the exact value is q d, so this is the
            // correctly rounded q * d the reference computes (a zero comes out +0 where the
            // reference may have -0, which changes no sum but an exact zero's sign)
#pragma unroll
            for (int b = 0; b < 4; ++b) wv[4 * i + b] = __builtin_fmaf(ubyte_f(u, b), d, off);
        }
    }
};

template <int E>
struct Weights<12, E> {  // Q4_K: y = (d sc) q - dmin m (src/quant.cpp:15-33); item: half a 32-value sub-block
    static constexpr size_t kRowBytes = (size_t)E / QFormat<12>::kValues * QFormat<12>::kBytes;
    u32x4_t hdr, q;  // the block's first 16 bytes (d, dmin, 12 scale bytes); the item's nibbles
    __device__ __forceinline__ void load(const uint8_t* row, int li) {
        const int v = (li & 15) * 16;
        const uint8_t* blk = row + 144 * (li >> 4);  // blocks are whole 16-byte pieces
        hdr = *reinterpret_cast<const u32x4_t*>(blk);
        q = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(blk + 16 + 32 * (v >> 6) + (v & 31)));
    }
    __device__ __forceinline__ void values(int li, float* wv) const {
#pragma clang fp contract(off)
        const int j = (li & 15) >> 1, hi4 = j & 1;  // sub-block: its 6-bit scale and min (src/quant.h:43-52)
        const float d = f16_bits(hdr.x), dmin = f16_bits(hdr.x >> 16);
        // bytes j%4 of the three words: sub-blocks 0..3 hold theirs in the low six bits of the first two,
        // 4..7 in the nibbles of the third and the top bits of the first two
        const uint32_t a = hdr.y >> (8 * (j & 3)), b = hdr.z >> (8 * (j & 3)), c = hdr.w >> (8 * (j & 3));
        const uint32_t sc = j < 4 ? a & 63u : (c & 15u) | ((a >> 2) & 0x30u);
        const uint32_t m = j < 4 ? b & 63u : ((c >> 4) & 15u) | ((b >> 2) & 0x30u);
        const float dl = d * (float)sc, ml = dmin * (float)m;
        const uint32_t qw[4] = {q.x, q.y, q.z, q.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t nib = opaque((qw[i] >> (4 * hi4)) & 0x0F0F0F0Fu);
            // dl * q is exact (17 x 4 significant bits), so the FMA rounds like dl * q - ml
#pragma unroll
            for (int k = 0; k < 4; ++k) wv[4 * i + k] = __builtin_fmaf(dl, ubyte_f(nib, k), -ml);
        }
    }
};

template <int E>
struct Weights<14, E> {  // Q6_K: y = (d sc) (q - 32) (src/quant.cpp:35-60); item: a 16-value group, one scale
    static constexpr size_t kRowBytes = (size_t)E / QFormat<14>::kValues * QFormat<14>::kBytes;
    u32x4_t ql, qh;
    uint32_t d16;
    int sc;
    __device__ __forceinline__ void load(const uint8_t* row, int li) {
        const uint8_t* blk = row + 210 * (li >> 4);
        const int v = (li & 15) * 16, h = v >> 7, g = (v >> 5) & 3, l = v & 31;
        ql = load16(blk + 64 * h + l + 32 * (g & 1));
        qh = load16(blk + 128 + 32 * h + l);
        sc = (int8_t)blk[192 + 8 * h + (l >> 4) + 2 * g];
        d16 = *reinterpret_cast<const uint16_t*>(blk + 208);
    }
    __device__ __forceinline__ void values(int li, float* wv) const {
#pragma clang fp contract(off)
        const int g = ((li & 15) >> 1) & 3;
        const float dsc = f16_bits(d16) * (float)sc;
        // dsc q - 32 dsc in one rounding (32 dsc is exact): the correctly rounded dsc (q - 32)
        const float off = -32.f * dsc;
        const uint32_t lw[4] = {ql.x, ql.y, ql.z, ql.w}, hw[4] = {qh.x, qh.y, qh.z, qh.w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t lo = (lw[i] >> (4 * (g >> 1))) & 0x0F0F0F0Fu;
            const uint32_t q6 = lo | (((hw[i] >> (2 * g)) & 0x03030303u) << 4);  // 0..63 per byte
#pragma unroll
            for (int b = 0; b < 4; ++b) wv[4 * i + b] = __builtin_fmaf(dsc, ubyte_f(q6, b), off);
        }
    }
};

// Sums of N values over the 32 lanes of each half-wave by a transposing butterfly: at each step a lane
// keeps half of its values and adds its partner's copy of that half, so N values take about N exchanges
// instead of 5 N.  v[k], k < n, of a lane then holds the sum of value at + k.
template <int M, int N>
__device__ __forceinline__ void half_wave_sums(float* v, int lane, int& at, int& n) {
    if constexpr (M >= 1) {
        constexpr int K = (N + 1) / 2;
        const bool up = (lane & M) != 0;
        if constexpr (N > 1) {
#pragma unroll
            for (int i = 0; i < K; ++i) {
                const float hi = i + K < N ? v[i + K] : 0.f;
                const float send = up ? v[i] : hi, keep = up ? hi : v[i];
                v[i] = keep + lane_xor<M>(send);
            }
            at += up ? K : 0;
            n = up ? n - K : min(n, K);
        } else {
            v[0] += lane_xor<M>(v[0]);
        }
        half_wave_sums<M / 2, K>(v, lane, at, n);
    }
}

// T the GGML weight type, NB activation rows, hidden size E, RB weight rows of a group in flight.
// Workgroup i takes output rows [i * rows, (i + 1) * rows): group g the rows g, g + kGroups, ... of it,
// RB at a time.
template <int T, int NB, int E, int RB>
__global__ __launch_bounds__((RowShape<T, E>::kThreads)) void k_qkv_project(const float* __restrict__ x, long x_stride,
                                                                           const float* __restrict__ gamma, float eps,
                                                                           const uint8_t* __restrict__ w, int n_out,
                                                                           int rows, float* __restrict__ out,
                                                                           long out_stride) {
    using S = RowShape<T, E>;
    using W = Weights<T, E>;
    constexpr int NV = S::kVals, HW = S::kLanes / 32, N = RB * NB;  // HW half-waves to a row group
    extern __shared__ __align__(16) float hs[];  // [NB][kHRow] normed activations
    __shared__ double ssum[S::kThreads / 64][NB];
    __shared__ float red[2][S::kThreads / 32][N];
    const int tid = threadIdx.x, lane = tid & 63, hwave = tid >> 5, wave = tid >> 6;
    const int grp = tid / S::kLanes, li = tid - grp * S::kLanes;
    const int row_lo = blockIdx.x * rows, row_hi = min(row_lo + rows, n_out);

    // ---- the activations and gammas first, 4 to a thread at a time, then RB rows of weights: loads return
    // in order, so the norm waits for the activations only and runs while the weights are on their way
    constexpr int kX = (E / 4 + S::kThreads - 1) / S::kThreads;
    float4 xv[NB][kX], gv[kX];
#pragma unroll
    for (int i = 0; i < kX; ++i) {
        const int e = 4 * min(tid + i * S::kThreads, E / 4 - 1);
        gv[i] = *reinterpret_cast<const float4*>(gamma + e);
#pragma unroll
        for (int b = 0; b < NB; ++b) xv[b][i] = *reinterpret_cast<const float4*>(x + (size_t)b * x_stride + e);
    }
    W wt[RB];
    // the row of this group's j-th turn; past the range the last row again (loaded, not used)
    auto row_at = [&](int j) { return min(row_lo + grp + j * S::kGroups, row_hi - 1); };
#pragma unroll
    for (int i = 0; i < RB; ++i) wt[i].load(w + (size_t)row_at(i) * W::kRowBytes, li);

    // ---- attention RMSNorm (src/ops.cpp:155-160: sum of squares in double,
    // inv = float(1 / sqrt(ss / E + eps)), h = (x * inv) * gamma)
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        double ss = 0.0;
#pragma unroll
        for (int i = 0; i < kX; ++i) {
            const float4 v = xv[b][i];
            if (tid + i * S::kThreads < E / 4)
                ss += ((double)v.x * (double)v.x + (double)v.y * (double)v.y) +
                      ((double)v.z * (double)v.z + (double)v.w * (double)v.w);
        }
        ss = wave_sum_f64(ss);
        if (lane == 0) ssum[wave][b] = ss;
    }
    lds_barrier();
    {
        // lane b of every four takes the root of activation row b
        const int mb = NB == 1 ? 0 : min(lane & 3, NB - 1);
        double ss = 0.0;
#pragma unroll
        for (int k = 0; k < S::kThreads / 64; ++k) ss += ssum[k][mb];
        const float inv = (float)(1.0 / sqrt(ss / (double)E + (double)eps));
#pragma unroll
        for (int b = 0; b < NB; ++b) {
            const float ib = __int_as_float(__builtin_amdgcn_readlane(__float_as_int(inv), b));
#pragma unroll
            for (int i = 0; i < kX; ++i) {
#pragma clang fp contract(off)
                const float4 v = xv[b][i], g = gv[i];
                const int e = 4 * (tid + i * S::kThreads);
                if (e < E)
                    *reinterpret_cast<float4*>(hs + b * S::kHRow + S::h_at(e)) =
                        make_float4((v.x * ib) * g.x, (v.y * ib) * g.y, (v.z * ib) * g.z, (v.w * ib) * g.w);
            }
        }
    }
    lds_barrier();
    float h[NB][NV];  // this lane's activations, for every row it works on
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int k = 0; k < NV; k += 4) {
            const float4 v = *reinterpret_cast<const float4*>(
                hs + b * S::kHRow + S::h_at(S::first(k / S::kPer, li) + k % S::kPer));
            h[b][k] = v.x, h[b][k + 1] = v.y, h[b][k + 2] = v.z, h[b][k + 3] = v.w;
        }

    // ---- the rows, RB at a time.  Every batch but the last loads each row's registers again as soon as
    // they are used, unconditionally (a branch around a load would make the waits behind it count the
    // worst case, that is, wait for everything)
    const int turns = (row_hi - row_lo + S::kGroups - 1) / S::kGroups;
    auto batch = [&](int j0, int buf, auto more) {
        float acc[N];
#pragma unroll
        for (int k = 0; k < N; ++k) acc[k] = 0.f;
#pragma unroll
        for (int i = 0; i < RB; ++i) {
            if (more || j0 + i < turns) {
                float wf[NV];
                wt[i].values(li, wf);
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    float a = wf[0] * h[b][0];
#pragma unroll
                    for (int k = 1; k < NV; ++k) a = fmaf(wf[k], h[b][k], a);
                    acc[i * NB + b] = a;
                }
            }
            if constexpr (more) wt[i].load(w + (size_t)row_at(j0 + RB + i) * W::kRowBytes, li);
            __builtin_amdgcn_sched_barrier(0);  // one row's values in registers at a time
        }
        int at = 0, n = N;
        half_wave_sums<16, N>(acc, lane, at, n);
#pragma unroll
        for (int k = 0; k < (N + 31) / 32; ++k)
            if (k < n) red[buf][hwave][at + k] = acc[k];
        lds_barrier();  // (two buffers: the next batch's stores meet no reader of this one)
        for (int t = tid; t < S::kGroups * N; t += S::kThreads) {
            const int g = t / N, v = t - g * N, i = v / NB, b = v - i * NB;
            const int row = row_lo + g + (j0 + i) * S::kGroups;
            float sum = 0.f;
#pragma unroll
            for (int k = 0; k < HW; ++k) sum += red[buf][g * HW + k][v];
            if (row < row_hi) out[(size_t)b * out_stride + row] = sum;
        }
    };
    int j0 = 0, buf = 0;
    for (; j0 + RB < turns; j0 += RB, buf ^= 1) batch(j0, buf, std::true_type{});
    batch(j0, buf, std::false_type{});
}

// ------------------------------------------------------------------ one activation row, a wave to two rows
// With a single activation row the sums need no sharing, and at the hidden sizes whose rows take ten waves
// above (160 or 320 lanes: 2560 and 5120) a wave per two output rows with every byte of them in flight is
// the faster layout: four waves to a workgroup, the normed activations read from LDS, no reduction beyond the
// wave.  So it is for F32 at 2048, whose 16 rows a CU are too few to keep rows in flight behind others, and
// for Q4_K at 4096.  Graph-timed in one run, this against the kernel above: F32 11.07 / 11.49 us at E 2560 and
// 24.36 / 25.50 at 5120, F16 6.72 / 6.98 and 14.47 / 15.00, Q8_0 6.51 / 7.88 and 13.23 / 14.98, Q4_K 5.52 /
// 6.16 and 11.28 / 11.47; F32 6.79 / 7.43 at 2048; Q4_K 7.82 / 8.22 at 4096, where Q8_0 takes 9.17 / 9.02.
// Q6_K stays above: staged through LDS like Q8_0 it took 8.09 / 8.13 at 2560 and 18.1 / 15.5 at 5120.
constexpr int kOneWaves = 4, kOneRows = 2;  // waves per workgroup, rows per wave

template <int T, int E>
constexpr bool project_one_row() {
    return (T != 14 && (E == 2560 || E == 5120)) || (T == 0 && E == 2048) || (T == 12 && E == 4096);
}

// RMSNorm of the activation row into hs (src/ops.cpp:155-160), kEl elements per thread; the caller's barrier
// makes it visible.
template <int E, int kEl>
__device__ __forceinline__ void norm_one(const float (&xv)[kEl], const float (&gv)[kEl], float eps, float* hs,
                                         double* ssum) {
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    double ss = 0.0;
#pragma unroll
    for (int i = 0; i < kEl; ++i) ss += (double)xv[i] * (double)xv[i];
    ss = wave_sum_f64(ss);
    if (lane == 0) ssum[wv] = ss;
    __syncthreads();
    ss = 0.0;
#pragma unroll
    for (int k = 0; k < kOneWaves; ++k) ss += ssum[k];
    const float inv = (float)(1.0 / sqrt(ss / (double)E + (double)eps));
#pragma unroll
    for (int i = 0; i < kEl; ++i) {
#pragma clang fp contract(off)
        hs[tid + i * 64 * kOneWaves] = (xv[i] * inv) * gv[i];
    }
}

// F32 and F16: lane l reads 16-byte pieces l, l + 64, ... of both rows.
template <int T, int E>
__global__ __launch_bounds__(64 * kOneWaves) void k_qkv_project_one(const float* __restrict__ x,
                                                                    const float* __restrict__ gamma, float eps,
                                                                    const uint8_t* __restrict__ w, int n_out,
                                                                    float* __restrict__ out) {
    constexpr int kPer = T == 1 ? 8 : 4, P = E / kPer / 64, kEl = E / (64 * kOneWaves);
    __shared__ __align__(16) float hs[E];
    __shared__ double ssum[kOneWaves];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int r0 = (blockIdx.x * kOneWaves + wv) * kOneRows;
    // the activation and gamma elements first, then every weight piece of the wave's rows: loads return in
    // order, so the norm waits for the activations only and overlaps the weight stream
    float xv[kEl], gv[kEl];
#pragma unroll
    for (int i = 0; i < kEl; ++i) gv[i] = gamma[tid + i * 64 * kOneWaves];
#pragma unroll
    for (int i = 0; i < kEl; ++i) xv[i] = x[tid + i * 64 * kOneWaves];
    u32x4_t wr[kOneRows][P];
#pragma unroll
    for (int rr = 0; rr < kOneRows; ++rr) {
        const uint8_t* row = w + (size_t)min(r0 + rr, n_out - 1) * E * (T == 1 ? 2 : 4);
#pragma unroll
        for (int p = 0; p < P; ++p)
            wr[rr][p] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(row) + p * 64 + lane);
    }
    norm_one<E>(xv, gv, eps, hs, ssum);
    __syncthreads();
    float acc[kOneRows] = {};
#pragma unroll
    for (int p = 0; p < P; ++p) {
        const int e0 = (p * 64 + lane) * kPer;
#pragma unroll
        for (int rr = 0; rr < kOneRows; ++rr) {
            float wf[kPer];
            if constexpr (T == 1) {
                f16x8(wr[rr][p], wf);
            } else {
                wf[0] = __uint_as_float(wr[rr][p].x), wf[1] = __uint_as_float(wr[rr][p].y);
                wf[2] = __uint_as_float(wr[rr][p].z), wf[3] = __uint_as_float(wr[rr][p].w);
            }
#pragma unroll
            for (int k = 0; k < kPer; k += 4) {
                const float4 h4 = *reinterpret_cast<const float4*>(hs + e0 + k);
                acc[rr] = fmaf(wf[k], h4.x, acc[rr]);
                acc[rr] = fmaf(wf[k + 1], h4.y, acc[rr]);
                acc[rr] = fmaf(wf[k + 2], h4.z, acc[rr]);
                acc[rr] = fmaf(wf[k + 3], h4.w, acc[rr]);
            }
        }
    }
#pragma unroll
    for (int rr = 0; rr < kOneRows; ++rr) {
        const float s = wave_sum(acc[rr]);
        if (lane == 0 && r0 + rr < n_out) out[r0 + rr] = s;
    }
}

// Q4_K and Q8_0: lanes of even and odd index take the two rows, lane l items l / 2, l / 2 + 32, ....  Q4_K
// items are whole 16-byte pieces and load straight into registers; Q8_0 rows (34-byte blocks) come in as
// coalesced pieces and are parked in a wave-private LDS area first.
template <int T, int E>
__global__ __launch_bounds__(64 * kOneWaves) void k_qkv_project_one_q(const float* __restrict__ x,
                                                                      const float* __restrict__ gamma, float eps,
                                                                      const uint8_t* __restrict__ w, int n_out,
                                                                      float* __restrict__ out) {
    using W = Weights<T, E>;
    constexpr int RB = (int)W::kRowBytes, kEl = E / (64 * kOneWaves), kItems = E / 512;
    constexpr int kPieces = (RB / 16 + 63) / 64;  // staged: 16-byte pieces per lane per row
    constexpr bool kStaged = T == 8;
    static_assert(RB % 16 == 0 && E % 512 == 0, "hidden size");
    __shared__ __align__(16) float hs[E];
    __shared__ __align__(16) uint8_t rows[kStaged ? kOneWaves * kOneRows * RB : 16];
    __shared__ double ssum[kOneWaves];
    const int tid = threadIdx.x, lane = tid & 63, wv = tid >> 6;
    const int r0 = (blockIdx.x * kOneWaves + wv) * kOneRows;
    float xv[kEl], gv[kEl];
#pragma unroll
    for (int i = 0; i < kEl; ++i) gv[i] = gamma[tid + i * 64 * kOneWaves];
#pragma unroll
    for (int i = 0; i < kEl; ++i) xv[i] = x[tid + i * 64 * kOneWaves];
    W it[kStaged ? 1 : kItems];
    u32x4_t pc[kOneRows][kStaged ? kPieces : 1];
    if constexpr (kStaged) {
#pragma unroll
        for (int rr = 0; rr < kOneRows; ++rr) {
            const uint8_t* row = w + (size_t)min(r0 + rr, n_out - 1) * RB;
#pragma unroll
            for (int k = 0; k < kPieces; ++k)  // clamped: the tail lanes reload the last piece
                pc[rr][k] = __builtin_nontemporal_load(reinterpret_cast<const u32x4_t*>(row) +
                                                       min(lane + 64 * k, RB / 16 - 1));
        }
    } else {
        const uint8_t* row = w + (size_t)min(r0 + (lane & 1), n_out - 1) * RB;
#pragma unroll
        for (int j = 0; j < kItems; ++j) it[j].load(row, (lane >> 1) + 32 * j);
    }
    norm_one<E>(xv, gv, eps, hs, ssum);
    uint8_t* my_rows = rows + wv * kOneRows * RB;
    if constexpr (kStaged) {
#pragma unroll
        for (int rr = 0; rr < kOneRows; ++rr)
#pragma unroll
            for (int k = 0; k < kPieces; ++k)
                if (lane + 64 * k < RB / 16) reinterpret_cast<u32x4_t*>(my_rows + rr * RB)[lane + 64 * k] = pc[rr][k];
    }
    __syncthreads();
    float acc = 0.f;
#pragma unroll
    for (int j = 0; j < kItems; ++j) {
        const int k = (lane >> 1) + 32 * j;
        float wf[16];
        if constexpr (kStaged) {
            const uint8_t* blk = my_rows + (lane & 1) * RB + 34 * (k >> 1);
            __builtin_memcpy(&it[0].q, blk + 2 + 16 * (k & 1), 16);  // 2-byte aligned
            it[0].d16 = *reinterpret_cast<const uint16_t*>(blk);
            it[0].values(k, wf);
        } else {
            it[j].values(k, wf);
        }
        // an item's activations are read once the sum before it is known: all items' at once would take the
        // registers of two waves a SIMD (Q4_K, E 5120: 12.4 against 11.1 us)
        int at = 16 * k;
        asm volatile("" : "+v"(at), "+v"(acc));
        const float4* hp = reinterpret_cast<const float4*>(hs + at);
#pragma unroll
        for (int q4 = 0; q4 < 4; ++q4) {
            const float4 hv = hp[q4];
            acc = fmaf(wf[4 * q4], hv.x, acc);
            acc = fmaf(wf[4 * q4 + 1], hv.y, acc);
            acc = fmaf(wf[4 * q4 + 2], hv.z, acc);
            acc = fmaf(wf[4 * q4 + 3], hv.w, acc);
        }
    }
    acc += lane_xor<2>(acc);  // sum over the 32 lanes of this lane's row (xor 2 .. 32 keep the parity)
    acc += lane_xor<4>(acc);
    acc += lane_xor<8>(acc);
    acc += lane_xor<16>(acc);
    acc += lane_xor<32>(acc);
    if (lane < 2 && r0 + lane < n_out) out[r0 + lane] = acc;
}

int qkv_project_max_rows(int E) {
    const int r = E > 0 ? kProjMaxLdsFloats / E : 0;
    return r < kProjMaxRows ? r : kProjMaxRows;
}

// 16-byte pieces per lane per row for the supported hidden sizes (0: not built)
static int qkv_project_pieces(int E, bool w_f16) {
    const int per = 64 * (w_f16 ? 8 : 4);
    if (E <= 0 || E % per) return 0;
    const int p = E / per;
    if (w_f16) return (p == 2 || p == 4 || p == 5 || p == 8 || p == 10 || p == 16 || p == 20) ? p : 0;
    return (p == 4 || p == 8 || p == 10 || p == 16 || p == 20) ? p : 0;
}

bool qkv_project_built(int E, int w_type) {
    if (w_type == 0 || w_type == 1) return qkv_project_pieces(E, w_type == 1) != 0;
    if (w_type != 8 && w_type != 12 && w_type != 14) return false;
    // the dense Qwen3 hidden sizes (whole 256-value super-blocks; a lane's item is 16 values)
    return E == 1024 || E == 2048 || E == 2560 || E == 4096 || E == 5120;
}

template <int T, int NB, int E>
static hipError_t launch_t(hipStream_t st, const float* x, long x_stride, const float* gamma, float eps,
                           const void* w, int n_out, float* out, long out_stride) {
    if constexpr (NB == 1 && project_one_row<T, E>()) {
        constexpr int kPerWg = kOneWaves * kOneRows;
        const dim3 grid((n_out + kPerWg - 1) / kPerWg);
        if constexpr (T <= 1)
            k_qkv_project_one<T, E><<<grid, 64 * kOneWaves, 0, st>>>(x, gamma, eps, static_cast<const uint8_t*>(w),
                                                                     n_out, out);
        else
            k_qkv_project_one_q<T, E><<<grid, 64 * kOneWaves, 0, st>>>(x, gamma, eps, static_cast<const uint8_t*>(w),
                                                                       n_out, out);
        return hipGetLastError();
    } else {
        using S = RowShape<T, E>;
        // one workgroup a CU
        const int rows = (n_out + 255) / 256, turns = (rows + S::kGroups - 1) / S::kGroups;
        // rows in flight: as many as the registers (256 or 168 a lane at 8 or 10 waves) take beside the
        // activations and one row's values, at most 8; fewer where the workgroup's rows then come out in even
        // batches
        constexpr int kRegs = sizeof(Weights<T, E>) / 4;
        constexpr int kBudget = S::kThreads <= 512 ? 160 : 112;
        constexpr int kFit = (kBudget - S::kVals * NB) / (kRegs + NB);
        // (two activation rows of block formats at ten waves: at most 3.  Graph-timed at 6 or 8 / 3, 6144 outputs
        // at E 2560 and 7168 at 5120: Q8_0 9.23 / 7.98 and 16.35 / 13.53 us, Q4_K 7.24 / 7.07 and 15.23 / 11.68;
        // Q6_K at 4 / 3 8.44 / 8.43 and 15.00 / 14.67)
        constexpr int kTop = T > 1 && NB == 2 && S::kThreads > 512 && kFit > 3 ? 3 : kFit;
        constexpr int kMost = kTop >= 8 ? 8 : kTop >= 6 ? 6 : kTop >= 4 ? 4 : kTop >= 3 ? 3 : 2;
        const int batches = (turns + kMost - 1) / kMost, want = (turns + batches - 1) / batches;
        constexpr size_t lds = (size_t)NB * S::kHRow * sizeof(float);
        auto go = [&](auto rb) {
            static std::atomic<bool> opted;
            if (const hipError_t e = opt_in_lds(opted, (const void*)k_qkv_project<T, NB, E, rb>, lds); e != hipSuccess)
                return e;
            k_qkv_project<T, NB, E, rb><<<(n_out + rows - 1) / rows, S::kThreads, lds, st>>>(
                x, x_stride, gamma, eps, static_cast<const uint8_t*>(w), n_out, rows, out, out_stride);
            return hipGetLastError();
        };
        if constexpr (kMost > 2) {
            if (want <= 2) return go(std::integral_constant<int, 2>{});
        }
        if constexpr (kMost > 3 && T > 1) {
            if (want <= 3) return go(std::integral_constant<int, 3>{});
        }
        if constexpr (kMost > 4) {
            if (want <= 4) return go(std::integral_constant<int, 4>{});
        }
        if constexpr (kMost > 6) {
            if (want <= 6) return go(std::integral_constant<int, 6>{});
        }
        return go(std::integral_constant<int, kMost>{});
    }
}

template <int T, int NB>
static hipError_t launch_e(hipStream_t st, const float* x, long x_stride, int E, const float* gamma, float eps,
                           const void* w, int n_out, float* out, long out_stride) {
#define EI_PROJ_E(EE) \
    case EE: return launch_t<T, NB, EE>(st, x, x_stride, gamma, eps, w, n_out, out, out_stride);
    switch (E) {
        EI_PROJ_E(1024) EI_PROJ_E(2048) EI_PROJ_E(2560) EI_PROJ_E(4096) EI_PROJ_E(5120)
        default: break;
    }
    if constexpr (T == 1 && NB * 8192 <= kProjMaxLdsFloats) {
        if (E == 8192) return launch_t<T, NB, 8192>(st, x, x_stride, gamma, eps, w, n_out, out, out_stride);
    }
    if constexpr (T == 1 && NB * 10240 <= kProjMaxLdsFloats) {
        if (E == 10240) return launch_t<T, NB, 10240>(st, x, x_stride, gamma, eps, w, n_out, out, out_stride);
    }
#undef EI_PROJ_E
    return hipErrorInvalidValue;
}

template <int T>
static hipError_t launch_w(hipStream_t st, const float* x, long x_stride, int B, int E, const float* gamma, float eps,
                           const void* w, int n_out, float* out, long out_stride) {
    switch (B) {
        case 1: return launch_e<T, 1>(st, x, x_stride, E, gamma, eps, w, n_out, out, out_stride);
        case 2: return launch_e<T, 2>(st, x, x_stride, E, gamma, eps, w, n_out, out, out_stride);
        case 3: return launch_e<T, 3>(st, x, x_stride, E, gamma, eps, w, n_out, out, out_stride);
        case 4: return launch_e<T, 4>(st, x, x_stride, E, gamma, eps, w, n_out, out, out_stride);
        default: return hipErrorInvalidValue;
    }
}

hipError_t launch_qkv_project(hipStream_t st, const float* x, long x_stride, int B, int E, const float* gamma,
                              float eps, const void* w, int w_type, int n_out, float* out, long out_stride) {
    switch (w_type) {
        case 0: return launch_w<0>(st, x, x_stride, B, E, gamma, eps, w, n_out, out, out_stride);
        case 1: return launch_w<1>(st, x, x_stride, B, E, gamma, eps, w, n_out, out, out_stride);
        case 8: return launch_w<8>(st, x, x_stride, B, E, gamma, eps, w, n_out, out, out_stride);
        case 12: return launch_w<12>(st, x, x_stride, B, E, gamma, eps, w, n_out, out, out_stride);
        case 14: return launch_w<14>(st, x, x_stride, B, E, gamma, eps, w, n_out, out, out_stride);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace ei
