// prefill.hip — causal GQA prefill attention on gfx950 bf16 matrix cores, fp32 operands in three planes.
//
// Both products run on v_mfma_f32_32x32x16_bf16 (fp32 accumulate; 16x the rate of the fp32
// 32x32x2 instruction) with every fp32 operand split into three bf16 planes that together hold
// all of its bits, x = h + m + l (values out of the planes' range are multiplied in fp32: see the
// split and the check after the key loop).  Six of the nine plane products are taken.  Of the three
// left out m.l and l.m are at most 2^-25 of |a||b| each and l.l 2^-34: together 2^-24 at worst, an
// fp32 rounding, and 2^-27.5 in the root mean square over all mantissas.  An instruction sums 16
// products before it rounds, so a 128-deep score takes 48 roundings, most of them of small
// terms, against 64 on the fp32 instruction.  Measured error of the output against 64 bits
// (2-norm): 3.3e-7 against 4.0e-7 with fp32 MFMA (2048-token prompt, H32/HKV8), 4.4e-7 against
// 5.2e-7 (8192 tokens), 6.1e-7 against 7.1e-7 (512 tokens at 7680, H16/HKV8); lower in every
// shape tried.  Online softmax in fp32 VALU between the two products.
//
// Each wave owns 32 queries of one head.  It computes the transposed score tile
//     S^T[key][query] = K . Q^T          (A = K planes from LDS, B = Q^T planes in registers)
// so that in the 32x32 accumulator layout every lane owns ONE query column and 16 key
// rows: the row max / row sum of the softmax need only the lane's own 16 values plus one
// exchange with lane^32.  The same registers, split into planes, are the B operand of
//     O^T[d][query] = V^T . P^T          (A = transposed V planes from LDS)
// because the accumulator row order (8*(r/4) + 4*(lane/32) + r%4) is used as the
// contraction order of the second product: step s of lane half hh takes registers 8s .. 8s+7,
// keys 16s + 4hh + {0..3, 8..11}, and the V planes are stored with those eight keys side by
// side.  Output block db (0..3) of O^T holds d = 32*db + i for accumulator row i.
//
// Workgroup = KS key groups x 4 query slots of one KV head.  A slot is one (query block,
// head) pair; slots are numbered s = qb*G + g over the G heads that share the KV head, and
// unit U of a KV head holds slots 4U..4U+3.  For G = 4 a unit is the four heads of one
// block, for G = 8 half of them, for G = 2 two heads of two neighbouring blocks, for G = 1
// four neighbouring blocks of the head, for odd G at most two neighbouring blocks: every
// wave of the unit shares every K/V tile, and the unit's key range ends at its last
// block's diagonal (a wave of an earlier block masks the few tiles past its own).  Slots
// past the last block repeat a valid row and write nothing.  Key group g takes the
// tiles kt = KS*i + g of the unit's causal range and keeps its own (m, l, O); the groups
// merge through LDS at the end of the unit.  When one unit pair per KV head would not
// fill the CUs (short chunks at long positions, GQA groups under 4 heads;
// ei_attn_prefill_split) the pair's key tiles are split over ksplit workgroups of equal cost
// (a share that crosses from one unit to the other pays a second pass), whose unnormalised
// shares k_prefill_combine merges.
//
// The key loop.  A tile (32 keys) is loaded by the four waves of its group, a quarter each, 16
// floats of K or V per lane, split in registers and stored as planes (K [key][d], V transposed
// [d][key]; rows padded to an odd number of 16-byte pieces).  Per half iteration a group either
// multiplies K by Q, while V of the same tile goes to its planes and K of the next is fetched, or
// runs the softmax and multiplies V by P, while the next K goes to its planes and the next V is
// fetched: one set of planes per group and one set of 16 landing registers suffice, and a fetch
// has half a phase and more to land.  The two groups run half an iteration apart, so of a SIMD's
// two waves one has matrix work while the other is in its softmax (1-3% faster than in step; the
// raised wave priority of the softmax half, whose chain is the longer one, another 3%).  Each
// matrix step refills its three LDS operands right after their last use (mfma_split).
//
// What bounds it: the matrix power of the part.  At 8192 tokens (H32/HKV8) the kernel runs 219
// TFLOP/s of attention = 1.31 PFLOP/s of bf16 MFMA at 1.65 GHz (the clock gives way under bf16
// load: a bare register-to-register MFMA loop on random bits reaches 1.53-1.63 PFLOP/s at
// 1.6-1.66 GHz), against 139 TFLOP/s on fp32 MFMA; 2048 tokens 285 -> 187 us a step, 512 tokens
// at 7680 (H16/HKV8) 268 -> 163 us.  The checks of the planes' range are 0-2% of that.  With parts taken out (timing only, before those checks): without the K/V
// split and its loads 2.14 ms of 2.53, without the loads alone 2.38, without operand reads as well as
// the split 2.04, without the exponentials too 1.98.
//
// q and the output pass through LDS too, so that global memory sees whole 512-byte rows:
// at the start of each unit the workgroup DMAs its 128 query rows (once, for both key
// groups) into a padded staging area and each wave reads its Q^T operand from there; at the
// end the finished rows are written there in row order and stored two rows per instruction.
//
// Softmax runs in the exp2 domain (scores x scale x log2 e, one FMA per score).  The
// running maximum is raised only when a tile's maximum exceeds it by more than kLazy
// (log2 units), so P <= 2^kLazy and O / l are rescaled rarely; the result is the same
// softmax (the common factor cancels in O / l).  The causal mask is applied only on the
// (at most two) tiles that cross the block's diagonal.
//
// Causal balance: unit U needs about (4U+4)/G + pos0/32 tiles, so a workgroup runs unit p
// and then unit nu-1-p; every workgroup has the same amount of work.  Workgroup id
// L -> kv head L % HKV first, so with 8 KV heads all blocks of one KV head share an
// XCD (and its L2) under the round-robin XCD dispatch.
#include <cstdlib>

#include "common.h"
#include "launch.h"

namespace ei {

typedef float floatx16 __attribute__((ext_vector_type(16)));

constexpr int kQB = 32;                          // queries per wave (and per block)
constexpr int kKT = 32;                          // keys per tile
constexpr int kKS_F = kHeadDim + 4;             // padded fp32 row of the staging area (floats)
// plane rows are padded to an odd number of 16-byte pieces: the lanes of an operand read, one row
// each, spread over all LDS banks
constexpr int kKRowB = 2 * kHeadDim + 16, kKPlane = kKT * kKRowB;  // K plane: [32 keys][128 d] bf16
constexpr int kVRowB = 2 * kKT + 16, kVPlane = kHeadDim * kVRowB;   // V plane, transposed: [128 d][32 keys] bf16
constexpr int kKS = 2;                           // key groups per workgroup
constexpr float kLazy = 8.f;                     // lazy-rescale threshold (log2 units)
constexpr int kXchF = 34;                        // floats per lane exchanged by the merge
constexpr int kSlots = 4;                        // query slots (waves) per key group
constexpr int kPassTiles = 5;                    // a pass's fixed cost, in tiles (key-share balance)

// n / d for small d (1..8) and n * d < 2^32 as one multiply-high: the per-pass index math
// runs on the scalar unit, which the eight waves of a CU share, so a division loop per use
// would cost thousands of cycles per pass.  m = ceil(2^32 / d); d = 1 is taken as is.
struct FastDiv {
    uint32_t m, d;
};
__device__ __forceinline__ FastDiv fast_div(uint32_t d) { return {d == 1 ? 0u : 0xFFFFFFFFu / d + 1u, d}; }
__device__ __forceinline__ int fdiv(int n, FastDiv f) {
    return f.d == 1 ? n : (int)__umulhi((uint32_t)n, f.m);
}
// Key shares.  A workgroup runs units `pair` and nu-1-pair (causal balance).  With ksplit
// shares, the pair's tiles, unit pair's then unit nu-1-pair's, are cut into ksplit contiguous
// shares of equal cost, where the boundary between the units counts as kPassTiles extra tiles:
// a share that crosses it runs two passes (q staging, first tiles, key-group merge and store
// twice), so it gets that many fewer tiles, and every other share runs one pass (3 to 8 tried, 512
// tokens at 0 / 1536, G = 4: 47.2 / 96.0 us at 3, 45.8 / 94.0 at 4 and 5, 47.5 / 93.9 at 6, 49.3 / 95.0 at 8).  Share
// `split` holds tiles [lo0, lo0 + r0) of unit pair and [lo1, lo1 + r1) of unit nu-1-pair; a
// unit without tiles in a share has no pass there and no partial, and k_prefill_combine,
// which evaluates the same cut, does not read one.  With ksplit = 1 the share is both units.
__device__ __forceinline__ int prefill_unit_tiles(int u, int pos0, int B, int nslot, FastDiv fG) {
    const int ql = fdiv(min(kSlots * u + kSlots - 1, nslot - 1), fG);  // the unit's last block
    return (pos0 + min(B, ql * kQB + kQB) + kKT - 1) / kKT;
}
__device__ __forceinline__ void prefill_share(int pair, int u_second, int split, FastDiv fK, int pos0, int B,
                                              int nslot, FastDiv fG, int& lo0, int& r0, int& lo1, int& r1) {
    const int n0 = prefill_unit_tiles(pair, pos0, B, nslot, fG);
    const int n1 = u_second != pair ? prefill_unit_tiles(u_second, pos0, B, nslot, fG) : 0;
    const int pen = n1 > 0 ? kPassTiles : 0;
    const int n_all = n0 + n1 + pen;
    auto real_tile = [&](int x) { return x <= n0 ? x : (x <= n0 + pen ? n0 : x - pen); };
    const int lo = real_tile(fdiv(split * n_all, fK)), hi = real_tile(fdiv((split + 1) * n_all, fK));
    lo0 = lo;
    r0 = max(min(hi, n0) - lo, 0);
    lo1 = max(lo, n0) - n0;
    r1 = max(hi - max(lo, n0), 0);
}

// LDS: both key groups' K planes from 0, and the merge exchange area from 0 as well (used only
// after the unit's last tile); after it both groups' V planes and, overlapping them, the staging
// area (the unit's 4 x 32 query rows, later its output rows, in fp32, padded).  K planes are stored
// while the query rows are staged, V planes once every wave has its query operand.
constexpr int kQStageF = 2 * kSlots * kXchF * 64;
constexpr int kLdsF = kQStageF + kSlots * kQB * kKS_F;
static_assert(kKS * 3 * kKPlane <= kQStageF * 4, "K planes below the staging area");
static_assert(kQStageF * 4 + kKS * 3 * kVPlane <= kLdsF * 4, "V planes within the LDS span");

// A value the optimiser may not carry across loop iterations: what is derived from it is computed
// where it is used (the vector registers of the key loop are full, hoisted addresses would spill).
__device__ __forceinline__ int unhoisted(int x) {
    asm volatile("" : "+v"(x));
    return x;
}
__device__ __forceinline__ float here(float x) {  // the same of a kernel argument
    asm volatile("" : "+s"(x));
    return x;
}
__device__ __forceinline__ float uniform(float x) {  // a wave-uniform value, in a scalar register
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}

// QK-norm + RoPE of two q rows in LDS (rope_dim = 128), eight lanes per row: lane k of a row
// holds elements 8k..8k+7 and their rotate-half partners 64+8k..64+8k+7.  Same arithmetic as the
// prologue's head-norm, which follows the reference CPU path (rmsnorm, src/ops.cpp:155-160; rope,
// src/model.cpp:23-32): sum of squares in double, inv = float(1/sqrt(ss/128 + eps)),
// y = (x*inv)*gamma, then (y_e, y_e+64) -> (y_e c - y_e+64 s, y_e s + y_e+64 c).  The double sum runs over the eight
// lanes' partial sums (a different order of exact products than the prologue's lane pairs; the
// float result is the same unless the double rounds across a float boundary).  Both rows are read
// before either is written, so their two chains of double arithmetic run side by side (one after
// the other they held each pass up by 0.6 us: a 2048-token step 187.0 against 185.8 us, a 512-token
// chunk at 1536 97.9 against 97.4).
__device__ __forceinline__ void norm_rope_q8(float* row0, float* row1, const float (&g)[16], const float4 (&t)[2][4],
                                             float eps, int k) {
#pragma clang fp contract(off)
    float* rows[2] = {row0, row1};
    float x[2][16], inv[2];
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const float4 a = *reinterpret_cast<const float4*>(rows[h] + 8 * k + 4 * i);
            const float4 b = *reinterpret_cast<const float4*>(rows[h] + 64 + 8 * k + 4 * i);
            x[h][4 * i] = a.x, x[h][4 * i + 1] = a.y, x[h][4 * i + 2] = a.z, x[h][4 * i + 3] = a.w;
            x[h][8 + 4 * i] = b.x, x[h][8 + 4 * i + 1] = b.y, x[h][8 + 4 * i + 2] = b.z, x[h][8 + 4 * i + 3] = b.w;
        }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        // float x float is exact in double, so fma(x, x, ss) rounds like ss + x*x
        double ss = 0.0;
#pragma unroll
        for (int i = 0; i < 16; ++i) ss = __builtin_fma((double)x[h][i], (double)x[h][i], ss);
        ss += lane_xor_f64<1>(ss);
        ss += lane_xor_f64<2>(ss);
        ss += lane_xor_f64<4>(ss);
        inv[h] = (float)(1.0 / sqrt(ss / (double)kHeadDim + (double)here(eps)));
    }
#pragma unroll
    for (int h = 0; h < 2; ++h) {
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const float c = (i & 1) ? t[h][i >> 1].z : t[h][i >> 1].x, sn = (i & 1) ? t[h][i >> 1].w : t[h][i >> 1].y;
            const float a = (x[h][i] * inv[h]) * g[i];
            const float b = (x[h][8 + i] * inv[h]) * g[8 + i];
            const float acs = a * c, bsn = b * sn;
            const float asn = a * sn, bcs = b * c;
            x[h][i] = acs - bsn;
            x[h][8 + i] = asn + bcs;
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            *reinterpret_cast<float4*>(rows[h] + 8 * k + 4 * i) =
                make_float4(x[h][4 * i], x[h][4 * i + 1], x[h][4 * i + 2], x[h][4 * i + 3]);
            *reinterpret_cast<float4*>(rows[h] + 64 + 8 * k + 4 * i) =
                make_float4(x[h][8 + 4 * i], x[h][8 + 4 * i + 1], x[h][8 + 4 * i + 2], x[h][8 + 4 * i + 3]);
        }
    }
}

// ------------------------------------------------------------------ three-plane split
// x = h + m + l with h, m, l in bf16: h = bf16(x), m = bf16(x - h), l = x - h - m, each rounded to
// nearest.  Both differences are exact (the residual of a 24-bit value rounded to 8 bits has at
// most 16 significant bits, the second at most 8), so the three planes hold every bit of x as long
// as none of them leaves bf16's range: from kPlaneMin up, where x's last bit is a normal bf16, to
// bf16's largest value.  What lies outside is noticed and multiplied in fp32.
typedef float f32x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
constexpr int kBufferDword3 = 0x00020000;  // raw 32-bit data, gfx9-family buffer resource word 3

__device__ __forceinline__ uint32_t pk_bf16(float a, float b) {
    return __builtin_bit_cast(uint32_t, __builtin_convertvector(f32x2{a, b}, bf16x2));
}
__device__ __forceinline__ void split_pair(float a, float b, uint32_t& h, uint32_t& m, uint32_t& l) {
#pragma clang fp contract(off)
    h = pk_bf16(a, b);
    const float ra = a - __uint_as_float(h << 16), rb = b - __uint_as_float(h & 0xFFFF0000u);
    m = pk_bf16(ra, rb);
    l = pk_bf16(ra - __uint_as_float(m << 16), rb - __uint_as_float(m & 0xFFFF0000u));
}
constexpr float kPlaneMin = 0x1p-100f;
// The planes of a small value are off by up to 2^-134, which counts for something only against a large
// partner.  From this value on an operand is taken to be one, so below it the smallest partner does
// not matter.
constexpr float kPlaneMax = 0x1p24f;
constexpr float kSmallSum = 0x1p-60f;
// |x| in the order of nonzero values, zero last
__device__ __forceinline__ uint32_t magnitude(uint32_t x) { return (x << 1) - 1u; }
__device__ __forceinline__ float of_magnitude(uint32_t m) {  // its |x|; infinite for zero
    return m == 0xFFFFFFFFu ? INFINITY : __uint_as_float((m >> 1) + 1u);
}
constexpr uint32_t kTinyMagnitude = (__builtin_bit_cast(uint32_t, kPlaneMin) << 1) - 1u;
struct Planes {  // eight values: one MFMA operand per plane
    u32x4 h, m, l;
};
__device__ __forceinline__ floatx16 mfma_bf16(u32x4 a, u32x4 b, floatx16 c) {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0,
                                                   0, 0);
}
// c += a . b without m.l, l.m and l.l (together at most 2^-24 of |a||b|).  a's planes are used up one
// after another, and next(x) refills plane x (2 l, 1 m, 0 h) with the next step's right after its last
// use: at least three matrix instructions cover each LDS read, in the registers of one step.
template <typename Next>
__device__ __forceinline__ void mfma_split(Planes& a, const Planes& b, floatx16& c, Next next) {
    constexpr int kAlu = 0x6;  // VALU and SALU work may move across, LDS reads and MFMAs stay in order
    c = mfma_bf16(a.l, b.h, c);
    __builtin_amdgcn_sched_barrier(kAlu);
    a.l = next(2);
    __builtin_amdgcn_sched_barrier(kAlu);
    c = mfma_bf16(a.m, b.m, c);
    c = mfma_bf16(a.m, b.h, c);
    __builtin_amdgcn_sched_barrier(kAlu);
    a.m = next(1);
    __builtin_amdgcn_sched_barrier(kAlu);
    c = mfma_bf16(a.h, b.l, c);
    c = mfma_bf16(a.h, b.m, c);
    c = mfma_bf16(a.h, b.h, c);
    __builtin_amdgcn_sched_barrier(kAlu);
    a.h = next(0);
    __builtin_amdgcn_sched_barrier(kAlu);
}

// kPaged: key t of the sequence sits in pool row btab[t >> bshift] << bshift | (t & mask), the
// block size 2^bshift >= 32, so a 32-key tile lies in one block and its rows are consecutive.
template <bool kNormQ, bool kPaged>
__global__ __launch_bounds__(64 * kSlots * kKS) void k_prefill(const float* __restrict__ q, long q_stride,
                                                           float* __restrict__ out, const float* __restrict__ kc,
                                                           const float* __restrict__ vc,
                                                           const int* __restrict__ pos_dev, int B, int H, int HKV,
                                                           float scale, int ksplit,
                                                           float* __restrict__ part_o, float* __restrict__ part_ml,
                                                           const float* __restrict__ q_gamma,
                                                           const float2* __restrict__ cs, float eps,
                                                           const int* __restrict__ btab, int bshift,
                                                           int max_blocks) {
    constexpr int D = kHeadDim;
    constexpr int GW = kSlots;
    extern __shared__ __align__(16) float smem[];

    const int L = blockIdx.x;
    const int kvh = L % HKV;
    const int rest = L / HKV;
    const int split = rest % ksplit;  // which contiguous share of each unit's key tiles
    const int pair = rest / ksplit;
    const int G = H / HKV;
    const FastDiv fG = fast_div((uint32_t)G), fK = fast_div((uint32_t)ksplit);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int wu = __builtin_amdgcn_readfirstlane(w);  // wave-uniform: keeps the branches scalar
    const int hw = wu % GW, grp = wu / GW;
    const int col = lane & 31, hh = lane >> 5;
    const int pos0 = *pos_dev;
    const size_t KD = (size_t)HKV * D;
    const float* kbase = kc + (size_t)kvh * D;
    const float* vbase = vc + (size_t)kvh * D;
    const uint32_t row_bytes = (uint32_t)(KD * sizeof(float));          // one cache row (all KV heads)
    // cache row of key t (wave-uniform t: one scalar load of the block table when paged)
    auto crow = [&](int t) -> uint32_t {
        // (a key past the table's blocks, outside the contract, reads the last entry: no fault)
        if constexpr (kPaged)
            return ((uint32_t)btab[min(t >> bshift, max_blocks - 1)] << bshift) | ((uint32_t)t & ((1u << bshift) - 1u));
        else return (uint32_t)t;
    };
    const int nb = (B + kQB - 1) / kQB;
    const int nslot = G * nb;                    // (block, head) slots of this KV head
    const int nu = (nslot + kSlots - 1) / kSlots;  // units
    char* const lds = reinterpret_cast<char*>(smem);
    char* const kpl = lds + grp * 3 * kKPlane;                 // this key group's K planes
    char* const vpl = lds + kQStageF * 4 + grp * 3 * kVPlane;  // and its V planes
    const float sl2 = scale * 1.44269504088896340736f;
    const uint32_t voff_k = (uint32_t)(8 * hw + (lane >> 3)) * row_bytes + 32u * (lane & 7);
    const uint32_t voff_v =
        (uint32_t)(16 * (lane >> 5) + 4 * ((lane >> 4) & 1)) * row_bytes + 4u * (32 * hw + 2 * (lane & 15));

    // q of unit u reaches LDS by LDS DMA, once per workgroup: row r = 32*slot + j holds query
    // qb*32 + j of the slot's head (one contiguous 512-byte DMA per row; rows past B and idle
    // slots are clamped to valid rows, never written out).  Both key groups then read their
    // Q^T operand from it and split it into planes: step t holds d = 16t + 8hh .. + 7 of query
    // qb*32 + col.
    float* qst = smem + kQStageF;
    const uint32_t voff_q = 16u * col;
    // wave wu stages rows 16*wu .. 16*wu+15 of unit u: half of slot wu/2, query rows r0 + min(j, jm)
    auto stage_rows = [&](int u, int& r0, int& jm, int& hq) {
        const int sl = kSlots * u + (wu >> 1);
        const int qsl = fdiv(sl, fG);
        const int qbs = sl < nslot ? qsl : nb - 1;
        r0 = min(qbs * kQB + (kQB / 2) * (wu & 1), B - 1);
        jm = B - 1 - r0;  // rows past B repeat the last row
        hq = kvh * G + sl - qsl * G;
    };
    auto stage_q = [&](int u) {
        // (scalar work is shared by the CU's eight waves, so the per-row address step is one add)
        int r0, jm, hq;
        stage_rows(u, r0, jm, hq);
        uint64_t sb = (uint64_t)(uintptr_t)(q + (size_t)r0 * q_stride + (size_t)hq * D);
        const uint32_t rs = (uint32_t)(q_stride * sizeof(float));
        const uint32_t lb = __builtin_amdgcn_readfirstlane(lds_addr(qst + (kQB / 2) * wu * kKS_F));
        if (hh == 0) {
#pragma unroll
            for (int j = 0; j < kQB / 2; ++j) {
                dma16_s(sb, voff_q, lb + j * (kKS_F * 4));
                if (j < jm) sb += rs;
            }
        }
    };
    Planes qp[8];
    // A score on planes is off by at most 2^-134 (|q| + |k|) per element, times the softmax scale: 2^-47
    // with K below kPlaneMax, q below 2^50 and the scale below 2^30, a larger scale taken off q's limit.
    // A wave with a q element past it takes its tiles in fp32 after the key loop.
    const float q_scale = uniform(__builtin_fabsf(sl2) < 0x1p30f ? fmaxf(1.f, __builtin_fabsf(sl2)) : INFINITY);
    uint64_t q_fp32 = 0;
    // raw q rows (kNormQ): QK-norm + RoPE in place, each wave on the 16 rows it staged, 8 lanes
    // per row, two rounds of 8 rows; gamma and both rounds' RoPE rows are loaded (load_norm)
    // while the q rows are still in flight, and used once they have landed (read_q)
    float qg[kNormQ ? 16 : 1];
    float4 qt[kNormQ ? 2 : 1][4];
    auto load_norm = [&](int u) {
        if constexpr (kNormQ) {
            int r0, jm, hq;
            stage_rows(u, r0, jm, hq);
            const int ln = unhoisted(lane), k = ln & 7, j = ln >> 3;
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                const float4 ga = *reinterpret_cast<const float4*>(q_gamma + 8 * k + 4 * i);
                const float4 gb = *reinterpret_cast<const float4*>(q_gamma + 64 + 8 * k + 4 * i);
                qg[4 * i] = ga.x, qg[4 * i + 1] = ga.y, qg[4 * i + 2] = ga.z, qg[4 * i + 3] = ga.w;
                qg[8 + 4 * i] = gb.x, qg[8 + 4 * i + 1] = gb.y, qg[8 + 4 * i + 2] = gb.z, qg[8 + 4 * i + 3] = gb.w;
            }
            const int p0 = *pos_dev + r0;
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const float2* row = cs + (size_t)(p0 + min(8 * h + j, jm)) * (kHeadDim / 2);
                const float4* tr = reinterpret_cast<const float4*>(row + 8 * k);
#pragma unroll
                for (int i = 0; i < 4; ++i) qt[h][i] = tr[i];
            }
        }
    };
    // q rows (and the norm's operands) have landed in this wave: the caller has waited
    auto read_q = [&]() {
        if constexpr (kNormQ) {
            const int k = lane & 7, j = lane >> 3;
            float* row = qst + ((kQB / 2) * wu + j) * kKS_F;
            norm_rope_q8(row, row + 8 * kKS_F, qg, qt, eps, k);
        }
        lds_barrier();
        const float* qs = qst + (hw * kQB + col) * kKS_F + 8 * hh;
        float most = 0.f;
        if constexpr (kNormQ) {  // a normed and rotated element is at most sqrt(2 * 128) gammas
#pragma unroll
            for (int i = 0; i < 16; ++i) most = fmaxf(most, 16.f * __builtin_fabsf(qg[i]));
        }
#pragma unroll
        for (int t = 0; t < 8; ++t) {
            const float4 x = *reinterpret_cast<const float4*>(qs + 16 * t);
            const float4 y = *reinterpret_cast<const float4*>(qs + 16 * t + 4);
#pragma unroll
            for (const float f : {x.x, x.y, x.z, x.w, y.x, y.y, y.z, y.w})
                if constexpr (!kNormQ) most = fmaxf(most, __builtin_fabsf(f));
            uint32_t h[4], m[4], l[4];
            split_pair(x.x, x.y, h[0], m[0], l[0]);
            split_pair(x.z, x.w, h[1], m[1], l[1]);
            split_pair(y.x, y.y, h[2], m[2], l[2]);
            split_pair(y.z, y.w, h[3], m[3], l[3]);
            qp[t] = {u32x4{h[0], h[1], h[2], h[3]}, u32x4{m[0], m[1], m[2], m[3]}, u32x4{l[0], l[1], l[2], l[3]}};
        }
        q_fp32 = __builtin_amdgcn_ballot_w64(!(most * q_scale < 0x1p50f));
    };
    const int u_second = nu - 1 - pair;  // the pass-1 unit (none when it equals pair)
    // this workgroup's share of the pair (prefill_share); wave-uniform: readfirstlane keeps the
    // values in scalar registers, the vector budget is full
    int lo0, r0, lo1, r1;
    prefill_share(pair, u_second, split, fK, pos0, B, nslot, fG, lo0, r0, lo1, r1);
    lo0 = __builtin_amdgcn_readfirstlane(lo0);
    r0 = __builtin_amdgcn_readfirstlane(r0);
    lo1 = __builtin_amdgcn_readfirstlane(lo1);
    r1 = __builtin_amdgcn_readfirstlane(r1);
    const int npass = (r0 > 0) + (r1 > 0);

    for (int pass = 0; pass < npass; ++pass) {
        const bool first_unit = pass == 0 && r0 > 0;  // this pass runs unit `pair`
        const int u = first_unit ? pair : u_second;
        const int sl = kSlots * u + hw;            // this wave's slot (wave-uniform)
        const bool live = sl < nslot;
        const int qb = fdiv(sl, fG), h = kvh * G + sl - qb * G;
        const int qb_last = fdiv(min(kSlots * u + kSlots - 1, nslot - 1), fG);  // the unit's last block
        const int b = qb * kQB + col;  // this lane's query row
        const int qpos = pos0 + b;

        const int T = pos0 + min(B, qb_last * kQB + kQB);  // keys seen by the unit's last query
        const int ntile = (T + kKT - 1) / kKT;
        const int nfull = live ? (pos0 + qb * kQB + 1) / kKT : ntile;  // tiles below this wave's diagonal
        const int kt_lo = first_unit ? lo0 : lo1;  // this workgroup's tiles of the unit: [kt_lo, kt_lo + nrange)
        const int nrange = first_unit ? r0 : r1;
        const int n_it = (nrange + kKS - 1) / kKS;
        const int n_mine = (nrange - grp + kKS - 1) / kKS;  // tiles of this key group

        // K and V of this group's i-th tile (kt = KS*i + grp): wave hw takes a quarter of each,
        // 16 floats per lane, into rg, and stores them as planes.  Rows past T read as zeros (masked out).
        //   K: row 8*hw + lane/8, d = 8c .. 8c+7 and 64 + 8c .. (c = lane%8): two 16-byte pieces
        //     of a row per plane
        //   V: d = 32*hw + 2*(lane%16) and the next, the eight keys of chunk lane/16 (step s =
        //     chunk/2, half hh = chunk%2 of the P.V operand: keys 16s + 4hh + {0..3, 8..11}): one
        //     16-byte piece of two transposed rows per plane
        float rg[16];
        // the tile's visible rows as a buffer: reads past the last one give zeros (masked out)
        auto tile_rsrc = [&](const float* cache, int t0) {
            return __builtin_amdgcn_make_buffer_rsrc(
                const_cast<float*>(cache) + (size_t)crow(t0) * KD, 0,
                (int)((uint32_t)(min(kKT, T - t0) - 1) * row_bytes + D * 4), kBufferDword3);
        };
        auto load_k = [&](int i) {
            const __amdgpu_buffer_rsrc_t rs = tile_rsrc(kbase, (kt_lo + kKS * i + grp) * kKT);
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, voff_k + 256 * (j >> 1) + 16 * (j & 1), 0, 0);
                rg[4 * j] = __uint_as_float(v.x), rg[4 * j + 1] = __uint_as_float(v.y);
                rg[4 * j + 2] = __uint_as_float(v.z), rg[4 * j + 3] = __uint_as_float(v.w);
            }
        };
        auto load_v = [&](int i) {
            const __amdgpu_buffer_rsrc_t rs = tile_rsrc(vbase, (kt_lo + kKS * i + grp) * kKT);
            const uint32_t off = unhoisted(voff_v);
#pragma unroll
            for (int j = 0; j < 8; ++j) {
                const u32x2 v =
                    __builtin_amdgcn_raw_buffer_load_b64(rs, off + (8 * (j >> 2) + (j & 3)) * row_bytes, 0, 0);
                rg[2 * j] = __uint_as_float(v.x), rg[2 * j + 1] = __uint_as_float(v.y);
            }
        };
        // a value of rg past kPlaneMax turns one of them into NaN, which reaches a sum of every wave that
        // multiplies it (ten operations; a branch would spill)
        auto check_planes = [&]() {
            float most = 0.f;
#pragma unroll
            for (int j = 0; j < 16; ++j) most = fmaxf(most, __builtin_fabsf(rg[j]));
            rg[0] = most < kPlaneMax ? rg[0] : __uint_as_float(0xFFFFFFFFu);  // (a NaN that is an inline constant)
        };
        // half x of the conversion of rg: eight values, one 16-byte piece of each plane
        auto conv_k = [&](int x) {
            uint32_t ch[4], cm[4], cl[4];
            if (x == 0) check_planes();
#pragma unroll
            for (int j = 0; j < 4; ++j) split_pair(rg[8 * x + 2 * j], rg[8 * x + 2 * j + 1], ch[j], cm[j], cl[j]);
            char* p = kpl + (8 * hw + (lane >> 3)) * kKRowB + 16 * (lane & 7) + 128 * x;
            *reinterpret_cast<u32x4*>(p) = u32x4{ch[0], ch[1], ch[2], ch[3]};
            *reinterpret_cast<u32x4*>(p + kKPlane) = u32x4{cm[0], cm[1], cm[2], cm[3]};
            *reinterpret_cast<u32x4*>(p + 2 * kKPlane) = u32x4{cl[0], cl[1], cl[2], cl[3]};
        };
        auto conv_v = [&](int x) {  // d + x
            uint32_t ch[4], cm[4], cl[4];
            if (x == 0) check_planes();
#pragma unroll
            for (int j = 0; j < 4; ++j) split_pair(rg[4 * j + x], rg[4 * j + 2 + x], ch[j], cm[j], cl[j]);
            char* p = vpl + (32 * hw + 2 * (lane & 15) + x) * kVRowB + 16 * (lane >> 4);
            *reinterpret_cast<u32x4*>(p) = u32x4{ch[0], ch[1], ch[2], ch[3]};
            *reinterpret_cast<u32x4*>(p + kVPlane) = u32x4{cm[0], cm[1], cm[2], cm[3]};
            *reinterpret_cast<u32x4*>(p + 2 * kVPlane) = u32x4{cl[0], cl[1], cl[2], cl[3]};
        };
        auto k_frag = [&](int t, int plane) {  // K[key col][16t + 8hh ..]
            return *reinterpret_cast<const u32x4*>(kpl + col * kKRowB + 16 * hh + 32 * t + plane * kKPlane);
        };
        auto v_frag = [&](int x, int plane) {  // step s = x/4, d = 32 (x%4) + col
            return *reinterpret_cast<const u32x4*>(vpl + (32 * (x & 3) + col) * kVRowB + 32 * (x >> 2) + 16 * hh +
                                                   plane * kVPlane);
        };

        if (pass > 0) lds_barrier();  // every wave has stored its rows from the staging area
        stage_q(u);
        load_norm(u);
        if (n_mine > 0) load_k(0);
        wait_vmcnt<0>();
        read_q();
        if (n_mine > 0) {
#pragma unroll
            for (int x = 0; x < 2; ++x) conv_k(x);
            load_v(0);
        }
        floatx16 o[4];
        float m, lsum;
        auto clear = [&]() {
#pragma unroll
            for (int db = 0; db < 4; ++db)
#pragma unroll
                for (int i = 0; i < 16; ++i) o[db][i] = 0.f;
            m = -INFINITY;
            lsum = 0.f;
        };
        // scores s of tile kt -> P (in place), the running maximum and sum, O rescaled if it rose
        auto softmax = [&](int kt, floatx16& s) {
            if (kt >= nfull) {  // tile crosses the diagonal (wave-uniform)
                const int k0 = unhoisted(kt * kKT + 4 * hh);
#pragma unroll
                for (int r = 0; r < 16; ++r)
                    if (k0 + 8 * (r >> 2) + (r & 3) > qpos) s[r] = -INFINITY;
            }
            float mx = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mx = fmaxf(mx, s[r]);
            const float ms = half_max(mx) * sl2;
            if (__builtin_amdgcn_ballot_w64(ms > m + kLazy)) {  // rare after the first tile
                const float mn = fmaxf(m, ms);
                const float corr = m == mn ? 1.f : __builtin_amdgcn_exp2f(m - mn);
                lsum *= corr;
#pragma unroll
                for (int db = 0; db < 4; ++db)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[db][r] *= corr;
                m = mn;
            }
            const float nb_ = m == -INFINITY ? 0.f : -m;
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                s[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], sl2, nb_));
                lsum += s[r];
            }
        };
        // The same two products in fp32 from the cache, for a wave that planes do not serve: see after the
        // key loop.  q comes from its row again, normed as in norm_rope_q8 if it is raw (each lane holds the
        // pairs (d, d + 64) of half its query's elements); values 16t + 8hh .. + 7 take the registers of
        // planes h and m.
        auto q_whole = [&]() {
            const int ln = unhoisted(lane), e0 = 8 * (ln >> 5);
            const int bq = min(qb * kQB + (ln & 31), B - 1);
            const float* row = q + (size_t)bq * q_stride + (size_t)h * D + e0;
#pragma unroll
            for (int t = 0; t < 8; ++t) {
                qp[t].h = *reinterpret_cast<const u32x4*>(row + 16 * t);
                qp[t].m = *reinterpret_cast<const u32x4*>(row + 16 * t + 4);
            }
            if constexpr (kNormQ) {
#pragma clang fp contract(off)
                double ss = 0.0;
#pragma unroll
                for (int t = 0; t < 8; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const double x = __uint_as_float(qp[t].h[j]), y = __uint_as_float(qp[t].m[j]);
                        ss = __builtin_fma(x, x, ss);
                        ss = __builtin_fma(y, y, ss);
                    }
                ss += lane_xor_f64<32>(ss);
                const float inv = (float)(1.0 / sqrt(ss / (double)kHeadDim + (double)here(eps)));
                const float2* tr = cs + (size_t)(pos0 + bq) * (kHeadDim / 2) + e0;
                auto turn = [&](uint32_t& lo, uint32_t& hi, int d) {  // elements d + 8hh and 64 further on
                    const float2 t = tr[d];
                    const float a = (__uint_as_float(lo) * inv) * q_gamma[d + e0];
                    const float e = (__uint_as_float(hi) * inv) * q_gamma[64 + d + e0];
                    const float ac = a * t.x, es = e * t.y, as = a * t.y, ec = e * t.x;
                    lo = __float_as_uint(ac - es), hi = __float_as_uint(as + ec);
                };
#pragma unroll
                for (int t = 0; t < 4; ++t)
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        uint32_t lo = qp[t].h[j], hi = qp[t + 4].h[j];
                        turn(lo, hi, 16 * t + j);
                        qp[t].h[j] = lo, qp[t + 4].h[j] = hi;
                        lo = qp[t].m[j], hi = qp[t + 4].m[j];
                        turn(lo, hi, 16 * t + 4 + j);
                        qp[t].m[j] = lo, qp[t + 4].m[j] = hi;
                    }
            }
        };
        auto qk_fp32 = [&](int i, floatx16& s) {
#pragma unroll
            for (int r = 0; r < 16; ++r) s[r] = 0.f;
            const __amdgpu_buffer_rsrc_t rs = tile_rsrc(kbase, (kt_lo + kKS * i + grp) * kKT);
            const int ln = unhoisted(lane);
            const uint32_t off = (ln & 31) * row_bytes + 32u * (ln >> 5);
#pragma unroll
            for (int t = 0; t < 8; ++t) {
#pragma unroll
                for (int j = 0; j < 4; ++j) {  // d = 16t + 8hh + 2j and the next
                    const u32x2 v = __builtin_amdgcn_raw_buffer_load_b64(rs, off + 64 * t + 8 * j, 0, 0);
                    const u32x4 qv = j < 2 ? qp[t].h : qp[t].m;
                    const float q0 = __uint_as_float(qv[2 * (j & 1)]), q1 = __uint_as_float(qv[2 * (j & 1) + 1]);
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(v.x), q0, s, 0, 0, 0);
                    s = __builtin_amdgcn_mfma_f32_32x32x2f32(__uint_as_float(v.y), q1, s, 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };
        auto pv_fp32 = [&](int i, const floatx16& p) {
            const __amdgpu_buffer_rsrc_t rs = tile_rsrc(vbase, (kt_lo + kKS * i + grp) * kKT);
            const uint32_t off = unhoisted(4 * hh) * row_bytes + 4u * col;
#pragma unroll
            for (int r = 0; r < 16; ++r) {  // lane half hh: key 8(r/4) + 4hh + r%4
#pragma unroll
                for (int db = 0; db < 4; ++db) {
                    const float v = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(
                        rs, off + (8 * (r >> 2) + (r & 3)) * row_bytes + 128 * db, 0, 0));
                    o[db] = __builtin_amdgcn_mfma_f32_32x32x2f32(v, p[r], o[db], 0, 0, 0);
                }
                __builtin_amdgcn_sched_barrier(0);
            }
        };

        clear();
        lds_barrier();  // every wave has its q (the staging area is free for the V planes); K planes stored
        // the groups run half an iteration apart: one multiplies K by Q while the other is in its
        // softmax, so a SIMD's two waves do not leave the matrix pipe idle together
        if (grp == 1) lds_barrier();
        for (int i = 0; i < n_it; ++i) {
            floatx16 s;
            if (i < n_mine) {
                // S^T = K . Q^T, while V(i) goes to its planes; then K(i+1) is fetched
#pragma unroll
                for (int r = 0; r < 16; ++r) s[r] = 0.f;
                Planes kf;
                kf.l = k_frag(0, 2), kf.m = k_frag(0, 1), kf.h = k_frag(0, 0);
#pragma unroll
                for (int t = 0; t < 8; ++t) {
                    if (t == 4 || t == 6) conv_v(t == 6);
                    mfma_split(kf, qp[t], s, [&](int p) { return t < 7 ? k_frag(t + 1, p) : u32x4{}; });
                }
                if (i + 1 < n_mine) load_k(i + 1);
            }
            lds_barrier();
            if (i < n_mine) {
                __builtin_amdgcn_s_setprio(1);
                softmax(kt_lo + kKS * i + grp, s);
                // O^T += V^T . P^T, while K(i+1) goes to its planes; then V(i+1) is fetched
                const bool more = i + 1 < n_mine;
                Planes vf, pp;
                vf.l = v_frag(0, 2), vf.m = v_frag(0, 1), vf.h = v_frag(0, 0);
#pragma unroll
                for (int x = 0; x < 8; ++x) {
                    if ((x & 3) == 0) {
                        uint32_t ph[4], pm[4], pl[4];
#pragma unroll
                        for (int j = 0; j < 4; ++j)
                            split_pair(s[2 * x + 2 * j], s[2 * x + 2 * j + 1], ph[j], pm[j], pl[j]);
                        pp = {u32x4{ph[0], ph[1], ph[2], ph[3]}, u32x4{pm[0], pm[1], pm[2], pm[3]},
                              u32x4{pl[0], pl[1], pl[2], pl[3]}};
                    }
                    if (x == 4 || x == 6) conv_k(x == 6);
                    mfma_split(vf, pp, o[x & 3], [&](int p) { return x < 7 ? v_frag(x + 1, p) : u32x4{}; });
                }
                if (more) load_v(i + 1);
                __builtin_amdgcn_s_setprio(0);
            }
            lds_barrier();
        }
        if (grp == 0) lds_barrier();

        // An infinite K or V value (or a finite one past bf16's range) has no planes to multiply:
        // the residual of inf is NaN, and inf times a zero residual is NaN where the fp32 product is
        // infinite or the key's weight is zero.  Such a tile, and one with a K or V value past kPlaneMax,
        // shows as a sum that is not finite.  A V value or a weight below kPlaneMin may have lost bits of
        // its third plane, 2^-134: with V below kPlaneMax, weights at most 2^kLazy and 2^20 keys, a sum from
        // kSmallSum up is off by less than 2^-30 of itself.  A smaller one has the wave look through its V
        // tiles, in the blocks of 32 columns with such a sum, because a column of zeros or small V throughout
        // give one too (8192 tokens: 10% with one column of zeros): it stands if no V value there is below
        // kPlaneMin and the largest one is too small for the weights' 2^-134 to show in it.  Otherwise, and
        // for a q past its limit, the wave takes its tiles again in fp32, whose outcome stands whatever it is.
        {
            float z = lsum * 0.f, least[4];  // per block of 32 columns
#pragma unroll
            for (int db = 0; db < 4; ++db) {
                least[db] = INFINITY;
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    z = __builtin_fmaf(o[db][r], 0.f, z);
                    least[db] = fminf(least[db], __builtin_fabsf(o[db][r]));
                }
            }
            const float least_all = fminf(fminf(least[0], least[1]), fminf(least[2], least[3]));
            uint64_t redo = q_fp32 | __builtin_amdgcn_ballot_w64(z != 0.f);
            // (a lane without a visible key has no sum: m stays -inf)
            if (!redo && __builtin_amdgcn_ballot_w64(least_all < kSmallSum && m != -INFINITY)) {
                uint32_t small = 0xFFFFFFFFu, tiny = 0xFFFFFFFFu;  // the smallest nonzero sum and V value
                if (m != -INFINITY) {
#pragma unroll
                    for (int db = 0; db < 4; ++db)
#pragma unroll
                        for (int r = 0; r < 16; ++r) small = min(small, magnitude(__float_as_uint(o[db][r])));
                }
                float most = 0.f;
#pragma unroll
                for (int db = 0; db < 4; ++db) {
                    if (!__builtin_amdgcn_ballot_w64(least[db] < kSmallSum && m != -INFINITY)) continue;
                    for (int i = 0; i < n_mine; ++i) {
                        const __amdgpu_buffer_rsrc_t rs = tile_rsrc(vbase, (kt_lo + kKS * i + grp) * kKT);
                        const int ln = unhoisted(lane);
                        const uint32_t off = (ln >> 3) * row_bytes + 16u * (ln & 7) + 128u * db;
#pragma unroll
                        for (int j = 0; j < kKT / 8; ++j) {
                            const u32x4 v = __builtin_amdgcn_raw_buffer_load_b128(rs, off + 8 * j * row_bytes, 0, 0);
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                tiny = min(tiny, magnitude(v[e]));
                                most = fmaxf(most, __builtin_fabsf(__uint_as_float(v[e])));
                            }
                        }
                    }
                }
                // the sums are off by up to 2^20 2^-134 most; a lane without a nonzero one has nothing to lose
                const float limit = wave_max(most) * 0x1p-84f;
                redo = __builtin_amdgcn_ballot_w64(tiny < kTinyMagnitude || limit > of_magnitude(small));
            }
            if (redo && live) {  // (a slot past the last block writes nothing)
                clear();
                q_whole();
                for (int i = 0; i < n_mine; ++i) {
                    floatx16 s;
                    qk_fp32(i, s);
                    softmax(kt_lo + kKS * i + grp, s);
                    pv_fp32(i, s);
                }
            }
        }

        // ---- merge the key groups through LDS (tile buffers are free after the barrier):
        // group g finalises output blocks db = 2g, 2g+1 and hands the other two to its partner
        float* xw = smem + w * (kXchF * 64) + lane;
        xw[0] = m;
        xw[64] = lsum;
        // (grp is wave-uniform: selects, not a dynamic register index)
        const floatx16 give0 = grp ? o[0] : o[2], give1 = grp ? o[1] : o[3];
        const floatx16 keep0 = grp ? o[2] : o[0], keep1 = grp ? o[3] : o[1];
#pragma unroll
        for (int i = 0; i < 16; ++i) {
            xw[(2 + i) * 64] = give0[i];
            xw[(18 + i) * 64] = give1[i];
        }
        lds_barrier();
        const float* xp = smem + ((1 - grp) * GW + hw) * (kXchF * 64) + lane;
        const float mp = xp[0], lp = xp[64];
        const float mt = fmaxf(m, mp);  // -inf only when this share holds no visible key for the query
        const float c0 = m == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(m - mt);
        const float cp = mp == -INFINITY ? 0.f : __builtin_amdgcn_exp2f(mp - mt);
        const float l = half_sum(lsum * c0 + lp * cp);
        // finished rows (normalised, or the unnormalised share for k_prefill_combine) go to the
        // staging area in row order, then every wave stores two whole 512-byte rows per instruction
        {
            const float inv = ksplit == 1 ? 1.f / l : 1.f;
            float* ost = qst + (hw * kQB + col) * kKS_F + 64 * grp + 4 * hh;
#pragma unroll
            for (int r = 0; r < 16; r += 4) {
                // O^T registers r .. r+3 of block db are d = 32 db + 8(r/4) + 4hh + 0 .. 3
                float v0[4], v1[4];
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    v0[j] = (keep0[r + j] * c0 + xp[(2 + r + j) * 64] * cp) * inv;
                    v1[j] = (keep1[r + j] * c0 + xp[(18 + r + j) * 64] * cp) * inv;
                }
                *reinterpret_cast<float4*>(ost + 2 * r) = make_float4(v0[0], v0[1], v0[2], v0[3]);
                *reinterpret_cast<float4*>(ost + 32 + 2 * r) = make_float4(v1[0], v1[1], v1[2], v1[3]);
            }
            if (ksplit > 1 && live && b < B && hh == 0 && grp == 0)
                *reinterpret_cast<float2*>(part_ml + ((size_t)split * B * H + (size_t)b * H + h) * 2) =
                    make_float2(mt, l);
        }
        lds_barrier();
        {
            const int sl = kSlots * u + (wu >> 1);  // wave wu stores rows 16*(wu&1).. of slot wu/2
            const int qbo = fdiv(sl, fG), ho = kvh * G + sl - qbo * G;
            float* dst0 = ksplit == 1 ? out : part_o + (size_t)split * B * H * D;
            const int ln = unhoisted(lane), hh0 = ln >> 5, c4 = 4 * (ln & 31);
#pragma unroll
            for (int j = 0; j < kQB / 4; ++j) {
                const int jj = (kQB / 2) * (wu & 1) + 2 * j + hh0;
                const int bo = qbo * kQB + jj;
                const float4 v = *reinterpret_cast<const float4*>(qst + ((wu >> 1) * kQB + jj) * kKS_F + c4);
                if (sl < nslot && bo < B)
                    *reinterpret_cast<float4*>(dst0 + ((size_t)bo * H + ho) * D + c4) = v;
            }
        }
    }
}

// Merge of the ksplit shares of every (query, head): grid ceil(B*H/4), 128 threads; thread
// = float4 column d4 of row (b, h).  o = sum_s 2^(m_s - M) O_s / sum_s 2^(m_s - M) l_s, empty
// shares (m = -inf, l = 0) skipped.
__global__ __launch_bounds__(128) void k_prefill_combine(const float* __restrict__ part_o,
                                                         const float* __restrict__ part_ml, float* __restrict__ out,
                                                         int rows, int ksplit, const int* __restrict__ pos_dev, int B,
                                                         int H, int HKV) {
    const int row = blockIdx.x * 4 + (threadIdx.x >> 5), d4 = threadIdx.x & 31;
    if (row >= rows) return;
    // the row's unit and pair, as k_prefill numbers them; the shares holding tiles of that unit
    const int G = H / HKV, b = row / H, hq = row - b * H, g = hq % G;
    const int nb = (B + kQB - 1) / kQB, nslot = G * nb, nu = (nslot + kSlots - 1) / kSlots;
    const int u = ((b / kQB) * G + g) / kSlots, pair = min(u, nu - 1 - u);
    const FastDiv fG = fast_div((uint32_t)G), fK = fast_div((uint32_t)ksplit);
    const int pos0 = *pos_dev;
    // the covered shares' (m, l) and accumulator pieces are loaded before any is used: one
    // round trip, and no read of a share without tiles of this unit
    float2 ml[kPrefillMaxSplit];
    float4 v[kPrefillMaxSplit];
#pragma unroll
    for (int s = 0; s < kPrefillMaxSplit; ++s) {
        ml[s] = make_float2(-INFINITY, 0.f);
        if (s >= ksplit) continue;
        int lo0, r0, lo1, r1;
        prefill_share(pair, nu - 1 - pair, s, fK, pos0, B, nslot, fG, lo0, r0, lo1, r1);
        if ((u == pair ? r0 : r1) == 0) continue;
        const size_t slot = (size_t)s * rows + row;
        ml[s] = *reinterpret_cast<const float2*>(part_ml + slot * 2);
        v[s] = *reinterpret_cast<const float4*>(part_o + slot * kHeadDim + 4 * d4);
    }
    float M = -INFINITY;
#pragma unroll
    for (int s = 0; s < kPrefillMaxSplit; ++s)
        if (s < ksplit) M = fmaxf(M, ml[s].x);
    float L = 0.f;
    float4 o = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int s = 0; s < kPrefillMaxSplit; ++s) {
        // an empty share adds nothing; one whose every score is NaN has m = -inf too, and its NaN l counts
        if (s >= ksplit || (ml[s].x == -INFINITY && ml[s].y == 0.f)) continue;
        const float wv = __builtin_amdgcn_exp2f(ml[s].x - M);
        L = fmaf(wv, ml[s].y, L);
        o.x = fmaf(wv, v[s].x, o.x);
        o.y = fmaf(wv, v[s].y, o.y);
        o.z = fmaf(wv, v[s].z, o.z);
        o.w = fmaf(wv, v[s].w, o.w);
    }
    const float inv = 1.f / L;
    o.x *= inv;
    o.y *= inv;
    o.z *= inv;
    o.w *= inv;
    *reinterpret_cast<float4*>(out + (size_t)row * kHeadDim + 4 * d4) = o;
}

static int prefill_grid1(int B, int H, int HKV) {
    const int G = H / HKV;
    const int nb = (B + kQB - 1) / kQB;
    const int nu = (G * nb + kSlots - 1) / kSlots;
    return ((nu + 1) / 2) * HKV;
}

int prefill_split(int B, int H, int HKV, int max_kv, bool fine) {
    // One workgroup per (unit pair, KV head), all with the same work, one per CU at a time
    // (134 KB of LDS): the launch takes ceil(g1 / 256) rounds.  Splitting every unit's key
    // tiles into k contiguous shares makes g1*k workgroups of 1/k the work, so the time goes
    // as ceil(g1*k / 256) / k.  The plan takes the k in 1..8 with the shortest time, a larger
    // k only when it gains >= 10% (each share adds a combine read and write), and keeps >= 4
    // tiles per share on average (max_kv bounds pos0 + B on the host, which does not see the
    // device-resident position).  The fine plan goes down to one tile per share: a tile now costs
    // about what a share does, and a small chunk leaves most CUs idle otherwise (64 rows at 300, G = 4:
    // 2 shares 40.8 us, 4 shares 32.7, 8 shares 27.1; 100 rows at 600: 5 shares 38.2, 8 shares 31.6; 16 rows at
    // 100: 1 share 23.1, 4 shares 20.8; 200 rows at 300, G = 8, paged: 3 shares 45.0, 4 shares 42.4).  It needs a
    // larger workspace, so a call takes it when its workspace holds it and the other plan when not.
    const int g1 = prefill_grid1(B, H, HKV);
    const long avg_tiles = ((long)max_kv - B / 2 + kKT - 1) / kKT;
    const long kmin_tiles = fine ? 1 : 4;
    long kmax = avg_tiles / kmin_tiles > 1 ? avg_tiles / kmin_tiles : 1;
    if (kmax > kPrefillMaxSplit) kmax = kPrefillMaxSplit;
    auto rounds = [&](long k) { return (double)((g1 * k + 255) / 256) / (double)k; };
    int best = 1;
    for (int k = 2; k <= kmax; ++k)
        if (rounds(k) < 0.9 * rounds(best)) best = k;
    if (const char* env = std::getenv("EI_PREFILL_SPLIT")) {  // tuning override (1..8)
        const int v = std::atoi(env);
        if (v >= 1 && v <= kPrefillMaxSplit) best = v;
    }
    return best;
}

static size_t align256(size_t x) { return (x + 255) & ~(size_t)255; }

size_t prefill_ws_bytes(int B, int H, int ksplit) {
    if (ksplit <= 1) return 0;
    const size_t rows = (size_t)B * H;
    return align256((size_t)ksplit * rows * kHeadDim * sizeof(float)) +
           align256((size_t)ksplit * rows * 2 * sizeof(float));
}

template <bool kNormQ, bool kPaged>
static hipError_t launch_prefill_kernel(hipStream_t st, unsigned grid, size_t lds, const float* q, long q_stride,
                                        float* out, const float* kc, const float* vc, const int* pos_dev, int B, int H,
                                        int HKV, float scale, int ksplit, float* part_o, float* part_ml,
                                        const float* q_gamma, const float* cs, float eps, const int* btab,
                                        int bshift, int max_blocks) {
    static std::atomic<bool> opted;
    if (const hipError_t e = opt_in_lds(opted, (const void*)k_prefill<kNormQ, kPaged>, lds); e != hipSuccess) return e;
    k_prefill<kNormQ, kPaged><<<grid, 64 * kSlots * kKS, lds, st>>>(q, q_stride, out, kc, vc, pos_dev, B, H, HKV, scale,
                                                                    ksplit, part_o, part_ml, q_gamma,
                                                                    reinterpret_cast<const float2*>(cs), eps, btab,
                                                                    bshift, max_blocks);
    return hipGetLastError();
}

hipError_t launch_prefill(hipStream_t st, const float* q, long q_stride, float* out, const float* kc,
                          const float* vc, const int* pos_dev, int B, int H, int HKV, float scale, int ksplit,
                          void* ws, const float* q_gamma, const float* cs, float eps, const int* block_table,
                          int block_shift, int max_blocks) {
    if (ksplit < 1) ksplit = 1;
    const unsigned grid = (unsigned)prefill_grid1(B, H, HKV) * ksplit;
    float* part_o = nullptr;
    float* part_ml = nullptr;
    if (ksplit > 1) {
        const size_t rows = (size_t)B * H;
        part_o = static_cast<float*>(ws);
        part_ml = reinterpret_cast<float*>(static_cast<char*>(ws) + align256((size_t)ksplit * rows * kHeadDim * 4));
    }
    const size_t lds = (size_t)kLdsF * sizeof(float);  // > 64 KB: opt in once
    static_assert(kLdsF * sizeof(float) <= 160 * 1024, "LDS budget");
    const bool nq = q_gamma != nullptr, pg = block_table != nullptr;
    hipError_t e;
    if (nq && pg) return hipErrorInvalidValue;  // not built: a paged step norms q in its prologue
    if (nq)
        e = launch_prefill_kernel<true, false>(st, grid, lds, q, q_stride, out, kc, vc, pos_dev, B, H, HKV, scale,
                                               ksplit, part_o, part_ml, q_gamma, cs, eps, nullptr, 0, 0);
    else if (pg)
        e = launch_prefill_kernel<false, true>(st, grid, lds, q, q_stride, out, kc, vc, pos_dev, B, H, HKV, scale,
                                               ksplit, part_o, part_ml, nullptr, nullptr, 0.f, block_table,
                                               block_shift, max_blocks);
    else
        e = launch_prefill_kernel<false, false>(st, grid, lds, q, q_stride, out, kc, vc, pos_dev, B, H, HKV, scale,
                                                ksplit, part_o, part_ml, nullptr, nullptr, 0.f, nullptr, 0, 0);
    if (e != hipSuccess) return e;
    if (ksplit > 1) {
        const int rows = B * H;
        k_prefill_combine<<<(rows + 3) / 4, 128, 0, st>>>(part_o, part_ml, out, rows, ksplit, pos_dev, B, H, HKV);
    }
    return hipGetLastError();
}

}  // namespace ei
