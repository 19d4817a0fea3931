// ESMM and ESTMM for fp32 operands on gfx950, on the bf16 matrix pipes and as exact as on the fp32 ones.  Unlike the reference,
// which rounds fp32 operands to fp16 before its WMMA (kernels/esmm_full.cu:128-130,167-169), nothing is rounded away.
//
// A fp32 value is the sum of three bf16 values, exactly: h = bf16(x), m = bf16(x - h), l = x - h - m (8 + 8 + 8 bits of
// significand, each rounded to nearest).  A product is then h h' + (h m' + m h') + (m m' + h l' + l h') and three terms below
// 2^-24 of it that are left out; each is exact in the matrix pipe's fp32.  v_mfma_f32_32x32x16_bf16 takes 32 cycles for 16
// contraction indices where v_mfma_f32_32x32x2_f32 takes 64 for two, so the six terms are 192 cycles against 512.
// Error against 64 bits, in brackets v_mfma_f32_32x32x2_f32, on 64 x 64 and 128 x 128 tiles: 448 products a result 2.2e-7 (3.8e-7)
// and 968 4.7e-7 (5.6e-7), lists of a few entries 5.4e-8 (6.3e-8); lower in each of 24 layers of 100 to 9000 tokens, 64 to 968 wide.
// GELU and GELU' are gelu_full's, as exact as through erff.
//
// What the split has to be careful with, it leaves to the fp32 pipe: a stage of operands that holds a magnitude of 2^63 and
// more (whose terms could overflow where the product does not), an infinity (0 times infinity in a term) or one value other than
// zero below 2^-100 (whose l would be a denormal bf16 value short of bits; its neighbours may be another result column's, so
// their size says nothing) is written to LDS unsplit and multiplied by v_mfma_f32_32x32x2_f32.  A NaN is one in either way.
// Cost of the check: one vector instruction per two values, and two per value more in a stage where a wavefront holds a zero or a small
// value (9216 tokens, 384 -> 1536, 8 experts, top-2, ESMM and ESTMM alone: 163 and 177 us; half of the values zeros 161 and 175; one in 10000
// of 1e-33, so that most stages go to the fp32 pipe, 231 and 300; all of them 357 and 392).
//
// Values are split once per workgroup, on their way from registers to LDS (6.5 vector instructions a value, about half the
// MFMA cycles of a 128 x 128 tile), not once per wavefront that reads them; rows are fetched into registers a stage ahead.
// One set of planes and two barriers a stage: 48 KB and eight wavefronts a workgroup, so that two (by registers; three by LDS) share a
// CU and one's split and barriers meet another's MFMAs.
// What bounds them: matrix and vector instructions, which overlap in part only (a launch without the split, or without the MFMAs,
// takes 0.9 and 0.6 of its time; without fetches 0.95).  At 9216 tokens, 384 -> 1536, 8 experts, top-2 (21.7 GFLOP a launch; before:
// v_mfma_f32_32x32x2_f32 fed by asynchronous copies, at 64 % of its pipe's rate), kernel times inside a training step: fc1 + GELU
// 245 -> 170 us, fc2 211 -> 136, dW 234 -> 143 and a fold of 19, dy1 248 -> 171, the step 1.44 -> 1.03 ms; 2048 rows, 8 experts:
// 128 -> 512 10.3 -> 9.7, 512 -> 128 15.5 -> 14.6.  Fetching two stages ahead, one barrier a stage with two sets of planes (one
// workgroup a CU), and splitting between a stage's MFMAs were measured too: 0 to 20 % slower.
//
// LDS tile formats, three planes (h, m, l) of each operand, a stage holds KD contraction indices:
//   KC  contraction index fastest in memory: [row][KD], fragments by ds_read_b128 (frag_kc)
//   KS  contraction index slowest in memory: [KD][W columns], fragments by ds_read_b64_tr_b16
// 16-byte pieces are permuted inside a row so that neither the writes nor the reads meet on a bank.
//
// Replaces esmm_shared_tensor_kernel_vectorized_accum_full (kernels/esmm_full.cu:58-246) and the
// ESMM / ESTMM tasks of fused_grad_*_kernel_vectorized_full (kernels/fused_ops_full.cu:117-371).
#include <algorithm>

#include "dma_common.h"
#include "small_bodies.h"

namespace hexa {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

// Workgroup tile: WR x WF wavefronts, every one multiplies RB x FB blocks of 32 x 32; KD contraction indices per stage, of which
// KG groups of wavefronts take a part each (and add their sums at the end).  WAVES: wavefronts per SIMD the registers are sized
// for (three planes of both operands: 48 KB of LDS).
template <int WR_, int WF_, int KG_, int RB_, int FB_, int KD_, int WAVES_> struct Tile {
    static constexpr int WR = WR_, WF = WF_, KG = KG_, NT = 64 * WR_ * WF_ * KG_, RB = RB_, FB = FB_, KD = KD_, WAVES = WAVES_;
    static constexpr int BM = 32 * RB_ * WR_, BN = 32 * FB_ * WF_, KSTEPS = KD_ / 16 / KG_;
    static constexpr int R_PLANE = BM * KD * 2, F_PLANE = BN * KD * 2, F_AT = 3 * R_PLANE, BYTES = F_AT + 3 * F_PLANE;
    static constexpr int RO = BM * KD / 8 / NT, FO = BN * KD / 8 / NT;      // octets a thread fetches and splits in a stage
    static_assert(RO * NT * 8 == BM * KD && FO * NT * 8 == BN * KD, "whole octets per thread");
    static_assert(KG <= 2 && (KG - 1) * WR * WF * RB * FB * 4096 <= BYTES, "one other group's sums fit into the planes");
};
using Wide = Tile<2, 4, 1, 2, 1, 32, 4>;
using Deep = Tile<2, 2, 2, 1, 1, 64, 4>;

// Eight neighbouring values of an operand: along the contraction (KC) or across it (KS).
struct Octet { f32x4 a, b; };

__device__ __forceinline__ float bits_f(unsigned u) { return __uint_as_float(u); }
__device__ __forceinline__ float largest(float m, float a, float b) {      // of |a|, |b| and m; a NaN is passed over
    float r;
    asm("v_max3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}
__device__ __forceinline__ float smallest(float m, float a, float b) {     // the same
    float r;
    asm("v_min3_f32 %0, %1, |%2|, |%3|" : "=v"(r) : "v"(m), "v"(a), "v"(b));
    return r;
}
constexpr float SPLIT_LOW = 0x1p-100f, SPLIT_HIGH = 0x1p63f;
struct Span { float low, high; };          // smallest and largest magnitude
// the planes of eight values
__device__ __forceinline__ void split(const Octet& v, u32x4& h, u32x4& m, u32x4& l, Span& span) {
    const float x[8] = {v.a.x, v.a.y, v.a.z, v.a.w, v.b.x, v.b.y, v.b.z, v.b.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const float a = x[2 * q], b = x[2 * q + 1];
        span.low = smallest(span.low, a, b);
        span.high = largest(span.high, a, b);
        const unsigned hw = pack2<__bf16>(a, b);
        const float ra = a - bits_f(hw << 16), rb = b - bits_f(hw & 0xffff0000u);
        const unsigned mw = pack2<__bf16>(ra, rb);
        h[q] = hw;
        m[q] = mw;
        l[q] = pack2<__bf16>(ra - bits_f(mw << 16), rb - bits_f(mw & 0xffff0000u));
    }
}
// the smallest magnitude other than zero, as bits of 2 |x| - 1, where a zero comes last
__device__ __forceinline__ unsigned smallest_but_zero(unsigned m, const Octet& v) {
    const float x[8] = {v.a.x, v.a.y, v.a.z, v.a.w, v.b.x, v.b.y, v.b.z, v.b.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) m = min(min(m, 2u * __float_as_uint(x[2 * q]) - 1u), 2u * __float_as_uint(x[2 * q + 1]) - 1u);
    return m;
}
// the same eight values unsplit: their upper and lower halves in the planes of h and m
__device__ __forceinline__ void halves(const Octet& v, u32x4& hi, u32x4& lo) {
    const float x[8] = {v.a.x, v.a.y, v.a.z, v.a.w, v.b.x, v.b.y, v.b.z, v.b.w};
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const unsigned a = __float_as_uint(x[2 * q]), b = __float_as_uint(x[2 * q + 1]);
        hi[q] = (a >> 16) | (b & 0xffff0000u);
        lo[q] = (a & 0xffffu) | (b << 16);
    }
}

// Where piece `oct` (eight values) of row r of an operand sits in a plane of width W, and which pieces a lane handles: octet i
// of thread tid is piece piece_of(tid) of row row_of(tid, i).
template <bool KS, int W, int KD, int NT = 64> struct Place {
    static constexpr int PPR = KS ? W / 8 : KD / 8, ROWS = NT / PPR;
    static __device__ __forceinline__ int row_of(int tid, int i) { return tid / PPR + i * ROWS; }
    static __device__ __forceinline__ int piece_of(int tid) { return tid % PPR; }
    static __device__ __forceinline__ int swizzle(int row) {
        if (!KS) return kc_swizzle<KD>(row);
        return W == 64 ? ((row >> 1) & 1) << 2 : (row & 3) << 2;     // the four rows a transposing read touches: other banks
    }
    static __device__ __forceinline__ int at(int row, int piece) { return row * PPR * 16 + ((piece ^ swizzle(row)) << 4); }
};

typedef __attribute__((address_space(3))) s16x4* lds_s16x4_t;
// the 32 x 16 fragment of a plane: rows col0 .. col0 + 31, contraction indices 16 ks + 8 (lane >> 5) + 0..7
template <bool KS, int W, int KD> __device__ __forceinline__ u32x4 fragment(const char* plane, int col0, int ks, int lane) {
    if constexpr (!KS) {
        return frag_kc<u32x4, KD>(plane, col0, ks, lane);
    } else {
        const int grp = lane >> 4, s = lane & 15;
        const int col = col0 + (grp & 1) * 16 + (s & 3) * 4, k = ks * 16 + (grp >> 1) * 8 + (s >> 2);
        union { u32x4 v; s16x4 h[2]; } r;
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            const char* p = plane + Place<true, W, KD>::at(k + 4 * half, col >> 3) + (col & 7) * 2;
            r.h[half] = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s16x4_t)(__attribute__((address_space(3))) const void*)p);
        }
        return r.v;
    }
}
__device__ __forceinline__ bf16x8 as_bf16(u32x4 v) {
    union { u32x4 u; bf16x8 b; } c;
    c.u = v;
    return c.b;
}
__device__ __forceinline__ float whole(u32x4 hi, u32x4 lo, int j) {
    return bits_f(j & 1 ? (hi[j >> 1] & 0xffff0000u) | (lo[j >> 1] >> 16) : (hi[j >> 1] << 16) | (lo[j >> 1] & 0xffffu));
}

// acc += F x R over the stage in LDS.  A lane ends up with row lane % 32 of R and, per group of four registers, 4 consecutive
// columns of F, from either instruction.
template <typename C, bool F_KS, bool R_KS>
__device__ __forceinline__ void multiply(const char* smem, int kg, int wr, int wf, int lane, f32x16 (&acc)[C::FB][C::RB]) {
    // the smallest terms first: of the first 16 products only the last addition rounds the whole sum
    constexpr int TERMS[6][2] = {{0, 2}, {2, 0}, {1, 1}, {0, 1}, {1, 0}, {0, 0}};
#pragma unroll
    for (int step = 0; step < C::KSTEPS; ++step) {
        const int ks = kg * C::KSTEPS + step;
        u32x4 r[C::RB][3];
#pragma unroll
        for (int i = 0; i < C::RB; ++i)
#pragma unroll
            for (int q = 0; q < 3; ++q) r[i][q] = fragment<R_KS, C::BM, C::KD>(smem + q * C::R_PLANE, (wr * C::RB + i) * 32, ks, lane);
#pragma unroll
        for (int j = 0; j < C::FB; ++j) {
            u32x4 f[3];
#pragma unroll
            for (int q = 0; q < 3; ++q) f[q] = fragment<F_KS, C::BN, C::KD>(smem + C::F_AT + q * C::F_PLANE, (wf * C::FB + j) * 32, ks, lane);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int t = 0; t < 6; ++t)
#pragma unroll
                for (int i = 0; i < C::RB; ++i) acc[j][i] = Mfma<__bf16>::run(as_bf16(f[TERMS[t][0]]), as_bf16(r[i][TERMS[t][1]]), acc[j][i]);
        }
    }
}
template <typename C, bool F_KS, bool R_KS>
__device__ __forceinline__ void multiply_whole(const char* smem, int kg, int wr, int wf, int lane, f32x16 (&acc)[C::FB][C::RB]) {
    for (int ks = kg * C::KSTEPS; ks < (kg + 1) * C::KSTEPS; ++ks) {
#pragma unroll
        for (int j = 0; j < C::FB; ++j) {
            u32x4 f[2];
#pragma unroll
            for (int q = 0; q < 2; ++q) f[q] = fragment<F_KS, C::BN, C::KD>(smem + C::F_AT + q * C::F_PLANE, (wf * C::FB + j) * 32, ks, lane);
#pragma unroll
            for (int i = 0; i < C::RB; ++i) {
                u32x4 r[2];
#pragma unroll
                for (int q = 0; q < 2; ++q) r[q] = fragment<R_KS, C::BM, C::KD>(smem + q * C::R_PLANE, (wr * C::RB + i) * 32, ks, lane);
#pragma unroll
                for (int k = 0; k < 8; ++k)
                    acc[j][i] = __builtin_amdgcn_mfma_f32_32x32x2f32(whole(f[0], f[1], k), whole(r[0], r[1], k), acc[j][i], 0, 0, 0);
            }
        }
    }
}

// The stages of a tile.  load(step, r, f) fetches a step's values into registers (the caller's addresses move on with it); the
// values of a step are fetched while the step before is multiplied, and split and written while the CU's other workgroups
// multiply.
template <typename C, bool F_KS, bool R_KS, typename L>
__device__ __forceinline__ void multiply_stages(int nk, bool busy, char* smem, int* sWhole, int tid, f32x16 (&acc)[C::FB][C::RB], L load) {
    using PR = Place<R_KS, C::BM, C::KD, C::NT>;
    using PF = Place<F_KS, C::BN, C::KD, C::NT>;
    const int lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave / (C::WR * C::WF), wr = wave / C::WF % C::WR, wf = wave % C::WF;
    Octet r[C::RO], f[C::FO];
    auto each = [&](auto&& put) {
#pragma unroll
        for (int i = 0; i < C::RO; ++i) put(r[i], smem + PR::at(PR::row_of(tid, i), PR::piece_of(tid)), C::R_PLANE);
#pragma unroll
        for (int i = 0; i < C::FO; ++i) put(f[i], smem + C::F_AT + PF::at(PF::row_of(tid, i), PF::piece_of(tid)), C::F_PLANE);
    };
    if (nk > 0) load(0, r, f);
    if (tid < 2) sWhole[tid] = 0;
    for (int kt = 0; kt < nk; ++kt) {
        __syncthreads();                                  // everyone is done reading the stage before
        Span span{1.f, 0.f};
        each([&](const Octet& v, char* to, int plane) {
            u32x4 h, m, l;
            split(v, h, m, l, span);
            *reinterpret_cast<u32x4*>(to) = h;
            *reinterpret_cast<u32x4*>(to + plane) = m;
            *reinterpret_cast<u32x4*>(to + 2 * plane) = l;
        });
        // (zeros are common: rows behind a list's end, tokens' own; they are told from small values only where there are any)
        bool odd = span.high >= SPLIT_HIGH;
        if (__builtin_amdgcn_ballot_w64(span.low < SPLIT_LOW) != 0) {
            unsigned low = ~0u;
            each([&](const Octet& v, char*, int) { low = smallest_but_zero(low, v); });
            odd |= low < 2u * __float_as_uint(SPLIT_LOW) - 1u;
        }
        // (one word for even and one for odd steps: the other one was last read before the barrier above)
        if (tid == 0) sWhole[(kt + 1) & 1] = 0;
        if (odd) sWhole[kt & 1] = 1;
        __syncthreads();
        if (__builtin_expect(__builtin_amdgcn_readfirstlane(sWhole[kt & 1]), 0)) {
            // (the stage is multiplied here, and the planes are left as zeros for what follows: two ways of adding to the
            // accumulators that meet behind a branch made the compiler copy them in every stage)
            __syncthreads();
            each([&](const Octet& v, char* to, int plane) {
                u32x4 hi, lo;
                halves(v, hi, lo);
                *reinterpret_cast<u32x4*>(to) = hi;
                *reinterpret_cast<u32x4*>(to + plane) = lo;
                *reinterpret_cast<u32x4*>(to + 2 * plane) = u32x4{0u, 0u, 0u, 0u};
            });
            __syncthreads();
            multiply_whole<C, F_KS, R_KS>(smem, kg, wr, wf, lane, acc);
            __syncthreads();
            each([&](const Octet&, char* to, int plane) {
                *reinterpret_cast<u32x4*>(to) = u32x4{0u, 0u, 0u, 0u};
                *reinterpret_cast<u32x4*>(to + plane) = u32x4{0u, 0u, 0u, 0u};
            });
            __syncthreads();
        }
        if (kt + 1 < nk) load(kt + 1, r, f);
        if (busy) multiply<C, F_KS, R_KS>(smem, kg, wr, wf, lane, acc);
    }
}

// The groups' sums added, in the first one's accumulators; whether this wavefront is of that group.
template <typename C> __device__ __forceinline__ bool combine(char* smem, int kg, int wave, int lane, f32x16 (&acc)[C::FB][C::RB]) {
    if constexpr (C::KG > 1) {
        f32x4* const at = reinterpret_cast<f32x4*>(smem) + (wave % (C::WR * C::WF)) * (C::RB * C::FB * 256) + lane;
        __syncthreads();                                 // the planes have been read
        if (kg > 0) {
#pragma unroll
            for (int b = 0; b < C::RB * C::FB; ++b)
#pragma unroll
                for (int g = 0; g < 4; ++g) {
                    const f32x16& v = acc[b / C::RB][b % C::RB];
                    at[(b * 4 + g) * 64] = f32x4{v[4 * g], v[4 * g + 1], v[4 * g + 2], v[4 * g + 3]};
                }
        }
        __syncthreads();
        if (kg > 0) return false;
#pragma unroll
        for (int b = 0; b < C::RB * C::FB; ++b)
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const f32x4 v = at[(b * 4 + g) * 64];
#pragma unroll
                for (int q = 0; q < 4; ++q) acc[b / C::RB][b % C::RB][4 * g + q] += v[q];
            }
    }
    return true;
}

struct Esmm32K {
    const float* x; const float* w; const float* bias; float* out; float* out_act; float* ws;
    const int32_t* token_ids; const int4* tile_info; const int32_t* tile_count;
    int T, K, N, mt_ub, ntn, slot_begin, nslots;
    int x_slot_rows, out_slot_rows;
    int accumulate, act, act_only;
    float* colsum;        // where set (tiles of HEXA_TILE_ROWS rows): [slot][row tile][column tile][BN] column sums of the stored result
};

template <bool W_IN_OUT, bool BIG, typename C>
__global__ __launch_bounds__(C::NT, C::WAVES) void esmm32_kernel(Esmm32K p) {
    constexpr int BM = C::BM, BN = C::BN, KD = C::KD, H = HEXA_TILE_ROWS / BM;   // H workgroup tiles per row tile of the routing
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    __shared__ int sTok[BM], sWhole[2];

    // Every XCD (workgroup ids go round-robin over the 8 of them) walks one contiguous eighth of the valid tiles,
    // column tiles fastest: an expert's weights are then fetched into one L2.
    int cum[9];
    cum[0] = 0;
#pragma unroll
    for (int q = 0; q < 8; ++q) cum[q + 1] = cum[q] + (q < p.nslots ? min(p.tile_count[p.slot_begin + q], p.mt_ub) : 0);
    const int valid = cum[8] * H * p.ntn;
    const int per = (valid + 7) >> 3;
    const int xcd = blockIdx.x & 7, loc = blockIdx.x >> 3;
    const int logical = xcd * per + loc;
    if (loc >= per || logical >= valid) return;
    const int piece_row = logical / p.ntn, nt = logical - piece_row * p.ntn;
    const int mtg = piece_row / H, half = piece_row - mtg * H;
    int sl = 0;
#pragma unroll
    for (int q = 1; q < 8; ++q) sl += (mtg >= cum[q] && q < p.nslots) ? 1 : 0;
    const int s = p.slot_begin + sl, mt = mtg - cum[sl];
    const int4 info = p.tile_info[(size_t)s * p.mt_ub + mt];
    const int e = info.x, row_start = info.y + half * BM, rows = min(BM, info.z - half * BM);
    if (rows <= 0) return;
    const int n0 = nt * BN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave / (C::WR * C::WF), wr = wave / C::WF % C::WR, wf = wave % C::WF;
    const int K = p.K, N = p.N;
    if (tid < BM) sTok[tid] = tid < rows ? p.token_ids[(size_t)s * p.T + row_start + tid] : -1;
    __syncthreads();

    // Sources of this lane's values: bases every lane shares plus 32-bit byte offsets (64-bit ones where an operand has
    // 4 GiB and more).  Lanes with nothing to fetch (rows past the tile's end, columns past N) read the first row or column:
    // what they produce is never stored.  Contraction indices past K are zeros in both operands.
    using Off = std::conditional_t<BIG, size_t, unsigned>;
    using PR = Place<false, BM, KD, C::NT>;
    using PF = Place<W_IN_OUT, BN, KD, C::NT>;
    const char* const xbase = reinterpret_cast<const char*>(p.x);
    const char* const wbase = reinterpret_cast<const char*>(p.w + (size_t)e * K * N);
    Off offR[C::RO], offF[C::FO];
    const int kR = PR::piece_of(tid) * 8;
    const int n1 = n0 + PF::piece_of(tid) * 8, second = n1 + 4 < N ? 16 : 0;     // W_IN_OUT: where the octet's second half is
#pragma unroll
    for (int i = 0; i < C::RO; ++i) offR[i] = (Off)((((size_t)p.x_slot_rows * s + max(sTok[PR::row_of(tid, i)], 0)) * K + kR) * 4);
#pragma unroll
    for (int i = 0; i < C::FO; ++i) {
        const int row = PF::row_of(tid, i);
        if (W_IN_OUT) offF[i] = (Off)(((size_t)row * N + (n1 < N ? n1 : 0)) * 4);
        else offF[i] = (Off)(((size_t)(n0 + row < N ? n0 + row : 0) * K + PF::piece_of(tid) * 8) * 4);
    }
    const Off stepF = W_IN_OUT ? (Off)KD * N * 4 : (Off)KD * 4;
    auto read4 = [](const char* base, Off off) { return *reinterpret_cast<const f32x4*>(base + (size_t)off); };
    auto load = [&](int step, Octet (&r)[C::RO], Octet (&f)[C::FO]) {
        const int left = K - step * KD;
        if (left >= KD) {
#pragma unroll
            for (int i = 0; i < C::RO; ++i) { r[i].a = read4(xbase, offR[i]); r[i].b = read4(xbase, offR[i] + 16); }
#pragma unroll
            for (int i = 0; i < C::FO; ++i) { f[i].a = read4(wbase, offF[i]); f[i].b = read4(wbase, offF[i] + (W_IN_OUT ? second : 16)); }
        } else {
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < C::RO; ++i) {
                r[i].a = zero; r[i].b = zero;
                if (kR < left) r[i].a = read4(xbase, offR[i]);
                if (kR + 4 < left) r[i].b = read4(xbase, offR[i] + 16);
            }
#pragma unroll
            for (int i = 0; i < C::FO; ++i) {
                const int k = W_IN_OUT ? PF::row_of(tid, i) : PF::piece_of(tid) * 8;
                f[i].a = zero; f[i].b = zero;
                if (k < left) f[i].a = read4(wbase, offF[i]);
                if (k + (W_IN_OUT ? 0 : 4) < left) f[i].b = read4(wbase, offF[i] + (W_IN_OUT ? second : 16));
            }
        }
#pragma unroll
        for (int i = 0; i < C::RO; ++i) offR[i] += KD * 4;
#pragma unroll
        for (int i = 0; i < C::FO; ++i) offF[i] += stepF;
    };

    f32x16 acc[C::FB][C::RB];
    zero_acc(acc);
    const bool busy = wr * 32 * C::RB < rows && n0 + wf * 32 * C::FB < N;     // the others have no row or no column of the tile
    multiply_stages<C, W_IN_OUT, false>((K + KD - 1) / KD, busy, smem, sWhole, tid, acc, load);
    constexpr bool COLSUM_OK = C::BM == HEXA_TILE_ROWS && C::WR == 2;
    const bool colsum = COLSUM_OK && p.colsum != nullptr;
    if (!combine<C>(smem, kg, wave, lane, acc) || (!busy && !colsum)) return;

    float cs[COLSUM_OK ? 16 * C::FB : 1];
#pragma unroll
    for (float& c : cs) c = 0.f;
    const bool to_ws = p.ws != nullptr && s > 0;
    float* const outp = to_ws ? p.ws : p.out;
    const bool accumulate = p.accumulate && !to_ws;
    const size_t row0 = to_ws ? (size_t)p.T * (s - 1) : (size_t)p.out_slot_rows * s;
#pragma unroll
    for (int i = 0; i < C::RB; ++i) {
        const int tok = sTok[(wr * C::RB + i) * 32 + (lane & 31)];
        if (tok < 0 || !busy) continue;
#pragma unroll
        for (int j = 0; j < C::FB; ++j) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = n0 + (wf * C::FB + j) * 32 + 8 * g + 4 * (lane >> 5);
                if (n >= N) continue;
                float4 v = make_float4(acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]);
                if (p.bias) {
                    const float4 b = *reinterpret_cast<const float4*>(p.bias + (size_t)e * N + n);
                    v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
                }
                const size_t off = (row0 + tok) * N + n;
                if (p.act == HEXA_ACT_GELU_BWD) {
                    const float4 y = *reinterpret_cast<const float4*>(p.out_act + off);
                    v.x *= gelu_grad_full(y.x); v.y *= gelu_grad_full(y.y); v.z *= gelu_grad_full(y.z); v.w *= gelu_grad_full(y.w);
                }
                float4* dst = reinterpret_cast<float4*>(outp + off);
                if (accumulate) {
                    const float4 old = *dst;
                    v.x += old.x; v.y += old.y; v.z += old.z; v.w += old.w;
                }
                if (!p.act_only) *dst = v;
                if constexpr (COLSUM_OK) {
                    float* const c = cs + j * 16 + 4 * g;
                    c[0] += v.x; c[1] += v.y; c[2] += v.z; c[3] += v.w;
                }
                if (p.act == HEXA_ACT_GELU)
                    *reinterpret_cast<float4*>(p.out_act + off) = make_float4(gelu_full(v.x), gelu_full(v.y), gelu_full(v.z), gelu_full(v.w));
            }
        }
    }
    // Column sums of the tile: the 32 lanes of a row block, then the two wavefronts of a column block.
    if constexpr (COLSUM_OK) {
        if (colsum) {
            __shared__ float sums[2][BN];
#pragma unroll
            for (float& c : cs)
#pragma unroll
                for (int m = 16; m > 0; m >>= 1) c += __shfl_xor(c, m);
            if ((lane & 31) == 0) {
#pragma unroll
                for (int c = 0; c < 16 * C::FB; ++c) sums[wr][(wf * C::FB + (c >> 4)) * 32 + 8 * ((c >> 2) & 3) + 4 * (lane >> 5) + (c & 3)] = cs[c];
            }
            __syncthreads();
            if (tid < BN) p.colsum[(((size_t)s * p.mt_ub + mt) * p.ntn + nt) * BN + tid] = sums[0][tid] + sums[1][tid];
        }
    }
}

struct Estmm32K {
    const float* pm; const float* qm; float* dw; float* scratch;
    const int32_t* token_ids; const int32_t* offsets;
    int T, k, E, M, N, mtn, ntn, parts;
    int p_slot_rows, q_slot_rows;
    int accumulate, group;
    long total;
};

template <bool BIG, typename C>
__global__ __launch_bounds__(C::NT, C::WAVES) void estmm32_kernel(Estmm32K p) {
    constexpr int BM = C::BM, BN = C::BN, KD = C::KD;
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    __shared__ int sLoad[256], sExpert, sWhole[2];

    const long logical = logical_tile(blockIdx.x, p.group);
    if (logical >= p.total) return;
    const int tiles = p.mtn * p.ntn;
    const int unit = (int)(logical / tiles), rem = (int)(logical - (long)unit * tiles);
    const int rank = unit / p.parts, part = unit - rank * p.parts;
    const int m0 = (rem / p.ntn) * BM, n0 = (rem % p.ntn) * BN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), kg = wave / (C::WR * C::WF), wr = wave / C::WF % C::WR, wf = wave % C::WF;
    const int M = p.M, N = p.N, E = p.E;

    // Heaviest expert first (workgroups are dispatched in id order), up to 256 experts; beyond that by index.
    int e = rank;
    if (E <= 256) {
        if (tid < E) {
            int t = 0;
            for (int s = 0; s < p.k; ++s) t += p.offsets[(size_t)s * (E + 1) + tid + 1] - p.offsets[(size_t)s * (E + 1) + tid];
            sLoad[tid] = t;
        }
        __syncthreads();
        if (tid < E) {
            const int mine = sLoad[tid];
            int r = 0;
            for (int x = 0; x < E; ++x) r += (sLoad[x] > mine || (sLoad[x] == mine && x < tid)) ? 1 : 0;
            if (r == rank) sExpert = tid;
        }
        __syncthreads();
        e = __builtin_amdgcn_readfirstlane(sExpert);
    }
    // The expert's steps of KD list entries, slot after slot (the last step of a slot's list may be partial), and this
    // workgroup's part of them.
    auto begin = [&](int s) { return p.offsets[(size_t)s * (E + 1) + e]; };
    auto end = [&](int s) { return p.offsets[(size_t)s * (E + 1) + e + 1]; };
    int all_steps = 0;
    for (int s = 0; s < p.k; ++s) all_steps += (end(s) - begin(s) + KD - 1) / KD;
    const int step0 = (int)((long)all_steps * part / p.parts);
    const int nk = (int)((long)all_steps * (part + 1) / p.parts) - step0;
    if (p.parts == 1 && p.accumulate && nk == 0) return;

    struct Cursor { int s, r, end; };           // position in the list of slot s
    auto seek = [&](Cursor c) {
        while (c.s < p.k && c.r >= c.end) {
            ++c.s;
            if (c.s < p.k) { c.r = begin(c.s); c.end = end(c.s); }
        }
        return c;
    };
    Cursor ids = seek(Cursor{0, begin(0), end(0)});
    for (int skip = step0; skip > 0 && ids.s < p.k;) {
        const int here = (ids.end - ids.r + KD - 1) / KD, take = min(here, skip);
        ids.r += take * KD;
        skip -= take;
        ids = seek(ids);
    }

    // Token ids are fetched a step before the rows they name.  Columns past the result's edge re-read the first ones of a row:
    // what they produce is never stored.  Rows past the end of a list are zeros in both operands.
    using Off = std::conditional_t<BIG, size_t, unsigned>;
    using PR = Place<true, BM, KD, C::NT>;
    using PF = Place<true, BN, KD, C::NT>;
    int idR[C::RO], idF[C::FO];
    Cursor rows = ids;
    auto fetch_ids = [&]() {
#pragma unroll
        for (int i = 0; i < C::RO; ++i) {
            const int r = ids.r + PR::row_of(tid, i);
            idR[i] = ids.s < p.k && r < ids.end ? p.token_ids[(size_t)ids.s * p.T + r] : 0;
        }
#pragma unroll
        for (int i = 0; i < C::FO; ++i) {
            const int r = ids.r + PF::row_of(tid, i);
            idF[i] = ids.s < p.k && r < ids.end ? p.token_ids[(size_t)ids.s * p.T + r] : 0;
        }
        rows = ids;
        if (ids.s < p.k) { ids.r += KD; ids = seek(ids); }
    };
    const int mR = m0 + PR::piece_of(tid) * 8, nF = n0 + PF::piece_of(tid) * 8;
    const unsigned colR = mR < M ? mR * 4u : 0u, colF = nF < N ? nF * 4u : 0u;
    const unsigned secondR = mR + 4 < M ? 16u : 0u, secondF = nF + 4 < N ? 16u : 0u;
    const Off pitchR = (Off)M * 4, pitchF = (Off)N * 4;
    auto read4 = [](const char* base, Off off) { return *reinterpret_cast<const f32x4*>(base + (size_t)off); };
    if (nk > 0) fetch_ids();
    auto load = [&](int step, Octet (&r)[C::RO], Octet (&f)[C::FO]) {
        const char* const pb = reinterpret_cast<const char*>(p.pm) + (size_t)p.p_slot_rows * rows.s * M * 4;
        const char* const qb = reinterpret_cast<const char*>(p.qm) + (size_t)p.q_slot_rows * rows.s * N * 4;
        const int left = rows.end - rows.r;
        Off offR[C::RO], offF[C::FO];
#pragma unroll
        for (int i = 0; i < C::RO; ++i) offR[i] = (Off)(unsigned)idR[i] * pitchR + colR;
#pragma unroll
        for (int i = 0; i < C::FO; ++i) offF[i] = (Off)(unsigned)idF[i] * pitchF + colF;
        if (left >= KD) {
#pragma unroll
            for (int i = 0; i < C::RO; ++i) { r[i].a = read4(pb, offR[i]); r[i].b = read4(pb, offR[i] + secondR); }
#pragma unroll
            for (int i = 0; i < C::FO; ++i) { f[i].a = read4(qb, offF[i]); f[i].b = read4(qb, offF[i] + secondF); }
        } else {
            const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int i = 0; i < C::RO; ++i) {
                r[i].a = zero; r[i].b = zero;
                if (PR::row_of(tid, i) < left) { r[i].a = read4(pb, offR[i]); r[i].b = read4(pb, offR[i] + secondR); }
            }
#pragma unroll
            for (int i = 0; i < C::FO; ++i) {
                f[i].a = zero; f[i].b = zero;
                if (PF::row_of(tid, i) < left) { f[i].a = read4(qb, offF[i]); f[i].b = read4(qb, offF[i] + secondF); }
            }
        }
        if (step + 1 < nk) fetch_ids();
    };

    f32x16 acc[C::FB][C::RB];
    zero_acc(acc);
    const bool busy = m0 + wr * 32 * C::RB < M && n0 + wf * 32 * C::FB < N;
    multiply_stages<C, true, true>(nk, busy, smem, sWhole, tid, acc, load);
    if (!combine<C>(smem, kg, wave, lane, acc)) return;

    const bool alone = p.parts == 1;
    float* const dst0 = alone ? p.dw + (size_t)e * M * N : p.scratch + ((size_t)part * E + e) * M * N;
#pragma unroll
    for (int i = 0; i < C::RB; ++i) {
        const int m = m0 + (wr * C::RB + i) * 32 + (lane & 31);
        if (m >= M) continue;
#pragma unroll
        for (int j = 0; j < C::FB; ++j) {
#pragma unroll
            for (int g = 0; g < 4; ++g) {
                const int n = n0 + (wf * C::FB + j) * 32 + 8 * g + 4 * (lane >> 5);
                if (n >= N) continue;
                float4 v = make_float4(acc[j][i][4 * g], acc[j][i][4 * g + 1], acc[j][i][4 * g + 2], acc[j][i][4 * g + 3]);
                float4* dst = reinterpret_cast<float4*>(dst0 + (size_t)m * N + n);
                if (alone && p.accumulate) {
                    const float4 old = *dst;
                    v.x += old.x; v.y += old.y; v.z += old.z; v.w += old.w;
                }
                *dst = v;
            }
        }
    }
}

template <bool IO, bool BIG, typename C> int launch_esmm32_t(Esmm32K& p, hipStream_t st) {
    p.ntn = div_up(p.N, C::BN);
    const long tiles = (long)p.nslots * p.mt_ub * (HEXA_TILE_ROWS / C::BM) * p.ntn;
    auto kernel = esmm32_kernel<IO, BIG, C>;
    if (int rc = ensure_smem(kernel, C::BYTES)) return rc;
    hipLaunchKernelGGL(kernel, dim3(round_up(tiles, 8)), dim3(C::NT), C::BYTES, st, p);
    HEXA_CHECK_LAUNCH("esmm32");
    return HEXA_OK;
}
template <bool BIG, typename C> int launch_estmm32_t(Estmm32K& p, hipStream_t st) {
    p.mtn = div_up(p.M, C::BM); p.ntn = div_up(p.N, C::BN);
    p.group = p.ntn;
    p.total = (long)p.E * p.parts * p.mtn * p.ntn;
    auto kernel = estmm32_kernel<BIG, C>;
    if (int rc = ensure_smem(kernel, C::BYTES)) return rc;
    hipLaunchKernelGGL(kernel, dim3(round_up(p.total, 8 * p.group)), dim3(C::NT), C::BYTES, st, p);
    HEXA_CHECK_LAUNCH("estmm32");
    return HEXA_OK;
}
// whether byte offsets into rows x cols floats (and a stage beyond) need more than 32 bits
bool too_large(size_t rows, size_t cols) { return (rows + 64) * cols * 4 >= ((size_t)1 << 32); }

}  // namespace

// 128 x 128 tiles where they come to one for most CUs and the lists fill them: 3000 rows, 1024 -> 2048, 4 experts 101
// against 125 us of 64 x 64 tiles, 23 x 8 tiles of its fc2 124 against 139, 8192 rows, 2048 -> 512 (64 x 4) 160 both; 64
// rows an expert 49 against 44, 4000 rows, 2048 -> 512 (31 x 4 tiles) 117 against 101
static bool esmm32_wide(const EsmmArgs& a, int slots) {
    return (long)slots * a.r.T / 128 * div_up(a.out_dim, 128) >= 180 && a.r.T >= 100 * a.r.E;
}
// Column sums come from the store loop of the 128 x 128 tiles, all slots in one launch: 9216 rows, top-2 of 8 experts, 384 x 1536, a
// pass over the stored result takes 21.5 us.
bool esmm32_colsum_supported(const EsmmArgs& a) {
    return a.act == HEXA_ACT_GELU_BWD && a.out_per_slot && a.r.k <= 8 && a.in_dim % 4 == 0 && a.out_dim % 4 == 0 && esmm32_wide(a, a.r.k);
}

int launch_esmm32(const EsmmArgs& a, hipStream_t st) {
    if ((a.in_dim & 3) || (a.out_dim & 3))
        HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "esmm (fp32): in_dim and out_dim must be multiples of 4 (got %d, %d)",
                  a.in_dim, a.out_dim);
    Esmm32K p;
    p.x = (const float*)a.x; p.w = (const float*)a.w; p.bias = (const float*)a.bias;
    p.out = (float*)a.out; p.out_act = (float*)a.out_act;
    p.token_ids = a.r.token_ids; p.tile_info = a.r.tile_info; p.tile_count = a.r.tile_count;
    p.T = a.r.T; p.K = a.in_dim; p.N = a.out_dim; p.mt_ub = a.r.mt_ub;
    p.x_slot_rows = a.x_per_slot ? a.r.T : 0;
    p.out_slot_rows = a.out_per_slot ? a.r.T : 0;
    p.act = a.act; p.act_only = a.act_only; p.colsum = a.colsum;
    // Summing the slots into one result: with scratch every slot runs in one launch (slot 0 into `out`, the others into
    // the scratch) and a small kernel adds them; without, one launch per slot adds into `out`.
    const bool sum = !a.out_per_slot && a.r.k > 1;
    p.ws = sum ? (float*)a.slot_ws : nullptr;
    const int per_launch = sum && !p.ws ? 1 : 8;
    for (int s = 0; s < a.r.k; s += per_launch) {
        p.slot_begin = s;
        p.nslots = std::min(per_launch, a.r.k - s);
        p.accumulate = (a.accumulate || (sum && !p.ws && s > 0)) ? 1 : 0;
        if (p.mt_ub == 0) continue;
        const bool io = a.w_layout == HEXA_W_IN_OUT;
        const bool big = too_large((size_t)a.r.T * (a.x_per_slot ? a.r.k : 1), a.in_dim) || too_large(a.in_dim, a.out_dim);
        const bool wide = esmm32_wide(a, p.nslots);
        auto go = [&](auto bg) {
            constexpr bool BIG = decltype(bg)::value;
            return wide ? (io ? launch_esmm32_t<true, BIG, Wide>(p, st) : launch_esmm32_t<false, BIG, Wide>(p, st))
                        : (io ? launch_esmm32_t<true, BIG, Deep>(p, st) : launch_esmm32_t<false, BIG, Deep>(p, st));
        };
        const int rc = big ? go(std::true_type()) : go(std::false_type());
        if (rc) return rc;
    }
    if (p.ws) return launch_sum_slots(a.out, a.slot_ws, a.r, a.out_dim, a.accumulate, HEXA_F32, st, a.sum_extra);
    if (a.colsum) return launch_colsum_fold(a, p.mt_ub, HEXA_TILE_ROWS, div_up(a.out_dim, Wide::BN), Wide::BN, st);
    return HEXA_OK;
}

// Tile and number of parts that every expert's token list is cut into.  Where 128 x 128 tiles come to two and more per CU they
// take whole lists.  With fewer, a launch is the walk over its longest list: such tiles cut lists of a thousand entries and
// more into parts, and below that 64 x 64 tiles until there are six workgroups per CU (or 128 entries a part).  Measured with
// one part of 64 x 64 tiles against this: 18432 entries, 8 experts, 1536 x 384 195 -> 178 us, 8192, 4, 2048 x 512 156 -> 133,
// 5000, 12, 800 x 200 72 -> 45; uncut 128 x 128 against 64 x 64 tiles at 12000, 32, 3072 x 768 402 against 537.
// The parts' scratch is 84 MB a result at the most: less than 768 + 512 blocks of 128 x 128 floats, or 2 * 1536 of 64 x 64.
static bool estmm32_wide(int T, int k, int E, int m_dim, int n_dim, int* parts) {
    const long t128 = (long)E * div_up(m_dim, 128) * div_up(n_dim, 128), t64 = (long)E * div_up(m_dim, 64) * div_up(n_dim, 64);
    const long avg = (long)T * k / std::max(1, E);
    const bool cut = t128 < 512 && avg >= 256, wide = t128 >= 512 || (t128 >= 200 && avg >= 1024);
    const long want = wide ? std::min<long>((768 + t128 - 1) / t128, avg / 256) : std::min<long>((1536 + t64 - 1) / t64, avg / 128);
    *parts = cut ? (int)std::max<long>(1, std::min<long>(8, want)) : 1;
    return wide;
}
int estmm32_parts(int T, int k, int E, int m_dim, int n_dim) {
    int parts;
    estmm32_wide(T, k, E, m_dim, n_dim, &parts);
    return parts;
}

int launch_estmm32(const EstmmArgs& a, hipStream_t st) {
    if ((a.m_dim & 3) || (a.n_dim & 3))
        HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "estmm (fp32): dims must be multiples of 4 (got %d, %d)", a.m_dim, a.n_dim);
    Estmm32K p;
    p.pm = (const float*)a.p; p.qm = (const float*)a.q; p.dw = (float*)a.dw; p.scratch = a.scratch;
    p.token_ids = a.r.token_ids; p.offsets = a.r.offsets;
    p.T = a.r.T; p.k = a.r.k; p.E = a.r.E; p.M = a.m_dim; p.N = a.n_dim;
    p.p_slot_rows = a.p_per_slot ? a.r.T : 0;
    p.q_slot_rows = a.q_per_slot ? a.r.T : 0;
    p.accumulate = a.accumulate;
    int parts;
    const bool wide = estmm32_wide(p.T, p.k, p.E, p.M, p.N, &parts) && !(parts > 1 && !a.scratch);
    p.parts = a.scratch ? std::max(1, std::min(parts, a.max_slots / p.E)) : 1;
    const bool big = too_large((size_t)p.T * (a.p_per_slot ? p.k : 1), p.M) || too_large((size_t)p.T * (a.q_per_slot ? p.k : 1), p.N);
    const int rc = big ? (wide ? launch_estmm32_t<true, Wide>(p, st) : launch_estmm32_t<true, Deep>(p, st))
                       : (wide ? launch_estmm32_t<false, Wide>(p, st) : launch_estmm32_t<false, Deep>(p, st));
    if (rc) return rc;
    return p.parts > 1 ? launch_fold(a.dw, a.scratch, (long)p.E * p.M * p.N, p.parts, HEXA_F32, a.accumulate, st) : HEXA_OK;
}

}  // namespace hexa
