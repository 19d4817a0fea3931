// ESMM and ESTMM in true fp32 on gfx950: v_mfma_f32_32x32x2_f32 (fp32 multiply, fp32 accumulate).  Unlike the
// reference, which rounds fp32 operands to fp16 before its WMMA (kernels/esmm_full.cu:128-130,167-169), nothing is
// rounded, so results agree with an fp32 matmul to ~1e-6.
//
// What bounds these kernels is the matrix pipeline: one such MFMA is 64 cycles for 4096 flop (131-145 TFLOP/s over the
// chip from registers, the clock falling with random operands).  A 64 x 64 tile's 32 contraction indices are 1024 cycles
// of each SIMD against 16 KB copied, so copies and LDS reads have time -- if they do not stand between the MFMAs:
//   * four wavefronts multiply (32 x 32 each) and four copy: tiles stream into LDS with the asynchronous copy
//     (global_load_lds_dwordx4), two or three stages, one barrier per stage;
//   * a multiplying wavefront reads half a stage while the MFMAs of the other half run, also across that barrier;
//   * tiles are small and three or four workgroups share a CU, so that one's start and end meet another's MFMAs and
//     256 CUs finish together; all routing slots of a slot-summed result run in one launch; an ESTMM with few tiles is
//     cut along its token lists.
// Measured at 9216 tokens, 384 -> 1536, 8 experts, top-2 (21.7 GFLOP a launch; before: 128 x 128 tiles through registers,
// two barriers per 16 indices, one launch per slot): fc1 + GELU 257 -> 237 us, fc2 465 -> 199, dW 446 -> 227, dy1 348 -> 242,
// dx 479 -> 197, and at 2048 tokens, 128 -> 512 28 -> 11, 58 -> 16, 92 -> 18 us.  128 x 64 tiles, copies issued between the
// MFMAs by the multiplying wavefronts, and one persistent workgroup pair per CU were measured too: 0 to 15 % slower.
//
// LDS tile formats (a stage holds 32 contraction indices):
//   KC  contraction index fastest in memory: [row][32 k], 128 B per row.  The MFMA takes one contraction index per
//       half-wavefront, and WHICH two indices it pairs is free: lanes 0..31 take k = 8g + j and lanes 32..63
//       k = 8g + 4 + j, so a lane's four indices of a group are one ds_read_b128.  16-byte piece p of a row sits at
//       position p ^ ((row >> 1) & 7): sixteen consecutive rows cover all 64 banks.
//   KS  contraction index slowest in memory: [32 k][W columns].  Lanes read single floats, two rows of k per
//       ds_read2st64_b32.  Piece ch of row k sits at ch ^ (8 * ((k >> 2) & 1)): the two half-wavefronts, four rows of k
//       apart, use different halves of the banks.
// The copy engine places lane i at LDS offset 16*i, so both swizzles choose which piece a lane fetches.
//
// Replaces esmm_shared_tensor_kernel_vectorized_accum_full (kernels/esmm_full.cu:58-246) and the
// ESMM / ESTMM tasks of fused_grad_*_kernel_vectorized_full (kernels/fused_ops_full.cu:117-371).
#include <algorithm>

#include "dma_common.h"
#include "small_bodies.h"

namespace hexa {
namespace {

constexpr int KD = 32;                  // contraction indices per stage
constexpr int NT = 512;                 // 2 x 2 wavefronts that multiply and four that copy
typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;

constexpr int BM = 64, BN = 64;         // workgroup tile: one 32 x 32 block per multiplying wavefront
constexpr int OPERAND_BYTES = 64 * KD * 4, STAGE_BYTES = 2 * OPERAND_BYTES;
constexpr int R_CPW = 2, CPW = 4;       // copies per wavefront and stage: two of each operand
// stages, and the wavefronts per SIMD the registers are sized for
template <int STAGES_, int WAVES_> struct Depth { static constexpr int STAGES = STAGES_, WAVES = WAVES_; };
using Deep = Depth<3, 6>;               // 48 KB: three workgroups per CU
using Many = Depth<2, 8>;               // 32 KB: four

// LDS reads in inline assembly: the compiler would order plain ones behind the copies in flight (see dma_common.h);
// not usable before frag_fence().
__device__ __forceinline__ f32x4 lds_read_f4(unsigned addr) {
    f32x4 r;
    asm volatile("ds_read_b128 %0, %1" : "=v"(r) : "v"(addr));
    return r;
}
template <int A, int B> __device__ __forceinline__ f32x2 lds_read_2f(unsigned addr) {   // units of 256 bytes
    f32x2 r;
    asm volatile("ds_read2st64_b32 %0, %1 offset0:%2 offset1:%3" : "=v"(r) : "v"(addr), "n"(A), "n"(B));
    return r;
}

// One 32-wide block of an operand for half a stage (HALF 0: k = 0..15, HALF 1: k = 16..31): at(g, j) is this lane's value
// for k = 16 HALF + 8g + 4(lane >> 5) + j.
struct FragKC {
    f32x4 v[2];
    // lane part of the address of group g of a stage
    static __device__ __forceinline__ unsigned lane_addr(int lane, int g) {
        const int row = lane & 31;
        return row * 128 + (((2 * g + (lane >> 5)) ^ ((row >> 1) & 7)) << 4);
    }
    template <int HALF> __device__ __forceinline__ void read(const unsigned (&la)[4], unsigned base) {
#pragma unroll
        for (int g = 0; g < 2; ++g) v[g] = lds_read_f4(la[2 * HALF + g] + base);
    }
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int g = 0; g < 2; ++g) asm volatile("" : "+v"(v[g]));
    }
    __device__ __forceinline__ float at(int g, int j) const { return v[g][j]; }
};
struct FragKS {                   // 64 columns per row of k: 256 bytes
    f32x2 v[2][2];
    static __device__ __forceinline__ unsigned lane_addr(int lane, int col0) {
        const int kh = lane >> 5, col = col0 + (lane & 31);
        return kh * 4 * 256 + ((((col >> 2) ^ (8 * kh)) << 4) | ((col & 3) << 2));
    }
    template <int HALF> __device__ __forceinline__ void read(unsigned addr) {
        constexpr int K0 = 16 * HALF;
        v[0][0] = lds_read_2f<K0, K0 + 1>(addr);      v[0][1] = lds_read_2f<K0 + 2, K0 + 3>(addr);
        v[1][0] = lds_read_2f<K0 + 8, K0 + 9>(addr);  v[1][1] = lds_read_2f<K0 + 10, K0 + 11>(addr);
    }
    __device__ __forceinline__ void pin() {
#pragma unroll
        for (int g = 0; g < 2; ++g) {
            asm volatile("" : "+v"(v[g][0]));
            asm volatile("" : "+v"(v[g][1]));
        }
    }
    __device__ __forceinline__ float at(int g, int j) const { return v[g][j >> 1][j & 1]; }
};
// half a stage of both operands: a wavefront's columns (F) and rows (R)
template <typename F, typename R> struct Half {
    F f;
    R r;
    __device__ __forceinline__ void fence() {        // the reads have returned; nothing that uses them moves ahead of this
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        f.pin();
        r.pin();
    }
    // acc (+)= F x R: a lane ends up with row lane%32 of R and, per group of four registers, 4 consecutive columns of F
    __device__ __forceinline__ void multiply(f32x16& acc) const {
#pragma unroll
        for (int g = 0; g < 2; ++g)
#pragma unroll
            for (int k = 0; k < 4; ++k) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(f.at(g, k), r.at(g, k), acc, 0, 0, 0);
    }
};
// A multiplying wavefront's nk stages of a tile.  load0 / load1(h) issue the reads of the current stage's halves, advance()
// makes the next stage the current one.  The half that follows is read while the MFMAs of the one before run, also across
// the barrier behind which the next stage may be read (and this one overwritten).
template <typename P, typename L0, typename L1, typename A>
__device__ __forceinline__ void multiply_stages(int nk, bool busy, f32x16& acc, L0 load0, L1 load1, A advance) {
    if (!busy) {
        for (int kt = 0; kt < nk; ++kt) { barrier_nofence(); advance(); }
        return;
    }
    P a, b;
    barrier_nofence();
    load0(a);
    for (int kt = 0; kt < nk; ++kt) {
        a.fence();
        load1(b);
        __builtin_amdgcn_sched_barrier(0);
        a.multiply(acc);
        __builtin_amdgcn_sched_barrier(0);
        b.fence();
        advance();
        if (kt + 1 < nk) {
            barrier_nofence();
            load0(a);
        }
        __builtin_amdgcn_sched_barrier(0);
        b.multiply(acc);
        __builtin_amdgcn_sched_barrier(0);
    }
}

// which piece a lane fetches in wavefront copy c: KC (8 rows per copy), KS (4 rows of k per copy)
__device__ __forceinline__ void kc32_lane(int c, int lane, int& row, int& piece) {
    row = 8 * c + (lane >> 3);
    piece = (lane & 7) ^ ((row >> 1) & 7);
}
__device__ __forceinline__ void ks32_lane(int c, int lane, int& kk, int& piece) {
    kk = 4 * c + (lane >> 4);
    piece = (lane & 15) ^ (8 * ((kk >> 2) & 1));
}

struct Esmm32K {
    const float* x; const float* w; const float* bias; float* out; float* out_act; float* ws;
    const int32_t* token_ids; const int4* tile_info; const int32_t* tile_count;
    int T, K, N, mt_ub, ntn, slot_begin, nslots;
    int x_slot_rows, out_slot_rows;
    int accumulate, act;
};

template <bool W_IN_OUT, bool WIDE, typename S>
__global__ __launch_bounds__(NT, S::WAVES) void esmm32_kernel(Esmm32K p) {
    constexpr int STAGES = S::STAGES, H = HEXA_TILE_ROWS / BM;   // H workgroup tiles per row tile of the routing
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    __shared__ int sTok[BM];

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
    const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3, wr = wave >> 1, wf = wave & 1;
    const bool copies = wave8 >= 4;
    const int K = p.K, N = p.N;
    if (tid < BM) sTok[tid] = tid < rows ? p.token_ids[(size_t)s * p.T + row_start + tid] : -1;
    __syncthreads();

    // Sources of this lane's copies: bases every lane shares plus 32-bit byte offsets (64-bit ones where an operand has
    // 4 GiB and more): a copy whose address is one register beside a scalar pair disturbs the MFMAs of the SIMD's other
    // wavefronts far less.  Lanes with nothing to fetch (rows past the tile's end, columns past N) re-read the first bytes
    // of the tensor: what they produce is never stored.  Contraction indices past K come from a block of zeros, in both
    // operands.
    using Off = std::conditional_t<WIDE, size_t, unsigned>;
    const char* const xbase = reinterpret_cast<const char*>(p.x);
    const char* const wbase = reinterpret_cast<const char*>(p.w + (size_t)e * K * N);
    Off off[CPW];
    int kOf[CPW];                              // the stage's contraction index the lane fetches
#pragma unroll
    for (int i = 0; i < CPW; ++i) {
        int row, piece;
        if (i < R_CPW) {
            kc32_lane(wave + 4 * i, lane, row, piece);
            const int tok = max(sTok[row], 0);
            kOf[i] = piece * 4;
            off[i] = (Off)((((size_t)p.x_slot_rows * s + tok) * K + piece * 4) * 4);
        } else if (W_IN_OUT) {
            ks32_lane(wave + 4 * (i - R_CPW), lane, row, piece);
            const int n = n0 + piece * 4;
            kOf[i] = row;
            off[i] = (Off)(((size_t)row * N + (n < N ? n : 0)) * 4);
        } else {
            kc32_lane(wave + 4 * (i - R_CPW), lane, row, piece);
            const int n = n0 + row;
            kOf[i] = piece * 4;
            off[i] = (Off)(((size_t)(n < N ? n : 0) * K + piece * 4) * 4);
        }
    }
    const Off stepF = W_IN_OUT ? (Off)KD * N * 4 : (Off)KD * 4;
    const int nk = (K + KD - 1) / KD;
    auto target = [&](int step, int i) {
        return smem + (step % STAGES) * STAGE_BYTES + (i < R_CPW ? (wave + 4 * i) * 1024 : OPERAND_BYTES + (wave + 4 * (i - R_CPW)) * 1024);
    };
    auto copy = [&](int step, int i) {            // copy i of a step that lies inside the contraction
        dma16((i < R_CPW ? xbase : wbase) + (size_t)off[i], target(step, i));
        off[i] += i < R_CPW ? (Off)(KD * 4) : stepF;
    };
    auto issue = [&](int step) {
        const int left = K - step * KD;
#pragma unroll
        for (int i = 0; i < CPW; ++i) {
            if (left >= KD) copy(step, i);
            else dma16(kOf[i] < left ? (i < R_CPW ? xbase : wbase) + (size_t)off[i] : reinterpret_cast<const char*>(g_zero_block), target(step, i));
        }
    };

    if (copies) {
#pragma unroll
        for (int st = 0; st < STAGES - 1; ++st)
            if (st < nk) issue(st);
        for (int kt = 0; kt < nk; ++kt) {
            wait_groups<CPW, STAGES - 2>(min(nk - 1 - kt, STAGES - 2));
            barrier_nofence();      // the copies of step kt are in LDS, and everyone is done reading step kt - 1
            if (kt + STAGES - 1 < nk) issue(kt + STAGES - 1);
        }
        return;
    }

    f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    const bool busy = wr * 32 < rows && n0 + wf * 32 < N;     // the others have no row or no column of the tile
    const unsigned lds0 = lds_addr(smem);
    unsigned la[4], ksF = 0, stage_at = lds0;
#pragma unroll
    for (int g = 0; g < 4; ++g) la[g] = FragKC::lane_addr(lane, g);
    if (W_IN_OUT) ksF = FragKS::lane_addr(lane, wf * 32);
    using Pair = Half<std::conditional_t<W_IN_OUT, FragKS, FragKC>, FragKC>;
    auto load = [&](Pair& h, auto half) {
        constexpr int HALF = decltype(half)::value;
        h.r.template read<HALF>(la, stage_at + wr * 32 * 128);
        if constexpr (W_IN_OUT) h.f.template read<HALF>(ksF + stage_at + OPERAND_BYTES);
        else h.f.template read<HALF>(la, stage_at + OPERAND_BYTES + wf * 32 * 128);
    };
    multiply_stages<Pair>(nk, busy, acc, [&](Pair& h) { load(h, std::integral_constant<int, 0>()); },
                          [&](Pair& h) { load(h, std::integral_constant<int, 1>()); },
                          [&]() { stage_at = stage_at + STAGE_BYTES == lds0 + STAGES * STAGE_BYTES ? lds0 : stage_at + STAGE_BYTES; });
    if (!busy) return;

    const int tok = sTok[wr * 32 + (lane & 31)];
    if (tok < 0) return;
    const bool to_ws = p.ws != nullptr && s > 0;
    float* const outp = to_ws ? p.ws : p.out;
    const bool accumulate = p.accumulate && !to_ws;
    const size_t row0 = to_ws ? (size_t)p.T * (s - 1) : (size_t)p.out_slot_rows * s;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int n = n0 + wf * 32 + 8 * g + 4 * (lane >> 5);
        if (n >= N) continue;
        float4 v = make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
        if (p.bias) {
            const float4 b = *reinterpret_cast<const float4*>(p.bias + (size_t)e * N + n);
            v.x += b.x; v.y += b.y; v.z += b.z; v.w += b.w;
        }
        const size_t off = (row0 + tok) * N + n;
        if (p.act == HEXA_ACT_GELU_BWD) {
            const float4 y = *reinterpret_cast<const float4*>(p.out_act + off);
            v.x *= gelu_grad_erf(y.x); v.y *= gelu_grad_erf(y.y); v.z *= gelu_grad_erf(y.z); v.w *= gelu_grad_erf(y.w);
        }
        float4* dst = reinterpret_cast<float4*>(outp + off);
        if (accumulate) {
            const float4 old = *dst;
            v.x += old.x; v.y += old.y; v.z += old.z; v.w += old.w;
        }
        *dst = v;
        if (p.act == HEXA_ACT_GELU)
            *reinterpret_cast<float4*>(p.out_act + off) = make_float4(gelu_erf(v.x), gelu_erf(v.y), gelu_erf(v.z), gelu_erf(v.w));
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

constexpr int RING = 8;      // steps whose token ids are in LDS (32 each)

template <bool WIDE, typename S>
__global__ __launch_bounds__(NT, S::WAVES) void estmm32_kernel(Estmm32K p) {
    constexpr int STAGES = S::STAGES, LEAD = STAGES - 1;
    static_assert(2 * LEAD <= RING, "ids are fetched LEAD steps ahead of the copies that need them");
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    __shared__ int sIds[RING * 32], sLoad[256], sExpert;

    const long logical = logical_tile(blockIdx.x, p.group);
    if (logical >= p.total) return;
    const int tiles = p.mtn * p.ntn;
    const int unit = (int)(logical / tiles), rem = (int)(logical - (long)unit * tiles);
    const int rank = unit / p.parts, part = unit - rank * p.parts;
    const int m0 = (rem / p.ntn) * BM, n0 = (rem % p.ntn) * BN;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave8 = __builtin_amdgcn_readfirstlane(tid >> 6), wave = wave8 & 3, wr = wave >> 1, wf = wave & 1;
    const bool copies = wave8 >= 4;
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
    // The expert's steps of 32 list entries, slot after slot (the last step of a slot's list may be partial), and this
    // workgroup's part of them.
    auto begin = [&](int s) { return p.offsets[(size_t)s * (E + 1) + e]; };
    auto end = [&](int s) { return p.offsets[(size_t)s * (E + 1) + e + 1]; };
    int all_steps = 0;
    for (int s = 0; s < p.k; ++s) all_steps += (end(s) - begin(s) + KD - 1) / KD;
    const int step0 = (int)((long)all_steps * part / p.parts);
    const int nk = (int)((long)all_steps * (part + 1) / p.parts) - step0;
    if (p.parts == 1 && p.accumulate && nk == 0) return;

    if (copies) {
        struct Cursor { int s, r, end; };           // position in the list of slot s
        auto seek = [&](Cursor c) {
            while (c.s < p.k && c.r >= c.end) {
                ++c.s;
                if (c.s < p.k) { c.r = begin(c.s); c.end = end(c.s); }
            }
            return c;
        };
        auto advance = [&](Cursor c) { c.r += KD; return seek(c); };
        Cursor start{0, begin(0), end(0)};
        start = seek(start);
        for (int skip = step0; skip > 0 && start.s < p.k;) {
            const int here = (start.end - start.r + KD - 1) / KD, take = min(here, skip);
            start.r += take * KD;
            skip -= take;
            start = seek(start);
        }
        // the stage's token a lane fetches from and the byte in its row (columns past the result's edge re-read the row's
        // first bytes: what they produce is never stored)
        using Off = std::conditional_t<WIDE, size_t, unsigned>;
        int tokOf[CPW];
        unsigned colOf[CPW];
#pragma unroll
        for (int i = 0; i < CPW; ++i) {
            int piece;
            if (i < R_CPW) ks32_lane(wave + 4 * i, lane, tokOf[i], piece);
            else ks32_lane(wave + 4 * (i - R_CPW), lane, tokOf[i], piece);
            const int col = (i < R_CPW ? m0 : n0) + piece * 4;
            colOf[i] = col < (i < R_CPW ? M : N) ? (unsigned)col * 4 : 0u;
        }
        const Off pitchP = (Off)M * 4, pitchQ = (Off)N * 4;
        const unsigned ids_at = lds_addr(sIds);
        const char* const zero = reinterpret_cast<const char*>(g_zero_block);
        // every copying wavefront fetches the 32 ids of a step itself (the same words), so its own count of outstanding
        // copies says when they are there
        auto issue_ids = [&](int step, const Cursor& c) {
            const int r = c.r + (lane & 31);
            const void* src = c.s < p.k && r < c.end ? (const void*)(p.token_ids + (size_t)c.s * p.T + r) : (const void*)zero;
            if (lane < 32) __builtin_amdgcn_global_load_lds((glb_ptr_t)src, (lds_ptr_t)(sIds + (step % RING) * 32), 4, 0, 0);
        };
        auto issue = [&](int step, const Cursor& c) {
            char* base = smem + (step % STAGES) * STAGE_BYTES;
            int tok[CPW];
#pragma unroll
            for (int i = 0; i < CPW; ++i) tok[i] = lds_read_i32(ids_at + ((step % RING) * 32 + tokOf[i]) * 4);
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const char* const pb = reinterpret_cast<const char*>(p.pm) + (size_t)p.p_slot_rows * c.s * pitchP;
            const char* const qb = reinterpret_cast<const char*>(p.qm) + (size_t)p.q_slot_rows * c.s * pitchQ;
            const int left = c.end - c.r;
#pragma unroll
            for (int i = 0; i < CPW; ++i) {
                int t = tok[i];
                asm volatile("" : "+v"(t));
                char* to = base + (i < R_CPW ? (wave + 4 * i) * 1024 : OPERAND_BYTES + (wave + 4 * (i - R_CPW)) * 1024);
                const char* from = (i < R_CPW ? pb : qb) + (size_t)((Off)(unsigned)t * (i < R_CPW ? pitchP : pitchQ) + colOf[i]);
                if (left >= KD) dma16((i < R_CPW ? pb : qb) + (size_t)((Off)(unsigned)t * (i < R_CPW ? pitchP : pitchQ) + colOf[i]), to);
                else dma16(tokOf[i] < left ? from : zero, to);
            }
        };
        if (nk > 0) {
            // groups of CPW + 1 copies: the rows of a step, then the ids LEAD steps further on
            Cursor ids = start, rows = start;
            for (int st = 0; st < LEAD; ++st) { issue_ids(st, ids); ids = advance(ids); }
            wait_vmcnt<0>();
#pragma unroll
            for (int st = 0; st < LEAD; ++st) {
                if (st < nk) {
                    issue(st, rows); rows = advance(rows);
                    issue_ids(st + LEAD, ids); ids = advance(ids);
                }
            }
            for (int kt = 0; kt < nk; ++kt) {
                wait_groups<CPW + 1, LEAD - 1>(min(nk - 1 - kt, LEAD - 1));
                barrier_nofence();
                if (kt + LEAD < nk) {
                    issue(kt + LEAD, rows); rows = advance(rows);
                    issue_ids(kt + 2 * LEAD, ids); ids = advance(ids);
                }
            }
        }
        return;
    }

    f32x16 acc;
#pragma unroll
    for (int v = 0; v < 16; ++v) acc[v] = 0.f;
    const bool busy = m0 + wr * 32 < M && n0 + wf * 32 < N;
    if (nk > 0) {
        const unsigned lds0 = lds_addr(smem), laR = FragKS::lane_addr(lane, wr * 32), laF = FragKS::lane_addr(lane, wf * 32) + OPERAND_BYTES;
        unsigned stage_at = lds0;
        using Pair = Half<FragKS, FragKS>;
        auto load = [&](Pair& h, auto half) {
            constexpr int HALF = decltype(half)::value;
            h.r.template read<HALF>(laR + stage_at);
            h.f.template read<HALF>(laF + stage_at);
        };
        multiply_stages<Pair>(nk, busy, acc, [&](Pair& h) { load(h, std::integral_constant<int, 0>()); },
                              [&](Pair& h) { load(h, std::integral_constant<int, 1>()); },
                              [&]() { stage_at = stage_at + STAGE_BYTES == lds0 + STAGES * STAGE_BYTES ? lds0 : stage_at + STAGE_BYTES; });
    }
    const int m = m0 + wr * 32 + (lane & 31);
    if (m >= M) return;

    const bool whole = p.parts == 1;
    float* const dst0 = (whole ? p.dw + (size_t)e * M * N : p.scratch + ((size_t)part * E + e) * M * N) + (size_t)m * N;
#pragma unroll
    for (int g = 0; g < 4; ++g) {
        const int n = n0 + wf * 32 + 8 * g + 4 * (lane >> 5);
        if (n >= N) continue;
        float4 v = make_float4(acc[4 * g], acc[4 * g + 1], acc[4 * g + 2], acc[4 * g + 3]);
        float4* dst = reinterpret_cast<float4*>(dst0 + n);
        if (whole && p.accumulate) {
            const float4 old = *dst;
            v.x += old.x; v.y += old.y; v.z += old.z; v.w += old.w;
        }
        *dst = v;
    }
}

template <bool IO, bool WIDE, typename S> int launch_esmm32_t(const Esmm32K& p, hipStream_t st) {
    auto kernel = esmm32_kernel<IO, WIDE, S>;
    constexpr int bytes = S::STAGES * STAGE_BYTES;
    if (int rc = ensure_smem(kernel, bytes)) return rc;
    const long tiles = (long)p.nslots * p.mt_ub * (HEXA_TILE_ROWS / BM) * p.ntn;
    hipLaunchKernelGGL(kernel, dim3(round_up(tiles, 8)), dim3(NT), bytes, st, p);
    HEXA_CHECK_LAUNCH("esmm32");
    return HEXA_OK;
}

template <bool WIDE> int launch_estmm32_t(Estmm32K& p, hipStream_t st) {
    auto kernel = estmm32_kernel<WIDE, Deep>;
    constexpr int bytes = Deep::STAGES * STAGE_BYTES;
    if (int rc = ensure_smem(kernel, bytes)) return rc;
    p.mtn = div_up(p.M, BM); p.ntn = div_up(p.N, BN);
    p.group = p.ntn;
    p.total = (long)p.E * p.parts * p.mtn * p.ntn;
    hipLaunchKernelGGL(kernel, dim3(round_up(p.total, 8 * p.group)), dim3(NT), bytes, st, p);
    HEXA_CHECK_LAUNCH("estmm32");
    return HEXA_OK;
}

// whether byte offsets into rows x cols floats (and a stage beyond) need more than 32 bits
bool too_large(size_t rows, size_t cols) { return (rows + 64) * cols * 4 >= ((size_t)1 << 32); }

}  // namespace

int launch_esmm32(const EsmmArgs& a, hipStream_t st) {
    if ((a.in_dim & 3) || (a.out_dim & 3))
        HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "esmm (fp32): in_dim and out_dim must be multiples of 4 (got %d, %d)",
                  a.in_dim, a.out_dim);
    Esmm32K p;
    p.x = (const float*)a.x; p.w = (const float*)a.w; p.bias = (const float*)a.bias;
    p.out = (float*)a.out; p.out_act = (float*)a.out_act;
    p.token_ids = a.r.token_ids; p.tile_info = a.r.tile_info; p.tile_count = a.r.tile_count;
    p.T = a.r.T; p.K = a.in_dim; p.N = a.out_dim; p.mt_ub = a.r.mt_ub;
    p.ntn = div_up(a.out_dim, 64);
    p.x_slot_rows = a.x_per_slot ? a.r.T : 0;
    p.out_slot_rows = a.out_per_slot ? a.r.T : 0;
    p.act = a.act;
    // Summing the slots into one result: with scratch every slot runs in one launch (slot 0 into `out`, the others into
    // the scratch) and a small kernel adds them; without, one launch per slot adds into `out`.
    const bool sum = !a.out_per_slot && a.r.k > 1;
    p.ws = sum ? (float*)a.slot_ws : nullptr;
    const int per_launch = sum && !p.ws ? 1 : 8;
    for (int s = 0; s < a.r.k; s += per_launch) {
        p.slot_begin = s;
        p.nslots = std::min(per_launch, a.r.k - s);
        p.accumulate = (a.accumulate || (sum && !p.ws && s > 0)) ? 1 : 0;
        if ((long)p.mt_ub * p.ntn == 0) continue;
        const bool io = a.w_layout == HEXA_W_IN_OUT;
        const bool wide = too_large((size_t)a.r.T * (a.x_per_slot ? a.r.k : 1), a.in_dim) || too_large(a.in_dim, a.out_dim);
        // With more tiles than three workgroups per CU take at once, four with two stages each hide more of each other's
        // starts and ends (fc2-type launch: 199 against 219 us; equal for fc1); below that a tile is on its own and a
        // third stage is worth 2 us of 18.
        const bool many = (long)p.nslots * a.r.T / BM * p.ntn > 768;
        const int rc = wide   ? (io ? launch_esmm32_t<true, true, Deep>(p, st) : launch_esmm32_t<false, true, Deep>(p, st))
                       : many ? (io ? launch_esmm32_t<true, false, Many>(p, st) : launch_esmm32_t<false, false, Many>(p, st))
                              : (io ? launch_esmm32_t<true, false, Deep>(p, st) : launch_esmm32_t<false, false, Deep>(p, st));
        if (rc) return rc;
    }
    if (p.ws) return launch_sum_slots(a.out, a.slot_ws, a.r, a.out_dim, a.accumulate, HEXA_F32, st, a.sum_extra);
    return HEXA_OK;
}

// Parts every expert's token list is cut into: with fewer than two 64 x 64 tiles per CU a launch is the walk over one
// list, so lists of 256 and more entries are cut until there are four workgroups per CU (or 128 entries a part).
int estmm32_parts(int T, int k, int E, int m_dim, int n_dim) {
    const long tiles = (long)E * div_up(m_dim, 64) * div_up(n_dim, 64), avg = (long)T * k / std::max(1, E);
    if (tiles >= 512 || avg < 256) return 1;
    return (int)std::max<long>(1, std::min<long>(8, std::min<long>((1024 + tiles - 1) / tiles, avg / 128)));
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
    p.parts = a.scratch ? std::max(1, std::min(estmm32_parts(p.T, p.k, p.E, p.M, p.N), a.max_slots / p.E)) : 1;
    const bool wide = too_large((size_t)p.T * (a.p_per_slot ? p.k : 1), p.M) || too_large((size_t)p.T * (a.q_per_slot ? p.k : 1), p.N);
    if (int rc = wide ? launch_estmm32_t<true>(p, st) : launch_estmm32_t<false>(p, st)) return rc;
    return p.parts > 1 ? launch_fold(a.dw, a.scratch, (long)p.E * p.M * p.N, p.parts, HEXA_F32, a.accumulate, st) : HEXA_OK;
}

}  // namespace hexa
