// ESMM for bf16 / fp16 on gfx950 with 256 x 256 tiles, for products large enough to fill the chip with them (the rule is
// use_big in gemm16_dma.hip; the sums are those of the 128 x 128 kernels, in the same order).
//
// What bounds the 128 x 128 kernels there is the way of the operands, not the matrix pipes: a 128 x 128 x 64 stage reads
// 32 KB from L2 and 64 KB from LDS for 2.1 MFLOP, and the CU's copy path (64 B a clock) is busy 64 to 72 % of the time.  A 256 x
// 256 tile halves both: eight wavefronts of 128 x 64 (4 x 2 blocks of 32 x 32, 128 accumulator registers) read each operand byte
// from LDS 4 and 2 times and copy 64 KB for 8.4 MFLOP.  One workgroup fills a CU's LDS (two stages of 64 KB), so nothing
// beside it hides its waits; the eight wavefronts are two groups of four (one of each group on a SIMD) that run half a stage
// apart, kept there by one barrier more for the second group: while one group multiplies, the other reads fragments
// and issues copies.  A stage is two halves of 64 rows per wavefront, whose four kinds of copies (upper and lower rows, even
// and odd columns) are issued where the half of the buffer they overwrite has been read by both groups, one stage ahead; waits
// count the younger copies and the stores of the tile before (s_waitcnt vmcnt), so nothing is drained between the tiles of plain and
// GELU launches.  GELU' waits for its block's y1 in every epilogue, and with it for the copies in front of it, which were issued
// a stage before; its fp16 instances with column sums spill one register (an address, reloaded once a tile).
//
// Measured: 8192 x 8192 x 8192 in bf16 1322 TFLOP/s in this schedule (1113 by the vendor's library on the same card); a
// stage takes 1.4 to 1.6 us per round of 256 tiles.  32768 rows, top-2 of 64 experts with a skewed load, 1024 -> 4096: plain 888 us
// before, 615 now; + GELU 1028, 740; fc2 787, 640; times GELU' with column sums 1010, 780.  What is left there is the
// results' way out (537 MB each, 100 us and more of them) with nothing to multiply in the meantime: a tile's accumulators
// hold half of the registers, so the next tile cannot begin before they are stored.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "pipe_common.h"
#include "small_bodies.h"

namespace hexa {
namespace {

constexpr int BIG_MAX_ROUNDS = 160;    // tiles one workgroup may walk (their records are kept in LDS)
constexpr int BIG_MAX_E = 2048;        // experts (their tile counts are summed up in the staging rows)
constexpr int BIG_ROW_RUN = 4;         // row tiles that are walked together, column tile by column tile

struct BigK {
    const void* x; const void* w; const void* bias; void* out; void* out_act; void* ws; float* colsum;
    const int32_t* token_ids; const int32_t* offsets;
    int T, K, N, E, nslots, ntn, x_per_slot, out_per_slot, bias_dt, stream_out, act_only;
    int wg_per_xcd;       // workgroups per XCD (grid = 8 * wg_per_xcd)
};

// The table of the activation of bf16 values: entry 2 * (magnitude bits - LO) + sign, as bf16 (GELU) or fp32 (GELU'), what
// the polynomial gives.  A wavefront's piece with a value outside (|x| >= 8, zeros, NaN) takes the polynomial, which costs 8 to
// 16 vector instructions a value more while the matrix pipes wait: 778 us without the table, 745 with it at the size above
// (GELU'  790, 740; with column sums 840, 785).  The wavefronts' staging has 8 rows instead of 16 to make room.
template <typename TC, int ACT> struct BigLut {
    static constexpr unsigned LO = ACT == HEXA_ACT_GELU_BWD ? 0x3900u : 0x3700u, R = LUT_M_HI - LO;      // from 2^-13 and 2^-17
    static constexpr int BYTES = !std::is_same<TC, __bf16>::value ? 0 : ACT == HEXA_ACT_GELU ? 2 * R * 2 : ACT == HEXA_ACT_GELU_BWD ? 2 * R * 4 : 0;
    static_assert(BYTES % 1024 == 0 && BYTES < 65536, "the stages' alignment; 16-bit table offsets");
};

struct BigHalf { static constexpr int HALF = 128 * 128, STAGE = 4 * HALF; };      // A0, A1, B0, B1: 128 rows or columns x 64 indices each
template <int LUT, bool BIAS, bool COLSUM> struct BigLds : BigHalf {
    static constexpr int CP = 64 * 2 + 16;                        // pitch of a wavefront's staged result row
    static constexpr int STAGES_AT = LUT;                         // (the table comes first: its offsets are LDS addresses)
    static constexpr int TOK_AT = STAGES_AT + 2 * STAGE;          // 2 x 256 token ids
    static constexpr int SLOT_AT = TOK_AT + 2 * 1024;             // 2 x 256 bytes: their slots
    static constexpr int BIAS_AT = SLOT_AT + 2 * 256;             // 2 x 256 bias elements
    static constexpr int INFO_AT = BIAS_AT + (BIAS ? 2 * 1024 : 0);
    static constexpr int RED_AT = INFO_AT + BIG_MAX_ROUNDS * 16;  // 2 x 256 partial column sums
    static constexpr int STAGING_AT = RED_AT + (COLSUM ? 2 * 1024 : 0);      // 8 x 8 rows
    static constexpr int BYTES = STAGING_AT + 8 * 8 * CP;
    static_assert(BYTES <= 160 * 1024, "LDS of a CU");
    static_assert((BIG_MAX_E + 1) * 4 <= 8 * 8 * CP, "the experts' first tiles");
};

template <int OFF = 0> __device__ __forceinline__ int lds_read_u8(unsigned addr) {
    int r;
    asm volatile("ds_read_u8 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
    return r;
}
__device__ __forceinline__ void lds_write_u8(unsigned addr, int v) { asm volatile("ds_write_b8 %0, %1" ::"v"(addr), "v"(v) : "memory"); }
// 16-byte store to an address of each lane's own (s_nop: see global_store128 of pipe_common.h)
__device__ __forceinline__ void global_store128(char* at, u32x4 v, bool streaming) {
    if (streaming) asm volatile("global_store_dwordx4 %0, %1, off nt\n\ts_nop 1" ::"v"(at), "v"(v) : "memory");
    else asm volatile("global_store_dwordx4 %0, %1, off\n\ts_nop 1" ::"v"(at), "v"(v) : "memory");
}

// a copy's wait: at most N (and EXTRA stores, where `lax`) younger operations may be outstanding
// (half: where only the activation is stored, half as many of them)
template <int N, int EXTRA, bool HALVES> __device__ __forceinline__ void wait_copies(bool more, bool lax, bool half) {
    if (!more) wait_vmcnt<0>();
    else if (HALVES && lax && half) wait_vmcnt<N + EXTRA / 2>();
    else if (lax) wait_vmcnt<N + EXTRA>();
    else wait_vmcnt<N>();
}

template <typename TC, bool W_IN_OUT, int ACT, bool COLSUM, bool TAIL>
__global__ __launch_bounds__(512, 2) void esmm16_big_kernel(BigK p) {
    using LT = BigLut<TC, ACT>;
    constexpr bool HAS_BIAS = ACT != HEXA_ACT_GELU_BWD;
    using L = BigLds<LT::BYTES, HAS_BIAS, COLSUM>;
    using V = typename Mfma<TC>::V;
    constexpr int BM = 256, BN = 256, BK = 64, HALF = L::HALF;
    constexpr bool IO_SUM = ACT == HEXA_ACT_NONE;                 // results may be summed over the slots
    constexpr int STORES = (ACT == HEXA_ACT_GELU ? 2 : 1) * 16;   // of a wavefront and full tile
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    const unsigned lds0 = lds_addr(smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 2, wf = wave & 3;
    const int K = p.K, N = p.N, nk = TAIL ? K / BK + 1 : K / BK;
    const bool streaming = p.stream_out != 0;
    const bool act_only = ACT == HEXA_ACT_GELU && p.act_only != 0;

    // An expert's rows are its lists of all slots, one behind the other: half a tile of its last 256 is empty on average, not half
    // a tile of each list's.  First tile of every expert:
    const int E = p.E, T = p.T, nslots = p.nslots;
    auto list_begin = [&](int s, int e) { return p.offsets[(size_t)s * (E + 1) + e]; };
    int* const sFirst = reinterpret_cast<int*>(smem + L::STAGING_AT);
    if (wave == 0) {
        const int share = (E + 63) >> 6, lo = min(E, lane * share), hi = min(E, lo + share);
        auto tiles_of = [&](int e) {
            int n = 0;
            for (int s = 0; s < nslots; ++s) n += list_begin(s, e + 1) - list_begin(s, e);
            return (n + BM - 1) / BM;
        };
        int sum = 0;
        for (int e = lo; e < hi; ++e) sum += tiles_of(e);
        int before = sum;
#pragma unroll
        for (int d = 1; d < 64; d <<= 1) {
            const int o = __shfl_up(before, d);
            if (lane >= d) before += o;
        }
        int at = before - sum;
        for (int e = lo; e < hi; ++e) { sFirst[e] = at; at += tiles_of(e); }
        if (lane == 63) sFirst[E] = at;
    }
    __syncthreads();
    // This workgroup's walk: XCD x owns one contiguous eighth of the tiles and its workgroups take them in turn.  Runs of four row
    // tiles of an expert are walked column tile by column tile: what the XCD multiplies at any time is about 4 x 8 tiles.
    const int valid = sFirst[E] * p.ntn;
    const int per = (valid + 7) >> 3;
    const int xcd = blockIdx.x & 7, wg = blockIdx.x >> 3;
    const int first = xcd * per + wg, lim = min(valid, (xcd + 1) * per);
    const int ntiles = first < lim ? (lim - first + p.wg_per_xcd - 1) / p.wg_per_xcd : 0;
    if (ntiles == 0) return;
    int4* sInfo = reinterpret_cast<int4*>(smem + L::INFO_AT);   // {expert, first row, rows | column tile << 10, row tile of all}
    for (int i = tid; i < ntiles; i += 512) {
        const int logical = first + i * p.wg_per_xcd;
        const int mt = logical / p.ntn;
        int e = 0;
        for (int d = BIG_MAX_E; d > 0; d >>= 1)
            if (e + d < E && sFirst[e + d] <= mt) e += d;         // the last expert whose first tile is not behind this one
        const int mine = sFirst[e + 1] - sFirst[e], j = logical - sFirst[e] * p.ntn;
        const int run = j / (BIG_ROW_RUN * p.ntn), in_run = j - run * BIG_ROW_RUN * p.ntn, high = min(BIG_ROW_RUN, mine - run * BIG_ROW_RUN);
        const int nt = in_run / high, row = run * BIG_ROW_RUN + in_run - nt * high;
        int n = 0;
        for (int s = 0; s < nslots; ++s) n += list_begin(s, e + 1) - list_begin(s, e);
        sInfo[i] = make_int4(e, row * BM, min(BM, n - row * BM) | (nt << 10), sFirst[e] + row);
    }
    __syncthreads();
    struct Rec { int e, row_start, rows, nt, mt; };
    auto tile_rec = [&](int r) {   // uniform: every lane reads the same record
        u32x4 v = lds_read128_async(lds0 + L::INFO_AT + r * 16);
        lds_wait();
        asm volatile("" : "+v"(v));
        const int z = __builtin_amdgcn_readfirstlane((int)v.z);
        Rec o;
        o.e = __builtin_amdgcn_readfirstlane((int)v.x); o.row_start = __builtin_amdgcn_readfirstlane((int)v.y);
        o.rows = z & 1023; o.nt = z >> 10; o.mt = __builtin_amdgcn_readfirstlane((int)v.w);
        return o;
    };
    // where row i of a tile is in the lists
    struct Entry { int slot; const int32_t* id; };
    auto entry = [&](const Rec& rec, int i) {
        Entry o{0, reinterpret_cast<const int32_t*>(g_zero_block)};
        int m = rec.row_start + i;
        if (i >= rec.rows) return o;
        for (int s = 0; s < nslots; ++s) {
            const int b = list_begin(s, rec.e), n = list_begin(s, rec.e + 1) - b;
            if (m >= 0 && m < n) { o.slot = s; o.id = p.token_ids + (size_t)s * T + b + m; }
            m -= n;
        }
        return o;
    };
    const char* const zero = reinterpret_cast<const char*>(g_zero_block);
    const int bias_esz = p.bias_dt == HEXA_F32 ? 4 : 2;

    // ---- copies: the stage they are for (tile ct, step cs), its two bases, every lane's offsets from them -----------------
    int ct = 0, cs = 0;
    bool more = true;
    unsigned cbuf = 0;
    const char* xk = nullptr; const char* wk = nullptr;
    unsigned offA[2][2], offB[2][2];
    int krow, kcol;                            // KC: row of the lane's first copy and its piece of 8 indices; KS: see ks_lane
    kc_lane<64>(wave, lane, krow, kcol);
    int skk, sch;
    ks_lane<128>(wave, lane, skk, sch);
    auto set_sources = [&](int r) {
        const Rec rec = tile_rec(r);
        int tok[2][2], slot[2][2];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                const int i = (r & 1) * BM + h * 128 + j * 64 + krow;
                tok[h][j] = lds_read_i32(lds0 + L::TOK_AT + i * 4);
                slot[h][j] = lds_read_u8(lds0 + L::SLOT_AT + i);
            }
        lds_wait();
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int j = 0; j < 2; ++j) {
                int t = tok[h][j];
                asm volatile("" : "+v"(t));
                asm volatile("" : "+v"(slot[h][j]));
                // (rows past the tile's end: token 0 of slot 0; what they produce is never stored)
                offA[h][j] = (unsigned)((((size_t)(p.x_per_slot ? T : 0) * slot[h][j] + t) * K + kcol * 8) * 2);
                int n;
                if (W_IN_OUT) {
                    n = rec.nt * BN + (2 * (sch >> 2) + h) * 32 + (sch & 3) * 8;
                    offB[h][j] = (unsigned)(((size_t)(skk + 32 * j) * N + (n < N ? n : 0)) * 2);
                } else {
                    const int row = j * 64 + krow;
                    n = rec.nt * BN + (2 * (row >> 5) + h) * 32 + (row & 31);
                    offB[h][j] = (unsigned)(((size_t)(n < N ? n : 0) * K + kcol * 8) * 2);
                }
            }
        xk = reinterpret_cast<const char*>(p.x);
        wk = reinterpret_cast<const char*>(p.w) + (size_t)rec.e * K * N * 2;
    };
    const int ktail = TAIL ? K % BK : 0;
    auto issueA = [&](int h) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            char* to = smem + L::STAGES_AT + cbuf + h * HALF + (wave + 8 * j) * 1024;
            if (TAIL && cs == nk - 1) dma16(kcol * 8 < ktail ? xk + (size_t)offA[h][j] : zero, to);
            else dma16(xk + (size_t)offA[h][j], to);
        }
    };
    auto issueB = [&](int h) {
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            char* to = smem + L::STAGES_AT + cbuf + (2 + h) * HALF + (wave + 8 * j) * 1024;
            if (TAIL && cs == nk - 1) dma16((W_IN_OUT ? skk + 32 * j : kcol * 8) < ktail ? wk + (size_t)offB[h][j] : zero, to);
            else dma16(wk + (size_t)offB[h][j], to);
        }
    };
    auto next_stage = [&]() {
        xk += BK * 2;
        wk += W_IN_OUT ? (size_t)BK * N * 2 : (size_t)BK * 2;
        cbuf ^= L::STAGE;
        if (++cs == nk) {
            cs = 0;
            if (++ct < ntiles) set_sources(ct);
            else more = false;
        }
    };
    // token ids and bias of tile r (waves 0..3: 64 ids each, wave 4: the bias)
    auto fetch_meta = [&](int r) {
        const Rec rec = tile_rec(r);
        if (wave < 4) {
            const Entry en = entry(rec, wave * 64 + lane);
            __builtin_amdgcn_global_load_lds((glb_ptr_t)en.id, (lds_ptr_t)(smem + L::TOK_AT + ((r & 1) * BM + wave * 64) * 4), 4, 0, 0);
            lds_write_u8(lds0 + L::SLOT_AT + (r & 1) * BM + wave * 64 + lane, en.slot);
        } else if (HAS_BIAS && wave == 4 && p.bias) {
            const int n = rec.nt * BN + lane * (16 / bias_esz);
            const bool ok = lane < BN * bias_esz / 16 && n < N;
            const void* src = ok ? (const void*)(reinterpret_cast<const char*>(p.bias) + ((size_t)rec.e * N + n) * bias_esz) : (const void*)zero;
            __builtin_amdgcn_global_load_lds((glb_ptr_t)src, (lds_ptr_t)(smem + L::BIAS_AT + (r & 1) * 1024), 16, 0, 0);
        }
    };

    // ---- fragments --------------------------------------------------------------------------------------------------------
    unsigned lp[4];                            // lane part of a KC fragment's address, by step of 16 indices
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) lp[ks] = lds0 + L::STAGES_AT + (lane & 31) * 128 + (((ks * 2 + (lane >> 5)) ^ kc_swizzle<64>(lane & 31)) << 4);
    unsigned sp;                               // the same of a KS fragment
    {
        const int grp = lane >> 4, sl = lane & 15;
        const int col = wf * 32 + (grp & 1) * 16 + (sl & 3) * 4, k = (grp >> 1) * 8 + (sl >> 2);
        sp = lds0 + L::STAGES_AT + 2 * HALF + k * 256 + (((col >> 3) ^ ((k & 3) << 2)) << 4) + (col & 7) * 2;
    }
    unsigned rbuf = 0;
    union Frag { V v; u32x4 q; s16x4 h[2]; };
    Frag a[2][4], b0[4], b1[4];
    auto readA = [&](auto hc) {
        constexpr int h = decltype(hc)::value;
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) {
            const unsigned at = lp[ks] + rbuf + wr * 8192;
            a[0][ks].q = lds_read128_async<h * HALF>(at);
            a[1][ks].q = lds_read128_async<h * HALF + 4096>(at);
        }
    };
    auto readB = [&](auto hc, Frag (&b)[4]) {
        constexpr int h = decltype(hc)::value;
        static_for<4>([&](auto kc) {
            constexpr int ks = decltype(kc)::value;
            if constexpr (W_IN_OUT) {
                const unsigned at = sp + rbuf;
                Frag& f = b[ks];
                asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(f.h[0]) : "v"(at), "n"(h * HALF + ks * 4096));
                asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(f.h[1]) : "v"(at), "n"(h * HALF + ks * 4096 + 1024));
            } else {
                b[ks].q = lds_read128_async<h * HALF + 2 * HALF>(lp[ks] + rbuf + wf * 4096);
            }
        });
    };
    int live_rows = 0, live_cols = 0;          // of the tile being multiplied
    f32x16 acc[2][2][2];                       // [half of rows][half of columns][32-row block]
    auto clear = [&]() {
#pragma unroll
        for (int x = 0; x < 8; ++x)
#pragma unroll
            for (int v = 0; v < 16; ++v) acc[x >> 2][(x >> 1) & 1][x & 1][v] = 0.f;
    };
    auto mma = [&](auto hac, auto hbc, Frag (&b)[4]) {
        constexpr int ha = decltype(hac)::value, hb = decltype(hbc)::value;
        __builtin_amdgcn_sched_barrier(0);
        if (ha * 128 + wr * 64 >= live_rows || (2 * wf + hb) * 32 >= live_cols) return;      // nothing of this block is stored
        __builtin_amdgcn_s_setprio(1);
#pragma unroll
        for (int ks = 0; ks < 4; ++ks)
#pragma unroll
            for (int i = 0; i < 2; ++i) acc[ha][hb][i] = Mfma<TC>::run(b[ks].v, a[i][ks].v, acc[ha][hb][i]);
        __builtin_amdgcn_s_setprio(0);
        __builtin_amdgcn_sched_barrier(0);
    };
    using I0 = std::integral_constant<int, 0>;
    using I1 = std::integral_constant<int, 1>;
    auto pinA = [&]() {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) { asm volatile("" : "+v"(a[0][ks].q)); asm volatile("" : "+v"(a[1][ks].q)); }
    };
    auto pinB = [&](Frag (&b)[4]) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) asm volatile("" : "+v"(b[ks].q));
    };

    // ---- tile 0's token ids and bias, the first stages -----------------------------------------------------------------------
    {
        const Rec rec = tile_rec(0);
        if (tid < BM) {
            const Entry en = entry(rec, tid);
            reinterpret_cast<int*>(smem + L::TOK_AT)[tid] = *en.id;
            reinterpret_cast<unsigned char*>(smem + L::SLOT_AT)[tid] = (unsigned char)en.slot;
            if constexpr (HAS_BIAS) {
                const int n = rec.nt * BN + tid;
                unsigned raw = 0;
                if (p.bias && n < N) {
                    if (bias_esz == 4) raw = reinterpret_cast<const unsigned*>(p.bias)[(size_t)rec.e * N + n];
                    else raw = reinterpret_cast<const unsigned short*>(p.bias)[(size_t)rec.e * N + n];
                }
                if (bias_esz == 4) reinterpret_cast<unsigned*>(smem + L::BIAS_AT)[tid] = raw;
                else reinterpret_cast<unsigned short*>(smem + L::BIAS_AT)[tid] = (unsigned short)raw;
            }
        }
        if constexpr (LT::BYTES > 0) {           // what the polynomials give for exactly these bf16 values
            for (unsigned i = tid; i < 2 * LT::R; i += 512) {
                const float xv = from_bits16<TC>((unsigned short)(((i & 1u) << 15) | (LT::LO + (i >> 1))));
                if (ACT == HEXA_ACT_GELU) reinterpret_cast<unsigned short*>(smem)[i] = (unsigned short)(pack2<TC>(gelu_poly(xv), 0.f) & 0xffff);
                else reinterpret_cast<float*>(smem)[i] = gelu_grad_poly(xv);
            }
        }
        __syncthreads();
    }
    set_sources(0);
    issueB(0); issueA(0); issueB(1); issueA(1);
    next_stage();
    issueB(0); issueA(0); issueB(1);
    clear();
    wait_vmcnt<8>();
    barrier_nofence();
    if (wr == 1) barrier_nofence();            // the second group runs half a phase behind the first

    bool lax = false;                          // the stores of a full tile are still younger than the copies waited for
    Rec done{};                                // COLSUM: the tile whose partial sums are in LDS
    auto write_colsum = [&]() {
        if (wr == 0) {
            const int c = wf * 64 + lane;
            int lo = lds_read_i32(lds0 + L::RED_AT + c * 4), hi = lds_read_i32(lds0 + L::RED_AT + 1024 + c * 4);
            lds_wait();
            asm volatile("" : "+v"(lo));
            asm volatile("" : "+v"(hi));
            p.colsum[((size_t)done.mt * p.ntn + done.nt) * BN + c] = __int_as_float(lo) + __int_as_float(hi);
        }
    };
    for (int r = 0; r < ntiles; ++r) {
        const Rec rec = tile_rec(r);
        live_rows = rec.rows;
        live_cols = N - rec.nt * BN;
        for (int kt = 0; kt < nk; ++kt) {
            // first half of the rows
            readA(I0());
            readB(I0(), b0);
            readB(I1(), b1);
            if (more) { issueA(1); next_stage(); }
            wait_copies<8, STORES, ACT == HEXA_ACT_GELU>(more, lax, act_only);
            lds_wait();
            pinA(); pinB(b0); pinB(b1);
            barrier_nofence();
            mma(I0(), I0(), b0);
            mma(I0(), I1(), b1);
            barrier_nofence();
            // second half
            readA(I1());
            if (more) { issueB(0); issueA(0); issueB(1); }
            if (kt == 0) {
                if (r + 1 < ntiles) fetch_meta(r + 1);
                if (COLSUM && r > 0) write_colsum();
            }
            wait_copies<8, STORES, ACT == HEXA_ACT_GELU>(more, lax, act_only);
            lax = false;
            lds_wait();
            pinA();
            barrier_nofence();
            mma(I1(), I1(), b1);
            mma(I1(), I0(), b0);
            barrier_nofence();
            rbuf ^= L::STAGE;
        }

        // ---- result: a wavefront's 128 x 64 values, 8 rows at a time through its own staging rows -----------------------------
        const int n0 = rec.nt * BN, rows = rec.rows;
        const bool slots_apart = p.ws != nullptr;         // slots above the first go to the scratch that is added afterwards
        const unsigned stg = lds0 + L::STAGING_AT + wave * 8 * L::CP;
        const unsigned put = stg + (lane & 7) * L::CP + (lane >> 5) * 8, get = stg + (lane >> 3) * L::CP + (lane & 7) * 16;
        const unsigned tok_at = lds0 + L::TOK_AT + ((r & 1) * BM + wr * 64 + (lane >> 3)) * 4;
        const unsigned slot_at = lds0 + L::SLOT_AT + (r & 1) * BM + wr * 64 + (lane >> 3);
        const int n = n0 + wf * 64 + (lane & 7) * 8;
        const bool col_ok = n < N;
        lax = rows == BM && n0 + BN <= N;
        float bv[8][4];
#pragma unroll
        for (int u = 0; u < 8; ++u) { bv[u][0] = 0.f; bv[u][1] = 0.f; bv[u][2] = 0.f; bv[u][3] = 0.f; }
        if (HAS_BIAS && p.bias) {
            const unsigned at = lds0 + L::BIAS_AT + (r & 1) * 1024 + (wf * 64 + 4 * (lane >> 5)) * bias_esz;
            if (bias_esz == 4) {
                u32x4 w[8];
                static_for<8>([&](auto uc) { constexpr int u = decltype(uc)::value; w[u] = lds_read128_async<u * 32>(at); });
                lds_wait();
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    asm volatile("" : "+v"(w[u]));
                    bv[u][0] = __uint_as_float(w[u].x); bv[u][1] = __uint_as_float(w[u].y); bv[u][2] = __uint_as_float(w[u].z); bv[u][3] = __uint_as_float(w[u].w);
                }
            } else {
                u32x2 w[8];
                static_for<8>([&](auto uc) { constexpr int u = decltype(uc)::value; w[u] = lds_read64_async<u * 16>(at); });
                lds_wait();
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    asm volatile("" : "+v"(w[u]));
                    bv[u][0] = lo16<TC>(w[u].x); bv[u][1] = hi16<TC>(w[u].x); bv[u][2] = lo16<TC>(w[u].y); bv[u][3] = hi16<TC>(w[u].y);
                }
            }
        }
        float colsum[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
        // result rows of a 32-row block: four per lane, 8 rows apart
        unsigned boff[2][4];
        bool ok[2][4], aside[2][4];
        u32x4 y[2][4];
        auto locate = [&](auto bc) {
            constexpr int b = decltype(bc)::value, ROW = (b >> 1) * 128 + (b & 1) * 32;    // (+ wr * 64)
            int tok[4], slot[4];
            static_for<4>([&](auto qc) {
                constexpr int q = decltype(qc)::value;
                tok[q] = lds_read32_async<(ROW + q * 8) * 4>(tok_at);
                slot[q] = lds_read_u8<ROW + q * 8>(slot_at);
            });
            lds_wait();
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                asm volatile("" : "+v"(tok[q]));
                asm volatile("" : "+v"(slot[q]));
                aside[b & 1][q] = slots_apart && slot[q] > 0;
                const unsigned row = (unsigned)tok[q] + (unsigned)T * (unsigned)(p.out_per_slot ? slot[q] : aside[b & 1][q] ? slot[q] - 1 : 0);
                ok[b & 1][q] = ROW + wr * 64 + q * 8 + (lane >> 3) < rows && col_ok;
                boff[b & 1][q] = ok[b & 1][q] ? row * (unsigned)N * 2u + (unsigned)n * 2u : 0u;
            }
            if (ACT == HEXA_ACT_GELU_BWD) {
#pragma unroll
                for (int q = 0; q < 4; ++q) y[b & 1][q] = global_load128_async(p.out_act, boff[b & 1][q]);
            }
        };
        constexpr int PASSES = ACT == HEXA_ACT_NONE ? 4 : 2;
        locate(I0());
        static_for<4>([&](auto bc) {
            constexpr int b = decltype(bc)::value, ha = b >> 1, i = b & 1;
            if constexpr (b < 3) locate(std::integral_constant<int, b + 1>());
            auto store = [&](int q, u32x4 v) {
                if (!ok[b & 1][q]) return;
                if (IO_SUM) global_store128(reinterpret_cast<char*>(aside[b & 1][q] ? p.ws : p.out) + boff[b & 1][q], v, streaming);
                else global_store128(p.out, boff[b & 1][q], v, streaming);
                if (COLSUM) {
#pragma unroll
                    for (int u = 0; u < 4; ++u) { colsum[2 * u] += lo16<TC>(v[u]); colsum[2 * u + 1] += hi16<TC>(v[u]); }
                }
            };
            // (a wavefront's LDS accesses happen in order: the next rows may follow the read of the ones before at once)
            static_for<4 / PASSES>([&](auto hc) {
                constexpr int q0 = decltype(hc)::value * PASSES;
                u32x4 val[PASSES];
                static_for<PASSES>([&](auto pc) {
                    constexpr int pass = decltype(pc)::value;
                    if (((lane >> 3) & 3) == q0 + pass) {
                        static_for<8>([&](auto uc) {
                            constexpr int u = decltype(uc)::value, hb = u >> 2, g = u & 3;
                            const f32x16& v = acc[ha][hb][i];
                            lds_write64<hb * 64 + g * 16>(put, pack4<TC>(v[4 * g] + bv[u][0], v[4 * g + 1] + bv[u][1], v[4 * g + 2] + bv[u][2], v[4 * g + 3] + bv[u][3]));
                        });
                    }
                    val[pass] = lds_read128_async(get);
                });
                lds_wait();
#pragma unroll
                for (int q = 0; q < PASSES; ++q) asm volatile("" : "+v"(val[q]));
                // (behind this block's y1: the stores of the block before, the next one's loads)
                if (ACT == HEXA_ACT_GELU_BWD && q0 == 0) {
                    if (lax) wait_vmcnt<(b > 0 ? 4 : 0) + (b < 3 ? 4 : 0)>();
                    else wait_vmcnt<(b < 3 ? 4 : 0)>();
#pragma unroll
                    for (int q = 0; q < 4; ++q) asm volatile("" : "+v"(y[b & 1][q]));
                }
#pragma unroll
                for (int qq = 0; qq < PASSES; ++qq) {
                    const int q = q0 + qq;
                    u32x4 x = val[qq], v = x;
                    if (ACT != HEXA_ACT_GELU_BWD && !act_only) store(q, x);
                    if (ACT != HEXA_ACT_NONE) {
                        // the activation of the value as stored (rounded): GELU of the result, or GELU' of y1 as a factor of it
                        const u32x4 arg = ACT == HEXA_ACT_GELU ? x : y[b & 1][q];
                        bool looked_up = false;
                        if constexpr (LT::BYTES > 0) {
                            unsigned at[4];
                            u16x2 far = {0, 0};
#pragma unroll
                            for (int u = 0; u < 4; ++u) at[u] = lut_offsets<LT::LO, ACT == HEXA_ACT_GELU ? 1 : 2>(arg[u], far);
                            // (every value of the wavefront's piece is in the table)
                            if (lds0 == 0 && __builtin_amdgcn_ballot_w64(max(far.x, far.y) >= (unsigned short)LT::R) == 0) {
                                unsigned g[8];
#pragma unroll
                                for (int u = 0; u < 4; ++u) {
                                    if (ACT == HEXA_ACT_GELU) {
                                        g[2 * u] = lds_read_u16_async<0>(at[u] & 0xffffu);
                                        g[2 * u + 1] = lds_read_u16_async<0>(at[u] >> 16);
                                    } else {
                                        g[2 * u] = (unsigned)lds_read32_async<0>(at[u] & 0xffffu);
                                        g[2 * u + 1] = (unsigned)lds_read32_async<0>(at[u] >> 16);
                                    }
                                }
                                lds_wait();
#pragma unroll
                                for (int u = 0; u < 8; ++u) asm volatile("" : "+v"(g[u]));
#pragma unroll
                                for (int u = 0; u < 4; ++u)
                                    v[u] = ACT == HEXA_ACT_GELU ? g[2 * u] | (g[2 * u + 1] << 16)
                                                                : pack2<TC>(lo16<TC>(x[u]) * __uint_as_float(g[2 * u]), hi16<TC>(x[u]) * __uint_as_float(g[2 * u + 1]));
                                looked_up = true;
                            }
                        }
                        if (!looked_up) {
#pragma unroll
                            for (int u = 0; u < 4; ++u)
                                v[u] = ACT == HEXA_ACT_GELU ? pack2<TC>(gelu_poly(lo16<TC>(arg[u])), gelu_poly(hi16<TC>(arg[u])))
                                                            : pack2<TC>(lo16<TC>(x[u]) * gelu_grad_poly(lo16<TC>(arg[u])), hi16<TC>(x[u]) * gelu_grad_poly(hi16<TC>(arg[u])));
                        }
                        if (ACT == HEXA_ACT_GELU_BWD) store(q, v);
                        else if (ok[b & 1][q]) global_store128(p.out_act, boff[b & 1][q], v, streaming);
                    }
                }
            });
        });
        if (COLSUM) {                          // the lanes that hold the same piece; the two groups are added after the next barriers
#pragma unroll
            for (int u = 0; u < 8; ++u)
#pragma unroll
                for (int m = 32; m >= 8; m >>= 1) colsum[u] += __shfl_xor(colsum[u], m);
            if (lane < 8) {
                const unsigned at = lds0 + L::RED_AT + wr * 1024 + (wf * 64 + lane * 8) * 4;
                lds_write128<0>(at, u32x4{__float_as_uint(colsum[0]), __float_as_uint(colsum[1]), __float_as_uint(colsum[2]), __float_as_uint(colsum[3])});
                lds_write128<16>(at, u32x4{__float_as_uint(colsum[4]), __float_as_uint(colsum[5]), __float_as_uint(colsum[6]), __float_as_uint(colsum[7])});
            }
            lds_wait();
            done = rec;
        }
        clear();
    }
    if (wr == 0) barrier_nofence();
    if (COLSUM) {
        barrier_nofence();
        write_colsum();
    }
}

template <typename TC, bool IO, int ACT, bool COLSUM, bool TAIL>
int launch_big_k(BigK& pk, int grid, hipStream_t st) {
    auto kernel = esmm16_big_kernel<TC, IO, ACT, COLSUM, TAIL>;
    constexpr int bytes = BigLds<BigLut<TC, ACT>::BYTES, ACT != HEXA_ACT_GELU_BWD, COLSUM>::BYTES;
    if (int rc = ensure_smem(kernel, bytes)) return rc;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(512), bytes, st, pk);
    HEXA_CHECK_LAUNCH("esmm16_big");
    return HEXA_OK;
}
template <typename TC, bool IO, int ACT, bool COLSUM>
int launch_big_t(BigK& pk, int grid, hipStream_t st) {
    return pk.K % 64 ? launch_big_k<TC, IO, ACT, COLSUM, true>(pk, grid, st) : launch_big_k<TC, IO, ACT, COLSUM, false>(pk, grid, st);
}
template <typename TC>
int launch_big_a(BigK& pk, int grid, bool io, int act, bool colsum, hipStream_t st) {
    if (io) return launch_big_t<TC, true, HEXA_ACT_NONE, false>(pk, grid, st);
    if (act == HEXA_ACT_GELU) return launch_big_t<TC, false, HEXA_ACT_GELU, false>(pk, grid, st);
    if (act == HEXA_ACT_GELU_BWD)
        return colsum ? launch_big_t<TC, false, HEXA_ACT_GELU_BWD, true>(pk, grid, st) : launch_big_t<TC, false, HEXA_ACT_GELU_BWD, false>(pk, grid, st);
    return launch_big_t<TC, false, HEXA_ACT_NONE, false>(pk, grid, st);
}

int big_units() {
    static int cus = 0;
    if (!cus) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || n < 8) n = 256;
        cus = n;
    }
    return cus;
}

// tiles of a launch at most: a partial one for every expert that has rows
long big_tiles_ub(const EsmmArgs& a) {
    const long rows = (long)a.r.T * a.r.k;
    return (rows / 256 + std::min<long>(a.r.E, rows)) * div_up(a.out_dim, 256);
}

}  // namespace

bool esmm16_big_supported(const EsmmArgs& a) {
    if (!(a.w_dt == a.x_dt && a.out_dt == a.x_dt && a.in_dim % 8 == 0 && a.out_dim % 8 == 0 && div_up(a.in_dim, 64) >= 4)) return false;
    if (a.r.k > 8 || a.accumulate || a.wide) return false;
    if (a.act != HEXA_ACT_NONE && (a.w_layout == HEXA_W_IN_OUT || !(a.out_per_slot || a.r.k == 1))) return false;
    if (a.colsum && a.act != HEXA_ACT_GELU_BWD) return false;
    if ((size_t)a.r.T * (a.x_per_slot ? a.r.k : 1) * a.in_dim * 2 >= ((size_t)1 << 32) || (size_t)a.in_dim * a.out_dim * 2 >= ((size_t)1 << 32) ||
        (size_t)a.r.T * a.r.k * a.out_dim * 2 >= ((size_t)1 << 32))
        return false;
    if (!(a.out_per_slot || a.r.k == 1 || a.slot_ws != nullptr)) return false;
    if (a.r.E > BIG_MAX_E || a.r.T >= 1 << 28) return false;
    const long total_ub = big_tiles_ub(a);
    const int wg_per_xcd = std::max(1, big_units() / 8);
    return ((total_ub + 7) / 8 + wg_per_xcd - 1) / wg_per_xcd <= BIG_MAX_ROUNDS;
}

int launch_esmm16_big(const EsmmArgs& a, hipStream_t st) {
    BigK pk;
    pk.x = a.x; pk.w = a.w; pk.bias = a.bias; pk.out = a.out; pk.out_act = a.out_act; pk.colsum = a.colsum;
    pk.token_ids = a.r.token_ids; pk.offsets = a.r.offsets;
    pk.T = a.r.T; pk.K = a.in_dim; pk.N = a.out_dim; pk.E = a.r.E; pk.nslots = a.r.k;
    pk.ntn = div_up(a.out_dim, 256);
    pk.x_per_slot = a.x_per_slot; pk.out_per_slot = a.out_per_slot;
    pk.bias_dt = a.bias_dt; pk.stream_out = option(OPT_ESMM_STREAM) != 2; pk.act_only = a.act_only;
    pk.ws = (!a.out_per_slot && a.r.k > 1) ? a.slot_ws : nullptr;
    const long total_ub = big_tiles_ub(a);
    if (total_ub == 0) return HEXA_OK;
    pk.wg_per_xcd = (int)std::min<long>(std::max(1, big_units() / 8), (total_ub + 7) / 8);
    const int grid = 8 * pk.wg_per_xcd;
    const bool io = a.w_layout == HEXA_W_IN_OUT;
    const int rc = a.x_dt == HEXA_BF16 ? launch_big_a<__bf16>(pk, grid, io, a.act, a.colsum != nullptr, st)
                                       : launch_big_a<_Float16>(pk, grid, io, a.act, a.colsum != nullptr, st);
    if (rc) return rc;
    if (pk.ws) return launch_sum_slots(a.out, a.slot_ws, a.r, a.out_dim, a.accumulate, a.out_dt, st, a.sum_extra);
    if (a.colsum) return launch_colsum_fold(a, (int)(total_ub / pk.ntn), HEXA_TILE_ROWS_L, pk.ntn, 256, st, true);
    return HEXA_OK;
}

}  // namespace hexa
