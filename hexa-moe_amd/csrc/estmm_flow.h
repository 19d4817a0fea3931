// ESTMM for bf16 / fp16 on gfx950: dw[e][m][n] = sum over the expert's (slot, token) list of P[row][m] * Q[row][n], in 128 x 128
// blocks by persistent workgroups of four wavefronts, four workgroups per CU.
//
// What bounds it: not one resource.  A block of 18432 rows, top-2 of 32 experts, 384 x 1536, has 36 steps of 32 list entries; the matrix pipes
// are busy a quarter of the time, LDS a fifth, and with the copies, the products or the stores taken out the launch keeps 80 to
// 95 % of its time.  A step is a chain -- copies land, barrier, fragments read, products -- between which a wavefront issues
// some 170 instructions for 8 products, and a SIMD issues something 83 % of the time where that number is 250.  So: as many
// workgroups as fit (four: 36 KB of LDS and 114 registers each; two with four stages of copies in flight take 25 % longer), and
// little to do per step:
//   - the workgroup's blocks and the stretches of token lists behind them are worked out once, into two tables in LDS; a step
//     then follows a cursor over the stretches, one after the other over the blocks' ends, so that the next block's first rows are
//     on their way while a result is stored, and no block pays for trips to the plan, the lists' ends and the ids;
//   - rows are fetched through a scalar base and a 32-bit lane offset, one multiply-add per copy (64-bit lane addresses, the
//     last step of a list only, have a form of their own);
//   - the token ids of a step are fetched three steps ahead by one wavefront and read one step ahead;
//   - a result leaves through the stage that has just been multiplied, 4 KB per wavefront and without barriers in between.
// The units come heaviest first from the plan and every second round is dealt out backwards.  The sums are those of the
// one-block kernel (gemm16_dma.hip), product by product: results are equal bit for bit.
//
// Measured against that kernel, us, dW1 and dW2: the size above in bf16 90, 89 before, 64, 64 now; 9216 rows, 32 experts, 384 x 1536 in fp32
// 47, 48 before, 37, 37; 4608 rows, 32 experts, 768 x 3072 75, 82 before, 53, 54; 3600 rows, 8 experts, 768 x 3072 in fp32 46, 53 before, 41, 41; 2999
// rows, top-3 of 13 experts, 264 x 1056, fp16 44, 43 before, 32, 32; 4608 rows, top-2 of 8 experts, 384 x 1536, fp16 58, 58 before, 39, 39; 32768
// rows, top-2 of 64 experts, 1024 x 4096, bf16 800, 830 before, 655, 657; with a skewed
// load 870, 890 before, 730, 723 (256 x 256 blocks with eight wavefronts 735, 730).
#pragma once
#include <algorithm>
#include <type_traits>
#include <utility>

#include "pipe_common.h"
#include "small_bodies.h"

namespace hexa {
namespace {

constexpr int FLOW_IDS = 4;            // steps whose token ids are in LDS
constexpr int FLOW_MAX_ITEMS = 64;     // blocks one workgroup may walk
constexpr int FLOW_MAX_SEGS = 128;     // lists of them
constexpr int FLOW_SORT_E = 256;       // experts that a workgroup sorts by itself where there is no plan

struct FlowLds {
    static constexpr int HALF = 32 * 256, STAGE = 2 * HALF;       // 32 list entries x 128 columns of either operand
    static constexpr int IDS_AT = 2 * STAGE;
    static constexpr int ITEMS_AT = IDS_AT + FLOW_IDS * 32 * 4;   // {expert, steps, block (flow_block), scratch slot or -1}
    static constexpr int SEGS_AT = ITEMS_AT + FLOW_MAX_ITEMS * 16;   // {first id, ids, slot, block (flow_block)}
    static constexpr int BYTES = SEGS_AT + FLOW_MAX_SEGS * 16;
    static_assert(4 * BYTES <= 160 * 1024, "four workgroups per CU where the kernel has no other LDS");
};

// a block's row and column of blocks in one word, 16 bits each
__host__ __device__ constexpr unsigned flow_block(int mb, int nb) { return (unsigned)mb | ((unsigned)nb << 16); }
__host__ __device__ constexpr int flow_row_block(unsigned b) { return (int)(b & 0xffffu); }
__host__ __device__ constexpr int flow_col_block(unsigned b) { return (int)(b >> 16); }
constexpr int FLOW_MAX_DIM = 65536 * 128;
static_assert(flow_row_block(flow_block(65535, 65535)) == 65535 && flow_col_block(flow_block(0, 65535)) == 65535 &&
              flow_col_block(flow_block(65535, 32768)) == 32768, "16 unsigned bits each");

struct FlowK {
    const void* pm; const void* qm; void* dw;
    const int32_t* token_ids; const int32_t* offsets;
    const int* plan; float* scratch;
    int T, k, E, M, N, mtn, ntn, p_slot_rows, q_slot_rows, accumulate, stream_dw, group, rounds, wg_per_xcd;
};

template <typename TC, bool OUT32>
__device__ __forceinline__ void estmm16_flow_body(const FlowK& p, int block, char* smem) {
    using L = FlowLds;
    using V = typename Mfma<TC>::V;
    constexpr int BM = 128, BN = 128, BK = 32;
    const unsigned lds0 = lds_addr(smem);
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), wr = wave >> 1, wf = wave & 1;
    const int M = p.M, N = p.N, T = p.T, k = p.k, per_e = p.mtn * p.ntn, rounds = p.rounds;

    // ---- the blocks of this workgroup and the stretches of token lists behind them -------------------------------------------
    int4* const sItem = reinterpret_cast<int4*>(smem + L::ITEMS_AT);
    int4* const sSeg = reinterpret_cast<int4*>(smem + L::SEGS_AT);
    int2* const sPart = reinterpret_cast<int2*>(smem);            // part, parts (in the stages, which are still empty)
    for (int j = tid; j < rounds; j += 256) {
        // units come heaviest first; every second round is walked backwards
        const int loc = block >> 3, at = j * p.wg_per_xcd + (j & 1 ? p.wg_per_xcd - 1 - loc : loc);
        const long logical = logical_tile(at * 8 + (block & 7), p.group);
        const int rank = (int)(logical / per_e), rem = (int)(logical - (long)rank * per_e);
        // (the dimension with fewer blocks inside: a run shares the longer operand's columns)
        const int mb = p.mtn < p.ntn ? rem % p.mtn : rem / p.ntn, nb = p.mtn < p.ntn ? rem / p.mtn : rem % p.ntn;
        sItem[j] = make_int4(-1, rank, (int)flow_block(mb, nb), -1);
    }
    __syncthreads();
    auto take = [&](int u0, int n, int e, int slot) {             // units u0 .. u0 + n - 1 are the parts of expert e
        for (int j = 0; j < rounds; ++j) {
            const int part = sItem[j].y - u0;
            if (part >= 0 && part < n) {
                sItem[j].x = e;
                sItem[j].w = slot >= 0 ? slot + part : -1;
                sPart[j] = make_int2(part, n);
            }
        }
    };
    if (p.plan) {
        for (int r = tid; r < p.E; r += 256) take(p.plan[2 * p.E + r], p.plan[p.E + r], p.plan[r], p.plan[3 * p.E + r]);
    } else if (p.E <= FLOW_SORT_E) {            // no plan: whole experts, the busiest first
        int* const sLoad = reinterpret_cast<int*>(sPart + FLOW_MAX_ITEMS);
        if (tid < p.E) {
            int n = 0;
            for (int s = 0; s < k; ++s) n += p.offsets[(size_t)s * (p.E + 1) + tid + 1] - p.offsets[(size_t)s * (p.E + 1) + tid];
            sLoad[tid] = n;
        }
        __syncthreads();
        if (tid < p.E) {
            const int mine = sLoad[tid];
            int r = 0;
            for (int x = 0; x < p.E; ++x) r += (sLoad[x] > mine || (sLoad[x] == mine && x < tid)) ? 1 : 0;
            take(r, 1, tid, -1);
        }
    } else {
        for (int r = tid; r < p.E; r += 256) take(r, 1, r, -1);
    }
    __syncthreads();
    for (int i = tid; i < rounds * k; i += 256) {
        const int j = i / k, s = i - j * k;
        const int4 it = sItem[j];
        int4 seg = make_int4(0, 0, s, it.z);
        if (it.x >= 0) {
            int before = 0, all = 0, beg = 0, end = 0;
            for (int q = 0; q < k; ++q) {
                const int b = p.offsets[(size_t)q * (p.E + 1) + it.x], n = p.offsets[(size_t)q * (p.E + 1) + it.x + 1];
                const int steps = (n - b + BK - 1) / BK;
                if (q < s) before += steps;
                if (q == s) { beg = b; end = n; }
                all += steps;
            }
            // this part's share of the steps, and what of it is in this list
            const int2 pt = sPart[j];
            const int from = (int)((long)all * pt.x / pt.y), to = (int)((long)all * (pt.x + 1) / pt.y);
            const int lo = max(before, from), hi = min(before + (end - beg + BK - 1) / BK, to);
            if (hi > lo) {
                seg.x = s * T + beg + (lo - before) * BK;
                seg.y = min(end, beg + (hi - before) * BK) - (beg + (lo - before) * BK);
            }
        }
        sSeg[i] = seg;
    }
    __syncthreads();
    // (a list's steps are those of its parts and slots; the expert's rank is no longer needed)
    for (int j = tid; j < rounds; j += 256) {
        int steps = 0;
        for (int s = 0; s < k; ++s) steps += (sSeg[j * k + s].y + BK - 1) / BK;
        sItem[j].y = steps;
    }
    __syncthreads();
    int todo = 0;                               // steps of this workgroup
    for (int j = 0; j < rounds; ++j) todo += __builtin_amdgcn_readfirstlane(sItem[j].y);
    __syncthreads();
    auto record = [&](unsigned at) {            // uniform: every lane reads the same record
        u32x4 v = lds_read128_async(at);
        lds_wait();
        asm volatile("" : "+v"(v));
        return make_int4(__builtin_amdgcn_readfirstlane((int)v.x), __builtin_amdgcn_readfirstlane((int)v.y),
                         __builtin_amdgcn_readfirstlane((int)v.z), __builtin_amdgcn_readfirstlane((int)v.w));
    };

    // ---- copies: where the token ids and the operands of the next step come from ------------------------------------------------
    const int nsegs = rounds * k;
    struct Cursor { int seg, r; int4 rec; };
    auto settle = [&](Cursor& c) {              // on to the next list if this one has been walked
        while (c.r >= c.rec.y && c.seg + 1 < nsegs) {
            ++c.seg;
            c.r = 0;
            c.rec = record(lds0 + L::SEGS_AT + c.seg * 16);
        }
    };
    Cursor ci{0, 0, record(lds0 + L::SEGS_AT)}, cd = ci;
    settle(ci);
    settle(cd);
    const char* const zero = reinterpret_cast<const char*>(g_zero_block);
    int si = 0, sd = 0;                         // steps of ids and of operands issued
    auto issue_ids = [&]() {                    // by one wavefront
        const unsigned at = (unsigned)(ci.rec.x + max(min(ci.r + lane, ci.rec.y - 1), 0)) * 4u;      // (past the end: not used)
        if (wave == (si & 3) && lane < 32)
            __builtin_amdgcn_global_load_lds((glb_ptr_t)(reinterpret_cast<const char*>(p.token_ids) + (size_t)at),
                                             (lds_ptr_t)(smem + L::IDS_AT + (si & (FLOW_IDS - 1)) * 128), 4, 0, 0);
        ++si;
        ci.r += BK;
        settle(ci);
    };
    int kk, ch;
    ks_lane<128>(wave, lane, kk, ch);           // this lane's copies fetch entries kk and kk + 16 of a step, column piece ch
    unsigned colP = 0, colQ = 0;
    const unsigned pitchP = (unsigned)M * 2u, pitchQ = (unsigned)N * 2u;
    const char* pb = nullptr; const char* qb = nullptr;
    auto set_columns = [&]() {
        pb = reinterpret_cast<const char*>(p.pm) + (size_t)(unsigned)(p.p_slot_rows * cd.rec.z) * pitchP;
        qb = reinterpret_cast<const char*>(p.qm) + (size_t)(unsigned)(p.q_slot_rows * cd.rec.z) * pitchQ;
        const int m = flow_row_block(cd.rec.w) * BM + ch * 8, n = flow_col_block(cd.rec.w) * BN + ch * 8;
        colP = m < M ? (unsigned)m * 2u : 0u;   // (past the result's edge: the row's first bytes; what they produce is not stored)
        colQ = n < N ? (unsigned)n * 2u : 0u;
    };
    set_columns();
    // ids of the step: read first, so that they are there when the fragments' reads behind them are still on their way
    int tok[2];
    auto read_ids = [&](int step) {
        const unsigned at = lds0 + L::IDS_AT + (step & (FLOW_IDS - 1)) * 128 + kk * 4;
        tok[0] = lds_read32_async<0>(at);
        tok[1] = lds_read32_async<64>(at);
    };
    auto issue_data = [&]() {
        char* to = smem + (sd & 1) * L::STAGE + wave * 1024;
        const int left = cd.rec.y - cd.r;
#pragma unroll
        for (int j = 0; j < 2; ++j) {
            asm volatile("" : "+v"(tok[j]));
            const unsigned offP = __umul24((unsigned)tok[j], pitchP) + colP, offQ = __umul24((unsigned)tok[j], pitchQ) + colQ;
            if (left >= BK) {
                dma16(pb + (size_t)offP, to + j * 4096);
                dma16(qb + (size_t)offQ, to + L::HALF + j * 4096);
                asm volatile("; whole step");   // (keeps the two forms apart: this one has 32-bit lane addresses)
            } else {                            // the last step of a list
                const bool ok = kk + 16 * j < left;
                dma16(ok ? pb + (size_t)offP : zero, to + j * 4096);
                dma16(ok ? qb + (size_t)offQ : zero, to + L::HALF + j * 4096);
            }
        }
        ++sd;
        cd.r += BK;
        if (cd.r >= cd.rec.y) {
            settle(cd);
            set_columns();
        }
    };

    // ---- fragments -----------------------------------------------------------------------------------------------------------------
    unsigned sa, sb;
    {
        const int grp = lane >> 4, sl = lane & 15, row = (grp >> 1) * 8 + (sl >> 2);
        auto at = [&](int col) { return lds0 + row * 256 + (((col >> 3) ^ ((row & 3) << 2)) << 4) + (col & 7) * 2; };
        const int c = (grp & 1) * 16 + (sl & 3) * 4;
        sa = at(wr * 64 + c);
        sb = at(wf * 64 + c) + L::HALF;
    }
    // (32 columns on: chunk 4 on, whose swizzle is that of the first with bit 2 the other way)
    const int on = (lane >> 2) & 1 ? -64 : 64;
    union Frag { V v; u32x4 q; s16x4 h[2]; };
    f32x16 acc[2][2];
    auto clear = [&]() { zero_acc(acc); };

    if (todo > 0) {
        issue_ids();
        issue_ids();
        wait_vmcnt<0>();
        barrier_nofence();
        read_ids(0);
        lds_wait();
        issue_data();
        issue_ids();
        read_ids(1);
        lds_wait();
    }
    int g = 0;                                  // the step that is multiplied
    bool lax = false;                           // the last block's stores are younger than the copies waited for
    constexpr int STORES = OUT32 ? 16 : 8;      // of a wavefront and whole block
    const bool streaming = p.stream_dw != 0, accumulate = p.accumulate != 0;
    for (int j = 0; j < rounds; ++j) {
        const int4 it = record(lds0 + L::ITEMS_AT + j * 16);
        if (it.x < 0) continue;
        clear();
        for (int kt = 0; kt < it.y; ++kt) {
            if (lax) wait_vmcnt<STORES>();
            else wait_vmcnt<0>();
            lax = false;
            barrier_nofence();
            const unsigned stage = (g & 1) * L::STAGE;
            const bool more = g + 1 < todo;
            Frag a[2][2], b[2][2];              // [step of 16][block of 32]
            const unsigned ra = sa + stage, rb = sb + stage;
            static_for<2>([&](auto kc) {
                constexpr int OFF = decltype(kc)::value * 4096;
#pragma unroll
                for (int i = 0; i < 2; ++i) {
                    Frag& fa = a[OFF / 4096][i];
                    Frag& fb = b[OFF / 4096][i];
                    const unsigned ta = ra + i * on, tb = rb + i * on;
                    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(fa.h[0]) : "v"(ta), "n"(OFF));
                    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(fa.h[1]) : "v"(ta), "n"(OFF + 1024));
                    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(fb.h[0]) : "v"(tb), "n"(OFF));
                    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(fb.h[1]) : "v"(tb), "n"(OFF + 1024));
                }
            });
            if (more) {
                issue_data();
                issue_ids();
                read_ids(g + 2);                // (landed with the copies of this step)
            }
            lds_wait();
#pragma unroll
            for (int x = 0; x < 4; ++x) { asm volatile("" : "+v"(a[x >> 1][x & 1].q)); asm volatile("" : "+v"(b[x >> 1][x & 1].q)); }
#pragma unroll
            for (int ks = 0; ks < 2; ++ks)
#pragma unroll
                for (int f = 0; f < 2; ++f)
#pragma unroll
                    for (int i = 0; i < 2; ++i) acc[f][i] = Mfma<TC>::run(b[ks][f].v, a[ks][i].v, acc[f][i]);
            ++g;
        }
        if (it.y == 0 && accumulate && it.w < 0) continue;
        asm volatile("s_nop 15\n\ts_nop 15");   // (the writes below are inline assembly: the products' results have to be in their registers)

        // ---- result: a wavefront's 64 x 64 values through its own 4 KB of the stage that has just been multiplied (its next
        // copies are issued behind the next step's barrier), 16 rows of 32 bits or 32 of 16 at a time.  The 16-byte pieces of a row
        // change places with the row's number, so that the lanes of a write, each in a row of its own, meet different banks.
        barrier_nofence();                      // every wavefront has read its fragments
        const int m0 = flow_row_block(it.z) * BM + wr * 64, n0 = flow_col_block(it.z) * BN + wf * 64;
        const bool whole = it.w < 0;
        const size_t per = (size_t)M * N;
        const unsigned stg = lds0 + ((g + 1) & 1) * L::STAGE + wave * 4096;
        int ln = lane;                          // (addresses worked out here, not kept over the whole kernel)
        asm volatile("" : "+v"(ln));
        auto passes = [&](auto f32c, auto store) {
            constexpr bool F32 = decltype(f32c)::value;
            constexpr int ROWS = F32 ? 16 : 32, PASSES = 32 / ROWS, LPR = F32 ? 16 : 8;      // lanes per row of a store
            const unsigned put = stg + (ln & (ROWS - 1)) * (16 * LPR);
            static_for<2 * PASSES>([&](auto pc) {
                constexpr int i = decltype(pc)::value / PASSES, pass = decltype(pc)::value % PASSES;
                if ((ln & 31) / ROWS == pass) {
                    static_for<8>([&](auto uc) {
                        constexpr int f = decltype(uc)::value >> 2, q = decltype(uc)::value & 3;
                        const f32x16& v = acc[f][i];
                        if constexpr (F32) lds_write128<0>(put + (((f * 8 + q * 2 + (ln >> 5)) ^ (ln & 15)) << 4), u32x4{__float_as_uint(v[4 * q]), __float_as_uint(v[4 * q + 1]), __float_as_uint(v[4 * q + 2]), __float_as_uint(v[4 * q + 3])});
                        else lds_write64<0>(put + (((f * 4 + q) ^ (ln & 7)) << 4) + (ln >> 5) * 8, pack4<TC>(v[4 * q], v[4 * q + 1], v[4 * q + 2], v[4 * q + 3]));
                    });
                }
                // (a wavefront's LDS accesses happen in order)
                u32x4 v[4];
                static_for<4>([&](auto qc) {
                    constexpr int q = decltype(qc)::value;
                    const int row = q * (64 / LPR) + ln / LPR;
                    v[q] = lds_read128_async(stg + row * (16 * LPR) + (((ln & (LPR - 1)) ^ (row & (LPR - 1))) << 4));
                });
                lds_wait();
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    asm volatile("" : "+v"(v[q]));
                    const int m = m0 + i * 32 + pass * ROWS + q * (64 / LPR) + ln / LPR, n = n0 + (ln & (LPR - 1)) * (F32 ? 4 : 8);
                    if (m < M && n < N) store((unsigned)m * (unsigned)N + (unsigned)n, v[q]);
                }
            });
        };
        if (!OUT32 && whole && !accumulate) {
            char* const to = reinterpret_cast<char*>(p.dw) + (size_t)it.x * per * 2;
            passes(std::false_type(), [&](unsigned at, u32x4 v) { global_store128(to, at * 2u, v, streaming); });
        } else {
            char* const to = whole ? reinterpret_cast<char*>(p.dw) + (size_t)it.x * per * (OUT32 ? 4 : 2)
                                   : reinterpret_cast<char*>(p.scratch) + (size_t)it.w * per * 4;
            passes(std::true_type(), [&](unsigned at, u32x4 v) {
                float o[4] = {__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w)};
                if (whole && accumulate) {      // (waits for every copy in flight, too)
                    if (OUT32) {
                        u32x4 old = global_load128_async(to, at * 4u);
                        wait_vmcnt<0>();
                        asm volatile("" : "+v"(old));
                        o[0] += __uint_as_float(old.x); o[1] += __uint_as_float(old.y); o[2] += __uint_as_float(old.z); o[3] += __uint_as_float(old.w);
                    } else {
                        unsigned long old;
                        asm volatile("global_load_dwordx2 %0, %1, %2" : "=v"(old) : "v"(at * 2u), "s"(to));
                        wait_vmcnt<0>();
                        asm volatile("" : "+v"(old));
                        const unsigned x = (unsigned)old, y = (unsigned)(old >> 32);
                        o[0] += lo16<TC>(x); o[1] += hi16<TC>(x); o[2] += lo16<TC>(y); o[3] += hi16<TC>(y);
                    }
                }
                if (OUT32 || !whole) {
                    global_store128(to, at * 4u, u32x4{__float_as_uint(o[0]), __float_as_uint(o[1]), __float_as_uint(o[2]), __float_as_uint(o[3])}, whole && streaming);
                } else {
                    const uint2 pk = pack4<TC>(o[0], o[1], o[2], o[3]);
                    const unsigned long w = (unsigned long)pk.x | ((unsigned long)pk.y << 32);
                    asm volatile("global_store_dwordx2 %0, %1, %2" ::"v"(at * 2u), "v"(w), "s"(to) : "memory");
                }
            });
        }
        // (at least STORES stores of this wavefront behind the copies of the next step)
        lax = !accumulate && m0 + 64 <= M && n0 + 64 <= N;
    }
}

// the kernel's arguments; returns the grid (0: nothing to do)
// (workgroups for four a CU.  The second of the shared backward launches holds three, see backward16_kernel: there, behind the ESMM's workgroups,
// the last quarter starts when others end.  With three a CU dealt: 26.4 us instead of 25.8 at 2304 rows, 56 instead of 57 at 9216.)
inline int flow_args(const EstmmArgs& a, FlowK& p) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 8) cus = 256;
    p.pm = a.p; p.qm = a.q; p.dw = a.dw; p.token_ids = a.r.token_ids; p.offsets = a.r.offsets; 
    p.T = a.r.T; p.k = a.r.k; p.E = a.r.E; p.M = a.m_dim; p.N = a.n_dim;
    p.mtn = div_up(a.m_dim, 128); p.ntn = div_up(a.n_dim, 128);
    p.p_slot_rows = a.p_per_slot ? a.r.T : 0;
    p.q_slot_rows = a.q_per_slot ? a.r.T : 0;
    p.accumulate = a.accumulate;
    p.stream_dw = option(OPT_ESMM_STREAM) != 2;
    // runs of about nine blocks on one XCD (1024 x 4096: 8 instead of 24, 760 -> 727 us with a skewed load; 384 x 1536: 9 instead of 3, 71 ->
    // 65; 256 x 1024: 6 instead of 2, 56 -> 46)
    const int inside = std::min(p.mtn, p.ntn);
    p.group = inside * run_length(OPT_ESTMM_GROUP, std::max(1, 9 / inside));
    const bool cut = a.plan && a.scratch && a.max_slots >= 2;
    p.plan = cut ? a.plan : nullptr;
    p.scratch = cut ? a.scratch : nullptr;
    // a list cut into n parts adds n - 1 units and holds n >= 2 of the slots
    const int units = a.r.E + (cut ? (int)std::min<long>(a.max_slots - 1, (long)a.r.E * (PLAN_MAX_PARTS - 1)) : 0);
    const long padded = round_up((long)units * p.mtn * p.ntn, 8 * p.group);
    p.wg_per_xcd = (int)std::min<long>(4 * (cus / 8), padded / 8);
    p.rounds = p.wg_per_xcd > 0 ? (int)((padded / 8 + p.wg_per_xcd - 1) / p.wg_per_xcd) : 0;
    return 8 * p.wg_per_xcd;
}

inline bool flow_rounds_fit(const FlowK& p, int k) { return p.rounds <= FLOW_MAX_ITEMS && p.rounds * k <= FLOW_MAX_SEGS; }

}  // namespace
}  // namespace hexa
