// Routing front end for gfx950: softmax + top-k + GShard auxiliary loss, and the loss's backward
// through the softmax (the gate projection itself is in gate.hip).  These are small HBM-/latency-bound kernels that replace a
// dozen framework launches per MoE depth (fp32 cast, a skinny fp32 GEMM, softmax, top-k select + sort,
// one-hot scatter, reductions).
//
// Reference: hexa_moe_cuda/hexa_moe/gates/top.py:17-19 (fp32 gate projection),
//            hexa_moe_cuda/hexa_moe/impls/cascaded_moe.py:515-531 (noise, softmax, loss selection),
//            hexa_moe_cuda/hexa_moe/impls/layers.py:476-484 (top-k), impls/losses.py:12-19 (GShard loss).
#include "hexa_internal.h"
#include "small_bodies.h"
#include "gate_bodies.h"
#include "dma_common.h"

namespace hexa {
namespace {

// ---- softmax + top-k + per-workgroup loss partials ----------------------------------------------------
// One token per lane, three passes over its logits row (max, sum of exp, scores + selection); the row
// is tiny (E floats) and stays in L1/L2.  Ties go to the lower expert index.
constexpr int MAX_TOPK = 8;

constexpr int ROUTER_TB = 64;   // tokens (= lanes) per workgroup of the softmax/top-k kernel

constexpr int ROUTER_LDS_E = 240;   // up to this many experts the workgroup's 64 x E tile is staged in LDS

// insertion of (cv, ci) into a descending list of k entries; strict '>' keeps the lower index on ties
template <int N> __device__ __forceinline__ void topk_insert(float (&best_v)[N], int (&best_i)[N], int k, float cv, int ci) {
#pragma unroll
    for (int j = 0; j < N; ++j) {
        if (j < k && cv > best_v[j]) {
            const float tv = best_v[j]; const int ti = best_i[j];
            best_v[j] = cv; best_i[j] = ci; cv = tv; ci = ti;
        }
    }
}

// One token per lane for any number of experts: every lane walks its own row in global memory (three passes,
// L1-resident) and the per-expert sums are wavefront reductions.  Used above ROUTER_LDS_E experts.
__global__ __launch_bounds__(ROUTER_TB) void router_fwd_kernel(float* __restrict__ scores, int32_t* __restrict__ idx,
                                                         float* __restrict__ part_me, float* __restrict__ part_cnt,
                                                         const float* __restrict__ logits,
                                                         const float* __restrict__ noise, float noise_scale,
                                                         int num_tokens, int E, int k) {
    extern __shared__ float sh[];          // me[E] column sums of the wavefront, cnt[E]
    float* s_me = sh;
    float* s_cnt = sh + E;
    for (int i = threadIdx.x; i < 2 * E; i += blockDim.x) sh[i] = 0.f;
    const int lane = threadIdx.x;
    const int t = blockIdx.x * ROUTER_TB + lane;
    const bool ok = t < num_tokens;
    __syncthreads();
    // The selection is total: a row of NaN scores (NaN or +Inf logits) beats no entry, so the list starts out
    // as experts 0..k-1 and such a token stays routed (torch.topk also returns valid ids for NaN rows); its
    // NaN then reaches the output through the token's own features and the loss through the score sums.
    float best_v[MAX_TOPK];
    int best_i[MAX_TOPK];
#pragma unroll
    for (int j = 0; j < MAX_TOPK; ++j) { best_v[j] = -INFINITY; best_i[j] = j; }
    const float* lr = logits + (size_t)(ok ? t : 0) * E;
    const float* nr = noise ? noise + (size_t)(ok ? t : 0) * E : nullptr;
    float mx = -INFINITY;
    for (int e = 0; e < E; ++e) mx = fmaxf(mx, nr ? lr[e] + noise_scale * nr[e] : lr[e]);
    float sum = 0.f;
    for (int e = 0; e < E; ++e) sum += expf((nr ? lr[e] + noise_scale * nr[e] : lr[e]) - mx);
    const float inv = 1.0f / sum;
    for (int e = 0; e < E; ++e) {        // uniform trip count: every lane takes part in the reductions
        const float v = nr ? lr[e] + noise_scale * nr[e] : lr[e];
        const float sc = ok ? expf(v - mx) * inv : 0.f;
        if (ok) scores[(size_t)t * E + e] = sc;
        topk_insert(best_v, best_i, k, sc, e);
        // column sum over the wavefront: xor butterfly, a fixed summation tree
        float r = sc;
#pragma unroll
        for (int m = 32; m > 0; m >>= 1) r += __shfl_xor(r, m);
        if (lane == 0) s_me[e] = r;
    }
    if (ok) {
#pragma unroll
        for (int j = 0; j < MAX_TOPK; ++j)
            if (j < k) idx[(size_t)t * k + j] = best_i[j];
        atomicAdd(&s_cnt[best_i[0]], 1.0f);            // exact: at most 64 ones per counter
    }
    __syncthreads();
    for (int e = threadIdx.x; e < E; e += blockDim.x) {
        part_me[(size_t)blockIdx.x * E + e] = s_me[e];
        part_cnt[(size_t)blockIdx.x * E + e] = s_cnt[e];
    }
}

// Up to ROUTER_LDS_E experts: FOUR lanes per token (256 threads for the workgroup's 64 tokens).  One lane per
// token leaves a 64-thread workgroup walking E-long dependent chains (max, exp and sum, selection) on a chip that
// holds a few hundred such workgroups at once -- latency, not work, sets the time (18.8 us against 8.8 us at
// 18432 tokens and 32 experts).  Lane q of a
// token owns the experts e = q, q + 4, ...; maxima, sums and the top-k lists are combined over the four lanes
// with quad shuffles.  The 64 x E tile sits token-major in LDS (pitch 4 x odd: the 64 lanes of a wavefront --
// 16 tokens x 4 -- hit every bank twice, the minimum), is loaded and written back with coalesced 16-byte
// accesses when E is a multiple of 4, and the per-expert sums run over it in token order.
constexpr int ROUTER_G = 4;
__host__ __device__ constexpr int router_pitch(int E) {
    int p = (E + 3) / 4;            // in units of 4 floats
    if ((p & 1) == 0) ++p;
    return 4 * p;
}

// hist (optional): [k][workgroups][E] ints, per slot the number of this workgroup's 64 tokens that chose each expert
// -- the histogram the routing pass starts from (units of 64 tokens), so that pass needs no counting launch.
// LDS of the four-lanes-per-token router: cnt[E], the tile [64][P] (with the load-importance loss a second one: logits
// without the noise, then Phi), then hist[k][E]
struct Router4Lds {
    float* cnt; float* tile; float* clean; int* hist; int P;
    __device__ __forceinline__ Router4Lds(float* sh, int E, bool li) : cnt(sh), tile(sh + ((E + 3) & ~3)), P(router_pitch(E)) {
        clean = tile + ROUTER_TB * P;
        hist = reinterpret_cast<int*>(li ? clean + ROUTER_TB * P : clean);
    }
};
__host__ __device__ constexpr size_t router4_lds_floats(int E, int k, bool hist, bool li) {
    return (size_t)((E + 3) & ~3) + (size_t)(li ? 2 : 1) * ROUTER_TB * router_pitch(E) + (hist ? (size_t)k * E : 0);
}

// What the load-importance loss (impls/losses.py:21-42) needs on top: thr[t] = the k-th choice's noisy LOGIT;
// s = softmax(logits) without noise (what `scores` then holds); importance[e] += s[e]; load[e] += Phi((s[e] - thr) / sigma).
struct LiK { float* thr; const float* noise; float noise_scale, inv_sigma; };
__device__ __forceinline__ float normal_cdf(float z) { return 0.5f * erfcf(-z * 0.70710678118654752f); }

// A lane's experts q, q + 4, ...: f(i, e) for each below E -- N of them at most, unrolled (the values can stay in registers), or any number
// (N = 0)
template <int N, typename F> __device__ __forceinline__ void lane_experts(int q, int E, F&& f) {
    if constexpr (N > 0) {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if (q + ROUTER_G * i < E) f(i, q + ROUTER_G * i);
    } else {
        for (int e = q; e < E; e += ROUTER_G) f(0, e);
    }
}

// Softmax, top-k, loss and histogram of one token by its four lanes.  N: see lane_experts; KMAX: the longest list.  (144 tokens of 32 experts,
// top-1: 7000 cycles with the values in LDS between the passes and lists of eight, 3400 so.)
template <bool LI, int N, int KMAX>
__device__ __forceinline__ void router4_rows(const Router4Lds& L, int32_t* __restrict__ idx, bool hist, int t0, int rows, int E, int k, const LiK& li) {
    constexpr bool REGS = N > 0;
    constexpr int NV = REGS ? N : 1;
    const int tid = threadIdx.x, r = tid >> 2, q = tid & 3;
    const int t = t0 + r;
    const bool ok = r < rows;
    float* row = L.tile + r * L.P;
    float v[NV];
    // The selection is total: a row of NaN scores (NaN or +Inf logits) beats no entry, so the lists start out as
    // the lanes' own experts in index order and such a token ends up with experts 0..k-1 (torch.topk also returns
    // valid ids for NaN rows); its NaN then reaches the output through the token's own features and the loss
    // through the score sums.
    float bv[KMAX];
    int bi[KMAX];
#pragma unroll
    for (int j = 0; j < KMAX; ++j) { bv[j] = -INFINITY; bi[j] = q + ROUTER_G * j; }
    // scores of the logits in `from` into `to`
    auto softmax = [&](const float* from, float* to, auto&& each) {
        if constexpr (REGS) lane_experts<N>(q, E, [&](int i, int e) { v[i] = from[e]; });
        float mx = -INFINITY;
        lane_experts<N>(q, E, [&](int i, int e) { mx = fmaxf(mx, REGS ? v[i] : from[e]); });
        mx = fmaxf(mx, __shfl_xor(mx, 1));
        mx = fmaxf(mx, __shfl_xor(mx, 2));
        float sum = 0.f;
        lane_experts<N>(q, E, [&](int i, int e) {
            const float ex = expf((REGS ? v[i] : from[e]) - mx);
            if (REGS) v[i] = ex;
            else to[e] = ex;
            sum += ex;
        });
        sum += __shfl_xor(sum, 1);         // (s0 + s1) + (s2 + s3) on every lane of the quad
        sum += __shfl_xor(sum, 2);
        const float inv = 1.0f / sum;
        lane_experts<N>(q, E, [&](int i, int e) {
            const float sc = (REGS ? v[i] : to[e]) * inv;
            to[e] = sc;
            each(e, sc);
        });
    };
    if (ok) softmax(row, row, [&](int e, float sc) { topk_insert(bv, bi, k, sc, e); });   // ascending e, strict '>': the lower index stays ahead on ties
    else lane_experts<N>(q, E, [&](int, int e) { row[e] = 0.f; });
    // merge the four lists: k rounds, each takes the best head (greater score; lower index on ties)
    int pick[KMAX];
#pragma unroll
    for (int j = 0; j < KMAX; ++j) {
        pick[j] = 0;
        if (j < k) {
            float hv = bv[0];
            int hi = bi[0];
#pragma unroll
            for (int m = 1; m <= 2; m <<= 1) {
                const float ov = __shfl_xor(hv, m);
                const int oi = __shfl_xor(hi, m);
                if (ov > hv || (ov == hv && oi < hi)) { hv = ov; hi = oi; }
            }
            pick[j] = hi;
            if (hi == bi[0]) {
#pragma unroll
                for (int m = 0; m + 1 < KMAX; ++m) { bv[m] = bv[m + 1]; bi[m] = bi[m + 1]; }
                bv[KMAX - 1] = -INFINITY;
                bi[KMAX - 1] = 0x7fffffff;
            }
        }
    }
    if (ok) {
#pragma unroll
        for (int j = 0; j < KMAX; ++j)
            if (j < k && (j & 3) == q) {
                idx[(size_t)t * k + j] = pick[j];
                if (hist) atomicAdd(&L.hist[j * E + pick[j]], 1);
            }
        if (!LI && q == 0) atomicAdd(&L.cnt[pick[0]], 1.0f);   // exact: at most 64 ones per counter
    }
    if (LI) {
        float* clean = L.clean + r * L.P;
        if (ok) {
            int last = 0;
#pragma unroll
            for (int j = 0; j < KMAX; ++j)
                if (j == k - 1) last = pick[j];
            float thr = clean[last];
            if (li.noise) thr += li.noise_scale * li.noise[(size_t)t * E + last];
            if (q == 0) li.thr[t] = thr;
            softmax(clean, row, [&](int e, float sc) { clean[e] = normal_cdf((sc - thr) * li.inv_sigma); });
        } else {
            lane_experts<N>(q, E, [&](int, int e) { clean[e] = 0.f; });
        }
    }
}

// the sum of a column of the tile in token order, its values read 32 at a time
__device__ __forceinline__ float router4_column(const float* col, int P) {
    float m = 0.f;
    for (int r0 = 0; r0 < ROUTER_TB; r0 += 32) {
        float v[32];
#pragma unroll
        for (int i = 0; i < 32; ++i) v[i] = col[(r0 + i) * P];
#pragma unroll
        for (int i = 0; i < 32; i += 8) asm volatile("" : "+v"(v[i]), "+v"(v[i + 1]), "+v"(v[i + 2]), "+v"(v[i + 3]), "+v"(v[i + 4]), "+v"(v[i + 5]), "+v"(v[i + 6]), "+v"(v[i + 7]));
#pragma unroll
        for (int i = 0; i < 32; ++i) m += v[i];
    }
    return m;
}

// Everything behind the tile of (noisy) logits: softmax, top-k, loss partials, histogram, scores out.  The tile
// holds rows [t0, t0 + rows) of the workgroup; the counters have been cleared; a barrier separates both from here.
// The workgroup has at least ROUTER_TB * ROUTER_G threads.  FEW: E <= 64, the lanes keep their scores in registers.
template <bool LI, bool FEW>
__device__ __forceinline__ void router4_body(const Router4Lds& L, float* __restrict__ scores, int32_t* __restrict__ idx,
                                             float* __restrict__ part_me, float* __restrict__ part_cnt,
                                             int32_t* __restrict__ hist, int t0, int rows, int E, int k, int nblocks, const LiK& li) {
    float* s_cnt = L.cnt;
    float* tile = L.tile;
    int* s_hist = L.hist;
    const int P = L.P;
    const int tid = threadIdx.x;
    const size_t g0 = (size_t)t0 * E;
    const int total = rows * E;
    if (tid < ROUTER_TB * ROUTER_G) {   // four lanes per token; further wavefronts of the workgroup help with the sums only
        if constexpr (FEW) {
            if (E <= 32 && k <= 2) router4_rows<LI, 8, 2>(L, idx, hist != nullptr, t0, rows, E, k, li);
            else if (k <= 2) router4_rows<LI, 16, 2>(L, idx, hist != nullptr, t0, rows, E, k, li);
            else router4_rows<LI, 16, MAX_TOPK>(L, idx, hist != nullptr, t0, rows, E, k, li);
        } else {
            router4_rows<LI, 0, MAX_TOPK>(L, idx, hist != nullptr, t0, rows, E, k, li);
        }
    }
    __syncthreads();
    // per-expert sums over the 64 tokens, in token order; the scores leave coalesced
    for (int e = tid; e < E; e += blockDim.x) {
        const float m = router4_column(tile + e, P);
        part_me[(size_t)blockIdx.x * E + e] = m;
        if (!LI) part_cnt[(size_t)blockIdx.x * E + e] = s_cnt[e];
    }
    if (LI)
        for (int e = (tid + 128) % blockDim.x; e < E; e += blockDim.x) {      // (other wavefronts than the sums above)
            const float m = router4_column(L.clean + e, P);
            part_cnt[(size_t)blockIdx.x * E + e] = m;
        }
    if (hist)
        for (int i = tid; i < k * E; i += blockDim.x) {
            const int j = i / E, e = i - j * E;
            hist[((size_t)j * nblocks + blockIdx.x) * E + e] = s_hist[i];
        }
    if ((E & 3) == 0) {
        for (int i = tid * 4; i < total; i += blockDim.x * 4) {
            const int rr = i / E, e = i - rr * E;
            *reinterpret_cast<float4*>(scores + g0 + i) = *reinterpret_cast<const float4*>(tile + rr * P + e);
        }
    } else {
        for (int i = tid; i < total; i += blockDim.x) {
            const int rr = i / E, e = i - rr * E;
            scores[g0 + i] = tile[rr * P + e];
        }
    }
}

template <bool LI>
__global__ __launch_bounds__(ROUTER_TB * ROUTER_G) void router_fwd4_kernel(
    float* __restrict__ scores, int32_t* __restrict__ idx, float* __restrict__ part_me, float* __restrict__ part_cnt,
    const float* __restrict__ logits, const float* __restrict__ noise, float noise_scale, int num_tokens, int E, int k,
    int32_t* __restrict__ hist, LiK li) {
    extern __shared__ float sh[];
    const Router4Lds L(sh, E, LI);
    const int P = L.P;
    float* tile = L.tile;
    const int tid = threadIdx.x;
    const int t0 = blockIdx.x * ROUTER_TB;
    const int rows = min(ROUTER_TB, num_tokens - t0);
    for (int i = tid; i < E; i += blockDim.x) L.cnt[i] = 0.f;
    if (hist)
        for (int i = tid; i < k * E; i += blockDim.x) L.hist[i] = 0;
    // ---- tile in: element i of the contiguous block [rows][E] ----
    const size_t g0 = (size_t)t0 * E;
    const int total = rows * E;
    if ((E & 3) == 0) {
        for (int i = tid * 4; i < total; i += blockDim.x * 4) {
            float4 v = *reinterpret_cast<const float4*>(logits + g0 + i);
            const int r = i / E, e = i - r * E;
            if (LI) *reinterpret_cast<float4*>(L.clean + r * P + e) = v;
            if (noise) {
                const float4 n = *reinterpret_cast<const float4*>(noise + g0 + i);
                v.x += noise_scale * n.x; v.y += noise_scale * n.y; v.z += noise_scale * n.z; v.w += noise_scale * n.w;
            }
            *reinterpret_cast<float4*>(tile + r * P + e) = v;
        }
    } else {
        for (int i = tid; i < total; i += blockDim.x) {
            float v = logits[g0 + i];
            const int r = i / E, e = i - r * E;
            if (LI) L.clean[r * P + e] = v;
            if (noise) v += noise_scale * noise[g0 + i];
            tile[r * P + e] = v;
        }
    }
    __syncthreads();
    router4_body<LI, false>(L, scores, idx, part_me, part_cnt, hist, t0, rows, E, k, gridDim.x, li);
}

// The gate's projection and the router in one launch for 16-bit or fp32 token tensors and up to GATE_ROUTER_MAX_E
// experts: the workgroup's 64 x E logits go from the matrix cores into the router's LDS tile (and out to `logits`,
// which the backward reads) instead of through a launch boundary.  The arithmetic is that of gate_fwd_kernel, sum
// for sum: a 32-token block's model dimension is cut into the same four quarters, one per wavefront, each
// accumulated by the same sequence of products and added in the same order, so the logits are bit-identical to
// hexa_gate_logits'.  Eight wavefronts (two token blocks) project; the first four then route.
constexpr int GATE_ROUTER_MAX_E = 64;
constexpr int GATE_ROUTER_NT = 2 * ROUTER_TB * ROUTER_G;
//
// A launch of few tokens is one workgroup's chain, 27500 cycles of it at 144 tokens (384 wide, 32 experts, bf16): operands 7300, products 7000 (two
// wavefronts of a SIMD, 48 fp32 products of 64 cycles each), partial sums and logits 2500, softmax and lists 3400, the rest merge, sums
// over the tokens and stores.  wg is the same for every workgroup, and a lane that reads its own row of it fetches 16 bytes of 32 lines an
// instruction: a trip's 24 pieces of 16 bytes of every row come by asynchronous copy, whole lines at a time, into LDS for the two token
// blocks.  The token rows, half the bytes and nobody else's, go to registers, all of a trip's loads in flight.  The partial sums take the
// operands' place in LDS.  Against both operands read by the lanes, a sixth of them in flight at once, and the scores in LDS between the passes
// with lists of eight: 13.4 -> 11.4 us there, 14.6 -> 12.2 at 2304 tokens, 21.3 -> 19.6 at 18432, 81 -> 71 at 32768 tokens, 1024 wide, 64 experts.
// Beside workgroups that round (38 to 75 million weights), whose traffic makes every trip to memory
// longer: 34.5 -> 26.4 at 9216 fp32 tokens, 39 -> 33 at 3600, 768 wide, 43 -> 34 at 18432.
//
// Workgroups past the routing ones round fp32 master weights to 16 bits (`round`): the routing workgroups are a chain of
// latencies that leaves the memory idle, and these are nothing but memory traffic.  ROUND says what the launch rounds:
// nothing, weights, or the tokens too (x_src into x).
constexpr int ROUND_NONE = 0, ROUND_WEIGHTS = 1, ROUND_TOKENS = 2;
constexpr int GR_PIECES = 4 * FWD_NB;                                    // 16-byte pieces of a wg row in a trip
constexpr int GR_QUARTER = 32 * GR_PIECES * 16, GR_BYTES = 4 * GR_QUARTER;   // of the four quarters of the model dimension
// Where wg's values come from.  DIRECT: few experts are few lines an instruction, and every lane reads its own row: no barrier between trips, no
// chunk multiplied that a quarter does not have.  STAGED: through LDS as above, trips cut where a quarter's chunks end.  WHOLE: no trip is cut
// (384, 768, 1152 columns); for rounded tokens an instance of its own, because beside cut trips it spills 28 registers and the cuts cost it 0.7 to
// 1 us of 13 to 17.  us of the launch, DIRECT | STAGED, 8 experts, 144, 3600 and 18432 tokens.  bf16 tokens: 128 wide 8.0, 8.7, 11.8 | 9.2, 9.9, 12.4; 768 wide
// 14.2, 15.3, 24.8 | 16.9, 17.8, 27.1; 1024 wide 16.4, 17.9, 29.5 | 21.0, 22.1, 33.9; 16 experts, 512 wide 12.2, 13.0, 20.2 | 14.9, 15.9, 22.8; 32 experts, 384 wide,
// 144 and 9216 tokens 11.7, 13.3 | 10.7, 12.3.  Rounded tokens beside 8 experts' weights, d x 4d: 128 wide 8.8, 10.3, 14.1 | 10.4, 11.6, 15.7; 512
// wide 20.1, 19.5, 28.4 | 23.1, 22.4, 29.6; 640 wide 24.2, 25.3, 42.7 | 26.3, 26.9, 41.2; 1024 wide 46.4, 46.6, 68.7 | 43.2, 44.2, 63.7; 4 experts, 1024 wide 29.9,
// 31.5, 58.8 | 32.7, 33.4, 59.5.  Against WHOLE: 384 wide 16.3, 16.6, 23.3 | 16.8, 17.2, 23.2, 16 experts 19.6, 19.6, 26.2 | 19.3, 19.4, 24.1; 768 wide 29.2, 33.4,
// 51.1 | 28.3, 31.1, 48.2; 1152 wide 53.7, 53.9, 80.6 | 47.7, 49.2, 74.2.
constexpr int GR_DIRECT = 0, GR_STAGED = 1, GR_WHOLE = 2;
constexpr int GR_DIRECT_E = 16;
constexpr int GR_AHEAD = 2;              // chunks in registers: one is under way while the other is multiplied
inline int gate_router_mode(int d, int E, bool tokens) {
    if (!tokens) return E <= GR_DIRECT_E ? GR_DIRECT : GR_STAGED;
    const bool whole = d % (4 * FWD_NB * 16) == 0;
    if (E <= GR_DIRECT_E && (whole ? E <= 8 && d <= 512 : d <= 512 || (d <= 1024 && E * d <= 5120))) return GR_DIRECT;
    return whole ? GR_WHOLE : GR_STAGED;
}
constexpr int GR_DIRECT_BYTES = 2 * 4 * 16 * 64 * 4;                     // the partial sums
static_assert(GR_BYTES >= GR_DIRECT_BYTES, "the partial sums fit in the operands' place");
static_assert(GR_BYTES >= 4 * ROUTER_TB * router_pitch(GATE_ROUTER_MAX_E) && GR_DIRECT_BYTES >= 4 * ROUTER_TB * router_pitch(GR_DIRECT_E),
              "the logits without the noise fit in the operands' place");
static_assert(GR_QUARTER % 2048 == 0, "copies of 1 KB, half of them by either token block's wavefront");
// piece p of row r sits in slot (p + r / 2) of its row: rows are 24 slots apart, 16 lanes read 16 different groups of four banks
__device__ __forceinline__ int gr_turn(int row) { return (row & 15) >> 1; }
template <typename T, bool LI, int ROUND, int MODE>
__global__ __launch_bounds__(GATE_ROUTER_NT, 4) void gate_router_kernel(
    float* __restrict__ logits, float* __restrict__ scores, int32_t* __restrict__ idx, float* __restrict__ part_me,
    float* __restrict__ part_cnt, std::conditional_t<ROUND == ROUND_TOKENS, T, const T>* __restrict__ x, const float* __restrict__ x_src,
    const float* __restrict__ wg, const float* __restrict__ noise,
    float noise_scale, int num_tokens, int d, int E, int k, int32_t* __restrict__ hist, int nblocks, LiK li, RoundAllK round) {
    extern __shared__ float sh[];
    __shared__ __attribute__((aligned(1024))) char operands[MODE == GR_DIRECT ? GR_DIRECT_BYTES : GR_BYTES];
    float (*part)[4][16][64] = reinterpret_cast<float (*)[4][16][64]>(operands);    // [token block][quarter of d][result register][lane]
    constexpr bool SRC32 = ROUND == ROUND_TOKENS;
    constexpr int NB = FWD_NB;
    constexpr bool WHOLE = MODE == GR_WHOLE;         // every quarter is whole trips, every chunk two pieces: nothing is asked for
    if (ROUND != ROUND_NONE && (int)blockIdx.x >= nblocks) {
        round_all_body(round, blockIdx.x - nblocks);
        return;
    }
    Router4Lds L(sh, E, false);
    if (LI) L.clean = reinterpret_cast<float*>(operands);    // (behind the projection; with a place of its own 64 experts left one workgroup a CU)
    const int P = L.P;
    float* tile = L.tile;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int t0 = blockIdx.x * ROUTER_TB;
    const int rows = min(ROUTER_TB, num_tokens - t0);
    for (int i = tid; i < E; i += blockDim.x) L.cnt[i] = 0.f;
    if (hist)
        for (int i = tid; i < k * E; i += blockDim.x) L.hist[i] = 0;
    // ---- the gate: logits of 64 tokens into the tile ----
    const int r = lane & 31, h = lane >> 5;
    const int blk = wave >> 2, quarter = wave & 3;
    const int pieces = d >> 3;                       // 8 contraction indices per piece
    const int chunks = (pieces + 1) >> 1;            // a chunk = one piece per half-wavefront
    const int c0 = (chunks * quarter) >> 2, c1 = (chunks * (quarter + 1)) >> 2;
    const bool tok_ok = t0 + 32 * blk + r < num_tokens;
    const size_t xat = (size_t)(tok_ok ? t0 + 32 * blk + r : 0) * d;
    using X = std::conditional_t<SRC32, float, T>;   // what is read
    const X* xrow;
    if constexpr (SRC32) xrow = x_src + xat;
    else xrow = x + xat;
    const char* const mine = operands + quarter * GR_QUARTER;
    for (int e0 = 0; e0 < (MODE == GR_DIRECT ? 1 : E); e0 += 32) {
        const bool exp_ok = e0 + r < E;
        f32x16 acc = zero16();
        // this lane's piece of a chunk as values; rounded tokens are stored, too: every piece of the workgroup's rows is some lane's once per block of
        // experts.  (The caller says which piece: from its own trip's h, see there.)
        auto values = [&](const Raw8<X>& from, int piece, bool ok, float (&a)[8]) {
#pragma unroll
            for (int i = 0; i < 8; ++i) a[i] = from.value(i);
            if constexpr (SRC32) {
                union { uint4 q; T t[8]; } o;
#pragma unroll
                for (int i = 0; i < 8; ++i) {
                    o.t[i] = (T)a[i];
                    a[i] = (float)o.t[i];
                }
                if (e0 == 0 && ok && (WHOLE || piece < pieces) && tok_ok) *reinterpret_cast<uint4*>(x + xat + (size_t)piece * 8) = o.q;
            }
        };
        if constexpr (MODE == GR_DIRECT && SRC32) {
            // Two chunks of an fp32 row are a line of 128 bytes and asked for together.  (One at a time and one ahead, as below, with a workgroup's lines as
            // large as the L1: 83 us instead of 71 at 32768 tokens, 1024 wide, 8 experts.)
            const float* const wrow = wg + (size_t)(exp_ok ? r : 0) * d;
            for (int c = c0; c < c1; c += 2) {
                Raw8<X> xv[2];
                Raw8<float> wv[2];
                float a[2][8];
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    const int piece = 2 * (c + u) + h;
                    const bool ok = c + u < c1 && piece < pieces;
                    xv[u].load(xrow + (ok ? piece : 0) * 8, ok && tok_ok);
                    wv[u].load(wrow + (ok ? piece : 0) * 8, ok && exp_ok);
                }
#pragma unroll
                for (int u = 0; u < 2; ++u) values(xv[u], 2 * (c + u) + h, c + u < c1, a[u]);
#pragma unroll
                for (int u = 0; u < 2; ++u)
#pragma unroll
                    for (int i = 0; i < 8; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[u][i], wv[u].value(i), acc, 0, 0, 0);
            }
        } else if constexpr (MODE == GR_DIRECT) {
            // (lanes without an expert or a token read another's: their column or row of the logits is nobody's)
            const X* const xblock = x + (size_t)t0 * d;
            const unsigned wat = (exp_ok ? r : 0) * d, tat = (tok_ok ? 32 * blk + r : 0) * d;
            Raw8<X> xv[GR_AHEAD];
            Raw8<float> wv[GR_AHEAD];
            auto fetch = [&](int u, int chunk) {
                chunk = min(chunk, c1 - 1);
                const unsigned at = (chunk * 2 + (2 * chunk + h < pieces ? h : 0)) * 8;
                wv[u].load(wg + (wat + at), true);
                xv[u].load(xblock + (tat + at), true);
            };
            auto multiply = [&](int u, int chunk) {
                wv[u].arrive();
                xv[u].arrive();
                float a[8];
                values(xv[u], 2 * chunk + h, true, a);
                const bool there = 2 * chunk + h < pieces;           // (the last chunk may have one piece)
#pragma unroll
                for (int i = 0; i < 8; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(there ? a[i] : 0.f, there ? wv[u].value(i) : 0.f, acc, 0, 0, 0);
            };
            if (c0 < c1) {
#pragma unroll
                for (int u = 0; u < GR_AHEAD; ++u) fetch(u, c0 + u);
                int c = c0;
                for (; c + GR_AHEAD <= c1; c += GR_AHEAD) {
#pragma unroll
                    for (int u = 0; u < GR_AHEAD; ++u) {
                        multiply(u, c + u);
                        fetch(u, c + u + GR_AHEAD);
                        asm volatile("" ::: "memory");
                    }
                }
#pragma unroll
                for (int u = 0; u < GR_AHEAD - 1; ++u)
                    if (c + u < c1) multiply(u, c + u);
            }
        } else {
        for (int c = 0; c < (chunks + 3) >> 2; c += NB) {            // (the quarters are of one length, or one chunk shorter)
            if (c > 0) __syncthreads();                              // the trip before has been read
            int ln = lane;               // (addresses worked out in every trip, not kept over all of them)
            asm volatile("" : "+v"(ln));
            const int r = ln & 31, h = ln >> 5;
            // this wavefront's half of its quarter's rows of wg, and its own token rows
#pragma unroll
            for (int i = 0; i < GR_QUARTER / 2048; ++i) {
                const int at = (blk * (GR_QUARTER / 2048) + i) * 64 + ln, row = at / GR_PIECES, slot = at - row * GR_PIECES;
                int p = slot - gr_turn(row);
                if (p < 0) p += GR_PIECES;
                const int col = (c0 + c) * 16 + p * 4;
                if (e0 + row >= E || (!WHOLE && c0 + c + (p >> 2) >= c1)) continue;     // (those columns of the logits are nobody's, those chunks not multiplied)
                const float* src = WHOLE || col < d ? wg + (size_t)(e0 + row) * d + col : reinterpret_cast<const float*>(g_gate_zeros);
                dma16(src, operands + quarter * GR_QUARTER + (blk * (GR_QUARTER / 2048) + i) * 1024);
            }
            Raw8<X> xv[NB];
#pragma unroll
            for (int u = 0; u < NB; ++u) {
                const int piece = 2 * (c0 + c + u) + h;
                const bool ok = WHOLE || (c0 + c + u < c1 && piece < pieces);
                xv[u].load(xrow + (ok ? piece : 0) * 8, ok && tok_ok);
            }
            wait_vmcnt<0>();                                         // this wavefront's copies have landed: the barrier waits for LDS accesses only
#pragma unroll
            for (int u = 0; u < NB; ++u) xv[u].arrive();
            __syncthreads();
            f32x4 b[2][2];               // a chunk's values of wg, read while the chunk before it is multiplied
            auto read = [&](int u) {
#pragma unroll
                for (int q = 0; q < 2; ++q) {
                    int slot = 4 * u + 2 * h + q + gr_turn(r);
                    if (slot >= GR_PIECES) slot -= GR_PIECES;
                    b[u & 1][q] = *reinterpret_cast<const f32x4*>(mine + (r * GR_PIECES + slot) * 16);
                }
            };
            auto multiply = [&](auto all) {                          // all: the quarter has chunks for the whole trip
                read(0);
#pragma unroll
                for (int u = 0; u < NB; ++u) {
                    if (!decltype(all)::value && c0 + c + u >= c1) break;
                    if (u + 1 < NB) read(u + 1);
                    asm volatile("" ::: "memory");       // (no further ahead: their registers)
                    float a[8];
                    values(xv[u], 2 * (c0 + c + u) + h, true, a);
#pragma unroll
                    for (int i = 0; i < 8; ++i) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[i], b[u & 1][i >> 2][i & 3], acc, 0, 0, 0);
                }
            };
            if constexpr (WHOLE) multiply(std::true_type());
            else if (!SRC32 && c0 + c + NB <= c1) multiply(std::true_type());
            else multiply(std::false_type());
        }
        }
        __syncthreads();                                             // the operands have been read
#pragma unroll
        for (int v = 0; v < 16; ++v) part[blk][quarter][v][lane] = acc[v];
        __syncthreads();
        // wavefront (blk, w) finishes result registers 4w .. 4w+3: token row 8w + 4h + q of the block, expert column r
#pragma unroll
        for (int q = 0; q < 4; ++q) {
            const int v = 4 * quarter + q;
            const float sum = ((part[blk][0][v][lane] + part[blk][1][v][lane]) + part[blk][2][v][lane]) + part[blk][3][v][lane];
            const int row = 32 * blk + 8 * quarter + 4 * h + q;
            if (exp_ok) tile[row * P + e0 + r] = sum;
        }
        __syncthreads();   // the partial sums have been consumed (the next expert block overwrites them)
    }
    // ---- the logits leave as they are; the noise joins the tile only ----
    const size_t g0 = (size_t)t0 * E;
    const int total = rows * E;
    if ((E & 3) == 0) {
        for (int i = tid * 4; i < total; i += blockDim.x * 4) {
            const int rr = i / E, e = i - rr * E;
            float4 v = *reinterpret_cast<const float4*>(tile + rr * P + e);
            *reinterpret_cast<float4*>(logits + g0 + i) = v;
            if (LI) *reinterpret_cast<float4*>(L.clean + rr * P + e) = v;
            if (noise) {
                const float4 n = *reinterpret_cast<const float4*>(noise + g0 + i);
                v.x += noise_scale * n.x; v.y += noise_scale * n.y; v.z += noise_scale * n.z; v.w += noise_scale * n.w;
                *reinterpret_cast<float4*>(tile + rr * P + e) = v;
            }
        }
    } else {
        for (int i = tid; i < total; i += blockDim.x) {
            const int rr = i / E, e = i - rr * E;
            const float v = tile[rr * P + e];
            logits[g0 + i] = v;
            if (LI) L.clean[rr * P + e] = v;
            if (noise) tile[rr * P + e] = v + noise_scale * noise[g0 + i];
        }
    }
    __syncthreads();
    router4_body<LI, true>(L, scores, idx, part_me, part_cnt, hist, t0, rows, E, k, nblocks, li);
}

// The GShard loss from the workgroup partials (see small_bodies.h) as a launch of its own.
__global__ __launch_bounds__(256) void router_loss_kernel(float* __restrict__ l_aux, float* __restrict__ me,
                                                          float* __restrict__ ce, const float* __restrict__ part_me,
                                                          const float* __restrict__ part_cnt, int nblocks,
                                                          int num_tokens, int E) {
    extern __shared__ float sh[];
    router_loss_body(sh, l_aux, me, ce, part_me, part_cnt, nblocks, num_tokens, E);
}

__global__ __launch_bounds__(256) void router_bwd_kernel(RouterBwdK p) {
    extern __shared__ float s_c[];
    router_bwd_body(s_c, p, blockIdx.x);
}


// ---- the load-importance loss above ROUTER_LDS_E experts ----------------------------------------------------
// One token per lane; the row (E floats) is walked in place, L1-resident.
__global__ __launch_bounds__(ROUTER_TB) void router_li_fwd_kernel(float* __restrict__ scores, int32_t* __restrict__ idx,
                                                                  float* __restrict__ thr_out,
                                                                  float* __restrict__ part_imp,
                                                                  float* __restrict__ part_load,
                                                                  const float* __restrict__ logits,
                                                                  const float* __restrict__ noise, float noise_scale,
                                                                  float inv_sigma, int num_tokens, int E, int k) {
    const int lane = threadIdx.x;
    const int t = blockIdx.x * ROUTER_TB + lane;
    const bool ok = t < num_tokens;
    const float* lr = logits + (size_t)(ok ? t : 0) * E;
    const float* nr = noise ? noise + (size_t)(ok ? t : 0) * E : nullptr;
    float best_v[MAX_TOPK];
    int best_i[MAX_TOPK];
#pragma unroll
    for (int j = 0; j < MAX_TOPK; ++j) { best_v[j] = -INFINITY; best_i[j] = j; }
    // noisy scores: selection only
    float mx = -INFINITY, cmx = -INFINITY;
    for (int e = 0; e < E; ++e) {
        const float c = lr[e];
        cmx = fmaxf(cmx, c);
        mx = fmaxf(mx, nr ? c + noise_scale * nr[e] : c);
    }
    float sum = 0.f, csum = 0.f;
    for (int e = 0; e < E; ++e) {
        const float c = lr[e];
        csum += expf(c - cmx);
        sum += expf((nr ? c + noise_scale * nr[e] : c) - mx);
    }
    const float inv = 1.0f / sum, cinv = 1.0f / csum;
    for (int e = 0; e < E; ++e) {
        const float v = nr ? lr[e] + noise_scale * nr[e] : lr[e];
        topk_insert(best_v, best_i, k, expf(v - mx) * inv, e);
    }
    int last = 0;
#pragma unroll
    for (int j = 0; j < MAX_TOPK; ++j)
        if (j == k - 1) last = best_i[j];
    float thr = 0.f;
    if (ok) {
        thr = nr ? lr[last] + noise_scale * nr[last] : lr[last];
        thr_out[t] = thr;
#pragma unroll
        for (int j = 0; j < MAX_TOPK; ++j)
            if (j < k) idx[(size_t)t * k + j] = best_i[j];
    }
    // clean scores, importance and load; uniform trip count: every lane takes part in the reductions
    for (int e = 0; e < E; ++e) {
        float sc = 0.f, ld = 0.f;
        if (ok) {
            sc = expf(lr[e] - cmx) * cinv;
            scores[(size_t)t * E + e] = sc;
            ld = normal_cdf((sc - thr) * inv_sigma);
        }
#pragma unroll
        for (int m = 32; m > 0; m >>= 1) { sc += __shfl_xor(sc, m); ld += __shfl_xor(ld, m); }
        if (lane == 0) {
            part_imp[(size_t)blockIdx.x * E + e] = sc;
            part_load[(size_t)blockIdx.x * E + e] = ld;
        }
    }
}

constexpr int ROUTER_LI_MAX_E = 1024;

__global__ __launch_bounds__(256) void router_li_loss_kernel(float* __restrict__ l_aux, float* __restrict__ importance,
                                                             float* __restrict__ load, float* __restrict__ g_imp,
                                                             float* __restrict__ g_load,
                                                             const float* __restrict__ part_imp,
                                                             const float* __restrict__ part_load, int nblocks, int E) {
    extern __shared__ double shd[];
    router_li_loss_body(shd, l_aux, importance, load, g_imp, g_load, part_imp, part_load, nblocks, E);
}

__global__ __launch_bounds__(256) void router_li_bwd_kernel(RouterBwdK p) {
    extern __shared__ float s_g[];
    router_li_bwd_body(s_g, p, blockIdx.x);
}

}  // namespace
}  // namespace hexa

using namespace hexa;

extern "C" int hexa_router_ws_floats(int T, int E, int64_t* out) {
    if (!out || T < 0 || E < 1) HEXA_FAIL(HEXA_ERR_ARG, "hexa_router_ws_floats: bad arguments");
    *out = (int64_t)2 * (T > 0 ? div_up(T, ROUTER_TB) : 1) * E;
    return HEXA_OK;
}

namespace hexa {
namespace {
// The LDS tile of the four-lanes-per-token router (with the routing histogram behind it) passes 64 KiB for many
// experts and a deep top-k, and so does the gate's kernel with the FIXED bytes that it declares itself: such a launch needs the kernel's
// dynamic-LDS limit raised first, once per kernel, to the MOST any supported (E, k) asks for.
template <auto KERNEL, size_t FIXED, size_t MOST> int allow_router_lds(size_t bytes) {
    static_assert(FIXED + MOST <= 160 * 1024, "LDS of a CU");
    static bool done = false;   // per kernel
    if (FIXED + bytes <= 64 * 1024 || done) return HEXA_OK;
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(KERNEL), hipFuncAttributeMaxDynamicSharedMemorySize, (int)MOST) != hipSuccess)
        HEXA_FAIL(HEXA_ERR_LAUNCH, "router: hipFuncSetAttribute(MaxDynamicSharedMemorySize=%d) failed", (int)MOST);
    done = true;
    return HEXA_OK;
}
}  // namespace
bool router_hist_supported(int E) { return E <= ROUTER_LDS_E; }
int router_tokens_per_workgroup() { return ROUTER_TB; }

// softmax + top-k + the loss partials (ws: hexa_router_ws_floats() floats); with `hist` (only where
// router_hist_supported) also the routing pass's histogram over units of 64 tokens.  thr: the load-importance loss (its
// partial sums are importance and load), null: GShard
int launch_router_fwd(float* scores, int32_t* idx, const float* logits, const float* noise, float noise_scale, int T, int E,
                      int k, float* ws, int32_t* hist, float* thr, float inv_sigma, hipStream_t st) {
    const int nb = div_up(T, ROUTER_TB);
    float* part_me = ws;
    float* part_cnt = ws + (size_t)nb * E;
    const LiK li{thr, noise, noise_scale, inv_sigma};
    if (E <= ROUTER_LDS_E) {
        const size_t lds = sizeof(float) * router4_lds_floats(E, k, hist != nullptr, thr != nullptr);
        constexpr size_t most = sizeof(float) * router4_lds_floats(ROUTER_LDS_E, MAX_TOPK, true, true);
        if (int rc = thr ? allow_router_lds<router_fwd4_kernel<true>, 0, most>(lds) : allow_router_lds<router_fwd4_kernel<false>, 0, most>(lds)) return rc;
        if (thr)
            hipLaunchKernelGGL(router_fwd4_kernel<true>, dim3(nb), dim3(ROUTER_TB * ROUTER_G), lds, st, scores, idx, part_me, part_cnt,
                               logits, noise, noise_scale, T, E, k, hist, li);
        else
            hipLaunchKernelGGL(router_fwd4_kernel<false>, dim3(nb), dim3(ROUTER_TB * ROUTER_G), lds, st, scores, idx, part_me, part_cnt,
                               logits, noise, noise_scale, T, E, k, hist, li);
    } else if (thr)
        hipLaunchKernelGGL(router_li_fwd_kernel, dim3(nb), dim3(ROUTER_TB), 0, st, scores, idx, thr, part_me, part_cnt,
                           logits, noise, noise_scale, inv_sigma, T, E, k);
    else
        hipLaunchKernelGGL(router_fwd_kernel, dim3(nb), dim3(ROUTER_TB), sizeof(float) * 2 * E, st, scores, idx,
                           part_me, part_cnt, logits, noise, noise_scale, T, E, k);
    HEXA_CHECK_LAUNCH("router_fwd");
    return HEXA_OK;
}

// gate projection + router in one launch (see gate_router_kernel); same results as hexa_gate_logits followed by
// launch_router_fwd.  round (may be null): weights to round beside it; x_src (may be null): fp32 tokens that the launch
// rounds into x on its way (a conversion launch of its own takes 8.8 us for 18432 x 384; this one takes 33 to 34 with them, beside 38 million weights)
bool gate_router_supported(int d, int E, int x_dt) {
    return E <= GATE_ROUTER_MAX_E && (d % 8) == 0 && (x_dt == HEXA_F32 || x_dt == HEXA_BF16 || x_dt == HEXA_F16);
}
namespace {
template <typename T, bool LI, int ROUND, int MODE>
int launch_gate_router_k(float* logits, float* scores, int32_t* idx, const void* x, const float* x_src, const float* wg, const float* noise, float noise_scale,
                         int T_, int d, int E, int k, float* ws, int32_t* hist, const LiK& li, RoundAllK* round, hipStream_t st) {
    const int nb = div_up(T_, ROUTER_TB);
    const size_t lds = sizeof(float) * router4_lds_floats(E, k, hist != nullptr, false);
    constexpr size_t fixed = MODE == GR_DIRECT ? GR_DIRECT_BYTES : GR_BYTES;
    constexpr size_t most = sizeof(float) * router4_lds_floats(MODE == GR_DIRECT ? GR_DIRECT_E : GATE_ROUTER_MAX_E, MAX_TOPK, true, false);
    if (int rc = allow_router_lds<gate_router_kernel<T, LI, ROUND, MODE>, fixed, most>(lds)) return rc;
    RoundAllK r{};
    if (round) r = *round;
    r.blocks = (int)((r.n + GATE_ROUTER_NT * 8 * ROUND_STEPS - 1) / (GATE_ROUTER_NT * 8 * ROUND_STEPS));
    using X = std::conditional_t<ROUND == ROUND_TOKENS, T*, const T*>;
    hipLaunchKernelGGL((gate_router_kernel<T, LI, ROUND, MODE>), dim3(nb + r.blocks), dim3(GATE_ROUTER_NT), lds, st, logits, scores, idx, ws,
                       ws + (size_t)nb * E, (X)x, x_src, wg, noise, noise_scale, T_, d, E, k, hist, nb, li, r);
    HEXA_CHECK_LAUNCH("gate_router");
    return HEXA_OK;
}
template <typename T, bool LI, int ROUND, typename... Args>
int launch_gate_router_t(int d, int E, Args... args) {
    const int mode = gate_router_mode(d, E, ROUND == ROUND_TOKENS);
    if (mode == GR_DIRECT) return launch_gate_router_k<T, LI, ROUND, GR_DIRECT>(args...);
    if constexpr (ROUND == ROUND_TOKENS)
        if (mode == GR_WHOLE) return launch_gate_router_k<T, LI, ROUND, GR_WHOLE>(args...);
    return launch_gate_router_k<T, LI, ROUND, GR_STAGED>(args...);
}
}  // namespace
int launch_gate_router(float* logits, float* scores, int32_t* idx, const void* x, const float* x_src, const float* wg, const float* noise,
                       float noise_scale, int T, int d, int E, int k, int x_dt, float* ws, int32_t* hist, float* thr, float inv_sigma,
                       RoundAllK* round, hipStream_t st) {
    const LiK li{thr, noise, noise_scale, inv_sigma};
#define HEXA_GATE_ROUTER(TYPE, S)                                                                                                     \
    return thr ? launch_gate_router_t<TYPE, true, S>(d, E, logits, scores, idx, x, x_src, wg, noise, noise_scale, T, d, E, k, ws, hist, li, round, st) \
               : launch_gate_router_t<TYPE, false, S>(d, E, logits, scores, idx, x, x_src, wg, noise, noise_scale, T, d, E, k, ws, hist, li, round, st)
    if (x_dt == HEXA_F32) HEXA_GATE_ROUTER(float, ROUND_NONE);
    const bool bf = x_dt == HEXA_BF16;
    if (bf && x_src) HEXA_GATE_ROUTER(__bf16, ROUND_TOKENS);
    if (bf && round) HEXA_GATE_ROUTER(__bf16, ROUND_WEIGHTS);
    if (bf) HEXA_GATE_ROUTER(__bf16, ROUND_NONE);
    if (x_src) HEXA_GATE_ROUTER(_Float16, ROUND_TOKENS);
    if (round) HEXA_GATE_ROUTER(_Float16, ROUND_WEIGHTS);
    HEXA_GATE_ROUTER(_Float16, ROUND_NONE);
#undef HEXA_GATE_ROUTER
}

int router_li_check(const char* who, int T, int E, int k, float sigma) {
    if (T < 1 || E < 2 || k < 1) HEXA_FAIL(HEXA_ERR_ARG, "%s: bad sizes T=%d E=%d k=%d (E >= 2 for a variance)", who, T, E, k);
    if (k > MAX_TOPK || k > E) HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "%s: top_k must be <= min(E, %d)", who, MAX_TOPK);
    if (!(sigma > 0.f)) HEXA_FAIL(HEXA_ERR_ARG, "%s: sigma must be > 0 (gate_noise / E of the reference)", who);
    if (E > ROUTER_LI_MAX_E) HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "%s: more than %d experts", who, ROUTER_LI_MAX_E);
    return HEXA_OK;
}
// the auxiliary loss from the router's partial sums: stats as in hexa_moe_depth_forward
int launch_router_loss(float* stats, bool li, const float* router_ws, int T, int E, hipStream_t st) {
    const int nb = div_up(T, ROUTER_TB);
    if (!li) {
        hipLaunchKernelGGL(router_loss_kernel, dim3(1), dim3(256), sizeof(float) * (2 * router_loss_chunks(E) * E + 256), st,
                           stats + 2 * E, stats, stats + E, router_ws, router_ws + (size_t)nb * E, nb, T, E);
        HEXA_CHECK_LAUNCH("router_loss");
        return HEXA_OK;
    }
    const size_t lds = sizeof(double) * router_li_loss_doubles(E);
    hipLaunchKernelGGL(router_li_loss_kernel, dim3(1), dim3(256), lds, st, stats + 4 * E, stats, stats + E, stats + 2 * E, stats + 3 * E,
                       router_ws, router_ws + (size_t)nb * E, nb, E);
    HEXA_CHECK_LAUNCH("router_li_loss");
    return HEXA_OK;
}
}  // namespace hexa

static int check_router_forward(int T, int E, int k, bool ptrs_ok) {
    if (T < 1 || E < 1 || k < 1) HEXA_FAIL(HEXA_ERR_ARG, "hexa_router_forward: bad sizes T=%d E=%d k=%d", T, E, k);
    if (k > MAX_TOPK || k > E) HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "hexa_router_forward: top_k must be <= min(E, %d)", MAX_TOPK);
    if (!ptrs_ok) HEXA_FAIL(HEXA_ERR_ARG, "hexa_router_forward: null pointer");
    if (E > 4096) HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "hexa_router_forward: more than 4096 experts");
    return HEXA_OK;
}

namespace hexa {
int router_forward_check(int T, int E, int k, bool ptrs_ok) { return check_router_forward(T, E, k, ptrs_ok); }
}

extern "C" int hexa_router_forward(float* scores, int32_t* idx, float* me, float* ce, float* l_aux,
                                   const float* logits, const float* noise, float noise_scale, int T, int E, int k,
                                   float* ws, void* stream) {
    if (int rc = check_router_forward(T, E, k, scores && idx && me && ce && l_aux && logits && ws)) return rc;
    hipStream_t st = (hipStream_t)stream;
    if (int rc = launch_router_fwd(scores, idx, logits, noise, noise_scale, T, E, k, ws, nullptr, nullptr, 0.f, st)) return rc;
    const int nb = div_up(T, ROUTER_TB);
    hipLaunchKernelGGL(router_loss_kernel, dim3(1), dim3(256), sizeof(float) * (2 * router_loss_chunks(E) * E + 256), st,
                       l_aux, me, ce, ws, ws + (size_t)nb * E, nb, T, E);
    HEXA_CHECK_LAUNCH("router_loss");
    return HEXA_OK;
}

extern "C" int hexa_router_backward(float* dlogits, const float* scores, const float* ce, const float* grad_l_aux,
                                    int T, int E, void* stream) {
    if (T < 1 || E < 1) HEXA_FAIL(HEXA_ERR_ARG, "hexa_router_backward: bad sizes");
    if (!dlogits || !scores || !ce || !grad_l_aux) HEXA_FAIL(HEXA_ERR_ARG, "hexa_router_backward: null pointer");
    if (E > 8192) HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "hexa_router_backward: more than 8192 experts");
    SmallTask t;
    t.kind = TASK_ROUTER_BWD; t.router_bwd = RouterBwdK{dlogits, scores, ce, grad_l_aux, T, E, nullptr, nullptr, nullptr, 0.f, 0}; t.blocks = div_up(T, 256);
    if (!defer_task(E <= BATCH_ROUTER_BWD_MAX_E ? defer_targets().router_bwd : nullptr, t)) {
        hipLaunchKernelGGL(router_bwd_kernel, dim3(t.blocks), dim3(256), sizeof(float) * E, (hipStream_t)stream, t.router_bwd);
        HEXA_CHECK_LAUNCH("router_bwd");
    }
    return HEXA_OK;
}

extern "C" int hexa_router_forward_load_importance(float* scores, int32_t* idx, float* thr, float* importance,
                                                   float* load, float* g_importance, float* g_load, float* l_aux,
                                                   const float* logits, const float* noise, float noise_scale,
                                                   float sigma, int T, int E, int k, float* ws, void* stream) {
    const char* who = "hexa_router_forward_load_importance";
    if (int rc = router_li_check(who, T, E, k, sigma)) return rc;
    if (!scores || !idx || !thr || !importance || !load || !g_importance || !g_load || !l_aux || !logits || !ws)
        HEXA_FAIL(HEXA_ERR_ARG, "%s: null pointer", who);
    hipStream_t st = (hipStream_t)stream;
    const int nb = div_up(T, ROUTER_TB);
    if (int rc = launch_router_fwd(scores, idx, logits, noise, noise_scale, T, E, k, ws, nullptr, thr, 1.0f / sigma, st)) return rc;
    hipLaunchKernelGGL(router_li_loss_kernel, dim3(1), dim3(256), sizeof(double) * router_li_loss_doubles(E), st, l_aux,
                       importance, load, g_importance, g_load, ws, ws + (size_t)nb * E, nb, E);
    HEXA_CHECK_LAUNCH("router_li_loss");
    return HEXA_OK;
}

extern "C" int hexa_router_backward_load_importance(float* dlogits, const float* scores, const float* thr,
                                                    const int32_t* idx, const float* g_importance,
                                                    const float* g_load, const float* grad_l_aux, float sigma, int T,
                                                    int E, int k, void* stream) {
    const char* who = "hexa_router_backward_load_importance";
    if (T < 1 || E < 2 || k < 1 || k > E) HEXA_FAIL(HEXA_ERR_ARG, "%s: bad sizes", who);
    if (!(sigma > 0.f)) HEXA_FAIL(HEXA_ERR_ARG, "%s: sigma must be > 0", who);
    if (!dlogits || !scores || !thr || !idx || !g_importance || !g_load || !grad_l_aux)
        HEXA_FAIL(HEXA_ERR_ARG, "%s: null pointer", who);
    if (E > 4096) HEXA_FAIL(HEXA_ERR_UNSUPPORTED, "%s: more than 4096 experts", who);
    SmallTask t;
    t.kind = TASK_ROUTER_BWD;
    t.router_bwd = RouterBwdK{dlogits, scores, g_importance, grad_l_aux, T, E, thr, idx, g_load, 1.0f / sigma, k};
    t.blocks = div_up(T, LI_BWD_TOKENS);
    if (!defer_task(2 * E <= BATCH_ROUTER_BWD_MAX_E ? defer_targets().router_bwd : nullptr, t)) {
        hipLaunchKernelGGL(router_li_bwd_kernel, dim3(t.blocks), dim3(256), sizeof(float) * 2 * E, (hipStream_t)stream, t.router_bwd);
        HEXA_CHECK_LAUNCH("router_li_bwd");
    }
    return HEXA_OK;
}
