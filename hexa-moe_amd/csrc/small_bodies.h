// Bodies of two single-workgroup kernels that also run as an extra workgroup of another launch (every launch
// of a small kernel costs 5-7 us of the step here, whatever it computes): the GShard loss from the router's
// per-workgroup partial sums, and the work plan of the balanced ESTMM.  Both are written for any workgroup size.
#pragma once
#include "small_tasks.h"

namespace hexa {

// me[e] = sum_t scores[t][e]; ce[e] = count[e] * E / T; l_aux = sum_e me[e]*ce[e] / T  (losses.py:12-19).
// lds: 2 * nch * E + blockDim.x floats, nch = router_loss_chunks(E).
__host__ __device__ inline int router_loss_chunks(int E) { return E <= 256 ? 32 : (8192 / E > 0 ? 8192 / E : 1); }

__device__ inline void router_loss_body(float* lds, float* __restrict__ l_aux, float* __restrict__ me,
                                        float* __restrict__ ce, const float* __restrict__ part_me,
                                        const float* __restrict__ part_cnt, int nblocks, int num_tokens, int E) {
    // per expert: nch threads sum nch contiguous ranges of the workgroup partials, then the range sums
    // are added in range order -- a fixed tree, independent of scheduling
    const int nch = router_loss_chunks(E), nthr = blockDim.x, tid = threadIdx.x;
    float* s_m = lds;
    float* s_c = lds + nch * E;
    float* red = lds + 2 * nch * E;
    const int per = (nblocks + nch - 1) / nch;
    for (int i = tid; i < nch * E; i += nthr) {
        const int c = i / E, e = i - c * E;
        const int b0 = c * per, b1 = min(nblocks, b0 + per);
        float m = 0.f, n = 0.f;
        for (int b = b0; b < b1; b += 8) {     // eight partials of each kind in flight per trip, added in order
            float pm[8], pc[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const size_t at = (size_t)min(b + u, b1 - 1) * E + e;
                pm[u] = part_me[at];
                pc[u] = part_cnt[at];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                m += (b + u < b1) ? pm[u] : 0.f;
                n += (b + u < b1) ? pc[u] : 0.f;
            }
        }
        s_m[i] = m;
        s_c[i] = n;
    }
    __syncthreads();
    float local = 0.f;
    for (int e = tid; e < E; e += nthr) {
        float m = 0.f, c = 0.f;
        for (int j = 0; j < nch; ++j) { m += s_m[j * E + e]; c += s_c[j * E + e]; }
        const float cev = c * ((float)E / (float)num_tokens);
        me[e] = m;
        ce[e] = cev;
        local += m * cev;
    }
    red[tid] = local;
    __syncthreads();
    if (tid == 0) {       // E products spread over the threads: their partial sums are added in thread order
        float t = 0.f;
        for (int i = 0; i < nthr; ++i) t += red[i];
        *l_aux = t / (float)num_tokens;
    }
}

// ---- plan of a balanced ESTMM launch ------------------------------------------------------------------
// One workgroup's walk over an expert's token list is serial, so the kernel is as slow as the
// busiest expert.  With scratch memory, experts with more than `cap` tokens are cut into up to
// PLAN_MAX_PARTS parts of equal step counts; a part is a unit of work like a whole small expert, its
// fp32 partial result goes to a scratch slot, and estmm_fixup_kernel adds an expert's slots in order
// (bit-reproducible).  Units are numbered heaviest expert first.  plan = 4 arrays of E ints in rank
// order -- expert, parts, first unit, first scratch slot -- followed by the number of units.
// lds: 2 * E ints.
constexpr int PLAN_MAX_PARTS = 8;
constexpr int PLAN_QUEUE_INTS = 16;    // work counters of the persistent ESTMM kernel behind the plan (8 queues, a finish count)
__host__ __device__ inline int estmm_plan_queue_at(int E) { return 4 * E + 1; }

// An expert's list is cut when it is longer than `cap` rows.  The persistent kernel hands items (an expert's or
// part's list x one 128 x 128 block of the result) longest-first to whichever workgroup is free, so a cut only pays
// when one item would be longer than a workgroup's share of the launch: rows of all lists x blocks per expert /
// workgroups (`tiles` = 0: unknown result size, the rule of the one-item-per-workgroup kernel: 1.5x the mean load).
__host__ __device__ inline int estmm_plan_cap(long T, int k, int E, int tiles = 0, int workgroups = 256) {
    const long avg = T * k / E;
    long c = (3 * avg + 1) / 2;
    if (tiles > 0) c = T * k * tiles / workgroups;
    return (int)(c > 256 ? c : 256);
}

__device__ inline void estmm_plan_from_loads(int* sp, int* __restrict__ plan, int E, int cap, int max_slots);

__device__ inline void estmm_plan_body(int* sp, int* __restrict__ plan, const int32_t* __restrict__ offsets, int E, int k,
                                       int cap, int max_slots) {
    int* load = sp;
    const int nthr = blockDim.x;
    for (int e = threadIdx.x; e < E; e += nthr) {
        int t = 0;
        for (int s = 0; s < k; ++s) t += offsets[(size_t)s * (E + 1) + e + 1] - offsets[(size_t)s * (E + 1) + e];
        load[e] = t;
    }
    __syncthreads();
    estmm_plan_from_loads(sp, plan, E, cap, max_slots);
}

// The plan from sp[0..E) = tokens per expert over all slots (written and published by the caller).
__device__ inline void estmm_plan_from_loads(int* sp, int* __restrict__ plan, int E, int cap, int max_slots) {
    int* load = sp;
    int* expert_of = sp + E;          // the expert at each rank
    const int nthr = blockDim.x;
    for (int e = threadIdx.x; e < E; e += nthr) {
        const int mine = load[e];
        int r = 0;
        for (int x = 0; x < E; ++x) {
            const int o = load[x];
            r += (o > mine || (o == mine && x < e)) ? 1 : 0;
        }
        expert_of[r] = e;
    }
    __syncthreads();
    if (threadIdx.x == 0) {          // E is small: a serial pass hands out units and scratch slots
        int unit = 0, slot = 0;
        for (int r = 0; r < E; ++r) {
            const int e = expert_of[r];
            int n = (load[e] + cap - 1) / cap;
            n = max(1, min(n, PLAN_MAX_PARTS));
            if (n > 1 && slot + n > max_slots) n = 1;
            plan[r] = e;
            plan[E + r] = n;
            plan[2 * E + r] = unit;
            plan[3 * E + r] = n > 1 ? slot : -1;
            unit += n;
            if (n > 1) slot += n;
        }
        plan[4 * E] = unit;
    }
    if (threadIdx.x < PLAN_QUEUE_INTS) plan[estmm_plan_queue_at(E) + threadIdx.x] = 0;
}

// ---- ESS: per-expert column sums of gathered rows (see ess.hip) --------------------------------------------------
template <typename T> struct Vec16;  // 16 bytes of T
template <> struct Vec16<float> { static constexpr int N = 4; };
template <> struct Vec16<__bf16> { static constexpr int N = 8; };
template <> struct Vec16<_Float16> { static constexpr int N = 8; };

template <typename T>
__device__ __forceinline__ void ess_body(const EssK& p, int block) {
    constexpr int V = Vec16<T>::N;
    constexpr int STRIP = 8 * V;  // columns per workgroup
    constexpr int U = 8;          // rows in flight per lane: 256 rows (32 KiB) per workgroup step
    __shared__ float red[4][STRIP];
    const int bx = block % p.gx, by = (block / p.gx) % p.gy, bz = block / (p.gx * p.gy);
    const int e = by;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int cl = lane & 7, rg = lane >> 3;
    const int col = bx * STRIP + cl * V;
    const bool col_ok = col < p.N;
    const T* dy = reinterpret_cast<const T*>(p.dy);

    float acc[V];
#pragma unroll
    for (int i = 0; i < V; ++i) acc[i] = 0.f;

    bool any = false;
    for (int s = 0; s < p.k; ++s) {
        int beg = p.offsets[(size_t)s * (p.E + 1) + e];
        int end = p.offsets[(size_t)s * (p.E + 1) + e + 1];
        any = any || end > beg;
        if (p.splits > 1) {
            const int part = (end - beg + p.splits - 1) / p.splits;
            beg = min(end, beg + bz * part);
            end = min(end, beg + part);
        }
        const int32_t* tok = p.token_ids + (size_t)s * p.T;
        const T* base = dy + (size_t)p.dy_slot_rows * s * p.N + col;
        // this lane's rows: beg + wave*8 + rg + 32*u + 256*step; the token ids of the next step are
        // fetched while the rows of the current one are in flight
        const int r_lane = beg + wave * 8 + rg;
        int ids[U];
#pragma unroll
        for (int u = 0; u < U; ++u) { const int r = r_lane + 32 * u; ids[u] = r < end ? tok[r] : -1; }
        for (int r0 = r_lane; r0 < end; r0 += 32 * U) {
            union { uint4 u; T e[V]; } v[U];
#pragma unroll
            for (int u = 0; u < U; ++u)
                v[u].u = (ids[u] >= 0 && col_ok) ? *reinterpret_cast<const uint4*>(base + (size_t)ids[u] * p.N)
                                                 : make_uint4(0u, 0u, 0u, 0u);
#pragma unroll
            for (int u = 0; u < U; ++u) { const int r = r0 + 32 * U + 32 * u; ids[u] = r < end ? tok[r] : -1; }
#pragma unroll
            for (int u = 0; u < U; ++u)
#pragma unroll
                for (int i = 0; i < V; ++i) acc[i] += Cvt<T>::to_f(v[u].e[i]);
        }
    }
#pragma unroll
    for (int i = 0; i < V; ++i) {
        float a = acc[i];
        a += __shfl_xor(a, 8);
        a += __shfl_xor(a, 16);
        a += __shfl_xor(a, 32);
        acc[i] = a;
    }
    if (rg == 0) {
#pragma unroll
        for (int i = 0; i < V; ++i) red[wave][cl * V + i] = acc[i];
    }
    __syncthreads();
    if (tid < STRIP) {
        const int c = bx * STRIP + tid;
        const float v = red[0][tid] + red[1][tid] + red[2][tid] + red[3][tid];
        if (p.splits > 1) {
            if (c < p.N) p.ws[((size_t)bz * p.E + e) * p.N + c] = v;
        } else if (c < p.N && (any || !p.accumulate)) {
            store_out(p.db, (size_t)e * p.N + c, v, p.db_dt, p.accumulate != 0);
        }
    }
}

// db (+)= ws[0] + ws[1] + ... in that order
__device__ __forceinline__ void ess_fold_body(const EssFoldK& p, int block) {
    if (p.by4) {
        const long i = ((long)block * 256 + threadIdx.x) * 4;
        if (i >= p.n) return;
        float4 part[8], v;
#pragma unroll
        for (int z = 0; z < 8; ++z)
            if (z < p.splits) part[z] = *reinterpret_cast<const float4*>(p.ws + (size_t)z * p.n + i);
        v = part[0];
#pragma unroll
        for (int z = 1; z < 8; ++z)
            if (z < p.splits) { v.x += part[z].x; v.y += part[z].y; v.z += part[z].z; v.w += part[z].w; }
        float4* const to = reinterpret_cast<float4*>(reinterpret_cast<float*>(p.db) + i);
        if (p.accumulate) { const float4 o = *to; v.x += o.x; v.y += o.y; v.z += o.z; v.w += o.w; }
        *to = v;
        return;
    }
    const long i = (long)block * 256 + threadIdx.x;
    if (i >= p.n) return;
    // all parts' loads in flight at once (at most 8 parts), added in part order
    float part[8];
#pragma unroll
    for (int z = 0; z < 8; ++z) part[z] = p.ws[(size_t)min(z, p.splits - 1) * p.n + i];
    float v = part[0];
#pragma unroll
    for (int z = 1; z < 8; ++z) v += z < p.splits ? part[z] : 0.f;
    store_out(p.db, (size_t)i, v, p.db_dt, p.accumulate != 0);
}

// out[i] += ws[0][i] + ws[1][i] + ... in fp32, slot order (the deterministic reduction behind the one-launch slot
// sum of ESMM).  `extra` (may be null): one more addend of out's shape, added last (the gate path's share of an
// input gradient).  A (token, slot) that is in no list -- its expert id was no expert's -- left its row of ws, or of out,
// as it was: where a list is short of T entries, sum_listed_slots adds the rows that were written (inlined: a call would
// give every kernel with this task a stack).
template <typename T>
__device__ __forceinline__ void sum_listed_slots(const SumSlotsK& p, int block) {
    constexpr int V = Vec16<T>::N;
    T* out = reinterpret_cast<T*>(p.out);
    const T* ws = reinterpret_cast<const T*>(p.ws);
    const int64_t nv = p.n / V;
    const int64_t stride = (int64_t)p.blocks * 256;
    const int lane = threadIdx.x & 63;
    // a wavefront looks its rows (consecutive ones) up in each slot's list, 64 entries at a time
    for (int64_t i0 = (int64_t)block * 256 + __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u); i0 < nv; i0 += stride) {
        const int64_t i = min(i0 + lane, nv - 1);
        const int row = (int)(i * V / p.N);
        const int lo = __builtin_amdgcn_readlane(row, 0), hi = __builtin_amdgcn_readlane(row, 63);
        float acc[V];
#pragma unroll
        for (int j = 0; j < V; ++j) acc[j] = 0.f;
        auto add = [&](const T* from) {
            union { uint4 u; T e[V]; } w;
            w.u = reinterpret_cast<const uint4*>(from)[i];
#pragma unroll
            for (int j = 0; j < V; ++j) acc[j] += Cvt<T>::to_f(w.e[j]);
        };
        for (int s = 0; s <= p.nws; ++s) {
            const int count = p.offsets[(size_t)s * (p.E + 1) + p.E];
            const int32_t* ids = p.token_ids + (size_t)s * p.T;
            bool listed = s == 0 && p.accumulate;
            for (int r0 = 0; r0 < count; r0 += 64) {
                const int id = r0 + lane < count ? ids[r0 + lane] : -1;
                for (unsigned long long m = __ballot(id >= lo && id <= hi); m; m &= m - 1)
                    listed = listed || __builtin_amdgcn_readlane(id, __ffsll((long long)m) - 1) == row;
            }
            if (listed) add(s == 0 ? out : ws + (size_t)(s - 1) * p.n);
        }
        if (p.extra) add(reinterpret_cast<const T*>(p.extra));
        union { uint4 u; T e[V]; } o;
#pragma unroll
        for (int j = 0; j < V; ++j) o.e[j] = Cvt<T>::from_f(acc[j]);
        if (i0 + lane < nv) reinterpret_cast<uint4*>(out)[i] = o.u;
    }
}

template <typename T>
__device__ __forceinline__ void sum_slots_body(const SumSlotsK& p, int block) {
    constexpr int V = Vec16<T>::N;
    const int lane = threadIdx.x & 63;
    // the length of slot `lane`'s list (more than 64 slots: the shortest one's)
    int len = p.T;
    if (p.offsets) {
        len = p.offsets[(size_t)min(lane, p.nws) * (p.E + 1) + p.E];
        if (p.nws >= 64)
            for (int s = lane + 64; s <= p.nws; s += 64) len = min(len, p.offsets[(size_t)s * (p.E + 1) + p.E]);
    }
    T* out = reinterpret_cast<T*>(p.out);
    const T* ws = reinterpret_cast<const T*>(p.ws);
    const int64_t nv = p.n / V;
    const int64_t stride = (int64_t)p.blocks * 256;
    for (int64_t i0 = (int64_t)block * 256 + __builtin_amdgcn_readfirstlane(threadIdx.x & ~63u); i0 < nv; i0 += stride) {
        const int64_t i = min(i0 + lane, nv - 1);
        union { uint4 u; T e[V]; } o, w;
        o.u = reinterpret_cast<const uint4*>(out)[i];
        float acc[V];
#pragma unroll
        for (int j = 0; j < V; ++j) acc[j] = Cvt<T>::to_f(o.e[j]);
        for (int s = 0; s < p.nws; ++s) {
            w.u = reinterpret_cast<const uint4*>(ws + (size_t)s * p.n)[i];
#pragma unroll
            for (int j = 0; j < V; ++j) acc[j] += Cvt<T>::to_f(w.e[j]);
        }
        if (p.extra) {
            w.u = reinterpret_cast<const uint4*>(p.extra)[i];
#pragma unroll
            for (int j = 0; j < V; ++j) acc[j] += Cvt<T>::to_f(w.e[j]);
        }
        // the lists' lengths are looked at here, before the first store and not before the first rows are on their way (with
        // a wait for them at the kernel's start a layer's two sums took 2 us each longer, 18432 tokens, d 384); the assembly
        // keeps the compiler from looking in front of the loop
        asm volatile("" : "+v"(len));
        if (__any(len != p.T)) return sum_listed_slots<T>(p, block);
#pragma unroll
        for (int j = 0; j < V; ++j) o.e[j] = Cvt<T>::from_f(acc[j]);
        if (i0 + lane >= nv) continue;
        // (fp32 tokens want an fp32 gradient: stored here, it spares a conversion of 5 us and its launch, 9216 x 384)
        if constexpr (V == 8) {
            if (p.wide) {
                float4* const to = reinterpret_cast<float4*>(p.wide + i * V);
                to[0] = make_float4(Cvt<T>::to_f(o.e[0]), Cvt<T>::to_f(o.e[1]), Cvt<T>::to_f(o.e[2]), Cvt<T>::to_f(o.e[3]));
                to[1] = make_float4(Cvt<T>::to_f(o.e[4]), Cvt<T>::to_f(o.e[5]), Cvt<T>::to_f(o.e[6]), Cvt<T>::to_f(o.e[7]));
                continue;
            }
        }
        reinterpret_cast<uint4*>(out)[i] = o.u;
    }
}

// d l_aux / d logits through the softmax (GShard loss): with c[e] = g * ce[e] / T,
//   dlogits[t][e] = scores[t][e] * (c[e] - sum_e' scores[t][e'] * c[e'])
// One token per thread.  s_c: E floats of LDS.
__device__ __forceinline__ void router_bwd_body(float* s_c, const RouterBwdK& p, int block) {
    const int E = p.E;
    const float g = *p.grad_l / (float)p.T;
    for (int e = threadIdx.x; e < E; e += blockDim.x) s_c[e] = g * p.ce[e];
    __syncthreads();
    const int t = block * blockDim.x + threadIdx.x;
    if (t >= p.T) return;
    const float* sr = p.scores + (size_t)t * E;
    float* dr = p.dlogits + (size_t)t * E;
    float dot = 0.f;
    if ((E & 3) == 0) {
        for (int e = 0; e < E; e += 4) {
            const float4 v = *reinterpret_cast<const float4*>(sr + e);
            dot += v.x * s_c[e] + v.y * s_c[e + 1] + v.z * s_c[e + 2] + v.w * s_c[e + 3];
        }
        for (int e = 0; e < E; e += 4) {
            const float4 v = *reinterpret_cast<const float4*>(sr + e);
            *reinterpret_cast<float4*>(dr + e) = make_float4(v.x * (s_c[e] - dot), v.y * (s_c[e + 1] - dot),
                                                             v.z * (s_c[e + 2] - dot), v.w * (s_c[e + 3] - dot));
        }
    } else {
        for (int e = 0; e < E; ++e) dot += sr[e] * s_c[e];
        for (int e = 0; e < E; ++e) dr[e] = sr[e] * (s_c[e] - dot);
    }
}

__device__ __forceinline__ float normal_pdf(float z) { return 0.3989422804014327f * expf(-0.5f * z * z); }

// d l_aux / d logits of the load-importance loss:  ds[e] = g_imp[e] + g_load[e] * pdf(z[e]) / sigma,  z[e] = (s[e] - thr) /
// sigma;  through the noise-free softmax  dlogits[e] = s[e] (ds[e] - sum_e' s[e'] ds[e']);  and through the
// threshold, which is the k-th choice's own logit:  dlogits[last] -= sum_e g_load[e] pdf(z[e]) / sigma.
// Four lanes per token (LI_BWD_TOKENS tokens per 256-thread workgroup).  s_g: 2 E floats of LDS.
constexpr int LI_BWD_TOKENS = 64;
__device__ __forceinline__ void router_li_bwd_body(float* s_g, const RouterBwdK& p, int block) {
    const int E = p.E, q = threadIdx.x & 3;
    const float g = *p.grad_l;
    for (int e = threadIdx.x; e < E; e += blockDim.x) { s_g[e] = g * p.ce[e]; s_g[E + e] = g * p.g_load[e] * p.inv_sigma; }
    __syncthreads();
    const int t = block * LI_BWD_TOKENS + (threadIdx.x >> 2);
    if (t >= p.T) return;
    const float* sr = p.scores + (size_t)t * E;
    float* dr = p.dlogits + (size_t)t * E;
    const float th = p.thr[t];
    const int last = p.idx[(size_t)t * p.k + (p.k - 1)];
    float dot = 0.f, dthr = 0.f;
    for (int e = q; e < E; e += 4) {
        const float sc = sr[e];
        const float w = s_g[E + e] * normal_pdf((sc - th) * p.inv_sigma);
        dot += sc * (s_g[e] + w);
        dthr -= w;
    }
#pragma unroll
    for (int m = 1; m <= 2; m <<= 1) { dot += __shfl_xor(dot, m); dthr += __shfl_xor(dthr, m); }
    for (int e = q; e < E; e += 4) {
        const float sc = sr[e];
        const float w = s_g[E + e] * normal_pdf((sc - th) * p.inv_sigma);
        dr[e] = sc * (s_g[e] + w - dot) + (e == last ? dthr : 0.f);
    }
}

// importance / load from the router's partial sums per workgroup (fixed order), the loss, and its derivative with
// respect to each importance[e] and load[e] (kept for the backward pass):
//   cv2(v) = var(v) / (mean(v)^2 + eps),  var unbiased;  d cv2 / d v[e] =
//   2 (v[e] - mean) / ((E-1)(mean^2 + eps))  -  var * 2 mean / (E (mean^2 + eps)^2)
// With a balanced router every v[e] is close to the mean, so v[e] - mean cancels almost all digits:
// the sums over workgroups and everything after them are carried in double (one workgroup, a few
// thousand operations).  256 threads; shd: router_li_loss_doubles(E) doubles of LDS.
__host__ __device__ inline int router_li_chunks(int E) { return E <= 32 ? 32 : (1024 / E > 0 ? 1024 / E : 1); }
__host__ __device__ inline size_t router_li_loss_doubles(int E) { return (size_t)2 * router_li_chunks(E) * E + 2 * E + 512; }
__device__ inline void router_li_loss_body(double* shd, float* __restrict__ l_aux, float* __restrict__ importance,
                                           float* __restrict__ load, float* __restrict__ g_imp, float* __restrict__ g_load,
                                           const float* __restrict__ part_imp, const float* __restrict__ part_load,
                                           int nblocks, int E) {
    const int nch = router_li_chunks(E);
    double* s_a = shd;                     // [nch][E] importance
    double* s_b = shd + nch * E;           // [nch][E] load
    double* v_a = shd + 2 * nch * E;
    double* v_b = v_a + E;
    double* red_a = v_b + E;               // [256] each
    double* red_b = red_a + 256;
    const int per = (nblocks + nch - 1) / nch;
    for (int i = threadIdx.x; i < nch * E; i += 256) {
        const int c = i / E, e = i - c * E;
        const int b0 = c * per, b1 = min(nblocks, b0 + per);
        double a = 0., b = 0.;
        for (int q = b0; q < b1; q += 8) {     // eight partials of each kind in flight per trip, added in order
            float pa[8], pb[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const size_t at = (size_t)min(q + u, b1 - 1) * E + e;
                pa[u] = part_imp[at];
                pb[u] = part_load[at];
            }
#pragma unroll
            for (int u = 0; u < 8; ++u)
                if (q + u < b1) { a += pa[u]; b += pb[u]; }
        }
        s_a[i] = a;
        s_b[i] = b;
    }
    __syncthreads();
    double la = 0., lb = 0.;
    for (int e = threadIdx.x; e < E; e += 256) {
        double a = 0., b = 0.;
        for (int j = 0; j < nch; ++j) { a += s_a[j * E + e]; b += s_b[j * E + e]; }
        v_a[e] = a; v_b[e] = b;
        importance[e] = (float)a; load[e] = (float)b;
        la += a; lb += b;
    }
    auto block_sum2 = [&](double x, double y, double& ox, double& oy) {
        red_a[threadIdx.x] = x; red_b[threadIdx.x] = y;
        __syncthreads();
        for (int s = 128; s > 0; s >>= 1) {
            if (threadIdx.x < s) { red_a[threadIdx.x] += red_a[threadIdx.x + s]; red_b[threadIdx.x] += red_b[threadIdx.x + s]; }
            __syncthreads();
        }
        ox = red_a[0]; oy = red_b[0];
        __syncthreads();
    };
    double sa, sb;
    block_sum2(la, lb, sa, sb);
    const double ma = sa / E, mb = sb / E;
    double qa = 0., qb = 0.;
    for (int e = threadIdx.x; e < E; e += 256) {
        const double da = v_a[e] - ma, db = v_b[e] - mb;
        qa += da * da; qb += db * db;
    }
    double ssa, ssb;
    block_sum2(qa, qb, ssa, ssb);
    const double var_a = ssa / (E - 1), var_b = ssb / (E - 1);
    const double den_a = ma * ma + 1e-10, den_b = mb * mb + 1e-10;
    if (threadIdx.x == 0) *l_aux = (float)(0.5 * (var_a / den_a + var_b / den_b));
    for (int e = threadIdx.x; e < E; e += 256) {
        g_imp[e] = (float)(0.5 * (2. * (v_a[e] - ma) / ((E - 1) * den_a) - var_a * 2. * ma / (E * den_a * den_a)));
        g_load[e] = (float)(0.5 * (2. * (v_b[e] - mb) / ((E - 1) * den_b) - var_b * 2. * mb / (E * den_b * den_b)));
    }
}

// One workgroup's share of a rounding task (ROUND_STEPS pieces of 8 elements per thread, all loads in flight).
constexpr int ROUND_STEPS = 4;
template <typename TC> __device__ __forceinline__ void round_all_as(const RoundAllK& p, int block) {
    const long base = (long)block * blockDim.x * 8 * ROUND_STEPS;
    float4 v[ROUND_STEPS][2];
#pragma unroll
    for (int i = 0; i < ROUND_STEPS; ++i) {
        const long at = base + (long)(i * blockDim.x + threadIdx.x) * 8;
        if (at < p.n) {
            v[i][0] = reinterpret_cast<const float4*>(p.src + at)[0];
            v[i][1] = reinterpret_cast<const float4*>(p.src + at)[1];
        }
    }
#pragma unroll
    for (int i = 0; i < ROUND_STEPS; ++i) {
        const long at = base + (long)(i * blockDim.x + threadIdx.x) * 8;
        if (at >= p.n) break;
        union { uint4 u; TC t[8]; } o;
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            o.t[4 * h] = (TC)v[i][h].x; o.t[4 * h + 1] = (TC)v[i][h].y;
            o.t[4 * h + 2] = (TC)v[i][h].z; o.t[4 * h + 3] = (TC)v[i][h].w;
        }
        *reinterpret_cast<uint4*>(reinterpret_cast<TC*>(p.dst) + at) = o.u;
    }
}
__device__ __forceinline__ void round_all_body(const RoundAllK& p, int block) {
    if (p.dt == HEXA_BF16) round_all_as<__bf16>(p, block);
    else round_all_as<_Float16>(p, block);
}

// dw[e] (+)= slot[0] + slot[1] + ... for the experts that the ESTMM plan cut into parts
constexpr int FIXUP_PIECES = 4;   // pieces of 1024 results per fix-up workgroup
__device__ __forceinline__ void estmm_fixup_body(const FixupK& p, int block) {
    // Workgroups (bx, j): piece bx of the result of the j-th expert whose list was cut.  A cut expert holds at least
    // two scratch slots, so the launch has max_slots / 2 values of j and not one per expert -- with 32 experts of
    // 3072 x 768 results and no list cut, one per expert was 74 thousand workgroups that only looked and left, 35 us.
    const int bx = block % p.gx, j = block / p.gx;
    const int E = p.E, lane = threadIdx.x & 63;
    int r = -1;
    for (int r0 = 0, seen = 0; r0 < E && r < 0; r0 += 64) {
        const bool cut = r0 + lane < E && p.plan[E + r0 + lane] > 1;
        unsigned long long m = __builtin_amdgcn_ballot_w64(cut);
        const int c = __builtin_popcountll(m);
        if (j < seen + c) {
            for (int q = j - seen; q > 0; --q) m &= m - 1;
            r = r0 + (int)__builtin_ctzll(m);
        }
        seen += c;
    }
    if (r < 0) return;
    const int n = p.plan[E + r];
    const int e = p.plan[r];
    const float* src0 = p.scratch + (size_t)p.plan[3 * E + r] * p.mn;
    // FIXUP_PIECES pieces of 1024 results per workgroup, one after the other
    for (int it = 0; it < FIXUP_PIECES; ++it) {
        const long i = (((long)bx * FIXUP_PIECES + it) * 256 + threadIdx.x) * 4;
        if (i >= p.mn) return;
        const float* src = src0 + i;
        // four parts' loads in flight at once, added in part order
        float4 v = make_float4(0.f, 0.f, 0.f, 0.f);
        for (int c0 = 0; c0 < n; c0 += 4) {
            float4 w[4];
#pragma unroll
            for (int c = 0; c < 4; ++c) w[c] = *reinterpret_cast<const float4*>(src + (size_t)min(c0 + c, n - 1) * p.mn);
#pragma unroll
            for (int c = 0; c < 4; ++c) {
                if (c0 + c < n) {
                    if (c0 + c == 0) v = w[0];
                    else { v.x += w[c].x; v.y += w[c].y; v.z += w[c].z; v.w += w[c].w; }
                }
            }
        }
        const size_t o = (size_t)e * p.mn + i;
        if (!p.accumulate) {   // one store of the four results (mn is a multiple of 4, so the piece is aligned)
            typedef __attribute__((ext_vector_type(4))) float f4;
            typedef __attribute__((ext_vector_type(2))) unsigned u2;
            if (p.dw_dt == HEXA_F32) {
                f4 w4 = {v.x, v.y, v.z, v.w};
                *reinterpret_cast<f4*>(reinterpret_cast<float*>(p.dw) + o) = w4;
            } else {
                union { __bf16 b[4]; _Float16 h[4]; u2 w; } pk;   // the conversions of store_out
                if (p.dw_dt == HEXA_BF16) { pk.b[0] = (__bf16)v.x; pk.b[1] = (__bf16)v.y; pk.b[2] = (__bf16)v.z; pk.b[3] = (__bf16)v.w; }
                else { pk.h[0] = (_Float16)v.x; pk.h[1] = (_Float16)v.y; pk.h[2] = (_Float16)v.z; pk.h[3] = (_Float16)v.w; }
                *reinterpret_cast<u2*>(reinterpret_cast<unsigned short*>(p.dw) + o) = pk.w;
            }
            continue;
        }
        store_out(p.dw, o, v.x, p.dw_dt, true);
        store_out(p.dw, o + 1, v.y, p.dw_dt, true);
        store_out(p.dw, o + 2, v.z, p.dw_dt, true);
        store_out(p.dw, o + 3, v.w, p.dw_dt, true);
    }
}

// db[e][n] (+)= the column sums an ESMM launch left per (slot, row tile, column tile), added in a fixed order.
// The tiles of a slot are listed expert after expert, so expert e's run starts at the number of tiles of the
// experts before it: every thread of the workgroup adds up ceil(rows / tile_rows) over a share of those experts
// (one round of loads instead of a bisection's chain of dependent ones).
__device__ __forceinline__ void colsum_fold_body(const ColsumFoldK& p, int block) {
    __shared__ int sFirst[8], sCount[8];        // per slot: first tile of expert e, its number of tiles
    __shared__ int red[256];
    const int bx = block % p.gx, e = block / p.gx, tid = threadIdx.x;
    const int runs = p.merged ? 1 : p.nslots;
    for (int s = 0; s < runs; ++s) {
        auto tiles_of = [&](int x) {
            int n = 0;
            for (int q = s; q < (p.merged ? p.nslots : s + 1); ++q) n += p.offsets[(size_t)q * (p.E + 1) + x + 1] - p.offsets[(size_t)q * (p.E + 1) + x];
            return (n + p.tile_rows - 1) / p.tile_rows;
        };
        int before = 0;
        for (int x = tid; x < e; x += 256) before += tiles_of(x);
        red[tid] = before;
        __syncthreads();
        for (int w = 128; w > 0; w >>= 1) {
            if (tid < w) red[tid] += red[tid + w];
            __syncthreads();
        }
        if (tid == 0) { sFirst[s] = red[0]; sCount[s] = tiles_of(e); }
        __syncthreads();
    }
    const int n = bx * 256 + tid;
    if (n >= p.N) return;
    const int nt = n / p.bn, nl = n - nt * p.bn;
    // Eight tiles' sums are added in pairs, and these groups like the digits of a binary counter: level l holds 2^l groups, so that no value
    // passes through a long chain of additions.  With the groups in a chain the fp32 sum was less exact than a pass over the stored rows from
    // 18000 rows of one expert on (65536 rows of mean 0.1 and deviation 1: 1.2e-7 of it, 3.6e-8 so, the pass 5.1e-8; 2304 rows of mean 0:
    // 9.1e-8 both ways, the pass 1.0e-7).
    constexpr int LEVELS = 8;
    float level[LEVELS] = {};
    int groups = 0;
    for (int s = 0; s < runs; ++s) {
        const int first = sFirst[s], last = min(first + sCount[s], p.mt_ub);
        // eight loads in flight per trip (a busy expert has a dozen tiles; one load per trip would pay the memory latency a dozen times)
        for (int mt = first; mt < last; mt += 8, ++groups) {
            float v[8];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = p.colsum[(((size_t)s * p.mt_ub + min(mt + u, last - 1)) * p.ntn + nt) * p.bn + nl];
#pragma unroll
            for (int u = 0; u < 8; ++u) v[u] = (mt + u < last) ? v[u] : 0.f;
            float group = ((v[0] + v[1]) + (v[2] + v[3])) + ((v[4] + v[5]) + (v[6] + v[7]));
#pragma unroll
            for (int l = 0; l < LEVELS; ++l) {
                const bool last_level = l + 1 == LEVELS;                     // (takes all there is)
                if (last_level || !(groups >> l & 1)) { level[l] = last_level ? level[l] + group : group; break; }
                group += level[l];
            }
        }
    }
    float sum = 0.f;
#pragma unroll
    for (int l = 0; l < LEVELS; ++l) sum += l + 1 == LEVELS || (groups >> l & 1) ? level[l] : 0.f;
    store_out(p.db, (size_t)e * p.N + n, sum, p.db_dt, p.accumulate != 0);
}

}  // namespace hexa
