// Helpers shared by the role-split persistent kernels (gemm16_pipe.hip: ESMM, gemm16_estmm_pipe.hip: ESTMM): LDS
// accesses as inline assembly with immediate offsets, global accesses with a base every lane shares plus a 32-bit
// lane offset, and the multiply wavefronts' software-pipelined stage product.
#pragma once
#include <type_traits>
#include <utility>

#include "dma_common.h"

namespace hexa {
namespace {

typedef __attribute__((ext_vector_type(4))) unsigned u32x4;
typedef __attribute__((ext_vector_type(2))) unsigned u32x2;

// LDS accesses with the constant part of the address as the instruction's immediate offset (0..65535), so
// that one address register serves a whole unrolled group of accesses
template <int OFF = 0> __device__ __forceinline__ void lds_write64(unsigned addr, uint2 v) {
    static_assert(OFF >= 0 && OFF < 65536, "LDS offset field");
    u32x2 w;
    w.x = v.x; w.y = v.y;
    asm volatile("ds_write_b64 %0, %1 offset:%2" ::"v"(addr), "v"(w), "n"(OFF) : "memory");
}
template <int OFF = 0> __device__ __forceinline__ void lds_write128(unsigned addr, u32x4 v) {
    static_assert(OFF >= 0 && OFF < 65536, "LDS offset field");
    asm volatile("ds_write_b128 %0, %1 offset:%2" ::"v"(addr), "v"(v), "n"(OFF) : "memory");
}
template <int OFF = 0> __device__ __forceinline__ u32x4 lds_read128_async(unsigned addr) {
    static_assert(OFF >= 0 && OFF < 65536, "LDS offset field");
    u32x4 r;
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
    return r;
}
template <int OFF = 0> __device__ __forceinline__ u32x2 lds_read64_async(unsigned addr) {
    static_assert(OFF >= 0 && OFF < 65536, "LDS offset field");
    u32x2 r;
    asm volatile("ds_read_b64 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
    return r;
}
template <int OFF = 0> __device__ __forceinline__ int lds_read32_async(unsigned addr) {
    static_assert(OFF >= 0 && OFF < 65536, "LDS offset field");
    int r;
    asm volatile("ds_read_b32 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
    return r;
}
// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>): a loop whose index is a constant expression
template <int... I, typename F> __device__ __forceinline__ void static_for_impl(std::integer_sequence<int, I...>, F&& f) {
    (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F> __device__ __forceinline__ void static_for(F&& f) {
    static_for_impl(std::make_integer_sequence<int, N>{}, f);
}
__device__ __forceinline__ void lds_wait() { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); }
// 16-byte store to base + off (a base every lane shares plus a 32-bit byte offset); `streaming` (uniform) adds the
// non-temporal hint.  A store of more than 8 bytes reads its data for two wait states after its issue; the compiler keeps
// vector instructions that overwrite it away from stores of its own, but does not look into inline assembly: s_nop 1.
__device__ __forceinline__ void global_store128(void* base, unsigned off, u32x4 v, bool streaming) {
    if (streaming) asm volatile("global_store_dwordx4 %0, %1, %2 nt\n\ts_nop 1" ::"v"(off), "v"(v), "s"(base) : "memory");
    else asm volatile("global_store_dwordx4 %0, %1, %2\n\ts_nop 1" ::"v"(off), "v"(v), "s"(base) : "memory");
}
// 16 bytes from base + off (one address register per lane)
__device__ __forceinline__ u32x4 global_load128_async(const void* base, unsigned off) {
    u32x4 r;
    asm volatile("global_load_dwordx4 %0, %1, %2" : "=v"(r) : "v"(off), "s"(base));
    return r;
}

// One stage's products for a wavefront that does nothing else: the fragments of contraction step ks+1 are read
// from LDS while the MFMAs of step ks run (with one such wavefront per SIMD there is no neighbour to fill the
// gap between a step's reads and its first MFMA: read-then-multiply keeps the matrix pipeline at about 60 %).
// All reads are inline assembly and return in order: the wait before step ks allows exactly the reads of step
// ks+1 to be outstanding, and every fragment passes through an empty statement behind that wait.
template <int N> __device__ __forceinline__ void lds_wait_but() { asm volatile("s_waitcnt lgkmcnt(%0)" ::"n"(N) : "memory"); }
// NRB: row blocks of this wavefront that hold anything (block i of KC rows is tile row 32 * (wr + WR * i) on,
// so that a tile of few rows keeps all wavefronts busy).
template <typename TC, typename C, bool F_KS, bool R_KS = false, int NRB = C::RB>
__device__ __forceinline__ void mma_stage_ahead(unsigned tileR, unsigned tileF, int wr, int wf, int lane, f32x16 (&acc)[C::FB][C::RB]) {
    using V = typename Mfma<TC>::V;
    constexpr int RW = 32 * C::RB, FW = 32 * C::FB, KD = C::BKC, NKS = KD / 16;
    constexpr int READS = (R_KS ? 2 * NRB : NRB) + (F_KS ? 2 * C::FB : C::FB);      // LDS read instructions per contraction step
    union Frag { V v; u32x4 q; s16x4 h[2]; };
    Frag f[2][C::FB], r[2][NRB];
    // what does not depend on the step: the row of a KC fragment and its swizzle, the column part of a KS one
    unsigned rbase[NRB]; int rsw[NRB];
    const int grp = lane >> 4, sl = lane & 15;
#pragma unroll
    for (int i = 0; i < NRB; ++i) {
        if (R_KS) {
            const int col = wr * RW + i * 32 + (grp & 1) * 16 + (sl & 3) * 4;
            rbase[i] = tileR + (col & 7) * 2;
            rsw[i] = col >> 3;
        } else {
            const int row = (wr + C::WR * i) * 32 + (lane & 31);
            rbase[i] = tileR + row * (2 * KD);
            rsw[i] = kc_swizzle<KD>(row);
        }
    }
    unsigned fbase[C::FB]; int fsw[C::FB];
#pragma unroll
    for (int j = 0; j < C::FB; ++j) {
        if (F_KS) {
            const int col = wf * FW + j * 32 + (grp & 1) * 16 + (sl & 3) * 4;
            fbase[j] = tileF + (col & 7) * 2;
            fsw[j] = col >> 3;
        } else {
            const int row = wf * FW + j * 32 + (lane & 31);
            fbase[j] = tileF + row * (2 * KD);
            fsw[j] = kc_swizzle<KD>(row);
        }
    }
    auto read_step = [&](int ks, Frag (&fs)[C::FB], Frag (&rs)[NRB]) {
        const int kch = ks * 2 + (lane >> 5);
#pragma unroll
        for (int j = 0; j < C::FB; ++j) {
            if (F_KS) {
                const int k = ks * 16 + (grp >> 1) * 8 + (sl >> 2);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int kk = k + half * 4;
                    fs[j].h[half] = lds_read_tr16(fbase[j] + kk * (2 * C::BN) + ((fsw[j] ^ ((kk & 3) << 2)) * 16));
                }
            } else {
                fs[j].q = lds_read128_async(fbase[j] + ((kch ^ fsw[j]) * 16));
            }
        }
#pragma unroll
        for (int i = 0; i < NRB; ++i) {
            if (R_KS) {
                const int k = ks * 16 + (grp >> 1) * 8 + (sl >> 2);
#pragma unroll
                for (int half = 0; half < 2; ++half) {
                    const int kk = k + half * 4;
                    rs[i].h[half] = lds_read_tr16(rbase[i] + kk * (2 * C::BM) + ((rsw[i] ^ ((kk & 3) << 2)) * 16));
                }
            } else {
                rs[i].q = lds_read128_async(rbase[i] + ((kch ^ rsw[i]) * 16));
            }
        }
    };
    read_step(0, f[0], r[0]);
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
        const int cur = ks & 1;
        if (ks + 1 < NKS) {
            read_step(ks + 1, f[cur ^ 1], r[cur ^ 1]);
            lds_wait_but<READS>();
        } else {
            lds_wait_but<0>();
        }
#pragma unroll
        for (int j = 0; j < C::FB; ++j) asm volatile("" : "+v"(f[cur][j].q));
#pragma unroll
        for (int i = 0; i < NRB; ++i) asm volatile("" : "+v"(r[cur][i].q));
#pragma unroll
        for (int j = 0; j < C::FB; ++j)
#pragma unroll
            for (int i = 0; i < NRB; ++i) acc[j][i] = Mfma<TC>::run(f[cur][j].v, r[cur][i].v, acc[j][i]);
    }
}

template <typename TC> __device__ __forceinline__ float lo16(unsigned w) { return from_bits16<TC>(w & 0xffff); }
template <typename TC> __device__ __forceinline__ float hi16(unsigned w) { return from_bits16<TC>(w >> 16); }

// Tables of GELU and GELU' over the bf16 values from a lowest magnitude up to 8 (see gemm16_pipe.hip)
constexpr unsigned LUT_M_HI = 0x4100;
typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ u16x2 as_u16x2(unsigned w) {
    union { unsigned u; u16x2 v; } c;
    c.u = w;
    return c.v;
}
__device__ __forceinline__ unsigned as_u32(u16x2 v) {
    union { unsigned u; u16x2 v; } c;
    c.v = v;
    return c.u;
}
// The table positions (as byte offsets, entries of 1 << SH bytes) of the two 16-bit values of w, packed in one word;
// `far` collects the largest distance from the table's first magnitude (a magnitude below it wraps to a huge
// one), so far >= the table's length says some value is outside.
template <unsigned LO, int SH> __device__ __forceinline__ unsigned lut_offsets(unsigned w, u16x2& far) {
    const u16x2 lo2 = {(unsigned short)LO, (unsigned short)LO};
    const u16x2 u = as_u16x2(w & 0x7fff7fffu) - lo2;
    far = __builtin_elementwise_max(far, u);
    const u16x2 sh = {(unsigned short)(SH + 1), (unsigned short)(SH + 1)};
    return as_u32(u << sh) | ((w >> (15 - SH)) & ((1u << SH) * 0x00010001u));
}
// (the 16-bit LDS loads that target one half of a register clear the other half on this chip, so two entries
// are read into two registers and joined with one shift-or)
template <int OFF> __device__ __forceinline__ unsigned lds_read_u16_async(unsigned addr) {
    unsigned r;
    asm volatile("ds_read_u16 %0, %1 offset:%2" : "=v"(r) : "v"(addr), "n"(OFF));
    return r;
}

}  // namespace
}  // namespace hexa
