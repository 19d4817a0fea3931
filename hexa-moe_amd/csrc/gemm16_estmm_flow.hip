// ESTMM for bf16 / fp16 (see estmm_flow.h) as a launch of its own.
#include "estmm_flow.h"

namespace hexa {
namespace {

template <typename TC, bool OUT32>
__global__ __launch_bounds__(256, 4) void estmm16_flow_kernel(FlowK p) {
    extern __shared__ __attribute__((aligned(1024))) char smem[];
    estmm16_flow_body<TC, OUT32>(p, blockIdx.x, smem);
}

template <typename TC, bool OUT32> int launch_flow_k(const FlowK& p, int grid, hipStream_t st) {
    auto kernel = estmm16_flow_kernel<TC, OUT32>;
    if (int rc = ensure_smem(kernel, FlowLds::BYTES)) return rc;
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(256), FlowLds::BYTES, st, p);
    HEXA_CHECK_LAUNCH("estmm16_flow");
    return HEXA_OK;
}

}  // namespace

bool estmm16_flow_supported(const EstmmArgs& a) {
    if (!(a.m_dim % 8 == 0 && a.n_dim % 8 == 0 && (a.dw_dt == a.pq_dt || a.dw_dt == HEXA_F32) && a.r.k <= 8 &&
          (size_t)a.r.T < ((size_t)1 << 24) && a.m_dim < FLOW_MAX_DIM && a.n_dim < FLOW_MAX_DIM &&
          (size_t)a.r.T * a.m_dim * 2 < ((size_t)1 << 32) && (size_t)a.r.T * a.n_dim * 2 < ((size_t)1 << 32) &&
          (size_t)a.m_dim * a.n_dim * 4 < ((size_t)1 << 32)))
        return false;
    FlowK p;
    flow_args(a, p);
    return flow_rounds_fit(p, a.r.k);
}

int launch_estmm16_flow(const EstmmArgs& a, hipStream_t st) {
    FlowK p;
    const int grid = flow_args(a, p);
    if (grid == 0) return HEXA_OK;
    const bool o32 = a.dw_dt == HEXA_F32;
    const int rc = a.pq_dt == HEXA_BF16 ? (o32 ? launch_flow_k<__bf16, true>(p, grid, st) : launch_flow_k<__bf16, false>(p, grid, st))
                                        : (o32 ? launch_flow_k<_Float16, true>(p, grid, st) : launch_flow_k<_Float16, false>(p, grid, st));
    return rc || !p.plan ? rc : launch_estmm_fixup(a, st);
}

}  // namespace hexa
