// prefill_gemm_q4_0.hip -- the prefill chunk's expert launches, Q4_0 experts.
#include "prefill_gemm.h"

namespace chimere {
template void pf_launch_experts<T_Q4_0>(const PfArgs&, int, hipStream_t);
}  // namespace chimere
