// prefill_gemm_iq3s.hip -- the prefill chunk's expert launches, IQ3_S experts.
#include "prefill_gemm.h"

namespace chimere {
template void pf_launch_experts<T_IQ3_S>(const PfArgs&, int, hipStream_t);
}  // namespace chimere
