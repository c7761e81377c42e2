// hessian_pass_f64.hip -- instantiations of the Hessian's rank-k passes (complex128
// amplitudes).
#include "hessian_pass.h"

namespace rpwa_amd {

hipError_t launch_hessian_passes_f64(bool dRows, const hp::PassArgs& a, int nWg, hipStream_t s)
{
	return hp::launch_passes<false>(dRows, a, nWg, s);
}

}  // namespace rpwa_amd
