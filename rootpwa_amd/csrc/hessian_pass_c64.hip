// hessian_pass_c64.hip -- instantiations of the Hessian's rank-k passes (complex64
// amplitudes).
#include "hessian_pass.h"

namespace rpwa_amd {

hipError_t launch_hessian_passes_c64(bool dRows, const hp::PassArgs& a, int nWg, hipStream_t s)
{
	return hp::launch_passes<true>(dRows, a, nWg, s);
}

}  // namespace rpwa_amd
