// The march schedule in FP32 (march_device.hpp).
#include "march_device.hpp"

namespace psa {

int launch_march(const psa_solver_desc *d, const StageArgs<float> &a, long long nsteps,
                 void *k1, void *k2, hipStream_t s) {
  return launch_march_t<float>(d, a, nsteps, k1, k2, s);
}

}  // namespace psa
