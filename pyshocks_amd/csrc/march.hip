// The march schedule in FP64 (march_device.hpp).
#include "march_device.hpp"

namespace psa {

int launch_march(const psa_solver_desc *d, const StageArgs<double> &a, long long nsteps,
                 void *k1, void *k2, hipStream_t s) {
  return launch_march_t<double>(d, a, nsteps, k1, k2, s);
}

}  // namespace psa
