// The kernels of one form of the resident steps, PVD_FORM (pvd_resident.hpp).
#include "pvd_resident.hpp"

namespace pvd {

// Two shapes: `small`, at most two rounds of 512 threads per workgroup (the step is latency then:
// fewer rounds to rank, 256 registers a wave), and W rounds of up to 1024 threads, which hold the
// population's whole range, 1.5 N0, wherever the LDS holds N0.  NTM 512 where a walker needs more than
// the 128 registers a wave of 1024 threads has.
template <>
Instance res_instance<PVD_FORM>(bool small) {
  using F = ResForm<PVD_FORM>;
  using R = F::R;
  const void* rest = (const void*)k_resident_rest<R, F::NP, F::IS, F::MS, F::NTM>;
  const int stride = res_stride<R, F::NP>();
  if (small) return Instance{(const void*)k_resident<R, F::NP, F::IS, F::MS, 2, 512, false>, rest, 2, 512, stride};
  return Instance{(const void*)k_resident<R, F::NP, F::IS, F::MS, F::W, F::NTM, true>, rest, F::W, F::NTM, stride};
}

}  // namespace pvd
