// A call that fails half way leaves nothing queued that would still write the
// context's pinned buffer.
#include "stubs.h"

namespace pol {
// as csrc/thermal.hip: per step a collide and a temperature pass; a reporting
// run ends with the fold, whose launch goes through even where one before it failed
hipError_t launch_thermal_steps(bool, const ThermalArgs& a, void* const*, void* const*, int&, int&, int nsteps, double*,
                                double* out, hipStream_t) {
  hipError_t e = hipSuccess;
  for (int n = 0; n < nsteps && e == hipSuccess; ++n) {
    e = launch([] {});
    const hipError_t t = launch([] {});
    if (e == hipSuccess) e = t;
    if (n + 1 == nsteps && a.report) (void)launch([=] { out[0] = out[1] = out[2] = out[3] = out[4] = 0.0; });
  }
  return e;
}
}  // namespace pol

int main() {
  Box box;
  double flux[8];
  for (int launches = 0; launches < 8; ++launches) {  // step, fold, step, fold, ...
    fail_after = launches;
    CHECK(pol_step_record(box.c, box.at(2), Box::state_bytes, 4, box.at(7), 0, flux, nullptr) == POL_ERR_HIP);
    CHECK(queued.empty());
  }
  CHECK(pol_step_record(box.c, box.at(2), Box::state_bytes, 4, box.at(7), 0, flux, nullptr) == POL_OK);
  CHECK(flux[0] == 0.5 && flux[3] == 0.5);

  pol_thermal_desc td{};
  td.omega = 1.0;
  td.options = POL_THERMAL_CONVECTION;
  pol_thermal_buffers tb{};
  tb.g[0] = box.at(8);
  tb.g[1] = box.at(9);
  tb.temperature[0] = box.at(10);
  tb.temperature[1] = box.at(11);
  tb.heat_source = box.at(12);
  tb.velocity = box.at(13);
  CHECK(pol_thermal_bind(box.c, &td, &tb) == POL_OK);
  double stats[4];
  int32_t bad;
  for (int launches = 0; launches < 4; ++launches) {
    fail_after = launches;
    CHECK(pol_thermal_step_with_velocity(box.c, 2, box.at(14), &bad, stats, nullptr) == POL_ERR_HIP);
    CHECK(queued.empty());
  }
  CHECK(pol_thermal_step_with_velocity(box.c, 2, box.at(14), &bad, stats, nullptr) == POL_OK);
  return 0;
}
