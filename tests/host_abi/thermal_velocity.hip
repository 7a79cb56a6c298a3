// Where the velocity of pol_thermal_step_with_velocity may lie.
#include "stubs.h"

namespace pol {
hipError_t launch_thermal_steps(bool, const ThermalArgs&, void* const*, void* const*, int& gcur, int& tcur, int nsteps,
                                double*, double*, hipStream_t) {
  gcur ^= nsteps & 1;
  tcur ^= nsteps & 1;
  return launch([] {});
}
}  // namespace pol

int main() {
  Box box;
  std::vector<float> mem(64 * Box::cells);
  auto plane = [&](int p, int cell = 0) { return mem.data() + p * Box::cells + cell; };
  const int last = (int)Box::cells - 1;
  pol_thermal_desc td{};
  td.omega = 1.0;
  td.options = POL_THERMAL_CONVECTION;
  pol_thermal_buffers tb{};
  tb.g[0] = plane(10);
  tb.g[1] = plane(20);
  tb.temperature[0] = plane(30);
  tb.temperature[1] = plane(32);
  tb.heat_source = plane(40);
  tb.velocity = plane(50);
  CHECK(pol_thermal_bind(box.c, &td, &tb) == POL_OK);
  auto step = [&](const void* v, int n = 2) {
    int32_t bad;
    return pol_thermal_step_with_velocity(box.c, n, v, &bad, nullptr, nullptr);
  };
  for (const float* v : {plane(50, 1), plane(50, -1), plane(52, last), plane(48, 1), plane(47, 1)})  // its own buffer
    CHECK(step(v) == POL_ERR_INVALID);
  for (const float* v : {plane(20), plane(24), plane(26, last), plane(17, 1)})  // written by the first step
    CHECK(step(v) == POL_ERR_INVALID);
  for (const float* v : {plane(40), plane(40, last), plane(37, 1)})
    CHECK(step(v) == POL_ERR_INVALID);
  CHECK(queued.empty());
  // the buffer itself, beside each, the populations that are read, the temperature
  for (const float* v : {plane(50), plane(47), plane(53), plane(27), plane(17), plane(37), plane(41), plane(11), plane(30)})
    CHECK(step(v) == POL_OK);
  // after an odd number of steps the other population buffer is written next
  CHECK(step(plane(50), 1) == POL_OK);
  CHECK(step(plane(11)) == POL_ERR_INVALID);
  CHECK(step(plane(21)) == POL_OK);
  return 0;
}
