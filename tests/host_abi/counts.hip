// Counters on the device after a call that failed between counting and the
// fold that takes the counts: the next call counts from zero.
#include "stubs.h"

namespace pol {
hipError_t launch_field_stats(bool, const StatsArgs&, hipStream_t) { return launch([] {}); }
hipError_t launch_pop_nonfinite(int, const StepArgs&, unsigned long long* out, const Grid&, hipStream_t) {
  return launch([=] { out[0] += 3; out[1] += 5; });
}
hipError_t launch_stats_final(const StatsArgs&, bool, double* out, unsigned long long* pop, hipStream_t) {
  return launch([=] {
    out[POL_STAT_FLUID_POP_NAN] = out[POL_STAT_FLUID_POP_INF] = 0.0;
    if (!pop) return;
    out[POL_STAT_FLUID_POP_NAN] = (double)pop[0];
    out[POL_STAT_FLUID_POP_INF] = (double)pop[1];
    pop[0] = pop[1] = 0;
  });
}
// one step that counts 7 fast cells, and its fold
hipError_t launch_thermal_steps(bool, const ThermalArgs& a, void* const*, void* const*, int&, int&, int, double*,
                                double* out, hipStream_t) {
  uint32_t* bad = a.bad;
  const bool report = a.report;
  hipError_t e = launch([=] {
    bad[0] = 0;
    if (report) bad[1] += 7;
  });
  if (e == hipSuccess && report)
    e = launch([=] {
      out[0] = out[1] = out[2] = 0.0;
      out[3] = bad[1];
      out[4] = bad[0];
      bad[1] = 0;
    });
  return e;
}
}  // namespace pol

int main() {
  Box box;
  pol_stats_opts o{};
  o.with_populations = 1;
  double out[POL_NSTAT];
  auto counts = [&](int nan, int inf) {
    CHECK(pol_field_stats(box.c, &o, out, nullptr, nullptr) == POL_OK);
    CHECK(out[POL_STAT_FLUID_POP_NAN] == nan && out[POL_STAT_FLUID_POP_INF] == inf);
  };
  counts(3, 5);
  for (int launches = 0; launches < 3; ++launches) {  // statistics, scan, fold
    fail_after = launches;
    CHECK(pol_field_stats(box.c, &o, out, nullptr, nullptr) == POL_ERR_HIP);
    counts(3, 5);
    counts(3, 5);
  }
  fail_after = 2;
  CHECK(pol_field_stats(box.c, &o, out, nullptr, nullptr) == POL_ERR_HIP);
  o.with_populations = 0;  // a call without the scan in between
  counts(0, 0);
  o.with_populations = 1;
  counts(3, 5);

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
  auto fast = [&] {
    CHECK(pol_thermal_step_with_velocity(box.c, 1, box.at(14), &bad, stats, nullptr) == POL_OK);
    CHECK(stats[3] == 7.0);
  };
  fast();
  for (int launches = 0; launches < 2; ++launches) {  // step, fold
    fail_after = launches;
    CHECK(pol_thermal_step_with_velocity(box.c, 1, box.at(14), &bad, stats, nullptr) == POL_ERR_HIP);
    CHECK(pol_thermal_step(box.c, 1, nullptr, nullptr) == POL_OK);
    fast();
    fast();
  }
  return 0;
}
