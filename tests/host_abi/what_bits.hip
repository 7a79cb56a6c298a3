// Bits of `what` that the header does not define do nothing: no launch sees
// them, and a reduction asked for beside them is the plain one.
#include "stubs.h"

namespace pol {
hipError_t launch_particles_couple(const ParticleArgs&, bool, hipStream_t) { return launch([] {}); }
hipError_t launch_particles_clear_footprint(const ParticleArgs&, hipStream_t) { return launch([] {}); }
hipError_t launch_particles_advance(const ParticleArgs&, hipStream_t) { return launch([] {}); }
hipError_t launch_add_field_fluid(bool, void*, const void*, const uint32_t*, uint32_t, hipStream_t) {
  return launch([] {});
}
}  // namespace pol

int main() {
  Box box(POL_FORCE_FIELD);
  constexpr uint32_t known = POL_WANT_MACRO | POL_WANT_REDUCE;
  double red[POL_NRED];
  pol_particle_desc pd{};
  pd.reaction = POL_REACTION_EXPLICIT;
  pd.dt = pd.max_disp = 1.0;
  pol_particle_buffers pb{};
  pb.reaction_field = box.at(12);
  CHECK(pol_particles_bind(box.c, &pd, &pb) == POL_OK);
  for (uint32_t asked : {POL_WANT_REDUCE, POL_WANT_MACRO, 0u, known})
    for (uint32_t bit = 0; bit < 32; ++bit) {
      if (known >> bit & 1u) continue;
      const uint32_t what = asked | 1u << bit;
      double* const r = what & POL_WANT_REDUCE ? red : nullptr;
      CHECK(pol_step_ex(box.c, 2, what, r, nullptr) == POL_OK);
      CHECK(pol_step_from(box.c, box.at(2), box.at(3), what, r, nullptr) == POL_OK);
      CHECK(pol_macroscopic(box.c, what, r, nullptr) == POL_OK);
      CHECK(pol_coupled_step(box.c, 1, what, r, nullptr) == POL_OK);
    }
  for (const pol::StepArgs& a : steps) CHECK((a.what & ~known) == 0u);
  // the recorded steps still ask for their flux
  steps.clear();
  double flux[2];
  CHECK(pol_step_record(box.c, box.at(2), Box::state_bytes, 3, box.at(7), 1, flux, nullptr) == POL_OK);
  CHECK(steps.size() == 3 && steps[0].what == 0u && steps[1].what == pol::WANT_FLUX && steps[2].what == pol::WANT_FLUX);
  return 0;
}
