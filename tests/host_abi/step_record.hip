// pol_step_record: what it refuses.
#include "stubs.h"

int main() {
  Box box;
  char* const f = box.at(2);
  const uint64_t S = Box::state_bytes;
  auto call = [&](uint64_t stride, int count, void* final_state) {
    return pol_step_record(box.c, f, stride, count, final_state, count, nullptr, nullptr);
  };
  // a step may not write into the state it reads
  CHECK(call(S, 1, f) == POL_ERR_INVALID);
  CHECK(call(S, 3, f + 2 * S) == POL_ERR_INVALID);
  CHECK(call(S, 3, f + 2 * S + 64) == POL_ERR_INVALID);
  CHECK(call(S, 3, f + 3 * S - 4) == POL_ERR_INVALID);
  CHECK(call(S, 3, f + S + 4) == POL_ERR_INVALID);
  // nor recorded states overlap
  CHECK(call(S - 4, 2, box.at(12)) == POL_ERR_INVALID);
  CHECK(call(64, 2, box.at(12)) == POL_ERR_INVALID);
  CHECK(steps.empty());
  // what lies beside them is fine: directly behind, before, a wider stride,
  // a stride that one state does not use, an earlier slot that is done with
  CHECK(call(S, 3, f + 3 * S) == POL_OK);
  CHECK(call(S, 3, f - S) == POL_OK);
  CHECK(call(2 * S, 3, f + 3 * S) == POL_OK);
  CHECK(call(0, 1, f + S) == POL_OK);
  CHECK(call(S, 3, f) == POL_OK);
  CHECK(steps.size() == 13);
  return 0;
}
