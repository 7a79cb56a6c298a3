// Creating a context waits for nothing.
#include "stubs.h"

int main() {
  queued.push_back([] {});  // work of the caller
  Box box;
  CHECK(blocking_copies == 0);
  CHECK(queued.size() == 1);
  return 0;
}
