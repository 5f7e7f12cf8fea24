// Host check of the work that goes with a later launch (hirensi_amd/csrc/hr_due.h).
#include "../../hirensi_amd/csrc/hr_due.h"

int main() {
  using namespace hr;
  Due<int> d;
  if (d.full() || d.get() != 0 || d.take() != 0) return 1;      // nothing due
  if (!d.put(7) || !d.full()) return 2;
  if (d.put(8) || d.get() != 7) return 3;                       // a second entry loses nothing
  if (d.take() != 7 || d.full() || d.get() != 0) return 4;      // taken once
  if (!d.put(9)) return 5;
  d.drop();
  if (d.full() || d.take() != 0) return 6;
  for (int stage = 0; stage <= 5; ++stage)                      // the other launches leave it to be flushed
    if (outputs_ride(stage) != (stage == 1)) return 7;
  return 0;
}
