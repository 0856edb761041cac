// gsis_wait.h -- the limit of a wait whose length depends on others' work (for
// device and host code).
#pragma once

namespace gsis {

// Over when `limit` ticks have passed in which `progress`, a number that changes
// as the work that is waited for goes on, stayed the same.
struct StallLimit {
  long long limit, since = 0, seen = 0;
  bool begun = false;
  constexpr explicit StallLimit(long long ticks) : limit(ticks) {}
  constexpr bool over(long long progress, long long now) {
    if (!begun || progress != seen) {
      begun = true;
      seen = progress;
      since = now;
    }
    return now - since > limit;
  }
};

}  // namespace gsis
