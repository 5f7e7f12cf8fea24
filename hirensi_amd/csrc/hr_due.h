// One piece of per-step work that goes with a later launch.  Plain C++, shared with the
// host-side check.
#pragma once

namespace hr {

// Holds at most one entry: a second one before the launch that takes the first would
// lose it, so it is refused.
template <class T>
class Due {
 public:
  bool put(const T& v) {
    if (full_) return false;
    v_ = v;
    full_ = true;
    return true;
  }
  bool full() const { return full_; }
  const T& get() const { return v_; }     // T{} where nothing is due
  T take() {
    const T v = v_;
    drop();
    return v;
  }
  void drop() {
    v_ = T{};
    full_ = false;
  }

 private:
  T v_{};
  bool full_ = false;
};

// Traces and slices are of the state that a step starts from: the launch of its first
// stage carries them, any other one finds them due beforehand.
constexpr bool outputs_ride(int stage) { return stage == 1; }

}  // namespace hr
