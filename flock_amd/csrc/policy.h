// policy.h -- the size-class policy's view of a whole batch (or server slice).  No device code.
#pragma once
#include <cstdint>

namespace flock {

// Over the instances whose tree and snapshot a 512-thread workgroup's LDS takes: add() each,
// then ask.  An instance's time on its workgroup grows about as (m+n)^2 with Dantzig pricing.
struct BatchShape {
  int max_v = 0;  // the largest m+n
  double v2 = 0, v3 = 0;
  int64_t count = 0;
  void add(int v) {
    max_v = v > max_v ? v : max_v;
    v2 += (double)v * v;
    v3 += (double)v * v * v;
    ++count;
  }
  // Whether Dantzig pricing, a sweep per pivot, wants 512 threads for every instance although
  // there are more instances than compute units.  A unit holds one 512-thread workgroup at a
  // time but three of 256, so 512 pay only for large instances (device ms at 256 / 512):
  //  - load, the units' share of all instances' time in units of the largest's, times the
  //    square of 420 / mean m+n (weighted by time; small instances lose more to the empty
  //    slots), is at most 1.8: the largest instance's chain of pivots sets the time (512 of
  //    [16,400] 16.0 / 14.1, 768 of [16,300] 7.8 / 6.5, 512 of [50,250] 5.4 / 4.8; not 1024
  //    of [16,256] 6.3 / 6.4, 257 of [130,140] 1.95 / 2.47, 1280 of [100,300] 16.4 / 17.0);
  //    instances much alike (time at the mean over 0.75 of the largest's) have to be 1.5 a
  //    unit, or units with two of them take twice as long as the others (257 of [400,430]
  //    32.1 / 36.3, 512 of them 67.0 / 60.9);
  //  - the mean is above 450 and there are 1.5 to 4 instances a unit: 512 threads use a full
  //    unit as well (768 of [210,240] 14.6 / 13.1, 1024 of [200,300] 26.2 / 24.5; not 768 of
  //    [180,220] 9.9 / 10.4, 1600 of [200,300] 37.3 / 38.6).
  // At most m+n = 400 nothing gains (512 of [16,200] 3.10 / 3.07, 1024 3.5 / 4.5).
  bool dantzig_wide(int units) const {
    if (max_v <= 400) return false;
    const double largest = (double)max_v * max_v, mean_v = v3 / v2, small = 420 / mean_v;
    const bool many = 2 * count >= 3 * (int64_t)units;
    const bool alike = v2 > 0.75 * largest * (double)count;
    const bool chain = v2 / (units * largest) * small * small <= 1.8 && (many || !alike);
    const bool full = mean_v > 450 && many && count <= 4 * (int64_t)units;
    return chain || full;
  }
};

}  // namespace flock
