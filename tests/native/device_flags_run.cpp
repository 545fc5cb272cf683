// Test helper: DeviceFlags (novaq_device_flags.h) from several threads.  Prints
// "ok" when every device's flag is its own, once set stays set, and none is lost
// where threads set different devices' flags at once.  Built with g++ by
// tests/test_device_flags.py.
#include <cstdio>
#include <thread>
#include <vector>

#include "../../novann_amd/csrc/novaq_device_flags.h"

int main() {
  for (int round = 0; round < 200; ++round) {
    novaq::DeviceFlags f;
    for (int d = -1; d < 70; ++d)
      if (f.test(d)) return std::printf("set at the start: %d\n", d), 1;
    std::vector<std::thread> t;
    for (int k = 0; k < 8; ++k)
      t.emplace_back([&f, k] {
        for (int d = k; d < 64; d += 8) {
          f.set(d);
          if (!f.test(d)) std::printf("lost: %d\n", d);
        }
      });
    for (auto& th : t) th.join();
    for (int d = 0; d < 64; ++d)
      if (!f.test(d)) return std::printf("lost: %d\n", d), 1;
    f.set(-1);
    f.set(64);
    if (f.test(-1) || f.test(64)) return std::printf("flag of no device\n"), 1;
  }
  novaq::DeviceFlags one;
  one.set(3);
  for (int d = 0; d < 64; ++d)
    if (one.test(d) != (d == 3)) return std::printf("not its own: %d\n", d), 1;
  std::printf("ok\n");
  return 0;
}
