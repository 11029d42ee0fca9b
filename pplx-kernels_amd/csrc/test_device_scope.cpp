// DeviceScope in processes that see no, one or several devices, whichever this one sees: HIP's three
// functions of the current device are this program's own.
//
//   test_device_scope <devices>      (what hipGetDeviceCount says; negative: it fails)
#include "a2a_device_scope.h"

#include <cstdio>
#include <cstdlib>

namespace {
int g_devices = 0, g_current = 0, g_gets = 0, g_sets = 0;
int g_failures = 0;

void expect(bool holds, const char *what) {
  if (!holds) ++g_failures;
  printf("  %s [%s]\n", holds ? "pass" : "FAIL", what);
}
}  // namespace

extern "C" {
hipError_t hipGetDeviceCount(int *n) {
  if (g_devices < 0) return hipErrorNoDevice;
  *n = g_devices;
  return hipSuccess;
}
hipError_t hipGetDevice(int *device) {
  ++g_gets;
  if (g_devices <= 0) return hipErrorNoDevice;
  *device = g_current;
  return hipSuccess;
}
hipError_t hipSetDevice(int device) {
  ++g_sets;
  if (device < 0 || device >= g_devices) return hipErrorInvalidDevice;
  g_current = device;
  return hipSuccess;
}
}

int main(int argc, char **argv) {
  g_devices = argc > 1 ? atoi(argv[1]) : 0;
  using pplx_amd::DeviceScope;
  if (g_devices <= 0) {
    for (int device = 0; device < 2; ++device) {
      DeviceScope scope(device);
      expect(!scope.ok(), "no device to select");
    }
    expect(g_sets == 0, "none selected");
  } else {
    {
      DeviceScope scope(0);
      expect(scope.ok() && g_current == 0 && g_sets == 0, "the current device");
      expect(g_gets == (g_devices == 1 ? 0 : 1), "asked for where there are several");
    }
    {
      DeviceScope scope(g_devices);
      expect(!scope.ok() && g_current == 0, "a device that is not there");
    }
    expect(g_current == 0 && g_sets == 1, "nothing to restore");
    for (int from = 0; from < g_devices; ++from) {
      for (int to = 0; to < g_devices; ++to) {
        g_current = from;
        g_sets = 0;
        {
          DeviceScope scope(to);
          expect(scope.ok() && g_current == to, "selected");
          {
            DeviceScope inner(from);
            expect(inner.ok() && g_current == from, "selected inside another");
          }
          expect(g_current == to, "the outer one's again");
        }
        expect(g_current == from && g_sets == (from == to ? 0 : 4), "restored");
      }
    }
  }
  printf(g_failures ? "%d FAILED\n" : "ALL PASSED\n", g_failures);
  return g_failures ? 1 : 0;
}
