// Which work a pass workgroup does.  No device code: also compiled for the host.
#pragma once
#include <hip/hip_runtime.h>

#ifndef TOTEM_XCD_REMAP
#define TOTEM_XCD_REMAP 1      // XCD-aware workgroup -> (probe, row/column group) mapping
#endif

namespace totem {

// Unit u (< K) of workgroup `bid` -> (probe item, group g of G per probe).
//
// Workgroups are dispatched round-robin over the 8 XCDs, each with its own L2.
// With the remap, XCD x works through the groups [x*G/8, (x+1)*G/8) of every probe in
// order: neighbouring column groups (which share 128-byte lines) run back to back on
// one L2, and each L2 only ever sees 1/8 of the propagator / a band of the transmission
// slice.  Any G with G/8 divisible by K gives a bijection; otherwise the plain
// probe-major order is used.  Taking one group of every probe of the launch in turn
// instead (so that consecutive workgroups of an XCD share a group's transmission rows
// or propagator columns) measured slower at every size (2048 points, 6 probes per
// launch: rows 91.5 -> 105 us, columns 108 -> 158 us; 1024: columns 88 -> 120 us).
template <int K = 1>
__host__ __device__ __forceinline__ void unit_map(int bid, int u, int G, int& item, int& g) {
#if TOTEM_XCD_REMAP
  if ((G & 7) == 0 && (G >> 3) % K == 0) {
    const int xcd = bid & 7, gp = G >> 3;
    const int q = (bid >> 3) * K + u;
    item = q / gp;
    g = xcd * gp + (q - item * gp);
    return;
  }
#endif
  const int q = bid * K + u;
  item = q / G;
  g = q - item * G;
}

}  // namespace totem
