// LDS of the routing kernels of many queries (route.hip) as their launches
// size it: host arithmetic without HIP, so that a CPU build can check it over
// every number of visible fines.
#pragma once

#include <stddef.h>

#if defined(__HIPCC__)
#define TAO_LDS_FN __host__ __device__ inline
#else
#define TAO_LDS_FN inline
#endif

namespace tao {

constexpr size_t kLdsBytes = 160 * 1024;   // of a CU: the most a workgroup can take

// Per-query routes: h rows, fine keys and page keys of a workgroup's query
// slots. A key row holds an odd number of words, so a column of them over the
// lanes spreads over the banks. Once the masses are formed the open pages (a
// bit each) and the selection lie where the h rows were.
struct RouteLds {
  int slots, fkeys, pkeys;           // slots; 16-bit keys of a row
  TAO_LDS_FN size_t bytes(int D) const {
    return (size_t)slots * (2 * (D + 8) + 2 * fkeys + 2 * pkeys);
  }
};
inline RouteLds route_lds(int slots, int max_epoch) {
  auto odd = [](int keys) { return 2 * (((keys + 1) / 2) | 1); };
  return RouteLds{slots, odd(max_epoch), odd(max_epoch / 8 + 1)};
}

// Turn routes of a prefill: sixteen turns a workgroup, each with its h row, a
// 32-bit key and a chosen page for every page or candidate (max_keys: the most
// of either that one turn has), and a bit for each page (static).
constexpr int kTurnSlots = 16;
constexpr int kTurnMaxEpoch = 2048;        // one byte numbers the pages
constexpr size_t kTurnOpenBytes = (size_t)kTurnSlots * (kTurnMaxEpoch / 8 / 32) * 4;

inline int turn_route_cap(int max_keys) { return max_keys | 1; }
inline size_t turn_route_bytes(int D, int cap) {
  return (size_t)kTurnSlots * (2 * (D + 8) + 5 * cap);
}
inline bool turn_route_fits(int D, int max_epoch, int max_keys) {
  return max_epoch >= 1 && max_epoch <= kTurnMaxEpoch && max_keys >= 1 &&
         turn_route_bytes(D, turn_route_cap(max_keys)) + kTurnOpenBytes <= kLdsBytes;
}

}  // namespace tao
