// lgv_em_tile.h -- the tiles of the Euler-Maruyama kernels (lgv_em.hip), by size.
#pragma once

#include <hip/hip_runtime.h>

namespace lgv {

constexpr int kEmBlock = 256;
constexpr int kEmSlots = 1024;  // blocks that the GPU holds at a time, about

// Tile of the two stencil marches: TX sites in x by TY rows in y, chunks of
// TZ planes in z.  A block's plane (tile plus a one-site ring, no corners)
// sits in LDS; each thread keeps its own column's planes z-1, z, z+1 in
// registers.
constexpr int kEmGrid = 400;  // (TY+2)(TX+2) <= 6 * 66
inline int em_div(int a, int b) { return (a + b - 1) / b; }

// TX: an even split of the row into at most 64.  From N = 100 on, where rows are
// whole 64-byte units, 64 or 48 instead, so that tiles are whole units too,
// unless that costs a tenth of the lanes at work (TY rows of N sites in nt tiles);
// 48 where no more lanes are at work with 64, and in rows of whole 256-byte units
// where 48 has a tenth more.  us per step forward / reverse, even -> 64, 48: 240^3
// 250 / 508 -> 230 / 440, 192 / 377; 304^3 510 / 1047 -> 447 / 858, 452 / 868;
// 368^3 862 / 1766 -> 786 / 1501, 772 / 1504; 288^3 393 / 799 -> 349 / 680, 388 /
// 744; 200^3 with Gaussian noise 196 / 313 -> -, 217 / 320; 72^3 15.0 / 28.4 ->
// 16.5 / 30.8, 16.4 / 29.1.
inline int em_width(int N) {
  const int even = em_div(N, em_div(N, 64));
  if (N < 100 || N % 8 != 0) return even;
  const int n48 = em_div(N, 48), n64 = em_div(N, 64);
  const int ty48 = kEmBlock / 48, ty64 = kEmBlock / 64, ty = kEmBlock / even;
  const bool w48 = 10 * ty48 * n64 >= (N % 32 == 0 ? 11 : 10) * ty64 * n48;
  // `even` takes n64 tiles
  if (9 * ty * (w48 ? n48 : n64) > 10 * (w48 ? ty48 : ty64) * n64) return even;
  return w48 ? 48 : 64;
}

// A block marches TZ planes after loading two: TZ of 8, 4, 2, 1 minimises the
// rounds of TZ + 2 planes (per step with 8 -> with the rule's: 33^3 Gaussian
// noise 24 -> 7.5 us (TZ 1), 64^3 15 -> 8.8 (TZ 1); 128^3 keeps 8).
inline void em_tile(int N, int &TX, int &TY, int &TZ) {
  TX = em_width(N);
  TY = kEmBlock / TX;
  if (TY > N) TY = N;
  const int tiles = em_div(N, TX) * em_div(N, TY);
  TZ = 8;
  for (int tz = 4; tz >= 1; tz /= 2)
    if (em_div(tiles * em_div(N, tz), kEmSlots) * (tz + 2) <
        em_div(tiles * em_div(N, TZ), kEmSlots) * (TZ + 2))
      TZ = tz;
  if (TZ > N) TZ = N;
}
inline int em_blocks(int N) {
  int TX, TY, TZ;
  em_tile(N, TX, TY, TZ);
  return em_div(N, TX) * em_div(N, TY) * em_div(N, TZ);
}

// Odd z chunks march downwards: two neighbouring chunks then start, or end, at
// their common boundary at the same time, and the plane that each reads from
// the other is still in the XCD's L2.  Where the GPU does not hold the blocks of
// two neighbouring chunks at a time, all march upwards.
inline bool em_alternates(int N, int TX, int TY) {
  return 2 * em_div(N, TX) * em_div(N, TY) <= kEmSlots;
}

// The tile of a launch, from the host: worked out in the kernels it is a chain
// of divisions before the first load (64^3 10.8 us a step, 11.5 so).
struct EmTile {
  int TX, TY, TZ;
  bool alternate;
};
inline EmTile em_tile(int N) {
  EmTile t;
  em_tile(N, t.TX, t.TY, t.TZ);
  t.alternate = em_alternates(N, t.TX, t.TY);
  return t;
}

}  // namespace lgv
