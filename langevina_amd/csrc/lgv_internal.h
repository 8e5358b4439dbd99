// lgv_internal.h -- structures shared by the kernels (lgv_kernels.hip) and
// the context / C-ABI layer (lgv_api.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <vector>

namespace lgv {

constexpr int kCUs = 256;  // MI355X
constexpr int kBlock = 256;  // threads per block of every sweep kernel but these:
constexpr int kPairBlock = 1024;  // k_hb_brick, k_hb_sweep

// Read-only (for the kernels) description of one replica.  The step
// coefficients (rdtg, rms, dt_ideal, tau) are computed on the host with the
// reference's expressions for the dt in use.
struct ReplicaParams {
  void *fields[2];    // two buffers of 10 planes x 2 parities x half elements
                      // (T = double/float); ReplicaState::cur_phi / cur_chg
                      // select where the live phi / charge planes are, the
                      // out-of-place kernels write the other buffer
  int N, NH;
  int64_t half;       // N^3 / 2
  double mass0, dmassdt, lambda, H, chi;
  double axx;         // pow(1/h, 2), Stepper.cxx:91-93
  double rdtg;        // sqrt(2 dt_hb gamma), Stepper.cxx:301
  double rms;         // sqrt(2 dt sigma), Stepper.cxx:456
  double dt_ideal;    // dt / scounts[1]
  double tau_ideal;   // dt_ideal / 2.0
  uint64_t base_key;
  int tile_cap, tile_tz;   // ideal-kernel tile (see ideal_tile)
  int hb_cap, hb_tz;       // phi-march tile (see hb_tile)
  int chg_cap, chg_chunk;  // charge-march tile (see charge_tile)
  int pair_y, pair_z;      // rows in y and planes of a block of both parities
  float chg_l2;            // see charge_l2
};

// -log2(e) / (2 chi) in single precision, with which the charge sweep forms
// exp(-dS) from dS 2 chi.  NaN, so that the double test decides, where that or
// dS 2 chi might leave the range of single precision: within 2^-100 .. 2^100 a
// dS 2 chi that overflows is a dS beyond 2^27, and one below 2^-126 a dS below
// 2^-26.
inline float charge_l2(double chi) {
  const double d = 2. * chi;
  return d >= 0x1p-100 && d <= 0x1p100 ? (float)(-0x1.71547652b82fep+0 * (1. / d))
                                       : __builtin_nanf("");
}

// Device-written state of one replica (clock, counters, per-step data).
struct ReplicaState {
  double t;
  uint64_t sweep_ctr;
  int cur_phi;       // buffer (0/1) holding the live phi planes
  int cur_chg;       // buffer (0/1) holding the live charge planes
  int pad;
  double E_old, E_new;
};

// The tile fields of ReplicaParams hold what a launch uses: the caller's
// request, or where that is 0 the choice of the rules (the resolve_ functions in
// lgv_api.hip, by replica size, storage type and the blocks of the launch).

// Tile of the fused ideal kernel: TXH half-columns x TY rows in x-y,
// marching over TZ planes in z.  (TY+2)(2 TXH+2) <= kIdealLds.  The
// one-site halo ring (2 TY + 4 TXH sites) may exceed the block's threads
// (64 half-columns x 4 rows: 264); its remainder then takes a second pass.
constexpr int kIdealLds = 800;
// FP32 fields keep the raw charges of the current plane in LDS as well, so
// their plane grid is held to the tiles of width <= 32 half-columns (at most
// 660 entries) and three blocks still fit one CU's LDS.
constexpr int kIdealLdsF32 = 660;
__host__ __device__ constexpr int ideal_lds(bool fp32) { return fp32 ? kIdealLdsF32 : kIdealLds; }
__host__ __device__ inline void ideal_tile(int N, int cap, int tz, int &TXH, int &TY, int &TZ) {
  const int NH = N / 2;
  TXH = NH < cap ? NH : cap;
  TY = kBlock / TXH;
  if (TY > N) TY = N;
  TZ = N < tz ? N : tz;
}

// Tile of the single-parity phi march: TXH half-columns x TY rows in x-y,
// chunks of TZ planes in z, valid while the packed grid fits
// (TY+2)(TXH+2) <= kHbMarchGrid and the ring 2 TY + 2 TXH <= kBlock.
__host__ __device__ inline void hb_tile(int N, int cap, int tz, int &TXH, int &TY, int &TZ) {
  const int NH = N / 2;
  TXH = NH < cap ? NH : cap;
  TY = 256 / TXH;
  if (TY > N) TY = N;
  TZ = N < tz ? N : tz;
}

// Its packed LDS grid: (TY+2)(TXH+2) entries.
constexpr int kHbMarchGrid = 400;

// Tile of the charge march kernel: TXH half-columns x TQ lines of the
// cross-section, chunks of C sites along the direction (C even), two blocks
// per tile (the even and the odd x of its half-columns).
__host__ __device__ inline void charge_tile(int N, int cap, int chunk, int &TXH, int &TQ,
                                            int &C) {
  const int NH = N / 2;
  TXH = NH < cap ? NH : cap;
  TQ = 256 / TXH;
  if (TQ > N) TQ = N;
  C = N < chunk ? N : chunk;
}

// Per-block monitor partials (o4_stepper_monitor counters).
struct MonSlot {
  long long down_counts, up_counts, up_yes, up_no;
  double down_dS, up_dS;
};

struct EnergySlot {
  double g_s, g_c, h_s, h_c, n_s, n_c;
};

// The blocks of a launch over several replicas, on the device: workgroup b is
// block local[b] of replica rep[b] (local == nullptr: block b - first[rep[b]]),
// and a replica's monitor slots start at first[replica].  rep == nullptr: all
// of replica 0.
struct LaunchBlocks {
  int *rep = nullptr, *local = nullptr, *first = nullptr;
};
struct Plan {
  int nblocks = 0;
  LaunchBlocks blocks;
  bool wide = false;    // 64-bit offsets: some plane of the launch (phi march: pair of planes)
                        // is >= 4 GiB
  bool stream = false;  // outputs written with non-temporal stores (see kCacheBytes)
  bool far = false;     // some replica's charge planes span >= 4 GiB (charge launch)
  // ideal launch: every replica's odd z chunks march downwards (see
  // ideal_alternates); an argument of the launch: read with a replica's tile, it
  // cost a step of 64^3 0.5 us
  bool alternate = true;
  bool xwave = false;   // charge launch: every replica has N = 128 or 256 (x rows per wave)
  std::vector<int> first;  // host copy of blocks.first
};

// The phi marches and the ideal kernel write their outputs with non-temporal
// stores where the outputs are next read by a later launch, after planes that
// together exceed the last-level cache have been swept, so that caching them
// only evicts lines that neighbouring tiles still read; and only where a tile's
// rows are whole lines (a non-temporal store of part of a line costs more than
// a cached one).  Ideal: fields (one buffer) above twice the cache, rows and
// tile rows of whole 128-byte lines, or of whole 64-byte halves of FP64 lattices
// that alone exceed it (ideal_unit); FP64 192^3 263 -> 259 us, 224^3 449 ->
// 437, 256^3 556 -> 534, FP32 256^3 324 -> 318; rows of 6.5 lines, 208^3, in
// tiles of 56 356 -> 337, of broken units, 52, 384 -> 413; 200^3, rows of 12.5
// halves, 308 -> 377; FP32 rows of halves 288^3 522 -> 536, in tiles of 36 644 ->
// 956.  Phi march: phi
// planes (one buffer) above the cache, rows and tile rows of whole 64-byte
// halves; FP64 208^3 94.5 -> 90.8 us, 224^3 119 -> 106, 256^3 170 -> 148,
// FP32 384^3 302 -> 291, but 256^3 FP32 (phi planes of just 256 MB) 86 -> 92,
// 280^3 FP64 (rows of 8.75 lines) 228 -> 242, 320^3 in tiles of 54 342 -> 394.
// k_hb_sweep: fields above twice the cache, rows of whole 64-byte halves; its own
// time changes little (256^3 128 -> 127 us, 224^3 87 -> 89), but the ideal and the
// charge kernel after it find more of their planes (256^3 551 -> 537, 329 -> 322;
// whole steps 192^3 1889 -> 1862, 224^3 3043 -> 3008, 256^3 4156 -> 4091; 160^3
// 1166 -> 1173, 200^3, rows of 6.25 lines, 2415 -> 2427).
constexpr uint64_t kCacheBytes = 256ull << 20;

// Width of an x tile of at most cap half-columns that splits a row of NH
// evenly: with a fixed width of 32 or 64 the last tile of a row whose length
// is no multiple of it is mostly empty (NH = 75 in tiles of 64: 59 % of the
// lanes at work; in two of 38, 99 %).
inline int even_width(int NH, int cap) {
  const int n = (NH + cap - 1) / cap;
  return (NH + n - 1) / n;
}

// The ideal kernel: blocks that the GPU holds at a time, and blocks of one z
// plane with tiles of width cap.
inline int ideal_slots(bool fp32) { return kCUs * (fp32 ? 3 : 2); }
inline int64_t ideal_plane_blocks(int N, int cap) {
  int TXH, TY, TZ;
  ideal_tile(N, cap, 1, TXH, TY, TZ);
  return (int64_t)((N / 2 + TXH - 1) / TXH) * ((N + TY - 1) / TY);
}
// Whether a lattice's fields alone exceed twice the cache.
inline bool ideal_large(int N, bool fp32) {
  return 10 * (uint64_t)N * N * N * (fp32 ? 4 : 8) > 2 * kCacheBytes;
}
// The unit in bytes whose multiples rows and tile rows have to be for
// non-temporal stores (see kCacheBytes).
inline int ideal_unit(int N, bool fp32) { return !fp32 && ideal_large(N, fp32) ? 64 : 128; }
// The width of its tiles where the caller asked for none: 32 half-columns where
// they divide the row (whole 128-byte lines of every component: 256^3 FP64 541
// us against 560 with 64) or need fewer tiles than the alternative; 16 for FP64
// rows of several tiles that those divide (160^3 174 -> 148 us, 224^3 443 ->
// 398; a FP32 row of 16 is half a line).  Rows of whole 64-byte units of a large
// lattice take such tiles: FP32 32 (288^3 583 -> 520, 480^3 2440 -> 2350), FP64
// the width with most lanes at work (TY rows of NH half-columns in nt tiles), on
// a tie the fewest, then the narrowest tiles (208^3 369 -> 337, 240^3 535 -> 490,
// 272^3 865 -> 715, 304^3 1160 -> 1010, 368^3 2107 -> 1780, 400^3 2640 -> 2320).
// Otherwise the widest even split that the kernel's plane grid holds (every ring
// column costs a line per row and component: 200^3 FP64 329 us with 50, 390 with
// 34, 435 with 25).
inline int ideal_width(int N, bool fp32) {
  const int NH = N / 2;
  if (NH > 64 && ideal_large(N, fp32) && NH % 16 == (fp32 ? 0 : 8)) {
    if (fp32) return 32;
    int best = 0, best_ty = 0, best_nt = 1;
    for (int cap = 32; cap <= 64; cap += 8) {
      const int TY = kBlock / cap, nt = (NH + cap - 1) / cap;
      const int gain = TY * best_nt - best_ty * nt;
      if (gain > 0 || (gain == 0 && nt < best_nt)) {
        best = cap;
        best_ty = TY;
        best_nt = nt;
      }
    }
    return best;
  }
  int width = 0;
  for (int cap = 64; cap >= 32 || !width; cap--) {
    int TXH, TY, TZ;
    ideal_tile(N, even_width(NH, cap), 1, TXH, TY, TZ);
    if ((TY + 2) * (2 * TXH + 2) <= ideal_lds(fp32)) {
      width = TXH;
      break;
    }
  }
  if (NH % 32 == 0 || ideal_plane_blocks(N, 32) < ideal_plane_blocks(N, width)) width = 32;
  if (!fp32 && NH % 32 == 16 && NH > width) width = 16;
  return width;
}

// Whether the ideal kernel's odd z chunks march downwards.  Two neighbouring
// chunks that run at the same time then start, or end, at their common boundary
// together, and the planes that each reads from the other are still in the XCD's
// L2 (256^3 FP64 545 -> 530 us, 240^3 554 -> 534).  They do where the GPU holds
// the blocks of both; otherwise the planes a chunk ends with are the first that
// the next one, marching the same way, reads (512^3 FP64 4230 -> 4110 us, 528^3
// 5100 -> 4950, 576^3 5950 -> 5850).
inline bool ideal_alternates(int N, int cap, bool fp32) {
  return 2 * ideal_plane_blocks(N, cap) <= ideal_slots(fp32);
}

// Width of the charge march's tiles: an even split of the row into at most 64.
// Where a replica's fields exceed the last-level cache and its rows are whole
// 64-byte units, tiles are too, or neighbouring tiles share a unit of every row
// and plane: 64, or 48 where that takes no more tiles (a block then has five
// lines instead of four).  Three launches, FP64, even -> 48 / 64: 176^3 475 ->
// 434 / 455 us, 272^3 1654 -> 1379 / 1413, 320^3 2614 -> 2213 / 2076, 352^3 3390
// -> 2829 / 2698, 528^3 9764 -> 10640 / 9563; FP32 224^3 575 -> 610 / 543, 480^3
// 5301 -> - / 4753; below the cache FP64 144^3 251 -> 264 / 298, FP32 160^3 209 ->
// 225 / 298.
inline int charge_width(int NH, bool fp32) {
  const int esz = fp32 ? 4 : 8;
  const uint64_t bytes = 80 * (uint64_t)NH * NH * NH * esz;  // ten planes of (2 NH)^3
  if (NH <= 64 || bytes <= kCacheBytes || NH * esz % 64 != 0) return even_width(NH, 64);
  return (NH + 47) / 48 == (NH + 63) / 64 ? 48 : 64;
}

// From this many sites on (all replicas) the phi half-sweeps run the z-march:
// it reads each value of the other parity once per launch where the
// one-thread-per-site kernel reads it up to four times, which costs that
// kernel traffic once the fields outgrow the 256 MB last-level cache; below,
// the per-site kernel's eight waves per SIMD (the march has four) count more.
// Whole steps, per site -> march: FP64 100^3 328 -> 332 us, 150^3 1134 -> 1169,
// 180^3 2058 -> 2070, 192^3 2124 -> 2082, 224^3 3840 -> 3636, 256^3 5006 ->
// 4371; FP32 128^3 410 -> 411, 180^3 1219 -> 1229, 192^3 1328 -> 1304, 224^3
// 2253 -> 2214, 256^3 2949 -> 2708.
// One FP64 lattice runs half-sweeps only as lone calls and as the last of an odd
// number, without a step's other kernels in the cache: two of them, site ->
// march, 192^3 123 -> 132 us, 200^3 139 -> 142, 204^3 181 -> 165 (a batch of 60 x
// 48^3 144 -> 127).
constexpr uint64_t kMarchSites = 7000000;
inline uint64_t phi_march_sites(bool fp32, int nreplicas) {
  return fp32 || nreplicas > 1 ? kMarchSites : 7500000;
}

// Pairs of phi sweeps run as launches of both parities, out of place (a pair
// leaves the live buffer where it was), below the first number of sites (all
// replicas) in bricks that fit kBrickLds bytes of LDS (k_hb_brick, two blocks of
// a CU), and FP64 fields from the second on in the march k_hb_sweep.
// Small lattices save launches.  Whole steps, half-sweeps -> bricks: FP64 16^3
// 100 -> 88 us, 32^3 106 -> 93, 64^3 151 -> 144, 80^3 231 -> 226, 84^3 248 ->
// 275, 5 x 48^3 230 -> 229; FP32 64^3 138 -> 128, 80^3 193 -> 189, 84^3 207 ->
// 209, 16 x 32^3 174 -> 165, 32 x 32^3 251 -> 246, 64 x 32^3 422 -> 457: above,
// the facing rows' extra decisions cost more than the launches saved.
// Large FP64 lattices are bound by the bytes of a half-sweep, which reads both
// parities and writes one; both parities in one pass read and write each value
// once.  Half-sweeps -> k_hb_sweep: 128^3 628 -> 648 us, 140^3 938 -> 938, 144^3
// 986 -> 967, 160^3 1267 -> 1176, 200^3 2509 -> 2414, 224^3 3221 -> 3057, 256^3
// 4319 -> 4162 (three contexts at once 4444 -> 4135 a step), 300^3 9159 -> 8372.
// FP32 fields move half the bytes and the march is bound by its decisions and
// one barrier per plane: 256^3 2664 -> 2911 us, 160^3 FP32 likewise slower.
constexpr uint64_t kBrickSites = 560000;
constexpr int kBrickLds = 64 << 10;
// In a batch, a replica below the side fills too few of a block's threads with
// its rows: 96 x 48^3 3004 -> 3278, but 16 x 64^3 1167 -> 1144, 8 x 96^3 2026 ->
// 1945, 2 x 160^3 2460 -> 2184.
constexpr uint64_t kPairMarchSites = 2900000;
constexpr int kPairMarchSide = 64;
// Rows that a block of k_hb_sweep owns: its threads less a facing row on either
// side; 0: the rows are too long for it.  A block of one row (sides above 512)
// decides three sites for each it keeps: step 514^3 FP64 56.1 ms, half-sweeps
// 49.9; 528^3 54.7, 48.5; 576^3 63.9, 56.4; of two rows 480^3 33.6, 33.7; 512^3
// 35.8, 36.8; 410^3 24.7, 25.4.
inline int pair_march_rows(int N) {
  const int rows = kPairBlock / (N / 2) - 2;
  return rows < 2 ? 0 : rows < N ? rows : N;
}

// A context of one lattice whose fields (one buffer) exceed this keeps the
// charge sweep after the phi sweeps rather than beside them; beside k_hb_sweep,
// which does not fill the memory system, the charge sweep gains up to more.
// Steps, after -> beside: 192^3 FP64 1913 -> 1876 us, 224^3 3019 -> 2965, 256^3
// 4131 -> 4073 (three contexts at once 4106 -> 4114), 300^3 8361 -> 8457; 256^3
// FP32 2703 -> 2702 (three contexts 2705 -> 2717).
constexpr uint64_t kOverlapBytes = 600ull << 20;
constexpr uint64_t kOverlapBytesPairMarch = 1300ull << 20;

// Largest side: N^3 must fit 32-bit site indices.
constexpr int kMaxN = 1536;

// Shape of the measurement pass (k_measure_tile): TX x TZ columns per
// wavefront, groups of nz tiles in z taken in turn, chunks of CY rows in y; ntx,
// ntz tiles and nch chunks.  The partial sums hold 25 N (nch ntx + words
// groups (nch + ntx)) doubles, at most 50 max(2^19, N^2).  While one tile a
// wavefront fits that, chunks are halved until the launch has 2048 wavefronts,
// which is what the GPU holds (256^3 FP64: 471 us with 1024, 385 with 2048, 383
// with 4096); small lattices stop at 16 N, where more partial sums cost as much
// as the shorter chunks give.  From N = 386 on nz and the chunk minimise the
// rounds of wavefronts, each of nz tiles of CY rows and about four rows' time
// for a tile's own sums (512^3 FP64: 512 wavefronts 7.5 ms, 2048 3.8).
struct MeasureShape {
  int TX, TZ, nz, CY, ntx, ntz, nch;
};
constexpr int64_t kMeasurePart = int64_t(1) << 19;
constexpr int kMeasureWaves = 2048;
__host__ __device__ inline int64_t measure_part_limit(int N) {
  const int64_t n2 = (int64_t)N * N;
  return 50 * (n2 > kMeasurePart ? n2 : kMeasurePart);
}
__host__ __device__ inline int measure_groups(const MeasureShape &s) {
  return (s.ntz + s.nz - 1) / s.nz;
}
__host__ __device__ inline int measure_words(const MeasureShape &s) { return s.nz > 1 ? 2 : 1; }
__host__ __device__ inline int64_t measure_waves(const MeasureShape &s) {
  return (int64_t)s.ntx * measure_groups(s) * s.nch;
}
__host__ __device__ inline int64_t measure_part(const MeasureShape &s, int N) {
  return 25 * (int64_t)N *
         ((int64_t)s.nch * s.ntx +
          (int64_t)measure_words(s) * measure_groups(s) * (s.nch + s.ntx));
}
inline MeasureShape measure_shape(int N) {
  MeasureShape s;
  s.ntx = (N + 63) / 64;
  s.TX = (N + s.ntx - 1) / s.ntx;
  s.TZ = 64 / s.TX;
  if (s.TZ > N) s.TZ = N;
  s.ntz = (N + s.TZ - 1) / s.TZ;
  s.nz = s.nch = 1;
  s.CY = N;
  if (measure_part(s, N) <= measure_part_limit(N)) {
    const int64_t waves = N < 128 ? 16 * N : kMeasureWaves;
    while (s.CY > 1 && measure_waves(s) < waves) {
      MeasureShape h = s;
      h.CY = (s.CY + 1) / 2;
      h.nch = (N + h.CY - 1) / h.CY;
      if (measure_part(h, N) > measure_part_limit(N)) break;
      s = h;
    }
    return s;
  }
  MeasureShape best = s;
  int64_t best_cost = INT64_MAX;
  for (s.nz = 2; s.nz < 2 * s.ntz; s.nz *= 2)
    for (s.CY = 4; s.CY < N + 4; s.CY += 4) {
      s.nch = (N + s.CY - 1) / s.CY;
      if (measure_part(s, N) > measure_part_limit(N)) continue;
      const int64_t rounds = (measure_waves(s) + kMeasureWaves - 1) / kMeasureWaves;
      const int64_t cost = rounds * s.nz * (s.CY + 4);
      if (cost < best_cost) {
        best_cost = cost;
        best = s;
      }
    }
  return best;
}

// Kernel launchers (lgv_kernels.hip).  fp32 selects the storage type.
// flip: the live-buffer flips of the earlier launches of the step, not yet
// in the replica state (bit 0 phi, bit 1 charges); launch_advance applies a
// step's net flip.
void launch_hb_phi(bool fp32, const Plan &plan, const ReplicaParams *P, ReplicaState *S,
                   int ieo, int ctr_off, int flip, MonSlot *mon, hipStream_t st);
void launch_hb_brick(bool fp32, const Plan &plan, int lds, const ReplicaParams *P,
                     ReplicaState *S, int ctr_off, int flip, MonSlot *mon, hipStream_t st);
void launch_hb_sweep(const Plan &plan, const ReplicaParams *P, ReplicaState *S, int ctr_off,
                     int flip, MonSlot *mon, hipStream_t st);
void launch_hb_march(bool fp32, const Plan &plan, const ReplicaParams *P, ReplicaState *S,
                     int ieo, int ctr_off, int flip, MonSlot *mon, hipStream_t st);
void launch_charge_march(bool fp32, const Plan &plan, const ReplicaParams *P, ReplicaState *S,
                         int ixyz, int ctr_off, int flip, MonSlot *mon, hipStream_t st);
void launch_ideal(bool fp32, const Plan &plan, const ReplicaParams *P, ReplicaState *S,
                  int flip, hipStream_t st);
void launch_energy(bool fp32, const Plan &plan, const ReplicaParams *P,
                   const ReplicaState *S, int flip, EnergySlot *slots, hipStream_t st);
void launch_energy_finish(int nrep, const Plan &plan, const ReplicaParams *P,
                          ReplicaState *S, const EnergySlot *slots, int which,
                          int ctr_off, MonSlot *mon_ideal, hipStream_t st);
void launch_advance(int nrep, ReplicaState *S, double dt, int advance_time,
                    uint64_t nctr, int flip, hipStream_t st);
void launch_set_time(int nrep, int replica, ReplicaState *S, double t, hipStream_t st);
// Field transfers go through a staging buffer of at most kStageBytes, in
// slabs of whole z-planes.
constexpr int64_t kStageBytes = int64_t(2) << 30;
__host__ __device__ inline int stage_planes(int N) {
  const int64_t plane = (int64_t)N * N * 10 * (int64_t)sizeof(double);
  const int64_t n = kStageBytes / plane;
  return n < 1 ? 1 : (n > N ? N : (int)n);
}
void launch_aos_to_rb(bool fp32, const ReplicaParams *P, const ReplicaState *S, int replica,
                      int N, int z0, int nz, const double *aos, hipStream_t st);
void launch_rb_to_aos(bool fp32, const ReplicaParams *P, const ReplicaState *S, int replica,
                      int N, int z0, int nz, double *aos, hipStream_t st);
// host_*: pinned host memory, written beside the device copies (launch_measure)
// or alone (launch_wall_dft), so that no transfer follows the kernels.
void launch_wall_dft(int N, const double *wall, const double *wallphase, double *host_wall_k,
                     double *host_wallphase_k, hipStream_t st);
void launch_measure(bool fp32, const ReplicaParams *P, const ReplicaState *S, int replica,
                    int N, double *part, double *wall, double *wallphase, double *host_wall,
                    double *host_wallphase, hipStream_t st);

}  // namespace lgv
