// lgv_api.hip -- the C ABI of include/lgv.h: context, replica storage,
// composition of PV2HBSplit::step from the kernels, host-side global engine
// (initial charges), monitors and measurement.
#include <algorithm>
#include <cfloat>
#include <array>
#include <cmath>
#include <complex>
#include <limits>
#include <cstdarg>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <memory>
#include <random>
#include <string>
#include <vector>

#include "lgv.h"
#include "lgv_device.h"
#include "lgv_internal.h"

using namespace lgv;

namespace {

thread_local std::string g_err;

int fail(int code, const char *fmt, ...) {
  char buf[512];
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(buf, sizeof buf, fmt, ap);
  va_end(ap);
  g_err = buf;
  return code;
}

#define HIPCHECK(expr)                                                          \
  do {                                                                          \
    hipError_t e_ = (expr);                                                     \
    if (e_ != hipSuccess)                                                       \
      return fail(LGV_ERR_HIP, "%s: %s (%s:%d)", #expr, hipGetErrorString(e_), \
                  __FILE__, __LINE__);                                          \
  } while (0)

// std::seed_seq{base}.generate(1 word): the seed NoiseGenerator gives rank 0
// (ModelG/NoiseGenerator.h:68-82).
uint32_t rank0_seed(int base) {
  std::seed_seq seq = {base};
  uint32_t out = 0;
  seq.generate(&out, &out + 1);
  return out;
}

// NoiseGenerator's engine and its normal() (libstdc++ 11 Marsaglia polar
// method with one cached value, bits/random.tcc:1802-1835).
struct HostNoise {
  Xoro g;
  double saved = 0.;
  int has_saved = 0;
  double normal() {
    if (has_saved) {
      has_saved = 0;
      return saved * 1.0 + 0.0;
    }
    double x, y, r2;
    do {
      x = 2.0 * canonical(xoro_next(g)) - 1.0;
      y = 2.0 * canonical(xoro_next(g)) - 1.0;
      r2 = x * x + y * y;
    } while (r2 > 1.0 || r2 == 0.0);
    const double mult = std::sqrt(-2 * std::log(r2) / r2);
    saved = x * mult;
    has_saved = 1;
    return (y * mult) * 1.0 + 0.0;
  }
};

}  // namespace

// Tiles a caller asked for; 0: the library's rule.
struct TileRequest {
  int ideal_cap = 0, ideal_tz = 0, hb_cap = 0, hb_tz = 0, chg_cap = 0, chg_chunk = 0;
};

// The kernel of launches of both parities: k_hb_brick, k_hb_sweep.
enum class TwoParity { kNone, kBricks, kMarch };

struct lgv_ctx {
  int device = 0;
  hipStream_t stream = nullptr;
  // the charge sweep of a step and the phi sweeps that follow the last ideal
  // substep run concurrently, one of them on stream2 (see enqueue_step)
  hipStream_t stream2 = nullptr;
  hipEvent_t ev_fork = nullptr, ev_join = nullptr;
  bool overlap = true;
  bool fp32 = false;
  unsigned s0 = 2, s1 = 3;
  bool nodiffuse = false, onlydiffuse = false, track_energy = false;
  int nrep = 0;
  std::vector<lgv_model_params> mp;
  std::vector<ReplicaParams> hp;
  std::vector<TileRequest> tiles;  // per replica; hp holds the resolved tiles
  std::vector<HostNoise> noise;
  ReplicaParams *dP = nullptr;
  ReplicaState *dS = nullptr;
  std::vector<void *> fields;
  Plan plan_half, plan_full, plan_ideal, plan_charge, plan_hb, plan_pair;
  bool wide = false;    // some plane is >= 4 GiB: kernels use 64-bit offsets
  uint64_t buffer_bytes = 0;  // one buffer's fields, all replicas
  int nt_stores = -1;  // non-temporal stores: -1 by the rule, 0 / 1 forced
  bool phi_march = false;  // the phi half-sweep runs the z-march kernel
  bool phi_march_auto = false;  // the size rule's choice (LGV_PHI_AUTO)
  // pairs of phi sweeps run as out-of-place launches of both parities
  // (LGV_PHI_AUTO), in the kernel that the size rule chose
  bool phi_pairs = false;
  TwoParity two_parity = TwoParity::kNone;
  int brick_lds = 0;  // bytes of LDS of a launch in bricks
  MonSlot *mon_phi = nullptr, *mon_pair = nullptr, *mon_charge = nullptr, *mon_ideal = nullptr;
  // monitor counts folded out of the per-block slots when a retile
  // reallocated them: [replica][phi, charge]
  std::vector<std::array<lgv_monitor, 2>> mon_carry;
  EnergySlot *eslots = nullptr;
  // Counters and live-buffer flips of lone sweeps that are not in the replicas'
  // state: the launches that follow start from them, so that such a sweep needs
  // no launch of its own to advance the state (six phi sweeps of 32^3: 70.8 ->
  // 51.8 us).
  uint64_t ctr = 0;
  int flip = 0;
  double coef_hb = NAN, coef_charge = NAN, coef_ideal = NAN;
  double *d_aos = nullptr;
  int maxN = 0;
  double *d_part = nullptr;  // partial sums of a measurement (see MeasureShape)
  double *d_meas = nullptr;  // walls and phase walls of one measurement (MeasBuf)
  // the same and their transforms in pinned host memory, which the kernels
  // write themselves
  double *h_meas = nullptr;
  bool use_graph = false;
  int graph_steps = 1;                 // steps per captured graph
  hipGraphExec_t graph_exec = nullptr;  // graph_steps steps
  hipGraphExec_t graph_one = nullptr;   // one step (the remainder of a run)
  double graph_dt = NAN;
  // HIP-event timing of kernel classes on the context stream
  bool timing = false;      // HIP-event timing configured (lgv_timing_enable)
  bool timing_now = false;  // the launches being enqueued are timed
  int timing_every = 1;     // time every k-th step of lgv_step / lgv_run
  uint64_t timing_ctr = 0;
  std::vector<hipEvent_t> ev_pool;
  size_t ev_used = 0;
  struct TimedLaunch {
    int cls, count;  // the launch counts as `count` of its class
    hipEvent_t e0, e1;
  };
  std::vector<TimedLaunch> ev_pairs;
  double t_ms[LGV_NCLASS] = {0};
  long long t_launch[LGV_NCLASS] = {0};
};

namespace {

// z-planes per staging slab; LGV_STAGE_PLANES (a test hook) lowers it.
int slab_planes(int N) {
  int n = stage_planes(N);
  if (const char *e = getenv("LGV_STAGE_PLANES")) {
    const int v = atoi(e);
    if (v >= 1 && v < n) n = v;
  }
  return n;
}

// Layout of one measurement in a packed buffer for side N: walls [3][11][N],
// phase walls [3][14][N], their transforms [3][11][nk][2] and [3][14][nk][2]
// (the device buffer holds the walls only).
struct MeasBuf {
  double *wall, *wallphase, *wallk, *wallphasek;
  static int64_t walls(int N) { return 3 * 25 * (int64_t)N; }
  static int64_t size(int N) { return walls(N) + 3 * 25 * (int64_t)(N / 2 + 1) * 2; }
  MeasBuf(double *base, int N) {
    const int64_t nk = N / 2 + 1;
    wall = base;
    wallphase = wall + 3 * 11 * (int64_t)N;
    wallk = wallphase + 3 * 14 * (int64_t)N;
    wallphasek = wallk + 3 * 11 * nk * 2;
  }
};

// A launch's work on one replica: its blocks, numbered plane after plane of
// `plane` blocks each (0: in no such order).
struct PlanWork {
  int64_t blocks;
  double plane;
};

// The order of a launch's blocks.  The dispatcher deals workgroups round-robin
// over the eight XCDs, each with its own L2, so workgroup b runs on XCD b % 8:
// blocks that read each other's edges are put on one XCD, close in time.
//  * A replica of at most a sixteenth of the launch goes to one XCD as a whole
//    (the largest first, each to the XCD with the least work).
//  * A larger one is cut into eight bands of every plane, each XCD taking its
//    band of plane after plane (where a plane's blocks don't divide by eight,
//    the band edges move by an eighth of a block from plane to plane, so that
//    the XCDs' shares even out); with fewer than eight blocks per plane into
//    eight slabs of planes.
// XCDs that run out of blocks take over the last ones of the longest list.
// local: block within its replica.
void xcd_order(const std::vector<PlanWork> &work, std::vector<int> &rep, std::vector<int> &local) {
  int64_t total = 0;
  for (const PlanWork &w : work) total += w.blocks;
  std::vector<std::pair<int, int>> list[8];
  std::vector<int> by_size(work.size());
  for (size_t r = 0; r < work.size(); r++) by_size[r] = (int)r;
  std::stable_sort(by_size.begin(), by_size.end(),
                   [&](int a, int b) { return work[a].blocks > work[b].blocks; });
  for (int r : by_size) {
    const PlanWork &w = work[r];
    if (16 * w.blocks <= total) {
      auto *least = &list[0];
      for (auto &l : list)
        if (l.size() < least->size()) least = &l;
      for (int64_t j = 0; j < w.blocks; j++) least->push_back({r, (int)j});
      continue;
    }
    const double span = w.plane >= 8. ? w.plane : (double)w.blocks;
    for (int64_t j = 0; j < w.blocks; j++) {
      const int64_t z = (int64_t)((double)j / span);
      const double u = (double)j - (double)z * span + .125 * (double)(5 * z & 7);
      const int x = w.plane > 0. ? (int)(8. * u / span) : (int)(j & 7);
      list[std::min(std::max(x, 0), 7)].push_back({r, (int)j});
    }
  }
  size_t head[8] = {0}, tail[8];
  for (int x = 0; x < 8; x++) tail[x] = list[x].size();
  rep.resize(total);
  local.resize(total);
  for (int64_t b = 0; b < total; b++) {
    int x = (int)(b & 7);
    std::pair<int, int> e;
    if (head[x] < tail[x]) {
      e = list[x][head[x]++];
    } else {
      for (int k = 0; k < 8; k++)
        if (tail[k] - head[k] > tail[x] - head[x]) x = k;
      e = list[x][--tail[x]];
    }
    rep[b] = e.first;
    local[b] = e.second;
  }
}

int upload(int **dev, const std::vector<int> &v) {
  HIPCHECK(hipMalloc(dev, v.size() * sizeof(int)));
  HIPCHECK(hipMemcpy(*dev, v.data(), v.size() * sizeof(int), hipMemcpyHostToDevice));
  return LGV_OK;
}

// ordered: the blocks in xcd_order, otherwise replica after replica.
int build_plan(Plan &plan, const std::vector<PlanWork> &work, bool wide, bool ordered = true) {
  plan.wide = wide;
  plan.first.clear();
  std::vector<int> rep, local;
  int64_t total = 0;
  for (size_t r = 0; r < work.size(); r++) {
    plan.first.push_back((int)total);
    total += work[r].blocks;
    if (!ordered) rep.resize(total, (int)r);
  }
  plan.nblocks = (int)total;
  if (ordered) xcd_order(work, rep, local);
  int rc = upload(&plan.blocks.first, plan.first);
  if (!rc && work.size() > 1) rc = upload(&plan.blocks.rep, rep);
  if (!rc && ordered) rc = upload(&plan.blocks.local, local);
  return rc;
}

// Releases a plan's device arrays (the stream must be idle).
int free_plan(Plan &plan) {
  for (int *p : {plan.blocks.rep, plan.blocks.local, plan.blocks.first})
    if (p) HIPCHECK(hipFree(p));
  plan = Plan{};
  return LGV_OK;
}

// The ideal kernel's tiles where the caller asked for none.  Width:
// ideal_width.  Depth: a block marches TZ planes and rotates one more on
// either side, and the GPU holds `slots` blocks at a time.  A launch of up to
// two rounds takes whole rounds of TZ planes, a longer one its blocks' share
// and a tail; TZ of 16, 8, 4, and 64, 32, 2, 1 within one round, minimises that
// (256^3 FP64: TZ 64, 512 blocks, 532 us, 16 538; 320^3 has two rounds of 64,
// 1145, and takes 16, 1112.  FP64, TZ 16, 8, 4: 256^3
// 537, 546, 575 us; 240^3 558, 522, 523; 192^3 261, 245, 249; 144^3 140, 125,
// 123; 100^3 63, 42, 38; 64^3 TZ 1 17 us, TZ 16 60).
void resolve_ideal_tiles(lgv_ctx *c) {
  const int slots = ideal_slots(c->fp32);
  for (int r = 0; r < c->nrep; r++) {
    ReplicaParams &p = c->hp[r];
    p.tile_cap = c->tiles[r].ideal_cap ? c->tiles[r].ideal_cap : ideal_width(p.N, c->fp32);
  }
  int best = 64;
  double best_cost = 1e300;
  const double tail = c->fp32 ? .15 : .25;
  for (int tz = 64; tz >= 1; tz /= 2) {
    int64_t blocks = 0;
    for (const ReplicaParams &p : c->hp)
      blocks += ideal_plane_blocks(p.N, p.tile_cap) * ((p.N + tz - 1) / tz);
    const double rounds = (double)blocks / slots;
    if (tz < 4 && rounds > 1.) break;
    if (tz > 16 && rounds > 1.) continue;
    const double cost = (rounds <= 2. ? std::ceil(rounds) : rounds + tail) * (tz + .5);
    if (cost < best_cost) {
      best = tz;
      best_cost = cost;
    }
  }
  for (int r = 0; r < c->nrep; r++)
    c->hp[r].tile_tz = c->tiles[r].ideal_tz ? c->tiles[r].ideal_tz : best;
}

// Whether rows of NH half-columns and of tiles of TXH are whole units of bytes.
bool whole_rows(const lgv_ctx *c, int NH, int TXH, int bytes) {
  const int esz = c->fp32 ? 4 : 8;
  return NH * esz % bytes == 0 && TXH * esz % bytes == 0;
}

// Blocks of the fused ideal kernel: one per (x-tile, y-tile, z-chunk) of
// every replica, with that replica's tile shape.
int build_ideal_plan(lgv_ctx *c) {
  resolve_ideal_tiles(c);
  std::vector<PlanWork> work;
  bool stream = c->buffer_bytes > 2 * kCacheBytes, alternate = true;
  for (int r = 0; r < c->nrep; r++) {
    const ReplicaParams &p = c->hp[r];
    alternate = alternate && ideal_alternates(p.N, p.tile_cap, c->fp32);
    int TXH, TY, TZ;
    ideal_tile(p.N, p.tile_cap, p.tile_tz, TXH, TY, TZ);
    if ((TY + 2) * (2 * TXH + 2) > ideal_lds(c->fp32))
      return fail(LGV_ERR_ARG, "replica %d: ideal tile %dx%d exceeds the LDS plane", r, TXH, TY);
    stream = stream && whole_rows(c, p.NH, TXH, ideal_unit(p.N, c->fp32));
    const int64_t plane = (int64_t)((p.NH + TXH - 1) / TXH) * ((p.N + TY - 1) / TY);
    work.push_back({plane * ((p.N + TZ - 1) / TZ), (double)plane});
  }
  if (c->plan_ideal.nblocks) HIPCHECK(hipStreamSynchronize(c->stream));
  int rc = free_plan(c->plan_ideal);
  if (rc) return rc;
  rc = build_plan(c->plan_ideal, work, c->wide);
  c->plan_ideal.stream = c->nt_stores < 0 ? stream : c->nt_stores;
  c->plan_ideal.alternate = alternate;
  return rc;
}

// The phi march's tiles where the caller asked for none.  Width: an even split
// of the row into at most 64 half-columns (wide rows keep the x-halo columns a
// small share of the lines that a plane touches), rounded up to a multiple of
// 16 where the tile keeps as many rows, so that tiles begin on whole lines
// (FP64 224^3 56 wide 120 us, 64 wide 119 and with non-temporal stores 106;
// 272^3 46 wide 215, 48 wide 206 and 198).  Depth: TZ of 16, 8, 4 that minimises
// the planes moved, blocks times TZ and the chunk's extra loads, over the GPU's
// 1024 resident blocks, plus half a block's time for the launch's end (FP64 TZ
// 16, 8, 4: 256^3 147, 144, 150 us; 128^3 26.4, 23.7, 24.2; 100^3 24.8, 16.8,
// 15.5).
void resolve_hb_tiles(lgv_ctx *c) {
  for (int r = 0; r < c->nrep; r++) {
    ReplicaParams &p = c->hp[r];
    const int w = even_width(p.NH, 64), w16 = (w + 15) / 16 * 16;
    p.hb_cap = c->tiles[r].hb_cap ? c->tiles[r].hb_cap
               : w < p.NH && kBlock / w16 == kBlock / w ? w16 : w;
  }
  int best = 16;
  double best_cost = 1e300;
  for (int tz = 16; tz >= 4; tz /= 2) {
    int64_t blocks = 0;
    for (const ReplicaParams &p : c->hp) {
      int TXH, TY, TZ;
      hb_tile(p.N, p.hb_cap, tz, TXH, TY, TZ);
      blocks += (int64_t)((p.NH + TXH - 1) / TXH) * ((p.N + TY - 1) / TY) * ((p.N + tz - 1) / tz);
    }
    const double cost = (tz + (c->fp32 ? 2 : 1)) * ((double)blocks / (4 * kCUs) + .5);
    if (cost < best_cost * 0.98) {
      best = tz;
      best_cost = cost;
    }
  }
  for (int r = 0; r < c->nrep; r++)
    c->hp[r].hb_tz = c->tiles[r].hb_tz ? c->tiles[r].hb_tz : best;
}

// Blocks of the phi march kernel: (x-tile, y-tile, z-chunk) per replica.
int build_hb_plan(lgv_ctx *c) {
  resolve_hb_tiles(c);
  std::vector<PlanWork> work;
  bool wide = c->wide, stream = c->buffer_bytes / 10 * 4 > kCacheBytes;
  for (int r = 0; r < c->nrep; r++) {
    const ReplicaParams &p = c->hp[r];
    wide = wide || 2 * (uint64_t)p.half * (c->fp32 ? 4 : 8) > 0xFFFFFFFFull;
    int TXH, TY, TZ;
    hb_tile(p.N, p.hb_cap, p.hb_tz, TXH, TY, TZ);
    if ((TY + 2) * (TXH + 2) > kHbMarchGrid || 2 * TY + 2 * TXH > kBlock)
      return fail(LGV_ERR_ARG, "replica %d: phi tile %dx%d does not fit", r, TXH, TY);
    stream = stream && whole_rows(c, p.NH, TXH, 64);
    const int64_t plane = (int64_t)((p.NH + TXH - 1) / TXH) * ((p.N + TY - 1) / TY);
    work.push_back({plane * ((p.N + TZ - 1) / TZ), (double)plane});
  }
  int rc = free_plan(c->plan_hb);
  if (rc) return rc;
  rc = build_plan(c->plan_hb, work, wide);
  c->plan_hb.stream = c->nt_stores < 0 ? stream : c->nt_stores;
  return rc;
}

// Rows of even sites that k_hb_brick decides for a brick of BY x BZ rows.
int brick_rows(int N, int by, int bz) {
  const int y = std::min(by, N), z = std::min(bz, N);
  return y * z + 2 * y + 2 * z;
}

// The bricks of k_hb_brick: of the BY x BZ rows whose even sites fit kBrickLds,
// those with the fewest decisions per CU, in wavefronts and whole rounds of 256
// blocks (64^3 FP64: 4 x 4 rows, 256 blocks, 24 wavefronts against the 16 that
// have no facing rows).  False: no brick fits.
bool resolve_bricks(lgv_ctx *c) {
  const int esz = c->fp32 ? 4 : 8;
  int best_y = 0, best_z = 0;
  double best = 1e300;
  for (int by = 1; by <= 16; by++)
    for (int bz = 1; bz <= by; bz++) {
      double blocks = 0., waves = 0.;
      bool fits = true;
      for (const ReplicaParams &p : c->hp) {
        const int rows = brick_rows(p.N, by, bz);
        fits = fits && rows * p.NH * 4 * esz <= kBrickLds;
        const double n = (double)((p.N + by - 1) / by) * ((p.N + bz - 1) / bz);
        blocks += n;
        waves += n * ((rows * p.NH + 63) / 64 +
                      (std::min(by, p.N) * std::min(bz, p.N) * p.NH + 63) / 64);
      }
      const double cost = waves / blocks * std::ceil(blocks / kCUs);
      if (fits && cost < best) {
        best = cost;
        best_y = by;
        best_z = bz;
      }
    }
  for (ReplicaParams &p : c->hp) {
    p.pair_y = best_y;
    p.pair_z = best_z;
    c->brick_lds = std::max(c->brick_lds, brick_rows(p.N, best_y, best_z) * p.NH * 4 * esz);
  }
  return best_y != 0;
}

// The tiles of k_hb_sweep: as many rows as its threads hold (pair_march_rows),
// and the depth TZ that minimises whole rounds of one block per CU, each of TZ
// planes and about five planes' time for the two more that it decides, its start
// and its end (256^3 FP64, per half-sweep: TZ 52, one round of 215 blocks, 131
// us; 24, two, 133; 16, three, 142; 8 160).
// False: the rows are too long.
bool resolve_pair_march(lgv_ctx *c) {
  for (ReplicaParams &p : c->hp) {
    p.pair_y = pair_march_rows(p.N);
    if (!p.pair_y) return false;
  }
  int best = 0;
  double best_cost = 1e300;
  for (int tz = 2; tz <= 64; tz++) {
    int64_t blocks = 0;
    for (const ReplicaParams &p : c->hp)
      blocks += (int64_t)((p.N + p.pair_y - 1) / p.pair_y) * ((p.N + tz - 1) / tz);
    const double cost = std::ceil((double)blocks / kCUs) * (tz + 5.);
    if (cost < best_cost) {
      best = tz;
      best_cost = cost;
    }
  }
  for (ReplicaParams &p : c->hp) p.pair_z = best;
  return true;
}

// Blocks of the launches of both parities, which exist where 32-bit offsets reach
// a component's pair of half-planes (the march FP64 only); other contexts, which
// no size rule sends there, run half-sweeps.
int build_pair_plan(lgv_ctx *c) {
  bool reach = !(c->fp32 && c->two_parity == TwoParity::kMarch);
  for (const ReplicaParams &p : c->hp)
    reach = reach && 2 * (uint64_t)p.half * (c->fp32 ? 4 : 8) <= 0xFFFFFFFFull;
  if (!reach || (c->two_parity == TwoParity::kBricks && !resolve_bricks(c)) ||
      (c->two_parity == TwoParity::kMarch && !resolve_pair_march(c)))
    c->two_parity = TwoParity::kNone;
  if (c->two_parity == TwoParity::kNone) return LGV_OK;
  std::vector<PlanWork> work;
  bool stream = c->buffer_bytes > 2 * kCacheBytes;
  for (const ReplicaParams &p : c->hp) {
    stream = stream && whole_rows(c, p.NH, p.NH, 64);
    const int64_t plane = (p.N + p.pair_y - 1) / p.pair_y;
    work.push_back({plane * ((p.N + p.pair_z - 1) / p.pair_z), (double)plane});
  }
  const int rc = build_plan(c->plan_pair, work, false);
  c->plan_pair.stream = stream;
  return rc;
}

// Whether the x sub-sweeps of every replica run whole rows per wavefront
// (charge_row_wave with two half-columns per lane or one): NH = 64 or 128 and
// a tile of 64 half-columns x 4 lines.
bool charge_rows(const lgv_ctx *c) {
  bool rows = true;
  for (const ReplicaParams &p : c->hp) {
    int TXH, TQ, C;
    charge_tile(p.N, p.chg_cap, 2, TXH, TQ, C);
    rows = rows && (p.NH == 64 || p.NH == 128) && TXH == 64 && TQ == 4;
  }
  return rows;
}

// The charge march's tiles where the caller asked for none.  Width:
// charge_width.  Chunk: a chunk of C sites
// updates C/2 + 1 first-parity pairs for its C/2 second-parity ones, and the
// GPU holds `slots` blocks at a time, so a launch takes about ceil(blocks /
// slots) rounds of C/2 + 1.5 pairs; C of 16, 8, 4, 2 minimises that.  Measured
// for C = 16, 8, 4, 2, FP64: 256^3 327, 329, 334, 462 us; 200^3 225, 213, 210,
// 219; 160^3 114, 105, 106, 126; 128^3 49, 50, 50, 64; 100^3 36, 31, 29, 33;
// 64^3 31, 21, 17, 16; FP32: 256^3 226, 242, 274, 401; 128^3 39, 36, 39, 50;
// 32^3 29, 18, 13, 10.
void resolve_charge_tiles(lgv_ctx *c) {
  for (int r = 0; r < c->nrep; r++) {
    ReplicaParams &p = c->hp[r];
    p.chg_cap = c->tiles[r].chg_cap ? c->tiles[r].chg_cap : charge_width(p.NH, c->fp32);
  }
  const int slots = kCUs * (!c->fp32 && charge_rows(c) ? 3 : 4);
  int best = 16;
  double best_cost = 1e300;
  for (int chunk = 16; chunk >= 2; chunk /= 2) {
    int64_t blocks = 0;
    for (const ReplicaParams &p : c->hp) {
      int TXH, TQ, C;
      charge_tile(p.N, p.chg_cap, chunk, TXH, TQ, C);
      blocks += (int64_t)2 * ((p.NH + TXH - 1) / TXH) * ((p.N + TQ - 1) / TQ) *
                ((p.N + C - 1) / C);
    }
    const double cost = ((blocks + slots - 1) / slots) * (chunk / 2 + 1.5);
    if (cost < best_cost * 0.98) {
      best = chunk;
      best_cost = cost;
    }
  }
  for (int r = 0; r < c->nrep; r++)
    c->hp[r].chg_chunk = c->tiles[r].chg_chunk ? c->tiles[r].chg_chunk : best;
}

// Blocks of the charge march kernel: (x-tile, line tile, chunk) per replica.
int build_charge_plan(lgv_ctx *c) {
  resolve_charge_tiles(c);
  std::vector<PlanWork> work;
  for (int r = 0; r < c->nrep; r++) {
    const ReplicaParams &p = c->hp[r];
    int TXH, TQ, C;
    charge_tile(p.N, p.chg_cap, p.chg_chunk, TXH, TQ, C);
    if (C % 2 != 0) return fail(LGV_ERR_ARG, "replica %d: charge chunk %d is odd", r, C);
    // two blocks per tile: the even and the odd x of its half-columns
    work.push_back({(int64_t)2 * ((p.NH + TXH - 1) / TXH) * ((p.N + TQ - 1) / TQ) *
                        ((p.N + C - 1) / C),
                    0.});
  }
  int rc = free_plan(c->plan_charge);
  if (rc) return rc;
  rc = build_plan(c->plan_charge, work, c->wide);
  c->plan_charge.xwave = charge_rows(c);
  // the twelve half-planes of the charges in one buffer resource need 32-bit
  // offsets (any size below 448^3 in FP64, 564^3 in FP32)
  const uint64_t esz = c->fp32 ? sizeof(float) : sizeof(double);
  c->plan_charge.far = c->wide;
  for (const ReplicaParams &p : c->hp)
    c->plan_charge.far = c->plan_charge.far || 12 * (uint64_t)p.half * esz > 0xFFFFFFFFull;
  return rc;
}

// Step coefficients with the reference's expressions:
//   EulerLangevinHB  rdtg = sqrt(2.*dt*gamma)          Stepper.cxx:301
//   ModelGChargeHB   rdtsigma = sqrt(2.*dt*sigma())    Stepper.cxx:456
//   IdealPV2         rotatePhi(dt/2.0)                 Stepper.cxx:73,169
bool same(double a, double b) { return a == b || (std::isnan(a) && std::isnan(b)); }

int ensure_coeffs(lgv_ctx *c, double dt_hb, double dt_charge, double dt_ideal) {
  if (same(dt_hb, c->coef_hb) && same(dt_charge, c->coef_charge) &&
      same(dt_ideal, c->coef_ideal))
    return LGV_OK;
  for (int r = 0; r < c->nrep; r++) {
    const lgv_model_params &m = c->mp[r];
    ReplicaParams &p = c->hp[r];
    p.rdtg = std::sqrt(2. * dt_hb * m.gamma);
    p.rms = std::sqrt(2. * dt_charge * (m.diffusion * m.chi));
    p.dt_ideal = dt_ideal;
    p.tau_ideal = dt_ideal / 2.0;
  }
  HIPCHECK(hipStreamSynchronize(c->stream));
  HIPCHECK(hipMemcpy(c->dP, c->hp.data(), c->nrep * sizeof(ReplicaParams),
                     hipMemcpyHostToDevice));
  c->coef_hb = dt_hb;
  c->coef_charge = dt_charge;
  c->coef_ideal = dt_ideal;
  return LGV_OK;
}

// Brackets one kernel (class cls) with events when timing is on.
struct Timed {
  lgv_ctx *c;
  int cls;
  hipEvent_t e1 = nullptr;
  Timed(lgv_ctx *cc, int k, int count = 1) : c(cc), cls(k) {
    if (!c->timing_now) return;
    if (c->ev_used + 2 > c->ev_pool.size()) {
      for (int i = 0; i < 64; i++) {
        hipEvent_t e;
        if (hipEventCreate(&e) != hipSuccess) { c->timing = c->timing_now = false; return; }
        c->ev_pool.push_back(e);
      }
    }
    hipEvent_t e0 = c->ev_pool[c->ev_used++];
    if (hipEventRecord(e0, c->stream) != hipSuccess) {  // timing is best effort
      c->timing = c->timing_now = false;
      return;
    }
    e1 = c->ev_pool[c->ev_used++];
    c->ev_pairs.push_back({cls, count, e0, e1});
  }
  ~Timed() {
    if (!e1) return;
    if (hipEventRecord(e1, c->stream) != hipSuccess) {
      c->timing = c->timing_now = false;
      c->ev_pairs.pop_back();  // the pair this object pushed: never resolved
    }
  }
};

// Resolves recorded event pairs into the per-class totals.
int drain_timing(lgv_ctx *c) {
  if (c->ev_pairs.empty()) return LGV_OK;
  HIPCHECK(hipStreamSynchronize(c->stream));
  for (auto &pr : c->ev_pairs) {
    float ms = 0.f;
    HIPCHECK(hipEventElapsedTime(&ms, pr.e0, pr.e1));
    c->t_ms[pr.cls] += ms;
    c->t_launch[pr.cls] += pr.count;
  }
  c->ev_pairs.clear();
  c->ev_used = 0;
  return LGV_OK;
}

// The launches of a step read the live buffers of the replica state XOR
// `flip` (bit 0 phi, bit 1 charges), the flips of the step's earlier
// launches; k_advance applies the step's net flip at its end, so no launch of
// a step writes the state's buffer bits.  Each enqueue_* returns the flips
// of its own launches.
int enqueue_ideal(lgv_ctx *c, int off, int flip) {
  if (c->timing_now && c->ev_used + 16 > 4096) drain_timing(c);
  if (c->track_energy) {
    Timed tm(c, LGV_CLASS_ENERGY);
    launch_energy(c->fp32, c->plan_full, c->dP, c->dS, flip, c->eslots, c->stream);
    launch_energy_finish(c->nrep, c->plan_full, c->dP, c->dS, c->eslots, 0, off,
                         c->mon_ideal, c->stream);
  }
  {
    Timed tm(c, LGV_CLASS_IDEAL);
    launch_ideal(c->fp32, c->plan_ideal, c->dP, c->dS, flip, c->stream);
  }
  if (c->track_energy) {
    Timed tm(c, LGV_CLASS_ENERGY);
    launch_energy(c->fp32, c->plan_full, c->dP, c->dS, flip ^ 3, c->eslots, c->stream);
    launch_energy_finish(c->nrep, c->plan_full, c->dP, c->dS, c->eslots, 1, off,
                         c->mon_ideal, c->stream);
  }
  return 3;  // out of place: phi and charges
}

// EulerLangevinHB::step (counters off, off+1 for the two parities), one
// in-place launch per parity: the z-march with the other parity's plane in
// LDS or the one-thread-per-site kernel, by the size rule (the march from
// phi_march_sites on) unless lgv_set_phi_kernel chose.  Per half-sweep, site
// against march, FP64: 64^3 8.9, 9.5 us; 100^3 16.8, 15.5; 160^3 42, 44; 192^3
// 67, 66; 224^3 147, 109; 256^3 221, 147; FP32: 160^3 33, 33; 224^3 79, 70;
// 256^3 116, 86.
bool use_march(const lgv_ctx *c) { return c->phi_march; }
const Plan &hb_plan(const lgv_ctx *c) { return use_march(c) ? c->plan_hb : c->plan_half; }
int enqueue_hb(lgv_ctx *c, int off, int flip, hipStream_t st) {
  for (int ieo = 0; ieo < 2; ieo++) {
    Timed tm(c, LGV_CLASS_PHI);
    if (use_march(c))
      launch_hb_march(c->fp32, c->plan_hb, c->dP, c->dS, ieo, off + ieo, flip, c->mon_phi, st);
    else
      launch_hb_phi(c->fp32, c->plan_half, c->dP, c->dS, ieo, off + ieo, flip, c->mon_phi, st);
  }
  return 0;  // in place
}

// n sweeps of EulerLangevinHB::step: pairs of out-of-place two-parity launches
// where the context has them (a pair leaves the live buffer where it was, as
// the in-place sweeps do), the others in place.
void enqueue_phi_sweeps(lgv_ctx *c, int n, int off, int flip, hipStream_t st) {
  int i = 0;
  if (c->phi_pairs) {
    for (; i < n - n % 2; i++) {
      Timed tm(c, LGV_CLASS_PHI, 2);  // two half-sweeps
      if (c->two_parity == TwoParity::kMarch)
        launch_hb_sweep(c->plan_pair, c->dP, c->dS, off + 2 * i, flip ^ (i & 1),
                        c->mon_pair, st);
      else
        launch_hb_brick(c->fp32, c->plan_pair, c->brick_lds, c->dP, c->dS, off + 2 * i,
                        flip ^ (i & 1), c->mon_pair, st);
    }
  }
  for (; i < n; i++) enqueue_hb(c, off + 2 * i, flip, st);
}

// ModelGChargeHB::step: the shuffle (counter off, drawn by every charge
// launch), then per direction both parities in one pass (counters
// off+1+2*ixyz and off+2+2*ixyz, as the unfused order), each launch writing
// the other charge buffer.
int enqueue_charge(lgv_ctx *c, int off, int flip, hipStream_t st) {
  for (int ixyz = 0; ixyz < 3; ixyz++) {
    Timed tm(c, LGV_CLASS_CHARGE);
    launch_charge_march(c->fp32, c->plan_charge, c->dP, c->dS, ixyz, off + 1 + 2 * ixyz,
                        flip ^ (ixyz & 1 ? 2 : 0), c->mon_charge, st);
  }
  return 2;  // three flips of the charge buffers
}

// The counter and the flips held on the host, for a launch sequence whose
// k_advance adds them to the replicas' state.
int take_state(lgv_ctx *c, int &flip) {
  const int n = (int)c->ctr;
  flip = c->flip;
  c->ctr = 0;
  c->flip = 0;
  return n;
}
// Adds them by a launch of their own: before a graph, whose offsets start at
// 0, and before launches that read the live buffers by the state alone.
void settle(lgv_ctx *c) {
  int flip;
  const int n = take_state(c, flip);
  if (n) launch_advance(c->nrep, c->dS, 0., 0, (uint64_t)n, flip, c->stream);
}

// PV2HBSplit::step (Stepper.cxx:542-580); returns the number of stream
// counters consumed, and those taken from the host's count.  The charge sweep
// reads and writes only the charges and the phi sweeps only phi, so after the
// last ideal substep the two run side by side on the context's two streams
// (fork and join by events, which a graph capture records as well).  Every
// sweep keeps its counter (random streams) and its monitor slots, so the
// result is the sequential one bit for bit.  Contexts of one large lattice
// (kOverlapBytes) keep the sequential order (their launches fill the GPU on
// their own), and so do timed steps (events on one stream).  On the
// stream the charge sweep, the longer of the two, follows the ideal launch
// without an event's wait and the phi sweeps take the second stream (steps
// with the charge sweep on the second stream -> on the first: 16^3 100 -> 92
// us, 64^3 155 -> 144, 100^3 334 -> 341 but three contexts at once 310 -> 309,
// 128^3 655 -> 637, 192^3 1896 -> 1874); in a graph the phi sweeps follow it
// and the charge sweep branches off (64^3 145 -> 138, 128^3 646 -> 626).  flip
// returns the step's net live-buffer flip.
int enqueue_step(lgv_ctx *c, int &flip, bool capture = false) {
  int off = take_state(c, flip);
  c->timing_now = c->timing && c->timing_ctr++ % c->timing_every == 0;
  // a timed step keeps one stream (events on it bracket every launch)
  const bool overlap = c->overlap && !c->timing_now && !c->onlydiffuse && !c->nodiffuse;
  bool forked = false, join_event = false;
  hipStream_t phi = c->stream, charge = c->stream;
  if (overlap) (capture ? charge : phi) = c->stream2;
  if (!c->onlydiffuse) {
    for (unsigned i1 = 0; i1 < c->s1; i1++) {
      flip ^= enqueue_ideal(c, off, flip);
      off += 1;
      forked = overlap && i1 + 1 == c->s1 && hipEventRecord(c->ev_fork, c->stream) == hipSuccess &&
               hipStreamWaitEvent(c->stream2, c->ev_fork, 0) == hipSuccess;
      // the phi sweeps that follow do not touch the charge bit of flip
      if (forked) flip ^= enqueue_charge(c, off + 2 * (int)c->s0, flip, charge);
      enqueue_phi_sweeps(c, (int)c->s0, off, flip, forked ? phi : c->stream);
      off += 2 * (int)c->s0;
      if (forked) join_event = hipEventRecord(c->ev_join, c->stream2) == hipSuccess;
    }
  }
  if (!c->nodiffuse) {
    if (!forked) flip ^= enqueue_charge(c, off, flip, c->stream);
    off += 7;
  }
  if (forked && (!join_event || hipStreamWaitEvent(c->stream, c->ev_join, 0) != hipSuccess))
    (void)hipStreamSynchronize(c->stream2);  // join on the host instead
  return off;
}

// computeDerivedObs's OAverage (measurer.cxx:288-300): mean of wallX rows
void volume_averages(const double *wall, int N, double *oavg) {
  for (int l = 0; l < 11; l++) {
    double s = 0.;
    for (int i = 0; i < N; i++) s += wall[l * N + i];
    oavg[l] = s / (double)N;
  }
}

// Complex numbers of rotate_to_vev.  Products as std::complex forms them, whose
// operator* also calls out of line to test every product for NaN (32 products
// per k: 90 us of a 256^3 measurement); the test is made here, and a NaN goes
// the library's way.
struct Cplx {
  double re, im;
};
inline Cplx operator*(const Cplx &a, const Cplx &b) {
  const Cplx p{a.re * b.re - a.im * b.im, a.re * b.im + a.im * b.re};
  if (__builtin_expect(p.re != p.re && p.im != p.im, 0)) {
    const std::complex<double> q =
        std::complex<double>(a.re, a.im) * std::complex<double>(b.re, b.im);
    return {q.real(), q.imag()};
  }
  return p;
}
inline Cplx operator+(const Cplx &a, const Cplx &b) { return {a.re + b.re, a.im + b.im}; }
inline Cplx operator-(const Cplx &a, const Cplx &b) { return {a.re - b.re, a.im - b.im}; }
inline Cplx operator-(const Cplx &a) { return {-a.re, -a.im}; }

// rotate_to_vev (measurer.cxx:231-286): rotates the k-space walls into the
// frame of the k = 0 phi direction.  wk[11][nk][2] -> rot[14][nk][2].
void rotate_to_vev(int nk, const double *wk, double *rot) {
  auto W = [&](int a, int k) { return Cplx{wk[(a * nk + k) * 2], wk[(a * nk + k) * 2 + 1]}; };
  auto contract = [](const Cplx *n, const Cplx *rho, Cplx *out) {
    out[0] = -(n[1] * rho[0]) - n[2] * rho[1] - n[3] * rho[2];
    out[1] = n[0] * rho[0] + n[3] * rho[4] - n[2] * rho[5];
    out[2] = n[0] * rho[1] - n[3] * rho[3] + n[1] * rho[5];
    out[3] = n[0] * rho[2] + n[2] * rho[3] - n[1] * rho[4];
  };
  Cplx n[4];
  double norm = 0.;
  for (int a = 0; a < 4; a++) {
    n[a] = W(a, 0);
    norm += n[a].re * n[a].re + n[a].im * n[a].im;
  }
  norm = std::sqrt(norm);
  if (norm < std::numeric_limits<double>::min()) {
    n[0] = {1, 0};
    n[1] = n[2] = n[3] = {0, 0};
  } else {
    for (int a = 0; a < 4; a++) n[a] = {n[a].re / norm, n[a].im / norm};
  }
  for (int k = 0; k < nk; k++) {
    Cplx phi[4], rho[6], drho[6], A[4], V[4];
    for (int a = 0; a < 4; a++) phi[a] = W(a, k);
    for (int ab = 0; ab < 6; ab++) rho[ab] = W(4 + ab, k);
    for (int l = 0; l < 3; l++) { drho[l] = rho[l + 3]; drho[l + 3] = rho[l]; }
    Cplx phis{0, 0};
    for (int a = 0; a < 4; a++) phis = phis + n[a] * phi[a];
    contract(n, rho, A);
    contract(n, drho, V);
    auto put = [&](int a, const Cplx &v) {
      rot[(a * nk + k) * 2] = v.re;
      rot[(a * nk + k) * 2 + 1] = v.im;
    };
    put(0, phis);
    for (int a = 0; a < 4; a++) {
      put(1 + a, phi[a] - n[a] * phis);
      put(5 + a, A[a]);
      put(9 + a, V[a]);
    }
    put(13, W(10, k));
  }
}

int check_launch() {
  HIPCHECK(hipGetLastError());
  return LGV_OK;
}

int check_replica(lgv_ctx *c, int r) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (r < 0 || r >= c->nrep) return fail(LGV_ERR_RANGE, "replica %d out of range [0,%d)", r, c->nrep);
  return LGV_OK;
}

}  // namespace

extern "C" {

const char *lgv_last_error(void) { return g_err.c_str(); }
int lgv_version(void) { return 1; }

int lgv_create(const lgv_config *cfg, lgv_ctx **out) {
  if (!cfg || !out) return fail(LGV_ERR_ARG, "null argument");
  *out = nullptr;
  if (cfg->nreplicas <= 0 || !cfg->replicas) return fail(LGV_ERR_ARG, "no replicas");
  if (cfg->precision != LGV_FP64 && cfg->precision != LGV_FP32)
    return fail(LGV_ERR_ARG, "precision must be LGV_FP64 or LGV_FP32");
  const unsigned s0 = cfg->scounts[0] ? cfg->scounts[0] : 2;
  const unsigned s1 = cfg->scounts[1] ? cfg->scounts[1] : 3;
  if (s0 > 64 || s1 > 64) return fail(LGV_ERR_ARG, "scounts too large");
  for (int r = 0; r < cfg->nreplicas; r++) {
    const lgv_model_params &m = cfg->replicas[r];
    if (m.NX < 4 || (m.NX & 1) || m.NX > kMaxN)
      return fail(LGV_ERR_ARG, "replica %d: NX=%d must be even and in [4, %d]", r, m.NX, kMaxN);
    if (!(m.chi > 0)) return fail(LGV_ERR_ARG, "replica %d: chi must be positive", r);
  }
  // on any failure below, everything allocated so far is released (the
  // error message of the failure is kept)
  auto cleanup = [](lgv_ctx *p) {
    const std::string msg = g_err;
    lgv_destroy(p);
    g_err = msg;
  };
  std::unique_ptr<lgv_ctx, decltype(cleanup)> c(new lgv_ctx, cleanup);
  c->device = cfg->device;
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamCreateWithFlags(&c->stream, hipStreamNonBlocking));
  HIPCHECK(hipStreamCreateWithFlags(&c->stream2, hipStreamNonBlocking));
  HIPCHECK(hipEventCreateWithFlags(&c->ev_fork, hipEventDisableTiming));
  HIPCHECK(hipEventCreateWithFlags(&c->ev_join, hipEventDisableTiming));
  c->fp32 = cfg->precision == LGV_FP32;
  c->s0 = s0;
  c->s1 = s1;
  c->nodiffuse = cfg->nodiffuse != 0;
  c->onlydiffuse = cfg->onlydiffuse != 0;
  c->track_energy = cfg->track_energy != 0;
  c->nrep = cfg->nreplicas;
  c->mp.assign(cfg->replicas, cfg->replicas + cfg->nreplicas);
  c->hp.resize(c->nrep);
  c->tiles.resize(c->nrep);
  c->noise.resize(c->nrep);
  const size_t esz = c->fp32 ? sizeof(float) : sizeof(double);
  std::vector<PlanWork> whalf, wfull;
  uint64_t buffer_bytes = 0;
  int minN = kMaxN;  // one buffer: 10 planes x 2 parities
  std::vector<ReplicaState> hs(c->nrep);
  for (int r = 0; r < c->nrep; r++) {
    const lgv_model_params &m = c->mp[r];
    const int N = m.NX;
    const int64_t half = (int64_t)N * N * N / 2;
    ReplicaParams &p = c->hp[r];
    memset(&p, 0, sizeof p);
    for (int b = 0; b < 2; b++) {
      void *field = nullptr;
      HIPCHECK(hipMalloc(&field, 20 * half * esz));
      HIPCHECK(hipMemset(field, 0, 20 * half * esz));
      c->fields.push_back(field);
      p.fields[b] = field;
    }
    p.N = N;
    p.NH = N / 2;
    p.half = half;
    p.mass0 = m.mass0;
    p.dmassdt = m.dmassdt;
    p.lambda = m.lambda;
    p.H = m.H;
    p.chi = m.chi;
    p.chg_l2 = charge_l2(m.chi);
    const double hx = (double)(m.LX > 0 ? m.LX : N) / N;
    p.axx = std::pow(1. / hx, 2);
    const uint32_t s32 = rank0_seed(m.seed);
    p.base_key = base_key(s32);
    c->noise[r].g = xoro_seeded((uint64_t)s32);
    hs[r] = ReplicaState{};
    hs[r].t = m.initialtime;
    whalf.push_back({(half + kBlock - 1) / kBlock, (double)N * p.NH / kBlock});
    wfull.push_back({(2 * half + kBlock - 1) / kBlock, 0.});
    if ((uint64_t)half * esz > 0xFFFFFFFFull) c->wide = true;
    buffer_bytes += (uint64_t)20 * half * esz;
    // test hook: LGV_FORCE_WIDE=1 runs the 64-bit-offset kernels on any size
    if (const char *fw = getenv("LGV_FORCE_WIDE")) c->wide = c->wide || atoi(fw) != 0;
    c->maxN = std::max(c->maxN, N);
    minN = std::min(minN, N);
  }
  c->buffer_bytes = buffer_bytes;
  c->phi_march_auto = buffer_bytes / (10 * esz) >= phi_march_sites(c->fp32, cfg->nreplicas);
  // test hook: LGV_NT_STORES=0/1 forces the store mode on any size, and with
  // FP64 fields the phi kernel that goes with it (1: the march)
  if (const char *nt = getenv("LGV_NT_STORES")) {
    c->nt_stores = atoi(nt) != 0;
    if (!c->fp32) c->phi_march_auto = c->nt_stores;
  }
  c->phi_march = c->phi_march_auto;
  // test hook: LGV_PHI_KERNEL=site/march forces the phi half-sweep kernel
  if (const char *pk = getenv("LGV_PHI_KERNEL")) {
    const std::string k(pk);
    if (k != "site" && k != "march")
      return fail(LGV_ERR_ARG, "LGV_PHI_KERNEL=%s: expected site or march", pk);
    c->phi_march = k == "march";
  }
  const uint64_t sites = buffer_bytes / (10 * esz);
  if (sites < kBrickSites) c->two_parity = TwoParity::kBricks;
  if (!c->fp32 && sites >= kPairMarchSites && minN >= kPairMarchSide)
    c->two_parity = TwoParity::kMarch;
  // test hook: LGV_PHI_PAIRS=0/1/2 takes no launches of both parities, bricks,
  // the march
  if (const char *pb = getenv("LGV_PHI_PAIRS"))
    c->two_parity = (TwoParity)std::min(std::max(atoi(pb), 0), 2);
  // one lattice whose launches each fill the GPU many times over gains
  // nothing from running the charge sweep beside the phi sweeps; smaller and
  // batched lattices do (kOverlapBytes)
  c->overlap = !(cfg->nreplicas == 1 &&
                 buffer_bytes > (c->two_parity == TwoParity::kMarch ? kOverlapBytesPairMarch
                                                                    : kOverlapBytes));
  // test hook: LGV_OVERLAP=0/1 forces the sequential / concurrent order
  if (const char *ov = getenv("LGV_OVERLAP")) c->overlap = atoi(ov) != 0;
  HIPCHECK(hipMalloc(&c->dS, c->nrep * sizeof(ReplicaState)));
  HIPCHECK(hipMemcpy(c->dS, hs.data(), c->nrep * sizeof(ReplicaState), hipMemcpyHostToDevice));
  int rc;
  if ((rc = build_plan(c->plan_half, whalf, c->wide)) != LGV_OK) return rc;
  if ((rc = build_plan(c->plan_full, wfull, c->wide, false)) != LGV_OK) return rc;
  if ((rc = build_ideal_plan(c.get())) != LGV_OK) return rc;
  if ((rc = build_charge_plan(c.get())) != LGV_OK) return rc;
  if ((rc = build_hb_plan(c.get())) != LGV_OK) return rc;
  if ((rc = build_pair_plan(c.get())) != LGV_OK) return rc;
  // the hooks that force a half-sweep kernel or its stores leave out the others
  c->phi_pairs =
      c->two_parity != TwoParity::kNone && !getenv("LGV_PHI_KERNEL") && c->nt_stores < 0;
  // the parameters as the plans' tile rules left them
  HIPCHECK(hipMalloc(&c->dP, c->nrep * sizeof(ReplicaParams)));
  HIPCHECK(hipMemcpy(c->dP, c->hp.data(), c->nrep * sizeof(ReplicaParams),
                     hipMemcpyHostToDevice));
  HIPCHECK(hipMalloc(&c->mon_phi, hb_plan(c.get()).nblocks * sizeof(MonSlot)));
  HIPCHECK(hipMemset(c->mon_phi, 0, hb_plan(c.get()).nblocks * sizeof(MonSlot)));
  if (c->two_parity != TwoParity::kNone) {
    HIPCHECK(hipMalloc(&c->mon_pair, c->plan_pair.nblocks * sizeof(MonSlot)));
    HIPCHECK(hipMemset(c->mon_pair, 0, c->plan_pair.nblocks * sizeof(MonSlot)));
  }
  HIPCHECK(hipMalloc(&c->mon_charge, c->plan_charge.nblocks * sizeof(MonSlot)));
  HIPCHECK(hipMemset(c->mon_charge, 0, c->plan_charge.nblocks * sizeof(MonSlot)));
  HIPCHECK(hipMalloc(&c->mon_ideal, c->nrep * sizeof(MonSlot)));
  HIPCHECK(hipMemset(c->mon_ideal, 0, c->nrep * sizeof(MonSlot)));
  c->mon_carry.assign(c->nrep, {lgv_monitor{}, lgv_monitor{}});
  HIPCHECK(hipMalloc(&c->eslots, c->plan_full.nblocks * sizeof(EnergySlot)));
  HIPCHECK(hipMalloc(&c->d_aos, (int64_t)stage_planes(c->maxN) * c->maxN * c->maxN * 10 *
                                     sizeof(double)));
  int64_t part = 0;
  for (const ReplicaParams &p : c->hp)
    part = std::max(part, measure_part(measure_shape(p.N), p.N));
  HIPCHECK(hipMalloc(&c->d_part, part * sizeof(double)));
  HIPCHECK(hipMalloc(&c->d_meas, MeasBuf::walls(c->maxN) * sizeof(double)));
  HIPCHECK(hipHostMalloc(&c->h_meas, MeasBuf::size(c->maxN) * sizeof(double), 0));
  HIPCHECK(hipDeviceSynchronize());
  *out = c.release();
  return LGV_OK;
}

int lgv_destroy(lgv_ctx *c) {
  if (!c) return LGV_OK;
  // releases everything even after a failure and reports the first one
  hipError_t first = hipSuccess;
  auto note = [&](hipError_t e) {
    if (first == hipSuccess && e != hipSuccess) first = e;
  };
  note(hipSetDevice(c->device));
  if (c->stream) note(hipStreamSynchronize(c->stream));
  if (c->stream2) note(hipStreamSynchronize(c->stream2));
  if (c->graph_exec) note(hipGraphExecDestroy(c->graph_exec));
  if (c->graph_one) note(hipGraphExecDestroy(c->graph_one));
  for (hipEvent_t e : c->ev_pool) note(hipEventDestroy(e));
  for (void *f : c->fields) note(hipFree(f));
  note(hipFree(c->dP));
  note(hipFree(c->dS));
  for (Plan *pl : {&c->plan_half, &c->plan_full, &c->plan_ideal, &c->plan_charge, &c->plan_hb,
                   &c->plan_pair}) {
    for (int *q : {pl->blocks.rep, pl->blocks.local, pl->blocks.first}) note(hipFree(q));
  }
  for (void *q : {(void *)c->mon_phi, (void *)c->mon_pair, (void *)c->mon_charge, (void *)c->mon_ideal,
                  (void *)c->eslots, (void *)c->d_aos, (void *)c->d_part,
                  (void *)c->d_meas})
    note(hipFree(q));
  if (c->h_meas) note(hipHostFree(c->h_meas));
  if (c->ev_fork) note(hipEventDestroy(c->ev_fork));
  if (c->ev_join) note(hipEventDestroy(c->ev_join));
  if (c->stream2) note(hipStreamDestroy(c->stream2));
  if (c->stream) note(hipStreamDestroy(c->stream));
  delete c;
  if (first != hipSuccess)
    return fail(LGV_ERR_HIP, "lgv_destroy: %s", hipGetErrorString(first));
  return LGV_OK;
}

int lgv_set_field(lgv_ctx *c, int r, const double *aos) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  if (!aos) return fail(LGV_ERR_ARG, "null field");
  HIPCHECK(hipSetDevice(c->device));
  const int N = c->hp[r].N;
  const int64_t P = (int64_t)N * N * 10;  // doubles per z-plane
  const int slab = slab_planes(N);
  settle(c);
  HIPCHECK(hipStreamSynchronize(c->stream));
  for (int z0 = 0; z0 < N; z0 += slab) {
    const int nz = std::min(slab, N - z0);
    HIPCHECK(hipMemcpy(c->d_aos, aos + z0 * P, nz * P * sizeof(double), hipMemcpyHostToDevice));
    launch_aos_to_rb(c->fp32, c->dP, c->dS, r, N, z0, nz, c->d_aos, c->stream);
    if ((rc = check_launch())) return rc;
    HIPCHECK(hipStreamSynchronize(c->stream));
  }
  return LGV_OK;
}

int lgv_get_field(lgv_ctx *c, int r, double *aos) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  if (!aos) return fail(LGV_ERR_ARG, "null field");
  HIPCHECK(hipSetDevice(c->device));
  const int N = c->hp[r].N;
  const int64_t P = (int64_t)N * N * 10;  // doubles per z-plane
  const int slab = slab_planes(N);
  settle(c);
  for (int z0 = 0; z0 < N; z0 += slab) {
    const int nz = std::min(slab, N - z0);
    launch_rb_to_aos(c->fp32, c->dP, c->dS, r, N, z0, nz, c->d_aos, c->stream);
    if ((rc = check_launch())) return rc;
    HIPCHECK(hipStreamSynchronize(c->stream));
    HIPCHECK(hipMemcpy(aos + z0 * P, c->d_aos, nz * P * sizeof(double), hipMemcpyDeviceToHost));
  }
  return LGV_OK;
}

int lgv_set_time(lgv_ctx *c, int r, double t) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (r >= c->nrep) return fail(LGV_ERR_RANGE, "replica out of range");
  HIPCHECK(hipSetDevice(c->device));
  launch_set_time(c->nrep, r, c->dS, t, c->stream);
  return check_launch();
}

int lgv_get_time(lgv_ctx *c, int r, double *t) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  HIPCHECK(hipSetDevice(c->device));
  ReplicaState s;
  HIPCHECK(hipStreamSynchronize(c->stream));
  HIPCHECK(hipMemcpy(&s, c->dS + r, sizeof s, hipMemcpyDeviceToHost));
  *t = s.t;
  return LGV_OK;
}

int lgv_step(lgv_ctx *c, double dt) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  HIPCHECK(hipSetDevice(c->device));
  int rc = ensure_coeffs(c, dt / (c->s0 * c->s1), dt, dt / (c->s1));
  if (rc) return rc;
  int flip;
  const int n = enqueue_step(c, flip);
  launch_advance(c->nrep, c->dS, dt, 0, (uint64_t)n, flip, c->stream);
  return check_launch();
}

// Releases the captured step graphs (they capture plans, tiles and dt).
static int drop_graphs(lgv_ctx *c) {
  for (hipGraphExec_t *g : {&c->graph_exec, &c->graph_one}) {
    if (*g) HIPCHECK(hipGraphExecDestroy(*g));
    *g = nullptr;
  }
  return LGV_OK;
}

// The per-block monitor slots follow the plans: before a replanning,
// fold_monitors adds them into the per-replica carry; realloc_monitors
// then allocates zeroed slots for the plans in use.
static int fold_monitors(lgv_ctx *c) {
  lgv_monitor m[3];
  for (int i = 0; i < c->nrep; i++) {
    int rc = lgv_monitor_get(c, i, m);
    if (rc) return rc;
    c->mon_carry[i] = {m[0], m[1]};
  }
  return LGV_OK;
}
static int realloc_monitors(lgv_ctx *c) {
  HIPCHECK(hipFree(c->mon_phi));
  HIPCHECK(hipFree(c->mon_charge));
  c->mon_phi = c->mon_charge = nullptr;
  HIPCHECK(hipMalloc(&c->mon_phi, hb_plan(c).nblocks * sizeof(MonSlot)));
  HIPCHECK(hipMemset(c->mon_phi, 0, hb_plan(c).nblocks * sizeof(MonSlot)));
  HIPCHECK(hipMalloc(&c->mon_charge, c->plan_charge.nblocks * sizeof(MonSlot)));
  HIPCHECK(hipMemset(c->mon_charge, 0, c->plan_charge.nblocks * sizeof(MonSlot)));
  if (c->mon_pair) HIPCHECK(hipMemset(c->mon_pair, 0, c->plan_pair.nblocks * sizeof(MonSlot)));
  return LGV_OK;
}

int lgv_use_graph(lgv_ctx *c, int enable) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (enable < 0 || enable > 1024) return fail(LGV_ERR_ARG, "graph steps %d out of range", enable);
  HIPCHECK(hipSetDevice(c->device));
  c->use_graph = enable != 0;
  if (enable > 0 && enable != c->graph_steps) {
    int rc = drop_graphs(c);
    if (rc) return rc;
    c->graph_steps = enable;
  }
  return LGV_OK;
}

int lgv_run(lgv_ctx *c, double dt, int nsteps) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (nsteps < 0) return fail(LGV_ERR_ARG, "nsteps < 0");
  HIPCHECK(hipSetDevice(c->device));
  int rc = ensure_coeffs(c, dt / (c->s0 * c->s1), dt, dt / (c->s1));
  if (rc) return rc;
  if (!c->use_graph || c->timing) {
    for (int i = 0; i < nsteps; i++) {
      int flip;
      const int n = enqueue_step(c, flip);
      launch_advance(c->nrep, c->dS, dt, 1, (uint64_t)n, flip, c->stream);
    }
    return check_launch();
  }
  settle(c);
  if (!c->graph_exec || c->graph_dt != dt) {
    if ((rc = drop_graphs(c))) return rc;
    // graph_steps steps in one graph, and (when that is more than one) one
    // step for the remainder of a run
    for (int g = 0; g < (c->graph_steps > 1 ? 2 : 1); g++) {
      const int k = g == 0 ? c->graph_steps : 1;
      hipGraph_t graph;
      HIPCHECK(hipStreamBeginCapture(c->stream, hipStreamCaptureModeThreadLocal));
      for (int i = 0; i < k; i++) {
        int flip;
        const int n = enqueue_step(c, flip, true);
        launch_advance(c->nrep, c->dS, dt, 1, (uint64_t)n, flip, c->stream);
      }
      HIPCHECK(hipStreamEndCapture(c->stream, &graph));
      // the captured graph is released whether or not it instantiates
      const hipError_t ei = hipGraphInstantiate(g == 0 ? &c->graph_exec : &c->graph_one,
                                                graph, nullptr, nullptr, 0);
      HIPCHECK(hipGraphDestroy(graph));
      if (ei != hipSuccess) {
        (g == 0 ? c->graph_exec : c->graph_one) = nullptr;
        drop_graphs(c);
        return fail(LGV_ERR_HIP, "hipGraphInstantiate: %s", hipGetErrorString(ei));
      }
    }
    c->graph_dt = dt;
  }
  const int K = c->graph_steps;
  for (int i = 0; i < nsteps / K; i++) HIPCHECK(hipGraphLaunch(c->graph_exec, c->stream));
  for (int i = 0; i < nsteps % K; i++) HIPCHECK(hipGraphLaunch(c->graph_one, c->stream));
  return check_launch();
}

int lgv_ideal_step(lgv_ctx *c, double dt) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  HIPCHECK(hipSetDevice(c->device));
  int rc = ensure_coeffs(c, c->coef_hb, c->coef_charge, dt);
  if (rc) return rc;
  c->timing_now = c->timing;  // single sweeps are always timed
  if (c->ctr >> 20) settle(c);
  c->flip ^= enqueue_ideal(c, (int)c->ctr, c->flip);
  c->ctr += 1;
  return check_launch();
}

int lgv_hb_phi_step(lgv_ctx *c, double dt) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  HIPCHECK(hipSetDevice(c->device));
  int rc = ensure_coeffs(c, dt, c->coef_charge, c->coef_ideal);
  if (rc) return rc;
  c->timing_now = c->timing;  // single sweeps are always timed
  if (c->ctr >> 20) settle(c);
  c->flip ^= enqueue_hb(c, (int)c->ctr, c->flip, c->stream);
  c->ctr += 2;
  return check_launch();
}

int lgv_charge_step(lgv_ctx *c, double dt) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  HIPCHECK(hipSetDevice(c->device));
  int rc = ensure_coeffs(c, c->coef_hb, dt, c->coef_ideal);
  if (rc) return rc;
  c->timing_now = c->timing;  // single sweeps are always timed
  if (c->ctr >> 20) settle(c);
  c->flip ^= enqueue_charge(c, (int)c->ctr, c->flip, c->stream);
  c->ctr += 7;
  return check_launch();
}

int lgv_init_gaussian_charges(lgv_ctx *c, int r) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  const int N = c->hp[r].N;
  const size_t V = (size_t)N * N * N;
  std::vector<double> u(V * 10);
  if ((rc = lgv_get_field(c, r, u.data()))) return rc;
  double sum[10] = {0};
  const double chi = c->mp[r].chi;
  HostNoise &ng = c->noise[r];
  for (size_t s = 0; s < V; s++)
    for (int L = 4; L < 10; L++) {
      u[s * 10 + L] = std::sqrt(chi) * ng.normal();
      sum[L] += u[s * 10 + L];
    }
  const double vol = (double)N * N * N;
  for (size_t s = 0; s < V; s++)
    for (int L = 4; L < 10; L++) u[s * 10 + L] -= sum[L] / vol;
  return lgv_set_field(c, r, u.data());
}

int lgv_thermalize(lgv_ctx *c, double dt, int nsteps) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  int rc;
  for (int r = 0; r < c->nrep; r++)
    if ((rc = lgv_init_gaussian_charges(c, r))) return rc;
  for (int i = 0; i < nsteps; i++) {
    const int substeps = 6;
    for (int j = 0; j < substeps; j++)
      if ((rc = lgv_hb_phi_step(c, dt / substeps))) return rc;
  }
  return LGV_OK;
}

int lgv_monitor_get(lgv_ctx *c, int r, lgv_monitor out[3]) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamSynchronize(c->stream));
  // phi half-sweeps, charge sweeps, two-parity phi sweeps
  MonSlot *src[3] = {c->mon_phi, c->mon_charge, c->mon_pair};
  const Plan *plan[3] = {&hb_plan(c), &c->plan_charge, &c->plan_pair};
  for (int k = 0; k < 2; k++) out[k] = c->mon_carry[r][k];
  for (int k = 0; k < 3; k++) {
    if (!src[k]) continue;
    const int b0 = plan[k]->first[r];
    const int b1 = r + 1 < c->nrep ? plan[k]->first[r + 1] : plan[k]->nblocks;
    std::vector<MonSlot> slots(b1 - b0);
    HIPCHECK(hipMemcpy(slots.data(), src[k] + b0, slots.size() * sizeof(MonSlot),
                       hipMemcpyDeviceToHost));
    lgv_monitor &m = out[k % 2];
    for (const MonSlot &s : slots) {
      m.down_counts += s.down_counts;
      m.up_counts += s.up_counts;
      m.up_yes += s.up_yes;
      m.up_no += s.up_no;
      m.down_dS += s.down_dS;
      m.up_dS += s.up_dS;
    }
  }
  MonSlot mi;
  HIPCHECK(hipMemcpy(&mi, c->mon_ideal + r, sizeof mi, hipMemcpyDeviceToHost));
  out[2] = lgv_monitor{mi.down_counts, mi.up_counts, mi.up_yes, mi.up_no, mi.down_dS, mi.up_dS};
  return LGV_OK;
}

int lgv_energy_get(lgv_ctx *c, int r, double out[2]) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamSynchronize(c->stream));
  ReplicaState s;
  HIPCHECK(hipMemcpy(&s, c->dS + r, sizeof s, hipMemcpyDeviceToHost));
  out[0] = s.E_old;
  out[1] = s.E_new;
  return LGV_OK;
}

int lgv_rng_get_state(lgv_ctx *c, int r, lgv_rng_state *st) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamSynchronize(c->stream));
  ReplicaState s;
  HIPCHECK(hipMemcpy(&s, c->dS + r, sizeof s, hipMemcpyDeviceToHost));
  st->s0 = c->noise[r].g.s0;
  st->s1 = c->noise[r].g.s1;
  st->saved_normal = c->noise[r].saved;
  st->has_saved_normal = c->noise[r].has_saved;
  st->sweep_ctr = s.sweep_ctr + c->ctr;
  return LGV_OK;
}

int lgv_rng_set_state(lgv_ctx *c, int r, const lgv_rng_state *st) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamSynchronize(c->stream));
  c->noise[r].g.s0 = st->s0;
  c->noise[r].g.s1 = st->s1;
  c->noise[r].saved = st->saved_normal;
  c->noise[r].has_saved = st->has_saved_normal;
  ReplicaState s;
  HIPCHECK(hipMemcpy(&s, c->dS + r, sizeof s, hipMemcpyDeviceToHost));
  s.sweep_ctr = st->sweep_ctr - c->ctr;
  HIPCHECK(hipMemcpy(c->dS + r, &s, sizeof s, hipMemcpyHostToDevice));
  return LGV_OK;
}

int lgv_measure(lgv_ctx *c, int r, double *wall, double *wallphase, double *oavg) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  if (!wall || !wallphase || !oavg) return fail(LGV_ERR_ARG, "null output");
  HIPCHECK(hipSetDevice(c->device));
  const int N = c->hp[r].N;
  const MeasBuf mb(c->d_meas, N), h(c->h_meas, N);
  settle(c);
  launch_measure(c->fp32, c->dP, c->dS, r, N, c->d_part, mb.wall, mb.wallphase, h.wall,
                 h.wallphase, c->stream);
  if ((rc = check_launch())) return rc;
  HIPCHECK(hipStreamSynchronize(c->stream));
  memcpy(wall, h.wall, 3 * 11 * N * sizeof(double));
  memcpy(wallphase, h.wallphase, 3 * 14 * N * sizeof(double));
  volume_averages(h.wall, N, oavg);
  return LGV_OK;
}

int lgv_timing_enable(lgv_ctx *c, int enable) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (enable < 0) return fail(LGV_ERR_ARG, "timing_enable %d < 0", enable);
  HIPCHECK(hipSetDevice(c->device));
  int rc = drain_timing(c);
  if (rc) return rc;
  c->timing = enable != 0;
  c->timing_now = c->timing;
  c->timing_every = enable > 1 ? enable : 1;
  c->timing_ctr = 0;
  for (int k = 0; k < LGV_NCLASS; k++) {
    c->t_ms[k] = 0.;
    c->t_launch[k] = 0;
  }
  return LGV_OK;
}

int lgv_timing_get(lgv_ctx *c, double ms[LGV_NCLASS], long long launches[LGV_NCLASS]) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  HIPCHECK(hipSetDevice(c->device));
  int rc = drain_timing(c);
  if (rc) return rc;
  for (int k = 0; k < LGV_NCLASS; k++) {
    ms[k] = c->t_ms[k];
    launches[k] = c->t_launch[k];
  }
  return LGV_OK;
}

int lgv_measure_full(lgv_ctx *c, int r, lgv_measurement *m) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  if (!m) return fail(LGV_ERR_ARG, "null measurement");
  HIPCHECK(hipSetDevice(c->device));
  const int N = c->hp[r].N, nk = N / 2 + 1;
  const MeasBuf mb(c->d_meas, N), h(c->h_meas, N);
  settle(c);
  launch_measure(c->fp32, c->dP, c->dS, r, N, c->d_part, mb.wall, mb.wallphase, h.wall,
                 h.wallphase, c->stream);
  launch_wall_dft(N, mb.wall, mb.wallphase, h.wallk, h.wallphasek, c->stream);
  if ((rc = check_launch())) return rc;
  HIPCHECK(hipStreamSynchronize(c->stream));
  if (m->wall) memcpy(m->wall, h.wall, 3 * 11 * (size_t)N * sizeof(double));
  if (m->wallphase) memcpy(m->wallphase, h.wallphase, 3 * 14 * (size_t)N * sizeof(double));
  if (m->oavg) volume_averages(h.wall, N, m->oavg);
  if (m->wall_k) memcpy(m->wall_k, h.wallk, 3 * 11 * (size_t)nk * 2 * sizeof(double));
  if (m->wallphase_k)
    memcpy(m->wallphase_k, h.wallphasek, 3 * 14 * (size_t)nk * 2 * sizeof(double));
  if (m->wall_k_rotated)
    for (int d = 0; d < 3; d++)
      rotate_to_vev(nk, h.wallk + (size_t)d * 11 * nk * 2,
                    m->wall_k_rotated + (size_t)d * 14 * nk * 2);
  return LGV_OK;
}

int lgv_set_mass(lgv_ctx *c, int r, double mass0, double dmassdt) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (r >= c->nrep) return fail(LGV_ERR_RANGE, "replica out of range");
  HIPCHECK(hipSetDevice(c->device));
  for (int i = 0; i < c->nrep; i++) {
    if (r >= 0 && i != r) continue;
    c->mp[i].mass0 = c->hp[i].mass0 = mass0;
    c->mp[i].dmassdt = c->hp[i].dmassdt = dmassdt;
  }
  HIPCHECK(hipStreamSynchronize(c->stream));
  HIPCHECK(hipMemcpy(c->dP, c->hp.data(), c->nrep * sizeof(ReplicaParams),
                     hipMemcpyHostToDevice));
  if (int rg = drop_graphs(c)) return rg;
  return LGV_OK;
}

int lgv_set_ideal_tile(lgv_ctx *c, int r, int txh_cap, int tz) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (r >= c->nrep) return fail(LGV_ERR_RANGE, "replica out of range");
  if (txh_cap < 2 || txh_cap > 64 || tz < 1 || tz > 1024)
    return fail(LGV_ERR_ARG, "tile cap %d / tz %d out of range", txh_cap, tz);
  HIPCHECK(hipSetDevice(c->device));
  const std::vector<TileRequest> old = c->tiles;
  for (int i = 0; i < c->nrep; i++) {
    if (r >= 0 && i != r) continue;
    c->tiles[i].ideal_cap = txh_cap;
    c->tiles[i].ideal_tz = tz;
  }
  int rc = build_ideal_plan(c);
  if (rc) {
    c->tiles = old;
    build_ideal_plan(c);
    return rc;
  }
  HIPCHECK(hipStreamSynchronize(c->stream));
  HIPCHECK(hipMemcpy(c->dP, c->hp.data(), c->nrep * sizeof(ReplicaParams),
                     hipMemcpyHostToDevice));
  if (int rg = drop_graphs(c)) return rg;
  return LGV_OK;
}

int lgv_get_ideal_tile(lgv_ctx *c, int r, int *txh_cap, int *tz) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  if (!txh_cap || !tz) return fail(LGV_ERR_ARG, "null argument");
  *txh_cap = c->hp[r].tile_cap;
  *tz = c->hp[r].tile_tz;
  return LGV_OK;
}

int lgv_set_sweep_tiles(lgv_ctx *c, int r, int hb_cap, int hb_tz, int chg_cap,
                        int chg_chunk) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (r >= c->nrep) return fail(LGV_ERR_RANGE, "replica out of range");
  auto bad = [](int v, int lo, int hi) { return v != 0 && (v < lo || v > hi); };
  if (bad(hb_cap, 4, 64) || bad(hb_tz, 1, 1024) || bad(chg_cap, 4, 64) ||
      bad(chg_chunk, 2, 1024) || chg_chunk % 2 != 0)
    return fail(LGV_ERR_ARG, "sweep tile %d/%d, %d/%d out of range", hb_cap, hb_tz, chg_cap,
                chg_chunk);
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamSynchronize(c->stream));
  if (int rm = fold_monitors(c)) return rm;
  const std::vector<TileRequest> old = c->tiles;
  for (int i = 0; i < c->nrep; i++) {
    if (r >= 0 && i != r) continue;
    c->tiles[i].hb_cap = hb_cap;
    c->tiles[i].hb_tz = hb_tz;
    c->tiles[i].chg_cap = chg_cap;
    c->tiles[i].chg_chunk = chg_chunk;
  }
  int rc = build_hb_plan(c);
  if (!rc) rc = build_charge_plan(c);
  if (rc) {
    c->tiles = old;
    build_hb_plan(c);
    build_charge_plan(c);
  }
  if (int rm = realloc_monitors(c)) return rm;
  HIPCHECK(hipMemcpy(c->dP, c->hp.data(), c->nrep * sizeof(ReplicaParams),
                     hipMemcpyHostToDevice));
  HIPCHECK(hipDeviceSynchronize());
  if (int rg = drop_graphs(c)) return rg;
  return rc;
}

int lgv_set_phi_kernel(lgv_ctx *c, int kernel) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  if (kernel != LGV_PHI_AUTO && kernel != LGV_PHI_SITE && kernel != LGV_PHI_MARCH)
    return fail(LGV_ERR_ARG, "phi kernel %d: expected LGV_PHI_AUTO, _SITE or _MARCH", kernel);
  const bool march = kernel == LGV_PHI_AUTO ? c->phi_march_auto : kernel == LGV_PHI_MARCH;
  const bool pairs = kernel == LGV_PHI_AUTO && c->two_parity != TwoParity::kNone;
  if (march == c->phi_march && pairs == c->phi_pairs) return LGV_OK;
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamSynchronize(c->stream));
  if (int rm = fold_monitors(c)) return rm;
  c->phi_march = march;
  c->phi_pairs = pairs;
  if (int rm = realloc_monitors(c)) return rm;
  HIPCHECK(hipDeviceSynchronize());
  return drop_graphs(c);
}

int lgv_get_phi_kernel(lgv_ctx *c, int *kernel) {
  if (!c || !kernel) return fail(LGV_ERR_ARG, "null argument");
  *kernel = c->phi_march ? LGV_PHI_MARCH : LGV_PHI_SITE;
  return LGV_OK;
}

int lgv_get_phi_pairs(lgv_ctx *c, int *kernel) {
  if (!c || !kernel) return fail(LGV_ERR_ARG, "null argument");
  *kernel = c->phi_pairs ? (int)c->two_parity : 0;
  return LGV_OK;
}

int lgv_monitor_reset(lgv_ctx *c) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamSynchronize(c->stream));
  HIPCHECK(hipMemset(c->mon_phi, 0, hb_plan(c).nblocks * sizeof(MonSlot)));
  HIPCHECK(hipMemset(c->mon_charge, 0, c->plan_charge.nblocks * sizeof(MonSlot)));
  if (c->mon_pair) HIPCHECK(hipMemset(c->mon_pair, 0, c->plan_pair.nblocks * sizeof(MonSlot)));
  HIPCHECK(hipMemset(c->mon_ideal, 0, c->nrep * sizeof(MonSlot)));
  HIPCHECK(hipDeviceSynchronize());
  for (auto &cr : c->mon_carry) cr = {lgv_monitor{}, lgv_monitor{}};
  return LGV_OK;
}

int lgv_synchronize(lgv_ctx *c) {
  if (!c) return fail(LGV_ERR_ARG, "null context");
  HIPCHECK(hipSetDevice(c->device));
  HIPCHECK(hipStreamSynchronize(c->stream));
  return LGV_OK;
}

int lgv_field_device_ptr(lgv_ctx *c, int r, void **ptr, int *elem_bytes) {
  int rc = check_replica(c, r);
  if (rc) return rc;
  *ptr = c->hp[r].fields[0];
  *elem_bytes = c->fp32 ? 4 : 8;
  return LGV_OK;
}

}  // extern "C"
