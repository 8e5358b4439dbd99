// lgv_kernels.hip -- HIP kernels of the ModelG time step for gfx950.
//
// Blocks are mapped to replicas through a launch plan, so one launch steps
// many independent lattices.  Fields live in the red-black
// structure-of-arrays layout of lgv_device.h, double-buffered: the phi
// half-sweeps update the live buffer in place (a checkerboard never reads what
// it writes); the phi launches of both parities, the charge launches and the
// fused ideal substep write the other buffer.
// All FP arithmetic is FP64 (FP32 storage is widened on load and rounded
// on store).  The Metropolis sweeps follow the reference's expression order
// bit for bit; the library is built with -ffp-contract=off.
#include <float.h>

#include "lgv_device.h"
#include "lgv_internal.h"

namespace lgv {

// `cur` packs the live buffer of the phi planes (bit 0) and of the charge
// planes (bit 1).  A select instead of p.fields[b]: a runtime index into the
// register copy of ReplicaParams would push the whole struct to scratch.
template <typename T>
__device__ __forceinline__ T *plane(const ReplicaParams &p, int cur, int c, int par) {
  const int b = c < 4 ? (cur & 1) : (cur >> 1);
  T *base = reinterpret_cast<T *>(b ? p.fields[1] : p.fields[0]);
  return base + ((int64_t)(c * 2 + par)) * p.half;
}
__device__ __forceinline__ int live(const ReplicaState &s) {
  return s.cur_phi | (s.cur_chg << 1);
}

// Lane 0's value of v, uniform over the wave (v_readfirstlane per word).  Also
// for values that are the same in every lane but were computed in vector
// registers: the compiler would treat whatever follows from them (plane bases,
// branches) as differing between lanes.
__device__ __forceinline__ int first_lane(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ uint64_t first_lane(uint64_t v) {
  const uint32_t lo = __builtin_amdgcn_readfirstlane((uint32_t)v);
  const uint32_t hi = __builtin_amdgcn_readfirstlane((uint32_t)(v >> 32));
  return ((uint64_t)hi << 32) | lo;
}
__device__ __forceinline__ float first_lane(float v) {
  return __uint_as_float(__builtin_amdgcn_readfirstlane(__float_as_uint(v)));
}
__device__ __forceinline__ double first_lane(double v) {
  return __longlong_as_double((long long)first_lane((uint64_t)__double_as_longlong(v)));
}

// Global-memory view of one plane for the sweep kernels.  The base is
// uniform over a block (it sits in SGPRs) and, with W == false, the element
// offset is a 32-bit byte offset, so every access is one global load/store
// in the saddr + 32-bit voffset form with no 64-bit address arithmetic.
// W == true (a plane of 4 GiB or more) widens the offset to 64 bits.
typedef __attribute__((address_space(1))) char gbyte;
template <typename T, bool W>
struct GPlane {
  gbyte *b;
  __device__ __forceinline__ static auto off(uint32_t i) {
    if constexpr (W) return (uint64_t)i * sizeof(T);
    else return (uint32_t)(i * (uint32_t)sizeof(T));
  }
  __device__ __forceinline__ T raw(uint32_t i) const {
    return *reinterpret_cast<const __attribute__((address_space(1))) T *>(b + off(i));
  }
  __device__ __forceinline__ double ld(uint32_t i) const { return (double)raw(i); }
  __device__ __forceinline__ void st(uint32_t i, double v) const {
    *reinterpret_cast<__attribute__((address_space(1))) T *>(b + off(i)) = (T)v;
  }
  // NTS: a non-temporal load, for a value no other thread reads
  template <bool NTS>
  __device__ __forceinline__ T get_raw(uint32_t i) const {
    if constexpr (NTS)
      return __builtin_nontemporal_load(
          reinterpret_cast<const __attribute__((address_space(1))) T *>(b + off(i)));
    else
      return raw(i);
  }
  template <bool NTS>
  __device__ __forceinline__ double get(uint32_t i) const { return (double)get_raw<NTS>(i); }
  // NTS: a non-temporal store (not kept in the caches)
  template <bool NTS>
  __device__ __forceinline__ void put_raw(uint32_t i, T v) const {
    if constexpr (NTS)
      __builtin_nontemporal_store(
          v, reinterpret_cast<__attribute__((address_space(1))) T *>(b + off(i)));
    else
      *reinterpret_cast<__attribute__((address_space(1))) T *>(b + off(i)) = v;
  }
  template <bool NTS>
  __device__ __forceinline__ void put(uint32_t i, double v) const {
    put_raw<NTS>(i, (T)v);
  }
};
template <typename T, bool W>
__device__ __forceinline__ GPlane<T, W> gplane(const ReplicaParams &p, int cur, int c, int par) {
  const int buf = c < 4 ? (cur & 1) : (cur >> 1);
  char *base = reinterpret_cast<char *>(buf ? p.fields[1] : p.fields[0]);
  return {(gbyte *)(base + (int64_t)(c * 2 + par) * p.half * (int64_t)sizeof(T))};
}
// The two field buffers of a replica read once into registers: a kernel
// that stores between its loads then forms every plane base from these
// values, where gplane(p, ...) would reload p.fields after each store (the
// compiler cannot prove that a field store misses the parameter block).
struct FieldBufs {
  char *f0, *f1;
  int64_t half_bytes;  // one half-plane
};
template <typename T>
__device__ __forceinline__ FieldBufs field_bufs(const ReplicaParams &p) {
  return {reinterpret_cast<char *>(p.fields[0]), reinterpret_cast<char *>(p.fields[1]),
          p.half * (int64_t)sizeof(T)};
}
template <typename T, bool W>
__device__ __forceinline__ GPlane<T, W> gplane(const FieldBufs &fb, int cur, int c, int par) {
  const int buf = c < 4 ? (cur & 1) : (cur >> 1);
  return {(gbyte *)((buf ? fb.f1 : fb.f0) + (int64_t)(c * 2 + par) * fb.half_bytes)};
}

// The charge planes of a replica: reads from the live buffer, writes to the
// other one.  W == false: the twelve half-planes of a buffer span less than 4
// GiB and are one buffer resource, so an access is one buffer instruction with
// the site's 32-bit byte offset in a vector register and the plane's offset
// in a scalar one: no address arithmetic per access and no scalar pair per
// plane (24 plane bases do not fit the scalar registers of the sweep).
// W == true: 64-bit addresses.
template <typename T, bool W>
struct ChargePlanes {
  FieldBufs fb;
  int cur;
  __device__ __forceinline__ ChargePlanes(const ReplicaParams &p, int cur_)
      : fb(field_bufs<T>(p)), cur(cur_) {}
  // component c of the six, parity par
  __device__ __forceinline__ T ld(int c, int par, uint32_t i) const {
    return gplane<T, true>(fb, cur, 4 + c, par).raw(i);
  }
  __device__ __forceinline__ void st(int c, int par, uint32_t i, T v) const {
    gplane<T, true>(fb, cur ^ 2, 4 + c, par).template put_raw<false>(i, v);
  }
};
template <typename T>
struct ChargePlanes<T, false> {
  __amdgpu_buffer_rsrc_t in, out;
  uint32_t half_bytes;
  __device__ __forceinline__ ChargePlanes(const ReplicaParams &p, int cur) {
    const FieldBufs fb = field_bufs<T>(p);
    half_bytes = first_lane((int)fb.half_bytes);
    auto resource = [&](char *f) __attribute__((always_inline)) {
      char *b = reinterpret_cast<char *>(
          first_lane((uint64_t)reinterpret_cast<uintptr_t>(f + 8 * fb.half_bytes)));
      // raw 32-bit format: reads past the twelve half-planes return zero
      return __builtin_amdgcn_make_buffer_rsrc(b, 0, (int)(12u * half_bytes), 0x00027000);
    };
    in = resource(cur >> 1 ? fb.f1 : fb.f0);
    out = resource(cur >> 1 ? fb.f0 : fb.f1);
  }
  __device__ __forceinline__ T ld(int c, int par, uint32_t i) const {
    const uint32_t s = (uint32_t)(c * 2 + par) * half_bytes;
    if constexpr (sizeof(T) == 4)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(in, i * 4u, s, 0));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(in, i * 8u, s, 0));
  }
  __device__ __forceinline__ void st(int c, int par, uint32_t i, T v) const {
    const uint32_t s = (uint32_t)(c * 2 + par) * half_bytes;
    typedef uint32_t b64 __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(T) == 4)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), out, i * 4u, s, 0);
    else
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(b64, v), out, i * 8u, s, 0);
  }
};

// The phi planes of a replica's live buffer for a march in z: an access names
// a component, a parity, a plane z and the lane's offset within the plane.
// W == false: one buffer resource per component (its two half-planes, less
// than 4 GiB); the plane's offset is scalar and the lane's stays in one vector
// register for the whole march.  That leaves no vector address arithmetic, and
// no address temporary that would first have to wait for a pending load into
// its register (measured in the FP32 march, where such waits for the loads of
// the plane after next come and go with the register allocation).
// W == true: a 64-bit base per component, parity and plane, and the lane's 32-bit
// offset within the plane (1024^3 FP32, two half-sweeps: 11.8 ms, 16.3 with the
// lane's index in the whole half-plane).
// NT: a value no other thread reads, not kept in the caches.
template <typename T, bool W>
struct PhiPlanes {
  gbyte *b;
  int64_t half_bytes;
  uint32_t plane_bytes;
  __device__ __forceinline__ PhiPlanes(const ReplicaParams &p, int cur) {
    const FieldBufs fb = field_bufs<T>(p);
    half_bytes = (int64_t)first_lane((uint64_t)fb.half_bytes);
    plane_bytes = (uint32_t)p.N * p.NH * (uint32_t)sizeof(T);
    b = (gbyte *)reinterpret_cast<char *>(
        first_lane((uint64_t)reinterpret_cast<uintptr_t>(cur & 1 ? fb.f1 : fb.f0)));
  }
  __device__ __forceinline__ GPlane<T, false> at(int l, int par, int z) const {
    return {b + (2 * l + par) * half_bytes + (int64_t)z * plane_bytes};
  }
  template <bool NT>
  __device__ __forceinline__ T ld(int l, int par, int z, uint32_t i) const {
    return at(l, par, z).template get_raw<NT>(i);
  }
  template <bool NT>
  __device__ __forceinline__ void st(int l, int par, int z, uint32_t i, T v) const {
    at(l, par, z).template put_raw<NT>(i, v);
  }
};
template <typename T>
struct PhiPlanes<T, false> {
  // no access (a load gives zero): past the end of the buffer resource, where the
  // hardware neither reads nor writes
  static constexpr uint32_t kNone = 0xFFFFFFFFu / sizeof(T);
  __amdgpu_buffer_rsrc_t f[4];
  uint32_t half_bytes, plane_bytes;
  __device__ __forceinline__ PhiPlanes(const ReplicaParams &p, int cur) {
    const FieldBufs fb = field_bufs<T>(p);
    half_bytes = first_lane((int)fb.half_bytes);
    plane_bytes = (uint32_t)p.N * p.NH * (uint32_t)sizeof(T);
    char *b = cur & 1 ? fb.f1 : fb.f0;
#pragma unroll
    for (int l = 0; l < 4; l++)
      f[l] = __builtin_amdgcn_make_buffer_rsrc(
          reinterpret_cast<char *>(
              first_lane((uint64_t)reinterpret_cast<uintptr_t>(b + 2 * l * fb.half_bytes))),
          0, (int)(2u * half_bytes), 0x00027000);
  }
  template <bool NT>
  __device__ __forceinline__ T ld(int l, int par, int z, uint32_t i) const {
    const uint32_t s = (uint32_t)z * plane_bytes + (par ? half_bytes : 0u);
    if constexpr (sizeof(T) == 4)
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(f[l], i * 4u, s, NT ? 2 : 0));
    else
      return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(f[l], i * 8u, s, NT ? 2 : 0));
  }
  template <bool NT>
  __device__ __forceinline__ void st(int l, int par, int z, uint32_t i, T v) const {
    const uint32_t s = (uint32_t)z * plane_bytes + (par ? half_bytes : 0u);
    typedef uint32_t b64 __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(T) == 4)
      __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(uint32_t, v), f[l], i * 4u, s,
                                            NT ? 2 : 0);
    else
      __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(b64, v), f[l], i * 8u, s,
                                            NT ? 2 : 0);
  }
};

// Replica r and block b of it that this workgroup is; returns the block's
// number in the launch (its monitor slot).  A launch of one replica reads
// nothing before the replica's parameters: a chain of loads at the start of a
// launch costs about 0.7 us a link.
__device__ __forceinline__ int block_of(const LaunchBlocks &blk, int &r, int &b) {
  r = blk.rep ? blk.rep[blockIdx.x] : 0;
  const int first = blk.rep ? blk.first[r] : 0;
  b = blk.local ? blk.local[blockIdx.x] : (int)blockIdx.x - first;
  return first + b;
}

__device__ __forceinline__ int wrapp(int a, int N) { return a == N ? 0 : a; }
__device__ __forceinline__ int wrapm(int a, int N) { return a < 0 ? N - 1 : a; }

// The lanes of the wavefront that hold a predicate, and back.  (The builtin,
// not __ballot, which rebuilds the mask with a select and a compare.)
__device__ __forceinline__ uint64_t lanes(bool pred) {
  return __builtin_amdgcn_ballot_w64(pred);
}
__device__ __forceinline__ bool in_lanes(uint64_t mask) {
  return __builtin_amdgcn_inverse_ballot_w64(mask);
}

// A thread's share of the monitor (o4_stepper_monitor).  The counts are those
// of the whole wavefront, popcounts of lane masks in scalar registers, so all
// active lanes carry the same values; the sums of dS are the lane's own.
struct Tally {
  uint32_t all = 0, down = 0, yes = 0;  // decisions, dS < 0, accepted dS >= 0
  double dSd = 0., dSu = 0.;
};
// n decisions of every lane that holds count
__device__ __forceinline__ void tally_all(Tally &m, int n, bool count) {
  m.all += n * __builtin_popcountll(lanes(count));
}
// One decision of the lanes in count: those in down had dS < 0, those in up
// were accepted with dS >= 0.
__device__ __forceinline__ void tally(Tally &m, double dS, uint64_t down, uint64_t up,
                                      uint64_t count) {
  uint32_t nd = __builtin_popcountll(down & count), ny = __builtin_popcountll(up & count);
  // one masked add each; written in plain C++ they become an add and two
  // selects
  if (in_lanes(down & count)) __asm__ volatile("v_add_f64 %0, %0, %1" : "+v"(m.dSd) : "v"(dS));
  if (in_lanes(up & count)) __asm__ volatile("v_add_f64 %0, %0, %1" : "+v"(m.dSu) : "v"(dS));
  // counted and summed here and now: otherwise the compiler keeps the masks
  // and dS of a dozen decisions (in spilled registers) for later
  __asm__ volatile("" : "+s"(nd), "+s"(ny));
  m.down += nd;
  m.yes += ny;
}

// Deterministic block reduction of the tallies; thread 0 adds the block
// total into the block's own slot (stream order makes this race-free).  The
// sums of dS are scaled by unit.
template <int B = kBlock>
__device__ void block_monitor_add(MonSlot *slot, const Tally &m, double unit = 1.) {
  __shared__ uint32_t sc[3][B / 64];
  __shared__ double sd[2][B / 64];
  double dSd = m.dSd, dSu = m.dSu;
  uint32_t c[3] = {m.all, m.down, m.yes};
  for (int o = 32; o > 0; o >>= 1) {
    dSd += __shfl_xor(dSd, o, 64);
    dSu += __shfl_xor(dSu, o, 64);
    // lanes without sites hold zeros, the others the wave's counts
    for (int i = 0; i < 3; i++) c[i] |= __shfl_xor(c[i], o, 64);
  }
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) {
    for (int i = 0; i < 3; i++) sc[i][w] = c[i];
    sd[0][w] = dSd; sd[1][w] = dSu;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    long long n[3] = {0, 0, 0};
    double d = 0, e = 0;
    for (int i = 0; i < B / 64; i++) {
      for (int k = 0; k < 3; k++) n[k] += sc[k][i];
      d += sd[0][i]; e += sd[1][i];
    }
    slot->down_counts += n[1];
    slot->up_counts += n[0] - n[1];
    slot->up_yes += n[2];
    slot->up_no += n[0] - n[1] - n[2];
    slot->down_dS += d * unit;
    slot->up_dS += e * unit;
  }
}

// ------------------------------------------------------------------------
// The Metropolis test canonical(u) < exp(x) for the draw u and x = -dS <= 0,
// decided as the double test decides it: the lanes that accept.  e is exp(x)
// in single precision: the callers round x log2(e) by at most three half-ulps
// (4.2e-6 of exp(x) for x > -23) and v_exp_f32 by one ulp.  r = float(u >> 32)
// is within 1 + 2^-24 r of canonical(u) 2^32, so D = e 2^32 - r in single
// precision is within 2e4 of (exp(x) - canonical(u)) 2^32 and its sign decides
// where |D| > 2^16.  The double draw and the double exp decide the rest (3e-5
// of the tests; with the earlier band of 1e-3 exp(x), a wavefront went there
// at every tenth decision), and for an e that is NaN.  Lanes that are in `sure`
// (dS < 0, e >= 1) accept; a NaN dS does not.
// The double test is out of line: inlined at every decision of a sweep
// kernel its exp makes up a sizeable part of the kernel's code.
__device__ __attribute__((noinline)) bool accept_exact(uint64_t u, double x) {
  return canonical(u) < exp(x);
}
constexpr float kLog2e = 0x1.715476p+0f;
template <typename X>
__device__ __forceinline__ uint64_t accept_draw(uint64_t u, float e, uint64_t sure, X x) {
  // the empty asm keeps the draw's top half a 32-bit value (otherwise it is
  // converted as a 64-bit one, six instructions instead of one)
  uint32_t h = (uint32_t)(u >> 32);
  __asm__("" : "+v"(h));
  const float D = __builtin_fmaf(e, 0x1p32f, -(float)h);
  uint64_t accept = lanes(D > 0.f);
  const uint64_t near = lanes(!(fabsf(D) > 0x1p16f));
  if (__builtin_expect(near != 0, 0)) {
    // the draw rebuilt from h (the same bits), so that u's top half need not
    // be kept beside h
    const uint64_t exact = lanes(accept_exact(((uint64_t)h << 32) | (uint32_t)u, x()));
    accept = (accept & ~near) | ((exact | sure) & near);
  }
  return accept;
}

// The Metropolis decision of one phi site (Stepper.cxx:330-370) in the
// reference's operand order: heff[l] is the neighbour sum of component l,
// ((x+1 + x-1) + (y+1 + y-1)) + (z+1 + z-1).  Returns the new value (the
// old one on reject) and adds the decision to the monitor where count.
__device__ __forceinline__ void hb_decide(const double phi_o[4], const double heff[4],
                                          double Lambda2, double lambda, double H, double rdtg,
                                          Xoro &g, double phi_new[4], Tally &m,
                                          bool count = true) {
  double hphi_o = 0., hphi_n = 0., s_o = 0., s_n = 0.;
  double phi_n[4];
#pragma unroll
  for (int l = 0; l < 4; l++) {
    phi_n[l] = phi_o[l] + rdtg * variance1(g);
    s_o += phi_o[l] * phi_o[l];
    s_n += phi_n[l] * phi_n[l];
    hphi_o += heff[l] * phi_o[l];
    hphi_n += heff[l] * phi_n[l];
  }
  hphi_o += (H * phi_o[0]);
  hphi_n += (H * phi_n[0]);
  const double dS = -(hphi_n - hphi_o) + Lambda2 * (s_n - s_o) +
                    lambda / 4. * (s_n * s_n - s_o * s_o);
  const uint64_t down = lanes(dS < 0);
  // the site's last draw: taken whether or not it is needed
  const uint64_t accept =
      accept_draw(xoro_next(g), __builtin_amdgcn_exp2f((float)dS * -kLog2e), down,
                  [&] { return -dS; });
  tally_all(m, 1, count);
  tally(m, dS, down, accept & ~down, lanes(count));
#pragma unroll
  for (int l = 0; l < 4; l++) phi_new[l] = in_lanes(accept) ? phi_n[l] : phi_o[l];
}

// One parity of EulerLangevinHB::step (ModelG/Stepper.cxx:309-386), one
// thread per site, in place.
template <typename T, bool W>
__global__ __launch_bounds__(kBlock) void k_hb_phi(const ReplicaParams *__restrict__ P,
                                                   const ReplicaState *__restrict__ S,
                                                   LaunchBlocks blk, int ieo,
                                                   int ctr_off, int flip,
                                                   MonSlot *__restrict__ mon) {
  int r, b;
  MonSlot *slot = mon + block_of(blk, r, b);
  const ReplicaParams &p = P[r];
  const uint32_t idx = (uint32_t)b * kBlock + threadIdx.x;
  Tally mt;
  if (idx < (uint64_t)p.half) {
    const uint32_t N = p.N, NH = p.NH;
    const uint32_t rowi = idx / NH, xh = idx - rowi * NH;
    const uint32_t z = rowi / N, y = rowi - z * N;
    const uint32_t x = site_x(xh, y, z, ieo);
    const int q = ieo ^ 1;
    const uint32_t row = rowi * NH;
    const uint32_t xp = x + 1 == N ? 0 : x + 1, xm = x == 0 ? N - 1 : x - 1;
    const uint32_t yp = y + 1 == N ? 0 : y + 1, ym = y == 0 ? N - 1 : y - 1;
    const uint32_t zp = z + 1 == N ? 0 : z + 1, zm = z == 0 ? N - 1 : z - 1;
    const uint32_t nb[6] = {row + (xp >> 1), row + (xm >> 1), (z * N + yp) * NH + xh,
                            (z * N + ym) * NH + xh, (zp * N + y) * NH + xh,
                            (zm * N + y) * NH + xh};
    const ReplicaState &s = S[r];
    const int cur = s.cur_phi ^ (flip & 1);  // phi planes only
    const double mass = p.mass0 + p.dmassdt * s.t;
    const double Lambda2 = 0.5 * (2. * 3. + mass);
    Xoro g = xoro_seeded(site_key(stream_key(p.base_key, s.sweep_ctr + ctr_off),
                                  (uint64_t)rowi * N + x));
    double phi_o[4], heff[4], phi_n[4];
#pragma unroll
    for (int l = 0; l < 4; l++) {
      const GPlane<T, W> fq = gplane<T, W>(p, cur, l, q);
      heff[l] = (fq.ld(nb[0]) + fq.ld(nb[1])) + (fq.ld(nb[2]) + fq.ld(nb[3])) +
                (fq.ld(nb[4]) + fq.ld(nb[5]));
      phi_o[l] = gplane<T, W>(p, cur, l, ieo).ld(idx);
    }
    hb_decide(phi_o, heff, Lambda2, p.lambda, p.H, p.rdtg, g, phi_n, mt);
#pragma unroll
    for (int l = 0; l < 4; l++) gplane<T, W>(p, cur, l, ieo).st(idx, phi_n[l]);
  }
  block_monitor_add(slot, mt);
}

__device__ __forceinline__ int wrapz(int z, int N) { return z < 0 ? z + N : (z >= N ? z - N : z); }

// Both parities of EulerLangevinHB::step (Stepper.cxx:309-386) in one launch,
// out of place: a block updates a brick of whole x rows, BY in y and BZ in z.
// It first decides the even sites of the brick and of the rows that face it
// (the neighbours of its odd sites; each decision has its own random stream,
// so the blocks that share a row make the same one), keeps them in LDS, and
// then decides its odd sites from there.  Small lattices spend most of a
// half-sweep on the launch and on one round of loads, so half the launches
// count more than deciding the facing rows again (a half-sweep of 32^3 6.6 ->
// 4.6 us, of 64^3 8.6 -> 7.1, half of a launch; 100^3 15.9 -> 16.7: kBrickSites).
// The first round of odd values is loaded before the even sites' decisions.
template <typename T>
__global__ __launch_bounds__(kPairBlock) void k_hb_brick(const ReplicaParams *__restrict__ P,
                                                          const ReplicaState *__restrict__ S,
                                                          LaunchBlocks blk, int ctr_off, int flip,
                                                          MonSlot *__restrict__ mon) {
  extern __shared__ double brick_lds[];
  T *even = reinterpret_cast<T *>(brick_lds);  // [4][rows][NH]
  int r, b;
  MonSlot *slot = mon + block_of(blk, r, b);
  const ReplicaParams &p = P[r];
  const ReplicaState &s = S[r];
  const int cur = s.cur_phi ^ (flip & 1), nxt = cur ^ 1;  // phi planes only
  const uint32_t N = p.N, NH = p.NH;
  const int nby = (N + p.pair_y - 1) / p.pair_y;
  const int y0 = b % nby * p.pair_y, z0 = b / nby * p.pair_z;
  const int h = min(p.pair_y, (int)N - y0), d = min(p.pair_z, (int)N - z0);
  // rows: the brick's, then the facing ones at y0 - 1, y0 + h, z0 - 1, z0 + d
  const int ni = h * d, fy0 = ni, fy1 = ni + d, fz0 = ni + 2 * d, fz1 = fz0 + h;
  const int rows = fz1 + h;
  const int comp = rows * (int)NH;
  const double mass = p.mass0 + p.dmassdt * s.t;
  const double Lambda2 = 0.5 * (2. * 3. + mass);
  const double lambda = p.lambda, H = p.H, rdtg = p.rdtg;
  const uint64_t key_e = stream_key(p.base_key, s.sweep_ctr + ctr_off);
  const uint64_t key_o = stream_key(p.base_key, s.sweep_ctr + ctr_off + 1);
  // i / NH for i < 2^16 as a multiplication (exact while i NH < 2^32)
  const uint32_t inv = 0xFFFFFFFFu / NH + 1;
  const int wave0 = first_lane((int)(threadIdx.x & ~63u)), lane = threadIdx.x & 63;
  Tally mt;
  // the odd site of round i0 and its value, loaded a round ahead (before the
  // even sites for the first one)
  const int odd = ni * (int)NH;
  T odd_o[4];
  auto odd_site = [&](int i0, uint32_t &rid, uint32_t &xh, int &dy, int &dz)
      __attribute__((always_inline)) {
    const uint32_t i = i0 + lane < odd ? i0 + lane : odd - 1;
    rid = __umulhi(i, inv);
    xh = i - rid * NH;
    dz = (int)rid / h;
    dy = (int)rid - dz * h;
    return ((z0 + dz) * N + y0 + dy) * NH + xh;
  };
  auto odd_load = [&](int i0) __attribute__((always_inline)) {
    uint32_t rid, xh;
    int dy, dz;
    const uint32_t idx = odd_site(i0, rid, xh, dy, dz);
#pragma unroll
    for (int l = 0; l < 4; l++) odd_o[l] = gplane<T, false>(p, cur, l, 1).raw(idx);
  };
  if (wave0 < odd) odd_load(wave0);
  // Every lane of a wavefront takes part in each of its rounds (the tallies
  // are the wavefront's): lanes past the end repeat the last site.
  for (int i0 = wave0; i0 < comp; i0 += kPairBlock) {
    const bool in = i0 + lane < comp;
    const uint32_t i = in ? i0 + lane : comp - 1;
    const uint32_t rid = __umulhi(i, inv), xh = i - rid * NH;
    int dy, dz;
    if ((int)rid < ni) { dz = (int)rid / h; dy = (int)rid - dz * h; }
    else if ((int)rid < fz0) { const bool up = (int)rid >= fy1; dz = (int)rid - (up ? fy1 : fy0); dy = up ? h : -1; }
    else { const bool up = (int)rid >= fz1; dy = (int)rid - (up ? fz1 : fz0); dz = up ? d : -1; }
    const uint32_t y = wrapz(y0 + dy, N), z = wrapz(z0 + dz, N);
    const uint32_t x = site_x(xh, y, z, 0);
    const uint32_t rowi = z * N + y, row = rowi * NH;
    const uint32_t xp = x + 1 == N ? 0 : x + 1, xm = x == 0 ? N - 1 : x - 1;
    const uint32_t yp = y + 1 == N ? 0 : y + 1, ym = y == 0 ? N - 1 : y - 1;
    const uint32_t zp = z + 1 == N ? 0 : z + 1, zm = z == 0 ? N - 1 : z - 1;
    const uint32_t nb[6] = {row + (xp >> 1), row + (xm >> 1), (z * N + yp) * NH + xh,
                            (z * N + ym) * NH + xh, (zp * N + y) * NH + xh,
                            (zm * N + y) * NH + xh};
    double phi_o[4], heff[4], phi_n[4];
#pragma unroll
    for (int l = 0; l < 4; l++) {
      const GPlane<T, false> f = gplane<T, false>(p, cur, l, 1);
      heff[l] = (f.ld(nb[0]) + f.ld(nb[1])) + (f.ld(nb[2]) + f.ld(nb[3])) +
                (f.ld(nb[4]) + f.ld(nb[5]));
      phi_o[l] = gplane<T, false>(p, cur, l, 0).ld(row + xh);
    }
    const bool mine = in && (int)rid < ni;
    Xoro g = xoro_seeded(site_key(key_e, (uint64_t)rowi * N + x));
    hb_decide(phi_o, heff, Lambda2, lambda, H, rdtg, g, phi_n, mt, mine);
#pragma unroll
    for (int l = 0; l < 4; l++) {
      even[l * comp + i] = (T)phi_n[l];
      if (mine) gplane<T, false>(p, nxt, l, 0).st(row + xh, phi_n[l]);
    }
  }
  __syncthreads();
  for (int i0 = wave0; i0 < odd; i0 += kPairBlock) {
    const bool in = i0 + lane < odd;
    uint32_t rid, xh;
    int dy, dz;
    const uint32_t idx = odd_site(i0, rid, xh, dy, dz);
    const uint32_t y = y0 + dy, z = z0 + dz;
    const uint32_t x = site_x(xh, y, z, 1);
    const uint32_t xp = x + 1 == N ? 0 : x + 1, xm = x == 0 ? N - 1 : x - 1;
    const uint32_t ryp = dy + 1 < h ? rid + 1 : fy1 + dz, rym = dy > 0 ? rid - 1 : fy0 + dz;
    const uint32_t rzp = dz + 1 < d ? rid + h : fz1 + dy, rzm = dz > 0 ? rid - h : fz0 + dy;
    double phi_o[4], heff[4], phi_n[4];
#pragma unroll
    for (int l = 0; l < 4; l++) phi_o[l] = odd_o[l];
    if (i0 + kPairBlock < odd) odd_load(i0 + kPairBlock);
#pragma unroll
    for (int l = 0; l < 4; l++) {
      const T *f = even + l * comp;
      heff[l] = ((double)f[rid * NH + (xp >> 1)] + (double)f[rid * NH + (xm >> 1)]) +
                ((double)f[ryp * NH + xh] + (double)f[rym * NH + xh]) +
                ((double)f[rzp * NH + xh] + (double)f[rzm * NH + xh]);
    }
    Xoro g = xoro_seeded(site_key(key_o, ((uint64_t)z * N + y) * N + x));
    hb_decide(phi_o, heff, Lambda2, lambda, H, rdtg, g, phi_n, mt, in);
    if (in) {
#pragma unroll
      for (int l = 0; l < 4; l++) gplane<T, false>(p, nxt, l, 1).st(idx, phi_n[l]);
    }
  }
  block_monitor_add<kPairBlock>(slot, mt);
}

// Both parities of EulerLangevinHB::step (Stepper.cxx:309-386) in one launch,
// out of place, marching z: a block owns BY whole x rows of each plane and the
// facing row on either side, one thread to a half-column.  Step k decides the
// even sites of plane z0 - 1 + k (on the facing rows as well) from the odd
// values of the planes around it, and then the odd sites of the plane before
// from the even ones.  In LDS lie the odd values of this plane and the last one
// and the new even values of the last two; one barrier per plane.
// It reads and writes each value once where two half-sweeps read both parities
// twice (counted at 256^3 FP64: 70 bytes a site, the half-sweeps 108), for
// which it decides the even sites of the facing rows and of two planes a chunk
// twice.  256^3 FP64: 256 us for both parities (two half-sweeps 295), 4.9 us a
// plane of a block; about 60 % of that are vector instructions (235 a decision,
// 28 wavefronts' decisions on four SIMDs), the rest the barrier's skew and LDS
// reads.  Whole rows need no ring in x; the 16 wavefronts, of which a facing
// row's have half the work, spread evenly over the SIMDs.
template <bool NTS>
__global__ __launch_bounds__(kPairBlock) void k_hb_sweep(const ReplicaParams *__restrict__ P,
                                                          const ReplicaState *__restrict__ S,
                                                          LaunchBlocks blk, int ctr_off, int flip,
                                                          MonSlot *__restrict__ mon) {
  using T = double;  // FP32 fields run half-sweeps (see kPairMarchSites)
  __shared__ T odd[2][4][kPairBlock], even[2][4][kPairBlock];
  int r, b;
  MonSlot *slot = mon + block_of(blk, r, b);
  const ReplicaParams &p = P[r];
  const ReplicaState &s = S[r];
  const int cur = first_lane(s.cur_phi ^ (flip & 1));  // phi planes only
  const int N = p.N, NH = p.NH;
  const int nby = (N + p.pair_y - 1) / p.pair_y;
  const int y0 = b % nby * p.pair_y, z0 = b / nby * p.pair_z;
  const int h = min(p.pair_y, N - y0), tz = min(p.pair_z, N - z0);
  const int t = threadIdx.x;
  const int j = (int)__umulhi((uint32_t)t, 0xFFFFFFFFu / NH + 1), xh = t - j * NH;
  const bool own = j < h + 2, inner = own && j >= 1 && j <= h;
  const int y = wrapz(y0 - 1 + j, N);
  const bool low = j == 0, outer = low || j == h + 1;  // rows that face the tile
  constexpr uint32_t kNone = PhiPlanes<T, false>::kNone;
  const uint32_t i_own = own ? (uint32_t)y * NH + xh : kNone;
  const uint32_t i_out =
      own && outer ? (uint32_t)wrapz(low ? y - 1 : y + 1, N) * NH + xh : kNone;
  const uint32_t i_inner = inner ? i_own : kNone;
  const int tu = outer && !low ? t : t + NH, td = low ? t : t - NH;  // rows above, below
  const double mass = p.mass0 + p.dmassdt * s.t;
  const double Lambda2 = 0.5 * (2. * 3. + mass);
  const double lambda = p.lambda, H = p.H, rdtg = p.rdtg;
  const uint64_t key_e = stream_key(p.base_key, s.sweep_ctr + ctr_off);
  const uint64_t key_o = stream_key(p.base_key, s.sweep_ctr + ctr_off + 1);
  const PhiPlanes<T, false> in(p, cur), out(p, cur ^ 1);
  Tally mt;
  auto ld4 = [&](int par, uint32_t i, int z, T v[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < 4; l++) v[l] = in.template ld<false>(l, par, z, i);
  };
  // the half-columns of row position c that hold x + 1 and x - 1 of a site with
  // x = 2 c + o, as steps from the thread's own slot
  auto step_up = [&](int o) __attribute__((always_inline)) {
    return o ? (xh + 1 == NH ? 1 - NH : 1) : 0;
  };
  auto step_down = [&](int o) __attribute__((always_inline)) {
    return o ? 0 : (xh == 0 ? NH - 1 : -1);
  };
  T o_next[4], o_far[4], e_old[4], e_far[4], o_out[4], o_outn[4];
  int z = wrapz(z0 - 1, N);  // plane of step k
  if (own) {
    T a[4], c[4];
    ld4(1, i_own, wrapz(z - 1, N), a);
    ld4(1, i_own, z, c);
    ld4(1, i_own, wrapz(z + 1, N), o_next);
    ld4(0, i_own, z, e_old);
    if (outer) ld4(1, i_out, z, o_out);
#pragma unroll
    for (int l = 0; l < 4; l++) {
      odd[1][l][t] = a[l];
      odd[0][l][t] = c[l];
    }
  }
  const bool wave_inner = lanes(inner) != 0;
  for (int k = 0; k < tz + 2; k++) {
    const int q = k & 1, zn = wrapz(z + 1, N);
    // every lane issues the same loads and stores, so that the wait for the
    // loads at the end of the step leaves the stores in flight
    const bool more = k < tz + 1;
    ld4(1, more ? i_own : kNone, wrapz(zn + 1, N), o_far);
    ld4(0, more ? i_own : kNone, zn, e_far);
    ld4(1, more ? i_out : kNone, zn, o_outn);
    __syncthreads();
    T e_new[4], o_new[4];
    const bool mid = k >= 1 && k <= tz;
    if (own) {
      const int o = (y + z) & 1;
      double phi_o[4], heff[4], phi_n[4];
      const int tp = t + step_up(o), tm = t + step_down(o);
#pragma unroll
      for (int l = 0; l < 4; l++) {
        double up = (double)odd[q][l][tu], dn = (double)odd[q][l][td];
        if (outer) (low ? dn : up) = (double)o_out[l];
        heff[l] = ((double)odd[q][l][tp] + (double)odd[q][l][tm]) + (up + dn) +
                  ((double)o_next[l] + (double)odd[q ^ 1][l][t]);
        phi_o[l] = (double)e_old[l];
      }
      Xoro g = xoro_seeded(site_key(key_e, ((uint64_t)z * N + y) * N + 2 * xh + o));
      hb_decide(phi_o, heff, Lambda2, lambda, H, rdtg, g, phi_n, mt, inner && mid);
#pragma unroll
      for (int l = 0; l < 4; l++) e_new[l] = (T)phi_n[l];
    }
#pragma unroll
    for (int l = 0; l < 4; l++) out.template st<NTS>(l, 0, z, mid ? i_inner : kNone, e_new[l]);
    const int zo = wrapz(z - 1, N);
    if (k >= 2 && wave_inner && own) {
      const int oo = (1 + y + zo) & 1;
      const int up = t + step_up(oo), dn = t + step_down(oo);
      double phi_o[4], heff[4], phi_n[4];
#pragma unroll
      for (int l = 0; l < 4; l++) {
        heff[l] = ((double)even[q ^ 1][l][up] + (double)even[q ^ 1][l][dn]) +
                  ((double)even[q ^ 1][l][tu] + (double)even[q ^ 1][l][td]) +
                  ((double)e_new[l] + (double)even[q][l][t]);
        phi_o[l] = (double)odd[q ^ 1][l][t];
      }
      Xoro go = xoro_seeded(site_key(key_o, ((uint64_t)zo * N + y) * N + 2 * xh + oo));
      hb_decide(phi_o, heff, Lambda2, lambda, H, rdtg, go, phi_n, mt, inner);
#pragma unroll
      for (int l = 0; l < 4; l++) o_new[l] = (T)phi_n[l];
    }
#pragma unroll
    for (int l = 0; l < 4; l++)
      out.template st<NTS>(l, 1, zo, k >= 2 ? i_inner : kNone, o_new[l]);
    // the slots of the next step: read by no other thread until the barrier
    // (the even ones of two planes ago, the odd ones of the last plane)
    if (own) {
#pragma unroll
      for (int l = 0; l < 4; l++) {
        even[q][l][t] = e_new[l];
        odd[q ^ 1][l][t] = o_next[l];
      }
    }
#pragma unroll
    for (int l = 0; l < 4; l++) {
      o_next[l] = o_far[l];
      e_old[l] = e_far[l];
      o_out[l] = o_outn[l];
    }
    z = zn;
  }
  block_monitor_add<kPairBlock>(slot, mt);
}

// One parity of EulerLangevinHB::step (Stepper.cxx:309-386), in place, by
// marching z through a TXH x TY tile of half-columns (the tile of hb_tile).
// The update parity ieo reads only the other parity q, which no thread of
// the launch writes: per plane, the q values of the tile and of a one-site
// ring sit in a packed LDS grid (one entry per half-column and row; two
// grids alternate, one barrier per plane), the q values of the thread's own
// half-column at z-1 and z+1 in registers.  Each q value is loaded once per
// plane (plus the ring), each decision is made once.
template <typename T, bool W, bool NTS>
__global__ __launch_bounds__(kBlock) void k_hb_march(const ReplicaParams *__restrict__ P,
                                                     const ReplicaState *__restrict__ S,
                                                     LaunchBlocks blk, int ieo,
                                                     int ctr_off, int flip,
                                                     MonSlot *__restrict__ mon) {
  constexpr int kGrid = kHbMarchGrid;
  // values held widened to FP64 (exact for FP32 fields): each is read by up
  // to four sites, so one conversion on the way in replaces four on the way out
  __shared__ double Q[2][4][kGrid];
  int r, tile;
  MonSlot *slot = mon + block_of(blk, r, tile);
  const ReplicaParams &p = P[r];
  const ReplicaState &s = S[r];
  const int cur = s.cur_phi ^ (flip & 1);  // phi planes only
  const int q = ieo ^ 1;
  const int N = p.N, NH = p.NH;
  int TXH, TY, TZ;
  hb_tile(N, p.hb_cap, p.hb_tz, TXH, TY, TZ);
  const int ntx = (NH + TXH - 1) / TXH, nty = (N + TY - 1) / TY;
  const int bx = tile % ntx, by = tile / ntx % nty, bz = tile / ntx / nty;
  const int xh0 = bx * TXH, y0 = by * TY, z0 = bz * TZ;
  const int tw = min(TXH, NH - xh0), th = min(TY, N - y0), tz = min(TZ, N - z0);
  const int GW = tw + 2;  // grid row width: half-columns xh0-1 .. xh0+tw
  const int t = threadIdx.x;
  const int tx = t % TXH, ty = t / TXH;
  const bool own = t < TXH * TY && ty < th && tx < tw;
  const int xh = xh0 + tx, y = y0 + ty;
  // ring entry of this thread: left/right half-column, rows above/below
  const bool halo = t < 2 * th + 2 * tw;
  int hlx, hly;
  if (t < th) { hlx = -1; hly = t; }
  else if (t < 2 * th) { hlx = tw; hly = t - th; }
  else if (t < 2 * th + tw) { hlx = t - 2 * th; hly = -1; }
  else { hlx = t - 2 * th - tw; hly = th; }
  const int hgxh = wrapz(xh0 + hlx, NH), hgy = wrapz(y0 + hly, N);
  const int hpos = (hly + 1) * GW + (hlx + 1);

  const double mass = p.mass0 + p.dmassdt * s.t;
  const double Lambda2 = 0.5 * (2. * 3. + mass);
  const double lambda = p.lambda, H = p.H, rdtg = p.rdtg;
  const uint64_t key = stream_key(p.base_key, s.sweep_ctr + ctr_off);
  Tally mt;
  const PhiPlanes<T, W> f(p, first_lane(cur));
  const uint32_t i_own = (uint32_t)y * NH + xh, i_halo = (uint32_t)hgy * NH + hgxh;
  auto ld4 = [&](uint32_t i, int zz, double v[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < 4; l++) v[l] = f.template ld<false>(l, q, zz, i);
  };
  // The loads of plane z+1 (the own half-column's q values at z+2, its own
  // update-parity value at z+1, the ring entry at z+1) are issued before
  // plane z's barrier, into the registers nq, nphi, nh as stored, so that
  // they are in flight during plane z's decisions.
  auto raw4 = [&](uint32_t i, int zz, T v[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < 4; l++) v[l] = f.template ld<false>(l, q, zz, i);
  };
  // the update parity's own value: read by this thread only
  auto own4 = [&](int zz, T v[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < 4; l++) v[l] = f.template ld<NTS>(l, ieo, zz, i_own);
  };
  // Plane z's new values are stored in iteration z+1, after the loads of
  // plane z+2 are issued and before the barrier: one in-order counter covers
  // loads and stores, so the next iteration's wait for those loads also
  // waits for these stores, which have had the decisions of plane z+1 to
  // complete (a store at the end of an iteration would be waited for at
  // once).  Only this thread reads its own sites.
  auto store4 = [&](int zz, const T v[4]) __attribute__((always_inline)) {
#pragma unroll
    for (int l = 0; l < 4; l++) f.template st<NTS>(l, ieo, zz, i_own, v[l]);
  };
  // FP32 fields: the loads run two planes ahead in two register sets (a
  // set holds half the bytes of an FP64 one, so one set in flight per wave
  // leaves the memory system short of requests; 256^3 half-sweep 94 -> 92
  // us, 119 registers, still four waves per SIMD); FP64: one plane ahead.
  constexpr int kDepth = sizeof(T) == 4 ? 2 : 1;
  double qm[4], qc[4], qp[4];  // q values of the own half-column at z-1, z, z+1
  // set s: the own q values at z+1, the own update-parity value at z and the
  // ring entry at z, for the planes z = z0 + s, z0 + s + kDepth, ...
  T nq[kDepth][4], nphi[kDepth][4], nh[kDepth][4];
  T pend[4];         // plane z-1's new values, stored at the top of iteration z
  if (own) {
    ld4(i_own, wrapz(z0 - 1, N), qm);
    ld4(i_own, z0, qc);
  }
#pragma unroll
  for (int sidx = 0; sidx < kDepth; sidx++) {
    if (sidx < tz) {  // plane z0 + sidx < z0 + tz <= N
      const int zs = z0 + sidx;
      if (own) {
        raw4(i_own, zs + 1 == N ? 0 : zs + 1, nq[sidx]);
        own4(zs, nphi[sidx]);
      }
      if (halo) raw4(i_halo, zs, nh[sidx]);
    }
  }
  // plane z0 + j from register set sq / sphi / sh, which then takes the
  // loads of plane z0 + j + kDepth
  auto plane = [&](int j, T (&sq)[4], T (&sphi)[4], T (&sh)[4]) __attribute__((always_inline)) {
    const int z = z0 + j;
    double(*g)[kGrid] = Q[j & 1];
    double phi_o[4];
    if (own) {
      const int pos = (ty + 1) * GW + (tx + 1);
#pragma unroll
      for (int l = 0; l < 4; l++) {
        qp[l] = sq[l];
        phi_o[l] = sphi[l];
        g[l][pos] = qc[l];
      }
    }
    if (halo) {
#pragma unroll
      for (int l = 0; l < 4; l++) g[l][hpos] = sh[l];
    }
    if (j + kDepth < tz) {  // plane zn = z + kDepth < z0 + tz <= N
      const int zn = z + kDepth;
      if (own) {
        raw4(i_own, zn + 1 == N ? 0 : zn + 1, sq);
        own4(zn, sphi);
      }
      if (halo) raw4(i_halo, zn, sh);
    }
    if (own && j > 0) store4(z - 1, pend);
    __syncthreads();
    if (own) {
      const int o = (ieo + y + z) & 1;  // x = 2 xh + o
      const int pos = (ty + 1) * GW + (tx + 1);
      double heff[4], phi_n[4];
#pragma unroll
      for (int l = 0; l < 4; l++)
        heff[l] = (g[l][pos + o] + g[l][pos - 1 + o]) +
                  (g[l][pos + GW] + g[l][pos - GW]) + (qp[l] + qm[l]);
      Xoro gg = xoro_seeded(site_key(key, ((uint64_t)z * N + y) * N + 2 * xh + o));
      hb_decide(phi_o, heff, Lambda2, lambda, H, rdtg, gg, phi_n, mt);
#pragma unroll
      for (int l = 0; l < 4; l++) {
        pend[l] = (T)phi_n[l];
        qm[l] = qc[l];
        qc[l] = qp[l];
      }
    }
  };
  // tz is the same for the whole block, so every thread makes the same calls
  // (and reaches the same barriers)
  for (int j = 0; j < tz; j += kDepth) {
    plane(j, nq[0], nphi[0], nh[0]);
    if constexpr (kDepth == 2) {
      if (j + 1 < tz) plane(j + 1, nq[kDepth - 1], nphi[kDepth - 1], nh[kDepth - 1]);
    }
  }
  if (own && tz > 0) store4(z0 + tz - 1, pend);
  block_monitor_add(slot, mt);
}


// ------------------------------------------------------------------------
// modelg_update_charge_pair (Stepper.cxx:419-441) for one component of one
// pair, applied as nA + (-q), nB + q; counts the decision when count.
// The constants of a charge sweep: the proposal width, the divisor d = 2 chi
// of dS with its rounded reciprocal, and -log2(e) / d in single precision (NaN
// where that won't do: charge_l2; formed here, it cost 0.3 of the 37.5 us of
// three launches at 64^3).
struct ChargeK {
  double rms, d, inv;
  float l2;
};
__device__ __forceinline__ ChargeK charge_k(const ReplicaParams &p) {
  const double d = 2. * p.chi;
  return {p.rms, d, 1. / d, p.chg_l2};
}
// x / d from the rounded reciprocal with one Markstein correction: q0 = x *
// inv, the residual x - q0 d exact with one FMA, q0 + residual * inv rounded
// once.  It equals the IEEE quotient for these divisors (no difference in
// 1.6e8 random dividends over eight values of chi, including the defaults;
// the CPU suite checks it); a one-ulp difference could only change a
// decision if the uniform draw fell within that ulp of exp(-dS).
__device__ __forceinline__ double div_by(double x, const ChargeK &k) {
  const double q0 = x * k.inv;
  return fma(fma(-q0, k.d, x), k.inv, q0);
}

// The decision goes by X = dS d: its sign is that of dS, the single-precision
// test needs exp2(X l2), the monitor sums X (scaled by inv at the end of the
// launch), and only the double test divides.
__device__ __forceinline__ void charge_pair(double nA, double nB, const ChargeK &k,
                                            Xoro &g, double &outA, double &outB, Tally &m,
                                            bool count) {
  const double q = k.rms * variance1(g);
  const double X = (nA - q) * (nA - q) + (nB + q) * (nB + q) - nA * nA - nB * nB;
  const uint64_t down = lanes(X < 0);
  // the uniform draw: the engine advances where it is needed
  uint64_t u = g.s0 + g.s1;
  __asm__ volatile("" : "+v"(u));  // formed before the engine moves on: no copy of its state
  if (!in_lanes(down)) (void)xoro_next(g);
  const uint64_t accept = accept_draw(u, __builtin_amdgcn_exp2f((float)X * k.l2), down,
                                      [&] { return -div_by(X, k); });
  tally(m, X, down, accept & ~down, lanes(count));
  outA = nA;
  outB = nB;
  if (in_lanes(accept)) {
    outA = nA - q;
    outB = nB + q;
  }
}

// The two sub-sweeps of one direction (the shuffled order always runs both
// parities of a direction back to back, Stepper.cxx:471-473) for one site
// A' of the second parity e2: along the direction its line reads
// L = A'-e, A', B' = A'+e, R = A'+2e.  First sub-sweep (parity e1): pairs
// (L, A') and (B', R), keyed by L and B'; second: pair (A', B') keyed by A'
// on the first sub-sweep's results.  Each first-parity pair is computed by
// the two threads that need it (identical counter streams, identical bits);
// the monitor counts it once, from the thread on its right.  Reads the live
// charge buffer, writes A' and B' into the other one.
template <typename T, bool W>
__device__ __forceinline__ void charge_line(const ReplicaParams &p, const ChargePlanes<T, W> &f,
                                            int dir, int e1, int e2, uint32_t xh, uint32_t y, uint32_t z,
                                            uint64_t k1, uint64_t k2, Tally &m) {
  const uint32_t N = p.N, NH = p.NH;
  const uint32_t x = site_x(xh, y, z, e2);
  // the four sites along the direction: L, A', B', R (parities e1 e2 e1 e2)
  const uint32_t a0 = dir == 0 ? x : (dir == 1 ? y : z);
  const uint32_t am = a0 == 0 ? N - 1 : a0 - 1;
  const uint32_t ap = a0 + 1 == N ? 0 : a0 + 1;
  const uint32_t app = ap + 1 == N ? 0 : ap + 1;
  uint32_t ii[4], lin[4];
#pragma unroll
  for (int k = 0; k < 4; k++) {
    const uint32_t a = k == 0 ? am : (k == 1 ? a0 : (k == 2 ? ap : app));
    const uint32_t xx = dir == 0 ? a : x, yy = dir == 1 ? a : y, zz = dir == 2 ? a : z;
    ii[k] = (zz * N + yy) * NH + (xx >> 1);
    lin[k] = (zz * N + yy) * N + xx;
  }
  const ChargeK ck = charge_k(p);
  Xoro gL = xoro_seeded(site_key(k1, lin[0]));
  Xoro gB = xoro_seeded(site_key(k1, lin[2]));
  Xoro gA = xoro_seeded(site_key(k2, lin[1]));
  tally_all(m, 12, true);
  // every load of the line before the first store (see charge_column)
  T w[6][4];
#pragma unroll
  for (int c = 0; c < 6; c++) {
    w[c][0] = f.ld(c, e1, ii[0]);
    w[c][1] = f.ld(c, e2, ii[1]);
    w[c][2] = f.ld(c, e1, ii[2]);
    w[c][3] = f.ld(c, e2, ii[3]);
  }
#pragma unroll
  for (int c = 0; c < 6; c++) {
    const double vL = w[c][0], vA = w[c][1], vB = w[c][2], vR = w[c][3];
    double tL, a1, b1, tR;
    charge_pair(vL, vA, ck, gL, tL, a1, m, true);
    charge_pair(vB, vR, ck, gB, b1, tR, m, false);
    // the first sub-sweep's results as stored (rounded in FP32 storage)
    a1 = (double)(T)a1;
    b1 = (double)(T)b1;
    double a2, b2;
    charge_pair(a1, b1, ck, gA, a2, b2, m, true);
    f.st(c, e2, ii[1], (T)a2);
    f.st(c, e1, ii[2], (T)b2);
  }
}

// The x direction with a whole row in one wavefront or in one aligned
// segment of seg lanes of it (NH = seg H; seg = NH <= 64 a power of two for
// H = 1, seg = 64 for H = 2): lane l of the segment owns the second-parity
// sites A'_h of half-columns h = l + 64 j, j < H.  First sub-sweep: the lane
// updates the pair (L_h, A'_h), L_h = A'_h - e_x.  The updated L_{h+1} is
// B'_h = A'_h + e_x; it comes from the lane that owns h + 1 (lane l + 1, or
// for the segment's last lane its lane 0, at j + 1 for H = 2, the row
// wrapping periodically).  Second sub-sweep: the lane updates (A'_h, B'_h)
// and writes both.  Every pair is computed once and counted once, from the
// same counter streams as charge_line.  Index logic checked on the CPU
// against the plain two sub-sweeps (exact integer stand-in, N = 4 ... 256).
template <typename T, bool W, int H>
__device__ __forceinline__ void charge_row_wave(const ReplicaParams &p, const ChargePlanes<T, W> &f,
                                                int e1, int e2, uint32_t y, uint32_t z, int lane, int seg,
                                                uint64_t k1, uint64_t k2, Tally &m) {
  static_assert(H == 1 || H == 2, "rows of up to 128 half-columns");
  const uint32_t N = p.N, NH = p.NH;
  const uint32_t row = z * N + y;
  const ChargeK ck = charge_k(p);
  // a1: updated A'_h; r: updated L_{h+1} from lane + 1; l0: lane 0's updated
  // L (H = 2 only); all as stored (T), which is how the second sub-sweep reads
  // them, so that FP32 fields hold and shuffle half the registers
  T a1[H][6], r[H][6], l0[H][6];
#pragma unroll
  for (int j = 0; j < H; j++) {
    const uint32_t h = lane + 64 * j;
    const uint32_t x = site_x(h, y, z, e2);
    const uint32_t xl = x == 0 ? N - 1 : x - 1;
    const uint32_t iA = row * NH + h, iL = row * NH + (xl >> 1);
    T wl[6], wa[6];  // as stored: converted where used
#pragma unroll
    for (int c = 0; c < 6; c++) {
      wl[c] = f.ld(c, e1, iL);
      wa[c] = f.ld(c, e2, iA);
    }
    Xoro gL = xoro_seeded(site_key(k1, row * N + xl));
    tally_all(m, 12, true);  // the six of this sub-sweep and the second's
#pragma unroll
    for (int c = 0; c < 6; c++) {
      double tl, ta;
      charge_pair((double)wl[c], (double)wa[c], ck, gL, tl, ta, m, true);
      // the first sub-sweep's results as stored (rounded in FP32 storage)
      const T tls = (T)tl;
      a1[j][c] = (T)ta;
      if constexpr (H == 1) {
        r[j][c] = __shfl(tls, (lane + 1) & (seg - 1), seg);
      } else {
        r[j][c] = __shfl(tls, (lane + 1) & 63, 64);
        l0[j][c] = first_lane(tls);  // lane 0's value, through scalar registers
      }
    }
  }
#pragma unroll
  for (int j = 0; j < H; j++) {
    const uint32_t h = lane + 64 * j;
    const uint32_t x = site_x(h, y, z, e2);
    const uint32_t xb = x + 1 == N ? 0 : x + 1;
    Xoro gA = xoro_seeded(site_key(k2, row * N + x));
#pragma unroll
    for (int c = 0; c < 6; c++) {
      // H = 2: lane 63's B'_h is lane 0's L of the next j (wrapping to j = 0)
      const double nb = (double)((H > 1 && lane == 63) ? l0[(j + 1) % H][c] : r[j][c]);
      double a2, b2;
      charge_pair((double)a1[j][c], nb, ck, gA, a2, b2, m, true);
      f.st(c, e2, row * NH + h, (T)a2);
      f.st(c, e1, row * NH + (xb >> 1), (T)b2);
    }
  }
}

// The same two sub-sweeps with every site loaded once and every pair
// computed once (except one first-parity pair per chunk end).  Blocks tile
// the lattice as TXH half-columns x TQ lines x a chunk of C sites (charge_tile):
//  * d = y or z: a thread owns the two columns x = 2xh, 2xh+1 along d and
//    marches d through its chunk.  Along a column the parity alternates; at
//    each step it updates the next first-parity pair (m, m+1) and then the
//    second-parity pair (m-1, m) from the previous pair's upper site, kept in
//    registers, and this pair's lower site.  The chunk owns the
//    second-parity pairs whose lower site lies in it and the first-parity
//    pairs whose lower site lies in it (the monitor counts those).
//  * d = x: pairs lie in rows; the thread runs charge_line for the row
//    (y, z) of each z of its chunk.
template <typename T, bool W, bool PIPE>
__device__ __forceinline__ void charge_column(const ReplicaParams &p, const ChargePlanes<T, W> &f,
                                              int dir, int e1, int e2, uint32_t x, uint32_t q, int c0,
                                              int c1, uint64_t k1, uint64_t k2, Tally &m) {
  const int N = p.N, NH = p.NH;
  const ChargeK ck = charge_k(p);
  // index / linear site of position m along the column
  auto at = [&](int m, uint32_t &ii, uint32_t &lin) __attribute__((always_inline)) {
    const uint32_t row = dir == 2 ? (uint32_t)m * N + q : q * N + (uint32_t)m;
    ii = row * NH + (x >> 1);
    lin = row * N + x;
  };
  // lower site of the first first-parity pair: c0-1 or c0
  const int mm0 = (int)((x + q + (uint32_t)(c0 + N - 1)) & 1) == e1 ? c0 - 1 : c0;
  // pair k: lower site m1 (parity e1), upper site m2 = m1 + 1 (parity e2)
  auto pair_at = [&](int k, int &m1, uint32_t &i1, uint32_t &l1, uint32_t &i2, uint32_t &l2)
      __attribute__((always_inline)) {
    const int mm = mm0 + 2 * k;
    m1 = mm < 0 ? mm + N : (mm >= N ? mm - N : mm);
    const int m2 = m1 + 1 == N ? 0 : m1 + 1;
    at(m1, i1, l1);
    at(m2, i2, l2);
  };
  // PIPE: pair k+1's loads are issued before pair k's arithmetic, into n1, n2
  // as stored, and pair k's results are stored in iteration k+1 after those
  // loads (one in-order counter covers loads and stores: a store issued
  // between a load and the wait for it would be waited for as well)
  T n1[6], n2[6], s0[6], s1[6];
  uint32_t si0 = 0, si1 = 0;
  auto load_pair = [&](uint32_t i1, uint32_t i2) __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 6; c++) {
      n1[c] = f.ld(c, e1, i1);
      n2[c] = f.ld(c, e2, i2);
    }
  };
  auto store_pending = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int c = 0; c < 6; c++) {
      f.st(c, e2, si0, s0[c]);
      f.st(c, e1, si1, s1[c]);
    }
  };
  const int npair = (c1 - c0) / 2;
  if (PIPE) {
    int m1;
    uint32_t i1, l1, i2, l2;
    pair_at(0, m1, i1, l1, i2, l2);
    load_pair(i1, i2);
  }
  T up[6];  // upper site of the previous first-parity pair, as stored
  for (int k = 0; k <= npair; k++) {
    const int mm = mm0 + 2 * k;
    int m1;
    uint32_t i1, l1, i2, l2;
    pair_at(k, m1, i1, l1, i2, l2);
    const bool own1 = mm >= c0 && mm < c1;
    tally_all(m, 6, own1);
    if (k > 0) tally_all(m, 6, true);
    Xoro g1 = xoro_seeded(site_key(k1, l1));
    Xoro g2;
    uint32_t i0 = 0, l0;
    if (k > 0) {
      const int m0 = m1 == 0 ? N - 1 : m1 - 1;
      at(m0, i0, l0);
      g2 = xoro_seeded(site_key(k2, l0));
    }
    T w1[6], w2[6];  // as stored: converted where used
    if (PIPE) {
#pragma unroll
      for (int c = 0; c < 6; c++) {
        w1[c] = n1[c];
        w2[c] = n2[c];
      }
      if (k < npair) {
        int mn;
        uint32_t j1, ln1, j2, ln2;
        pair_at(k + 1, mn, j1, ln1, j2, ln2);
        load_pair(j1, j2);
      }
      if (k > 1) store_pending();
    } else {
      // every load of the pair is issued before the first store: the
      // compiler cannot prove that the stores (other buffer) miss the loaded
      // planes and would otherwise wait for each component's load after the
      // previous store
#pragma unroll
      for (int c = 0; c < 6; c++) {
        w1[c] = f.ld(c, e1, i1);
        w2[c] = f.ld(c, e2, i2);
      }
    }
#pragma unroll
    for (int c = 0; c < 6; c++) {
      double a, b;
      charge_pair((double)w1[c], (double)w2[c], ck, g1, a, b, m, own1);
      // as stored (rounded in FP32 storage)
      const T as = (T)a, bs = (T)b;
      if (k > 0) {
        double o0, o1;
        charge_pair((double)up[c], (double)as, ck, g2, o0, o1, m, true);
        if (PIPE) {
          s0[c] = (T)o0;
          s1[c] = (T)o1;
        } else {
          f.st(c, e2, i0, (T)o0);
          f.st(c, e1, i1, (T)o1);
        }
      }
      up[c] = bs;
    }
    if (PIPE && k > 0) {
      si0 = i0;
      si1 = i1;
    }
  }
  if (PIPE && npair > 0) store_pending();
}

template <typename T, bool W, bool XW>
__global__ __launch_bounds__(kBlock)
__attribute__((amdgpu_waves_per_eu(sizeof(T) == 8 && XW ? 3 : 4))) void k_charge_march(const ReplicaParams *__restrict__ P,
                                                         const ReplicaState *__restrict__ S,
                                                         LaunchBlocks blk,
                                                         int ixyz, int ctr_off, int flip,
                                                         MonSlot *__restrict__ mon) {
  int r, tile;
  MonSlot *slot = mon + block_of(blk, r, tile);
  const ReplicaParams &p = P[r];
  const ReplicaState &s = S[r];
  const int N = p.N, NH = p.NH;
  int TXH, TQ, C;
  charge_tile(N, p.chg_cap, p.chg_chunk, TXH, TQ, C);
  const int nbx = (NH + TXH - 1) / TXH, nbq = (N + TQ - 1) / TQ;
  const int sx = tile & 1;
  int b = tile >> 1;
  const int bx = b % nbx;
  b /= nbx;
  const int bq = b % nbq, bc = b / nbq;
  const int t = threadIdx.x;
  const uint32_t xh = bx * TXH + t % TXH, q = bq * TQ + t / TXH;
  const int c0 = bc * C, c1 = min(c0 + C, N);
  Tally mt;
  if (xh < (uint32_t)NH && q < (uint32_t)N && t < TXH * TQ) {
    const ChargePlanes<T, W> f(p, first_lane(live(s) ^ flip));
    // the shuffled sub-sweep order of ModelGChargeHB::step
    // (Stepper.cxx:461-468) from the sweep's shuffle stream, the counter
    // before the first direction's two; every thread draws the same order
    int order[5];
    {
      Xoro g = xoro_seeded(site_key(stream_key(p.base_key, s.sweep_ctr + ctr_off - 1 - 2 * ixyz), 0));
      shuffle_orders(g, order);
    }
    const int dir = first_lane(ixyz == 0 ? order[0] : (ixyz == 1 ? order[1] : order[2]));
    const int e1 = first_lane(order[3]), e2 = e1 ^ 1;
    const uint64_t k1 = first_lane(stream_key(p.base_key, s.sweep_ctr + ctr_off));
    const uint64_t k2 = first_lane(stream_key(p.base_key, s.sweep_ctr + ctr_off + 1));
    // d = x: the chunk's planes, of which this block takes a share
    const int len = c1 - c0;
    if (XW && dir == 0) {  // every replica of the launch has NH = 64 or 128
      // whole rows in one wavefront (TXH = 64, TQ = 4: wave w takes row q);
      // the chunk's planes are split over the 2 nbx blocks of the row
      const int lane = t & 63, part = 2 * bx + sx;
      const int zs = c0 + part * len / (2 * nbx), ze = c0 + (part + 1) * len / (2 * nbx);
      for (int z = zs; z < ze; z++) {
        if (NH == 64)
          charge_row_wave<T, W, 1>(p, f, e1, e2, q, (uint32_t)z, lane, 64, k1, k2, mt);
        else
          charge_row_wave<T, W, 2>(p, f, e1, e2, q, (uint32_t)z, lane, 64, k1, k2, mt);
      }
    } else if (dir == 0) {
      const int zs = c0 + sx * len / 2, ze = c0 + (sx + 1) * len / 2;
      if (TXH == NH && NH <= 64 && (NH & (NH - 1)) == 0) {
        // whole rows in aligned segments of NH lanes: with TXH = NH thread t
        // takes half-column t % NH of the tile's row t / NH, and NH divides
        // the wavefront, so a row never straddles two waves
        for (int z = zs; z < ze; z++)
          charge_row_wave<T, W, 1>(p, f, e1, e2, q, (uint32_t)z, (int)xh, NH, k1, k2, mt);
      } else {
        for (int z = zs; z < ze; z++)
          charge_line<T, W>(p, f, 0, e1, e2, xh, q, (uint32_t)z, k1, k2, mt);
      }
    } else {
      charge_column<T, W, XW>(p, f, dir, e1, e2, 2 * xh + sx, q, c0, c1, k1, k2, mt);
    }
  }
  block_monitor_add(slot, mt, 1. / (2. * p.chi));
}

// ------------------------------------------------------------------------
// IdealPV2::step_no_reject (Stepper.cxx:68-176) fused into one pass:
// rotate by dt/2, kick the charges with the rotated neighbours, rotate by
// dt/2 with the kicked charges.  A block owns a TXH x TY x-y tile (both
// parities of each half-column) and marches over TZ planes; the rotated phi
// of the current plane and a one-site x-y halo (recomputed from the raw
// fields) sit in LDS, the rotated phi of the plane above in registers and of
// the plane below in thread-private LDS slots.  Reads the live buffer,
// writes the other one.
template <typename T, bool W>
__device__ __forceinline__ void load_site(const ReplicaParams &p, int cur, int x, int y, int z,
                                          double f[10]) {
  const int par = (x + y + z) & 1;
  const uint32_t i = ((uint32_t)z * p.N + y) * p.NH + (x >> 1);
#pragma unroll
  for (int c = 0; c < 10; c++) f[c] = gplane<T, W>(p, cur, c, par).ld(i);
}

// FP32 fields: at least 3 waves per SIMD (168 registers)
template <typename T, bool W, bool NTS>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(sizeof(T) == 4 ? 3 : 1)))
void k_ideal_fused(const ReplicaParams *__restrict__ P, const ReplicaState *__restrict__ S,
                   LaunchBlocks blk, int flip, int alternate) {
  __shared__ double lds[4][ideal_lds(sizeof(T) == 4)];
  // rotated phi of plane z-1 at the thread's own sites: thread-private slots
  __shared__ double lprv[2][4][kBlock];
  int r, tile;
  block_of(blk, r, tile);
  // a reference, not a copy: a private copy would be staged in scratch memory
  const ReplicaParams &p = P[r];
  const int cur = live(S[r]) ^ flip, nxt = cur ^ 3;
  const int N = p.N, NH = p.NH;
  int TXH, TY, TZ;
  ideal_tile(N, p.tile_cap, p.tile_tz, TXH, TY, TZ);
  const int ntx = (NH + TXH - 1) / TXH, nty = (N + TY - 1) / TY;
  const int bx = tile % ntx, by = tile / ntx % nty, bz = tile / ntx / nty;
  const int xh0 = bx * TXH, y0 = by * TY, z0 = bz * TZ;
  const int tw = min(TXH, NH - xh0), th = min(TY, N - y0), tz = min(TZ, N - z0);
  const int LW = 2 * tw + 2;  // LDS row width
  const int t = threadIdx.x;
  const int tx = t % TXH, ty = t / TXH;
  const bool own = ty < th && tx < tw;
  const int xh = xh0 + tx, y = y0 + ty;
  // the one-site ring around the tile (no corners): ring site j = t, t + kBlock, ..
  // (a second pass only when the ring has more sites than the block threads)
  const int nh = 2 * th + 4 * tw;
  // ring site j: global (x, y) and LDS slot
  auto ring_site = [&](int j, int &gx, int &gy, int &pos) __attribute__((always_inline)) {
    int hlx, hly;
    if (j < th) { hlx = -1; hly = j; }
    else if (j < 2 * th) { hlx = 2 * tw; hly = j - th; }
    else if (j < 2 * th + 2 * tw) { hlx = j - 2 * th; hly = -1; }
    else { hlx = j - 2 * th - 2 * tw; hly = th; }
    gx = 2 * xh0 + hlx;
    gx = gx < 0 ? gx + N : (gx >= N ? gx - N : gx);
    gy = y0 + hly;
    gy = gy < 0 ? gy + N : (gy >= N ? gy - N : gy);
    pos = (hly + 1) * LW + (hlx + 1);
  };
  int rgx = 0, rgy = 0, rpos = 0;  // this thread's first ring site
  if (t < nh) ring_site(t, rgx, rgy, rpos);
  const double h = 0.5 * (p.tau_ideal / p.chi);
  const double axx = p.axx, H0 = p.H, dt = p.dt_ideal;

  // FP64 fields carry the raw charges of planes z and z+1 in registers (two
  // waves per SIMD).  FP32 fields keep those of plane z in thread-private
  // LDS slots (as stored, in FP32) and those of plane z+1 in registers from
  // their load to the end of the iteration, which keeps three waves per
  // SIMD; re-reading plane z's charges at kick time instead made the kernel
  // read 1.92x its algorithmic bytes (the re-reads miss the 4 MB L2).
  constexpr bool kCarry = sizeof(T) == 8;
  __shared__ T chq[kCarry ? 1 : 2][kCarry ? 1 : 6][kCarry ? 1 : kBlock];
  // The thread's two own sites of a plane are indexed by parity (pp), not by
  // x offset: a parity's plane base is the same for every lane, so the loads
  // and stores use one scalar base and 32-bit offsets.  The site of parity pp
  // sits at x = 2 xh + ((pp + y + z) & 1); its z +- 1 neighbours have parity
  // pp ^ 1 in the same half-column.
  double cen[2][4], nex[2][4];  // rotated phi at the own sites of planes z, z+1
  double chg[2][6];             // raw charges of plane z (kCarry only)
  T chn[2][6];                  // raw charges of plane z+1, as stored
  auto rotate_own = [&](int z, double out[2][4], T ch[2][6]) __attribute__((always_inline)) {
    if (!own) return;
    const uint32_t i = ((uint32_t)z * N + y) * NH + xh;
    // both sites' loads before the first rotation: one wait for the pair
    T raw[2][10];
#pragma unroll
    for (int pp = 0; pp < 2; pp++)
#pragma unroll
      for (int c = 0; c < 10; c++) raw[pp][c] = gplane<T, W>(p, cur, c, pp).raw(i);
#pragma unroll
    for (int pp = 0; pp < 2; pp++) {
      double f[10];
#pragma unroll
      for (int c = 0; c < 10; c++) f[c] = (double)raw[pp][c];
      rotate_site_fast(f, f + 4, f + 7, h);
#pragma unroll
      for (int c = 0; c < 4; c++) out[pp][c] = f[c];
#pragma unroll
      for (int c = 0; c < 6; c++) ch[pp][c] = (T)f[4 + c];
    }
  };
  auto fill_lds = [&](int z, const double o[2][4]) __attribute__((always_inline)) {
    if (own) {
#pragma unroll
      for (int pp = 0; pp < 2; pp++) {
        const int sx = (pp + y + z) & 1;
#pragma unroll
        for (int c = 0; c < 4; c++) lds[c][(ty + 1) * LW + (2 * tx + sx + 1)] = o[pp][c];
      }
    }
    auto ring_fill = [&](int gx, int gy, int pos) __attribute__((always_inline)) {
      double f[10];
      load_site<T, W>(p, cur, gx, gy, z, f);
      rotate_site_fast(f, f + 4, f + 7, h);
#pragma unroll
      for (int c = 0; c < 4; c++) lds[c][pos] = f[c];
    };
    // the second pass of a ring of more sites than threads
    for (int j = t + kBlock; j < nh; j += kBlock) {
      int gx, gy, pos;
      ring_site(j, gx, gy, pos);
      ring_fill(gx, gy, pos);
    }
  };

  // With `alternate` (0 or 1) odd chunks march downwards.  Below, planes "z-1" and
  // "z+1" are those behind and ahead of z.
  const bool down = bz & alternate;
  const int dz = down ? -1 : 1, zs = down ? z0 + tz - 1 : z0;
  rotate_own(wrapz(zs - dz, N), nex, chn);
  if (own) {
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int c = 0; c < 4; c++) lprv[s][c][t] = nex[s][c];
  }
  rotate_own(zs, cen, chn);
  // the charges of the first plane: registers (FP64) or the thread's LDS slots (FP32)
  if (own) {
#pragma unroll
    for (int s = 0; s < 2; s++)
#pragma unroll
      for (int c = 0; c < 6; c++) {
        if constexpr (kCarry) chg[s][c] = (double)chn[s][c];
        else chq[s][c][t] = chn[s][c];
      }
  }
  if (t < nh) {
    double f[10];
    load_site<T, W>(p, cur, rgx, rgy, zs, f);
    rotate_site_fast(f, f + 4, f + 7, h);
#pragma unroll
    for (int c = 0; c < 4; c++) lds[c][rpos] = f[c];
  }
  fill_lds(zs, cen);
  for (int k = 0; k < tz; k++) {
    const int z = zs + k * dz;
    const int zn = wrapz(z + dz, N);
    rotate_own(zn, nex, chn);
    // The raw fields, as stored, of the thread's first ring site of plane z+1
    // are loaded before the kick of plane z, so that their latency overlaps the
    // kick (FP32: ten registers more, which the waves-per-SIMD bound of 3 holds
    // at 168 with three spilled; 256^3 FP32 347 -> 329 us, 2 waves 360 us)
    T rraw[10];
    const bool ring1 = t < nh && k + 1 < tz;
    if (ring1) {
      const uint32_t ri = ((uint32_t)zn * N + rgy) * NH + (rgx >> 1);
      const int rpar = (rgx + rgy + zn) & 1;
#pragma unroll
      for (int c = 0; c < 10; c++) rraw[c] = gplane<T, W>(p, cur, c, rpar).raw(ri);
    }
    __syncthreads();
    if (own) {
      const uint32_t i = ((uint32_t)z * N + y) * NH + xh;
#pragma unroll
      for (int pp = 0; pp < 2; pp++) {
        // held to 1e-12 like the rotations: contraction into FMA allowed
#pragma clang fp contract(fast)
        const int lx = 2 * tx + ((pp + y + z) & 1) + 1, ly = ty + 1;
        // The kick of Stepper.cxx:112-163, summed per direction there, is
        // linear in the neighbours: with S the sum of the six neighbours'
        // rotated phi, the axial kick is axx (cp0 S_l - cp_l S0) - H cp_l
        // and the vector kick axx (cp_s1 S_s2 - cp_s2 S_s1), (s1, s2) the
        // cyclic successors of s (every direction shares axx).
        const double *zp = nex[pp ^ 1];
        double cp[4], S[4], A[3], V[3];
#pragma unroll
        for (int c = 0; c < 4; c++) {
          cp[c] = cen[pp][c];
          S[c] = (lds[c][ly * LW + lx + 1] + lds[c][ly * LW + lx - 1]) +
                 (lds[c][(ly + 1) * LW + lx] + lds[c][(ly - 1) * LW + lx]) +
                 (zp[c] + lprv[pp ^ 1][c][t]);
        }
        const int par = pp;
        // the charges of plane z, unchanged by the first rotation
#pragma unroll
        for (int l = 0; l < 3; l++) {
          if constexpr (kCarry) {
            A[l] = chg[pp][l];
            V[l] = chg[pp][3 + l];
          } else {
            A[l] = (double)chq[pp][l][t];
            V[l] = (double)chq[pp][3 + l][t];
          }
        }
#pragma unroll
        for (int l = 0; l < 3; l++)
          A[l] += dt * (axx * (cp[0] * S[l + 1] - cp[l + 1] * S[0]) - H0 * cp[l + 1]);
#pragma unroll
        for (int s3 = 0; s3 < 3; s3++) {
          const int s1 = (s3 + 1) % 3, s2 = (s3 + 2) % 3;
          V[s3] += dt * (axx * (cp[1 + s1] * S[1 + s2] - cp[1 + s2] * S[1 + s1]));
        }
        rotate_site_fast(cp, A, V, h);
#pragma unroll
        for (int c = 0; c < 4; c++) gplane<T, W>(p, nxt, c, par).template put<NTS>(i, cp[c]);
#pragma unroll
        for (int c = 0; c < 3; c++) gplane<T, W>(p, nxt, 4 + c, par).template put<NTS>(i, A[c]);
#pragma unroll
        for (int c = 0; c < 3; c++) gplane<T, W>(p, nxt, 7 + c, par).template put<NTS>(i, V[c]);
      }
    }
    __syncthreads();
    if (ring1) {
      double rf[10];
#pragma unroll
      for (int c = 0; c < 10; c++) rf[c] = (double)rraw[c];
      rotate_site_fast(rf, rf + 4, rf + 7, h);
#pragma unroll
      for (int c = 0; c < 4; c++) lds[c][rpos] = rf[c];
    }
    if (k + 1 < tz) fill_lds(zn, nex);
#pragma unroll
    for (int s = 0; s < 2; s++) {
#pragma unroll
      for (int c = 0; c < 4; c++) {
        if (own) lprv[s][c][t] = cen[s][c];
        cen[s][c] = nex[s][c];
      }
      if (own) {
#pragma unroll
        for (int c = 0; c < 6; c++) {
          if constexpr (kCarry) chg[s][c] = (double)chn[s][c];
          else chq[s][c][t] = chn[s][c];
        }
      }
    }
  }
}

// ------------------------------------------------------------------------
// IdealPV2::computeEnergy (Stepper.cxx:204-268): per-block compensated
// partial sums of grad2, hEn and nab2.
template <typename T>
__global__ __launch_bounds__(kBlock) void k_energy(const ReplicaParams *__restrict__ P,
                                                   const ReplicaState *__restrict__ S,
                                                   LaunchBlocks blk,
                                                   int flip, EnergySlot *__restrict__ slots) {
  const int bid = blockIdx.x;
  int r, b;
  block_of(blk, r, b);
  const ReplicaParams p = P[r];
  const int cur = live(S[r]) ^ flip;
  int64_t idx = (int64_t)b * kBlock + threadIdx.x;
  double g2 = 0., hE = 0., n2 = 0.;
  if (idx < 2 * p.half) {
    const int par = idx >= p.half;
    idx -= par * p.half;
    const int N = p.N, NH = p.NH;
    const int xh = (int)(idx % NH);
    const int64_t rowi = idx / NH;
    const int y = (int)(rowi % N), z = (int)(rowi / N);
    const int x = site_x(xh, y, z, par);
    const int q = par ^ 1;
    const int64_t ixp = rowi * NH + (wrapp(x + 1, N) >> 1);
    const int64_t iyp = ((int64_t)z * N + wrapp(y + 1, N)) * NH + xh;
    const int64_t izp = ((int64_t)wrapp(z + 1, N) * N + y) * NH + xh;
    for (int s = 0; s < 4; s++) {
      const double phimid = (double)plane<T>(p, cur, s, par)[idx];
      const T *o = plane<T>(p, cur, s, q);
      double d;
      d = (double)o[izp] - phimid; g2 += d * d;
      d = (double)o[iyp] - phimid; g2 += d * d;
      d = (double)o[ixp] - phimid; g2 += d * d;
      if (s == 0) hE = phimid * p.H;
    }
    for (int s = 0; s < 3; s++) { const double v = (double)plane<T>(p, cur, 7 + s, par)[idx]; n2 += v * v; }
    for (int s = 0; s < 3; s++) { const double a = (double)plane<T>(p, cur, 4 + s, par)[idx]; n2 += a * a; }
  }
  KSum kg{g2, 0.}, kh{hE, 0.}, kn{n2, 0.};
  for (int o = 32; o > 0; o >>= 1) {
    KSum tt;
    tt.s = __shfl_xor(kg.s, o, 64); tt.c = __shfl_xor(kg.c, o, 64); ksum_merge(kg, tt);
    tt.s = __shfl_xor(kh.s, o, 64); tt.c = __shfl_xor(kh.c, o, 64); ksum_merge(kh, tt);
    tt.s = __shfl_xor(kn.s, o, 64); tt.c = __shfl_xor(kn.c, o, 64); ksum_merge(kn, tt);
  }
  __shared__ KSum sh[3][kBlock / 64];
  const int w = threadIdx.x >> 6;
  if ((threadIdx.x & 63) == 0) { sh[0][w] = kg; sh[1][w] = kh; sh[2][w] = kn; }
  __syncthreads();
  if (threadIdx.x == 0) {
    KSum a = sh[0][0], b = sh[1][0], c = sh[2][0];
    for (int i = 1; i < kBlock / 64; i++) {
      ksum_merge(a, sh[0][i]); ksum_merge(b, sh[1][i]); ksum_merge(c, sh[2][i]);
    }
    slots[bid] = EnergySlot{a.s, a.c, b.s, b.c, c.s, c.c};
  }
}

// Combines a replica's energy partials; which = 0 stores E_old, 1 stores
// E_new and applies IdealPV2::step's statistics (Stepper.cxx:37-55): if
// deltaE > 0 one uniform is drawn and compared with exp(-deltaE).
__global__ void k_energy_finish(const ReplicaParams *P, ReplicaState *S,
                                const int *blk_first, int nrep, int nblocks,
                                const EnergySlot *slots, int which, int ctr_off,
                                MonSlot *mon_ideal) {
  const int r = blockIdx.x;
  if (r >= nrep) return;
  const int b0 = blk_first[r];
  const int b1 = (r + 1 < nrep) ? blk_first[r + 1] : nblocks;
  KSum g{0, 0}, h{0, 0}, n{0, 0};
  for (int b = b0 + (int)threadIdx.x; b < b1; b += 64) {
    ksum_merge(g, KSum{slots[b].g_s, slots[b].g_c});
    ksum_merge(h, KSum{slots[b].h_s, slots[b].h_c});
    ksum_merge(n, KSum{slots[b].n_s, slots[b].n_c});
  }
  for (int o = 32; o > 0; o >>= 1) {
    KSum t;
    t.s = __shfl_xor(g.s, o, 64); t.c = __shfl_xor(g.c, o, 64); ksum_merge(g, t);
    t.s = __shfl_xor(h.s, o, 64); t.c = __shfl_xor(h.c, o, 64); ksum_merge(h, t);
    t.s = __shfl_xor(n.s, o, 64); t.c = __shfl_xor(n.c, o, 64); ksum_merge(n, t);
  }
  if (threadIdx.x != 0) return;
  const ReplicaParams &p = P[r];
  double e = 0;
  e += 0.5 / p.chi * ksum_value(n);
  e += 0.5 * ksum_value(g);
  e -= ksum_value(h);
  if (which == 0) {
    S[r].E_old = e;
    return;
  }
  S[r].E_new = e;
  const double deltaE = e - S[r].E_old;
  MonSlot &m = mon_ideal[r];
  if (deltaE > 0) {
    Xoro gg = xoro_seeded(site_key(stream_key(p.base_key, S[r].sweep_ctr + ctr_off), 0));
    const double prob = uniform01(gg);
    if (prob > exp(-deltaE)) { m.up_counts++; m.up_no++; }
    else { m.up_counts++; m.up_yes++; m.up_dS += deltaE; }
  } else {
    m.down_counts++;
    m.down_dS += deltaE;
  }
}

// ------------------------------------------------------------------------
// The end of a step (or of a single sweep): the clock, the stream counter
// and the live buffers.  The kernels of a step take the buffer flips of the
// launches before them as an argument (flip: bit 0 phi, bit 1 charges, XORed
// into the state's live bits) and this kernel applies the step's net flip.
__global__ void k_advance(ReplicaState *S, int nrep, double dt, int advance_time,
                          uint64_t nctr, int flip) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrep) return;
  if (advance_time) S[r].t += dt;
  S[r].sweep_ctr += nctr;
  S[r].cur_phi ^= flip & 1;
  S[r].cur_chg ^= (flip >> 1) & 1;
}

__global__ void k_set_time(ReplicaState *S, int nrep, int replica, double t) {
  const int r = blockIdx.x * blockDim.x + threadIdx.x;
  if (r >= nrep) return;
  if (replica < 0 || r == replica) S[r].t = t;
}

// ------------------------------------------------------------------------
// o4fields [z][y][x][10] <-> red-black planes of the live buffer.
template <typename T>
__global__ void k_aos_to_rb(const ReplicaParams *P, const ReplicaState *S, int replica,
                            int z0, int nz, const double *aos) {
  const ReplicaParams &p = P[replica];
  const int cur = live(S[replica]);
  const int N = p.N;
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // within the slab
  if (s >= (int64_t)nz * N * N) return;
  const int x = (int)(s % N);
  const int64_t yz = s / N + (int64_t)z0 * N;
  const int y = (int)(yz % N), z = (int)(yz / N);
  const int par = (x + y + z) & 1;
  const int64_t i = yz * p.NH + (x >> 1);
  for (int c = 0; c < 10; c++) plane<T>(p, cur, c, par)[i] = (T)aos[s * 10 + c];
}

template <typename T>
__global__ void k_rb_to_aos(const ReplicaParams *P, const ReplicaState *S, int replica,
                            int z0, int nz, double *aos) {
  const ReplicaParams &p = P[replica];
  const int cur = live(S[replica]);
  const int N = p.N;
  const int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;  // within the slab
  if (s >= (int64_t)nz * N * N) return;
  const int x = (int)(s % N);
  const int64_t yz = s / N + (int64_t)z0 * N;
  const int y = (int)(yz % N), z = (int)(yz / N);
  const int par = (x + y + z) & 1;
  const int64_t i = yz * p.NH + (x >> 1);
  for (int c = 0; c < 10; c++) aos[s * 10 + c] = (double)plane<T>(p, cur, c, par)[i];
}

// ------------------------------------------------------------------------
// Measurer observables of one site (measurer.cxx:245-269 and :351-392):
// o[0..10] = phi, A, V, phi^2; o[11..24] = |phi|, n, A', V', |phi|^2.
__device__ __forceinline__ void contract_rho(const double n[4], const double rho[6],
                                             double out[4]) {
  out[0] = -(n[1] * rho[0]) - n[2] * rho[1] - n[3] * rho[2];
  out[1] = n[0] * rho[0] + n[3] * rho[4] - n[2] * rho[5];
  out[2] = n[0] * rho[1] - n[3] * rho[3] + n[1] * rho[5];
  out[3] = n[0] * rho[2] + n[2] * rho[3] - n[1] * rho[4];
}

template <typename T>
__device__ __forceinline__ void site_obs(const T raw[10], double o[25]) {
  double f[10];
#pragma unroll
  for (int c = 0; c < 10; c++) o[c] = f[c] = (double)raw[c];
  double phi2 = 0.0;
#pragma unroll
  for (int l = 0; l < 4; l++) phi2 += f[l] * f[l];
  const double sigma = sqrt(phi2);
  double n[4];
  if (phi2 > 100. * DBL_MIN) {
    // f / sigma from the reciprocal with one Markstein correction: the
    // quotient rounded once, three instructions instead of ten.  Where phi2
    // overflows, inv = 0 and the residual takes a finite sigma: f / inf = 0.
    const double inv = 1. / sigma, finite = fmin(sigma, DBL_MAX);
#pragma unroll
    for (int l = 0; l < 4; l++) {
      const double q = f[l] * inv;
      n[l] = fma(fma(-q, finite, f[l]), inv, q);
    }
  } else {
    n[0] = 1; n[1] = 0; n[2] = 0; n[3] = 0;
  }
  const double rho[6] = {f[4], f[5], f[6], f[7], f[8], f[9]};
  const double drho[6] = {f[7], f[8], f[9], f[4], f[5], f[6]};
  o[10] = phi2;
  o[11] = sigma;
#pragma unroll
  for (int l = 0; l < 4; l++) o[12 + l] = n[l];
  contract_rho(n, rho, o + 16);
  contract_rho(n, drho, o + 20);
  o[24] = sigma * sigma;
}

// a += x with the rounding error of the addition collected in a.c: Knuth's
// two-sum, six additions and no comparison (ksum_add takes a branch or
// selects).  The same error term as ksum_add's.
__device__ __forceinline__ void two_sum_add(KSum &a, double x) {
  const double s = a.s + x;
  const double bx = s - a.s;
  a.c += (a.s - (s - bx)) + (x - bx);
  a.s = s;
}
__device__ __forceinline__ void ksum_xor_merge(KSum &a, int o) {
  KSum b;
  b.s = __shfl_xor(a.s, o, 64);
  b.c = __shfl_xor(a.c, o, 64);
  two_sum_add(a, b.s);
  a.c += b.c;
}

// The three walls' slice sums in one pass over the fields (measurer.cxx:
// 10-229).  A wavefront takes 64 columns (x, z), TX x TZ of them in use, and
// marches y through a chunk of CY rows: a lane keeps the 25 observables of its
// column summed over y in registers (from which the x and z walls follow), and
// each row's sums over the columns (the y wall) are taken through the
// wavefront's own LDS table, two lanes to an observable.  No wavefront waits
// for another.  All sums are compensated, by a two-sum that holds for any order
// of magnitudes (sums that started at a bias made from the first row's
// magnitudes took three operations less an addition, 256^3 FP64 444 us against
// 464, FP32 365 against 425, but were plain ones where a later row was larger).
// Partial sums, (sum, correction) pairs where a wavefront takes the nz > 1 z
// tiles of a group in turn:
//   px[(chunk, z group)][25][N][words]  over the group's planes, the chunk's rows,
//   pz[(chunk, x tile)][25][N]  over the tile's columns and the chunk's rows,
//   py[(x tile, z group)][25][N][words]  over the group's columns.
// What bounds it is bytes in flight: two rows' loads ahead of the sums at two
// wavefronts per SIMD keep 80 KB per CU under way.
constexpr int kMeasureCols = 64;
// the padding puts the rows that a half-wavefront reads at once on different banks
typedef double MeasureTable[25][kMeasureCols + 2];

template <typename T>
__global__ __launch_bounds__(kBlock) __attribute__((amdgpu_waves_per_eu(2)))
void k_measure_tile(const ReplicaParams *__restrict__ P, const ReplicaState *__restrict__ S,
                    int replica, MeasureShape sh, double *__restrict__ px,
                    double *__restrict__ py, double *__restrict__ pz) {
  __shared__ MeasureTable tab[kBlock / 64];
  const ReplicaParams &p = P[replica];
  const int cur = first_lane(live(S[replica]));
  const gbyte *phi = (const gbyte *)(cur & 1 ? p.fields[1] : p.fields[0]),
              *chg = (const gbyte *)(cur >> 1 ? p.fields[1] : p.fields[0]);
  const int N = p.N, NH = p.NH;
  const int64_t half = p.half;
  const int wave = first_lane((int)threadIdx.x >> 6), lane = threadIdx.x & 63;
  MeasureTable &q = tab[wave];
  int b = (int)blockIdx.x * (kBlock / 64) + wave;
  const int ngz = measure_groups(sh);
  if (b >= sh.ntx * ngz * sh.nch) return;  // whole wavefronts; no barrier follows
  const int bx = b % sh.ntx;
  b /= sh.ntx;
  const int gz = b % ngz, by = b / ngz;
  const int tx = lane % sh.TX, tz = lane / sh.TX;
  const int x0 = bx * sh.TX, tw = min(sh.TX, N - x0);
  const int y0 = by * sh.CY, y1 = min(y0 + sh.CY, N);
  const int words = measure_words(sh);
  double *xrow = px + (int64_t)(by * ngz + gz) * 25 * N * words;
  double *yrow = py + (int64_t)(bx * ngz + gz) * 25 * N * words;
  // adds a tile's sum to the group's, which this lane alone reads and writes
  auto put = [&](double *w, KSum a, int bz) __attribute__((always_inline)) {
    if (words == 1) {
      w[0] = ksum_value(a);
    } else {
      if (bz > gz * sh.nz) {
        two_sum_add(a, w[0]);
        a.c += w[1];
      }
      w[0] = a.s;
      w[1] = a.c;
    }
  };
  // this lane's part in the table's row sums: row k, entries s, s + 2, ...
  const int k = lane >> 1, s = lane & 1;
  // the table is written and read by one wavefront: its LDS operations stay
  // in order, and the compiler must keep them so
  auto table_ready = [] __attribute__((always_inline)) {
    __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    __builtin_amdgcn_wave_barrier();
  };
  for (int bz = gz * sh.nz; bz < min((gz + 1) * sh.nz, sh.ntz); bz++) {
    const int z0 = bz * sh.TZ, th = min(sh.TZ, N - z0);
    const int x = x0 + tx, z = z0 + tz;
    const bool own = tx < tw && tz < th, ragged = !__all(own);
    T raw[2][10];
    auto load = [&](int y, T *r) __attribute__((always_inline)) {
      // lanes without a column read site 0 and count zero
      const int64_t i = own ? ((x + y + z) & 1) * half + ((int64_t)z * N + y) * NH + (x >> 1) : 0;
#pragma unroll
      for (int c = 0; c < 10; c++)
        r[c] = reinterpret_cast<const __attribute__((address_space(1))) T *>(
            c < 4 ? phi : chg)[c * 2 * half + i];
    };
    auto observe = [&](const T *r, double *o) __attribute__((always_inline)) {
      site_obs(r, o);
      if (ragged) {
#pragma unroll
        for (int i = 0; i < 25; i++) o[i] = own ? o[i] : 0.;
      }
    };
    load(y0, raw[0]);
    if (y0 + 1 < y1) load(y0 + 1, raw[1]);
    KSum acc[25];
#pragma unroll
    for (int i = 0; i < 25; i++) acc[i] = KSum{0., 0.};
    auto take = [&](int y, T *r) __attribute__((always_inline)) {
      double o[25];
      observe(r, o);
      if (y + 2 < y1) load(y + 2, r);
#pragma unroll
      for (int i = 0; i < 25; i++) {
        q[i][lane] = o[i];
        two_sum_add(acc[i], o[i]);
      }
      table_ready();
      if (k < 25) {
        KSum a{0., 0.};
        const double *row = &q[k][s];
#pragma unroll
        for (int i = 0; i < kMeasureCols; i += 2) two_sum_add(a, row[i]);
        ksum_xor_merge(a, 1);
        if (s == 0) put(yrow + ((int64_t)k * N + y) * words, a, bz);
      }
      table_ready();
    };
    for (int y = y0; y < y1; y += 2) {
      take(y, raw[0]);
      if (y + 1 < y1) take(y + 1, raw[1]);
    }
    // the columns' sums over the chunk, then over the tile's planes / columns
#pragma unroll
    for (int i = 0; i < 25; i++) q[i][lane] = ksum_value(acc[i]);
    table_ready();
    if (tz == 0 && tx < tw) {
      for (int i = 0; i < 25; i++) {
        KSum a{0., 0.};
        for (int r = 0; r < th; r++) two_sum_add(a, q[i][r * sh.TX + tx]);
        put(xrow + ((int64_t)i * N + x) * words, a, bz);
      }
    }
    double *zrow = pz + (int64_t)(by * sh.ntx + bx) * 25 * N;
    for (int j = lane >> 3; j < 25 * th; j += 8) {  // eight lanes to a row sum
      const int i = j / th, r = j - i * th;
      KSum a{0., 0.};
      for (int c = lane & 7; c < tw; c += 8) two_sum_add(a, q[i][r * sh.TX + c]);
      ksum_xor_merge(a, 1);
      ksum_xor_merge(a, 2);
      ksum_xor_merge(a, 4);
      if ((lane & 7) == 0) zrow[(int64_t)i * N + z0 + r] = ksum_value(a);
    }
    table_ready();
  }
}

// wall_d[k][n] = (compensated sum of the partial sums of (d, k, n)) / N^2.  A
// block takes 64 consecutive n (coalesced) of one (d, k); its thread groups g
// take the partial sums g, g + kReduceGroups, ... and are merged in group order.
constexpr int kReduceGroups = 16;
__global__ __launch_bounds__(64 * kReduceGroups) void k_measure_reduce(int N, MeasureShape sh,
                                                        const double *__restrict__ px,
                                                        const double *__restrict__ py,
                                                        const double *__restrict__ pz,
                                                        double *__restrict__ wall,
                                                        double *__restrict__ wallphase,
                                                        double *__restrict__ host_wall,
                                                        double *__restrict__ host_wallphase) {
  __shared__ KSum part[kReduceGroups][64];
  const int nb = (N + 63) / 64;
  const int lane = threadIdx.x & 63, g = threadIdx.x >> 6;
  const int k = blockIdx.x / nb % 25, d = blockIdx.x / nb / 25;
  const int n = (blockIdx.x % nb) * 64 + lane;
  const int ngz = measure_groups(sh);
  const int entries = d == 0 ? sh.nch * ngz : (d == 1 ? sh.ntx * ngz : sh.nch * sh.ntx);
  const int64_t stride = 25 * (int64_t)N, at = (int64_t)k * N + n;
  KSum acc{0., 0.};
  if (n < N) {
    const double *src = d == 0 ? px : (d == 1 ? py : pz);
    if (d != 2 && measure_words(sh) == 2) {
#pragma unroll 8
      for (int e = g; e < entries; e += kReduceGroups) {
        two_sum_add(acc, src[(e * stride + at) * 2]);
        acc.c += src[(e * stride + at) * 2 + 1];
      }
    } else {
#pragma unroll 8
      for (int e = g; e < entries; e += kReduceGroups) two_sum_add(acc, src[e * stride + at]);
    }
  }
  part[g][lane] = acc;
  __syncthreads();
  if (g == 0 && n < N) {
    for (int i = 1; i < kReduceGroups; i++) ksum_merge(acc, part[i][lane]);
    const double val = ksum_value(acc) / (double)((int64_t)N * N);
    const int64_t at_wall = ((int64_t)d * 11 + k) * N + n,
                  at_phase = ((int64_t)d * 14 + (k - 11)) * N + n;
    if (k < 11) wall[at_wall] = host_wall[at_wall] = val;
    else wallphase[at_phase] = host_wallphase[at_phase] = val;
  }
}

// measurer_fft::execute_row (measurer.h:33-41): FFTW's r2c forward
// transform divided by N, out[k] = (1/N) sum_x in[x] e^{-2 pi i k x / N},
// k = 0..N/2, as a direct DFT with exactly reduced twiddles and compensated
// sums.  A block takes kDftK values of k of one row (3 x 25 rows), 16 lanes
// to each: one thread per k was a chain of N dependent sums (256^3: 24 us).
constexpr int kDftK = 16;
__global__ __launch_bounds__(256) void k_wall_dft(int N, const double *__restrict__ wall,
                                                  const double *__restrict__ wallphase,
                                                  double *__restrict__ wall_k,
                                                  double *__restrict__ wallphase_k) {
  // twiddles cos/sin(2 pi m / N), m = 0 .. N-1, once per block
  __shared__ double tc[kMaxN], ts[kMaxN];
  for (int m = threadIdx.x; m < N; m += blockDim.x) sincospi(2.0 * m / N, &ts[m], &tc[m]);
  __syncthreads();
  const int nk = N / 2 + 1, nkb = (nk + kDftK - 1) / kDftK;
  const int row = blockIdx.x / nkb;  // d*25 + obs
  const int k = (blockIdx.x % nkb) * kDftK + (threadIdx.x >> 4), l = threadIdx.x & 15;
  const int d = row / 25, o = row % 25;
  const double *in = o < 11 ? wall + ((int64_t)d * 11 + o) * N
                            : wallphase + ((int64_t)d * 14 + (o - 11)) * N;
  KSum re{0., 0.}, im{0., 0.};
  if (k < nk) {
    const int step = (int)((int64_t)k * 16 % N);
    int m = (int)((int64_t)k * l % N);  // k x mod N
    for (int x = l; x < N; x += 16) {
      two_sum_add(re, in[x] * tc[m]);
      two_sum_add(im, -(in[x] * ts[m]));
      m += step;
      if (m >= N) m -= N;
    }
  }
  for (int b = 1; b < 16; b *= 2) {
    ksum_xor_merge(re, b);
    ksum_xor_merge(im, b);
  }
  if (k < nk && l == 0) {
    double *out = o < 11 ? wall_k + (((int64_t)d * 11 + o) * nk + k) * 2
                         : wallphase_k + (((int64_t)d * 14 + (o - 11)) * nk + k) * 2;
    out[0] = ksum_value(re) / N;
    out[1] = ksum_value(im) / N;
  }
}

// ======================================================================== launchers

void launch_wall_dft(int N, const double *wall, const double *wallphase, double *wall_k,
                     double *wallphase_k, hipStream_t st) {
  const int nkb = (N / 2 + 1 + kDftK - 1) / kDftK;
  k_wall_dft<<<3 * 25 * nkb, 256, 0, st>>>(N, wall, wallphase, wall_k, wallphase_k);
}

static inline unsigned nblk(int64_t n, int b) { return (unsigned)((n + b - 1) / b); }

// W: some plane of the launch is 4 GiB or larger (64-bit element offsets).
// The same over the store mode as well (plan.stream).
#define LGV_DISPATCH_S(KERNEL, GRID, ST, ...)                                             \
  do {                                                                                    \
    if (plan.stream) {                                                                    \
      if (fp32) {                                                                         \
        if (plan.wide) KERNEL<float, true, true><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);   \
        else KERNEL<float, false, true><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);            \
      } else {                                                                            \
        if (plan.wide) KERNEL<double, true, true><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);  \
        else KERNEL<double, false, true><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);           \
      }                                                                                   \
    } else {                                                                              \
      if (fp32) {                                                                         \
        if (plan.wide) KERNEL<float, true, false><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);  \
        else KERNEL<float, false, false><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);           \
      } else {                                                                            \
        if (plan.wide) KERNEL<double, true, false><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__); \
        else KERNEL<double, false, false><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);          \
      }                                                                                   \
    }                                                                                     \
  } while (0)

#define LGV_DISPATCH(KERNEL, GRID, ST, ...)                                           \
  do {                                                                                \
    if (fp32) {                                                                       \
      if (plan.wide) KERNEL<float, true><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);       \
      else KERNEL<float, false><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);                \
    } else {                                                                          \
      if (plan.wide) KERNEL<double, true><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);      \
      else KERNEL<double, false><<<GRID, kBlock, 0, ST>>>(__VA_ARGS__);               \
    }                                                                                 \
  } while (0)

void launch_hb_phi(bool fp32, const Plan &plan, const ReplicaParams *P, ReplicaState *S,
                   int ieo, int ctr_off, int flip, MonSlot *mon, hipStream_t st) {
  LGV_DISPATCH(k_hb_phi, plan.nblocks, st, P, S, plan.blocks, ieo,
               ctr_off, flip, mon);
}

void launch_hb_sweep(const Plan &plan, const ReplicaParams *P, ReplicaState *S, int ctr_off,
                     int flip, MonSlot *mon, hipStream_t st) {
  if (plan.stream)
    k_hb_sweep<true><<<plan.nblocks, kPairBlock, 0, st>>>(P, S, plan.blocks, ctr_off, flip, mon);
  else
    k_hb_sweep<false><<<plan.nblocks, kPairBlock, 0, st>>>(P, S, plan.blocks, ctr_off, flip, mon);
}

void launch_hb_brick(bool fp32, const Plan &plan, int lds, const ReplicaParams *P,
                     ReplicaState *S, int ctr_off, int flip, MonSlot *mon, hipStream_t st) {
  if (fp32)
    k_hb_brick<float><<<plan.nblocks, kPairBlock, lds, st>>>(P, S, plan.blocks, ctr_off, flip, mon);
  else
    k_hb_brick<double><<<plan.nblocks, kPairBlock, lds, st>>>(P, S, plan.blocks, ctr_off, flip, mon);
}

void launch_hb_march(bool fp32, const Plan &plan, const ReplicaParams *P, ReplicaState *S,
                     int ieo, int ctr_off, int flip, MonSlot *mon, hipStream_t st) {
  LGV_DISPATCH_S(k_hb_march, plan.nblocks, st, P, S, plan.blocks, ieo,
               ctr_off, flip, mon);
}

void launch_charge_march(bool fp32, const Plan &plan, const ReplicaParams *P, ReplicaState *S,
                         int ixyz, int ctr_off, int flip, MonSlot *mon, hipStream_t st) {
  // the row-per-wavefront x path costs registers (3 waves per SIMD instead of
  // 4), so it is compiled in only for launches whose replicas all use it
  const int g = plan.nblocks;
#define LGV_CHARGE(TT, WW, XX)                                                         \
  k_charge_march<TT, WW, XX><<<g, kBlock, 0, st>>>(P, S, plan.blocks, ixyz, ctr_off, flip, mon)
  if (plan.xwave) {
    if (fp32) { if (plan.far) LGV_CHARGE(float, true, true); else LGV_CHARGE(float, false, true); }
    else { if (plan.far) LGV_CHARGE(double, true, true); else LGV_CHARGE(double, false, true); }
  } else {
    if (fp32) { if (plan.far) LGV_CHARGE(float, true, false); else LGV_CHARGE(float, false, false); }
    else { if (plan.far) LGV_CHARGE(double, true, false); else LGV_CHARGE(double, false, false); }
  }
#undef LGV_CHARGE
}

void launch_ideal(bool fp32, const Plan &plan, const ReplicaParams *P, ReplicaState *S,
                  int flip, hipStream_t st) {
  LGV_DISPATCH_S(k_ideal_fused, plan.nblocks, st, P, S, plan.blocks, flip, (int)plan.alternate);
}

void launch_energy(bool fp32, const Plan &plan, const ReplicaParams *P,
                   const ReplicaState *S, int flip, EnergySlot *slots, hipStream_t st) {
  if (fp32)
    k_energy<float><<<plan.nblocks, kBlock, 0, st>>>(P, S, plan.blocks, flip, slots);
  else
    k_energy<double><<<plan.nblocks, kBlock, 0, st>>>(P, S, plan.blocks, flip, slots);
}

void launch_energy_finish(int nrep, const Plan &plan, const ReplicaParams *P,
                          ReplicaState *S, const EnergySlot *slots, int which,
                          int ctr_off, MonSlot *mon_ideal, hipStream_t st) {
  k_energy_finish<<<nrep, 64, 0, st>>>(P, S, plan.blocks.first, nrep, plan.nblocks, slots,
                                       which, ctr_off, mon_ideal);
}

void launch_advance(int nrep, ReplicaState *S, double dt, int advance_time, uint64_t nctr,
                    int flip, hipStream_t st) {
  k_advance<<<nblk(nrep, 64), 64, 0, st>>>(S, nrep, dt, advance_time, nctr, flip);
}

void launch_set_time(int nrep, int replica, ReplicaState *S, double t, hipStream_t st) {
  k_set_time<<<nblk(nrep, 64), 64, 0, st>>>(S, nrep, replica, t);
}

void launch_aos_to_rb(bool fp32, const ReplicaParams *P, const ReplicaState *S, int replica,
                      int N, int z0, int nz, const double *aos, hipStream_t st) {
  const int64_t V = (int64_t)nz * N * N;
  if (fp32) k_aos_to_rb<float><<<nblk(V, 256), 256, 0, st>>>(P, S, replica, z0, nz, aos);
  else k_aos_to_rb<double><<<nblk(V, 256), 256, 0, st>>>(P, S, replica, z0, nz, aos);
}

void launch_rb_to_aos(bool fp32, const ReplicaParams *P, const ReplicaState *S, int replica,
                      int N, int z0, int nz, double *aos, hipStream_t st) {
  const int64_t V = (int64_t)nz * N * N;
  if (fp32) k_rb_to_aos<float><<<nblk(V, 256), 256, 0, st>>>(P, S, replica, z0, nz, aos);
  else k_rb_to_aos<double><<<nblk(V, 256), 256, 0, st>>>(P, S, replica, z0, nz, aos);
}

void launch_measure(bool fp32, const ReplicaParams *P, const ReplicaState *S, int replica,
                    int N, double *part, double *wall, double *wallphase, double *host_wall,
                    double *host_wallphase, hipStream_t st) {
  const MeasureShape sh = measure_shape(N);
  double *px = part, *pz = px + (int64_t)sh.nch * measure_groups(sh) * measure_words(sh) * 25 * N,
         *py = pz + (int64_t)sh.nch * sh.ntx * 25 * N;
  const unsigned tiles = (unsigned)measure_waves(sh);
  const unsigned blocks = nblk(tiles, kBlock / 64);  // a wavefront to a tile
  if (fp32) k_measure_tile<float><<<blocks, kBlock, 0, st>>>(P, S, replica, sh, px, py, pz);
  else k_measure_tile<double><<<blocks, kBlock, 0, st>>>(P, S, replica, sh, px, py, pz);
  k_measure_reduce<<<3 * 25 * ((N + 63) / 64), 64 * kReduceGroups, 0, st>>>(
      N, sh, px, py, pz, wall, wallphase, host_wall, host_wallphase);
}

}  // namespace lgv
