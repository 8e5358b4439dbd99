"""The rules that choose shapes by size (langevina_amd/csrc/lgv_internal.h and
lgv_em_tile.h), compiled as they stand: what they give over the whole range of sides."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIP_INCLUDE = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    """rule(body): runs a C++ main body with the header and returns the rows
    of numbers it prints."""
    def run(body):
        d = tmp_path_factory.mktemp("rules")
        src, exe = d / "rules.cpp", d / "rules"
        src.write_text('#include <cstdio>\n#include "lgv_em_tile.h"\n#include "lgv_internal.h"\nusing namespace lgv;\n'
                       "int main() {\n" + body + "\n}\n")
        subprocess.run(["g++", "-std=c++17", "-O1", "-D__HIP_PLATFORM_AMD__", "-I", HIP_INCLUDE,
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "langevina_amd", "csrc"), str(src), "-o",
                        str(exe)], check=True, capture_output=True, text=True)
        out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
        return [[int(v) for v in line.split()] for line in out.splitlines()]
    return run


def test_measurement_fills_the_gpu_at_every_side(rule):
    rows = rule("""
  for (int N = 4; N <= kMaxN; N += 2) {
    const MeasureShape s = measure_shape(N);
    printf("%d %d %d %d %d %d %d %d %lld %lld\\n", N, s.TX, s.TZ, s.nz, s.CY, s.ntx, s.ntz, s.nch,
           (long long)measure_part(s, N), (long long)measure_part_limit(N));
  }""")
    assert len(rows) == (1536 - 4) // 2 + 1
    for N, TX, TZ, nz, CY, ntx, ntz, nch, part, limit in rows:
        assert TX * TZ <= 64 and nz >= 1 and CY >= 1, N
        for n, tiles, size in ((N, ntx, TX), (N, ntz, TZ), (N, nch, CY)):
            assert (tiles - 1) * size < n <= tiles * size, N
        assert part <= limit == 50 * max(2 ** 19, N * N), N
        # wavefronts: what the GPU holds, of a lattice that has them, or nearly
        # that with no second round of a few
        waves = ntx * -(-ntz // nz) * nch
        assert waves >= (1700 if N >= 128 else min(16 * N, ntx * ntz * N)), (N, waves)
        if nz > 1:
            assert -(-waves // 2048) * 2048 <= 1.25 * waves, (N, waves)


def test_a_block_of_both_parities_owns_two_rows_or_none(rule):
    rows = rule("""
  for (int N = 4; N <= kMaxN; N += 2) printf("%d %d\\n", N, pair_march_rows(N));""")
    for N, own in rows:
        threads = (own + 2) * (N // 2)
        assert own == 0 if N > 512 else 2 <= own <= N and threads <= 1024, N


def test_charge_tiles_of_large_lattices_are_whole_units(rule):
    """Where the fields exceed the 256 MiB cache and a row is whole 64-byte units,
    a tile is too, with most lanes at work; elsewhere rows split evenly."""
    rows = rule("""
  for (int N = 4; N <= kMaxN; N += 2)
    for (int f = 0; f < 2; f++) printf("%d %d %d\\n", N, f, charge_width(N / 2, f));""")
    for N, fp32, w in rows:
        NH, esz = N // 2, 4 if fp32 else 8
        n = -(-NH // w)
        if NH > 64 and 10 * N ** 3 * esz > 2 ** 28 and NH * esz % 64 == 0:
            assert w in (48, 64) and w * esz % 64 == 0, (N, fp32)
            assert n == -(-NH // 64), (N, fp32)
        else:
            assert w <= 64 and n == -(-NH // 64) and w * n - NH < n, (N, fp32)


def test_ideal_tiles_of_large_lattices_are_whole_units(rule):
    """Where a lattice's fields exceed twice the 256 MiB cache and a row is whole
    64-byte units, an ideal tile's rows are too (and FP64 ones are then stored
    past the caches); every tile fits the kernel's plane grid."""
    rows = rule("""
  for (int N = 4; N <= kMaxN; N += 2)
    for (int f = 0; f < 2; f++) {
      const int w = ideal_width(N, f);
      int TXH, TY, TZ;
      ideal_tile(N, w, 1, TXH, TY, TZ);
      printf("%d %d %d %d %d %d %d\\n", N, f, w, TXH, TY, ideal_lds(f), ideal_unit(N, f));
    }""")
    for N, fp32, w, TXH, TY, lds, unit in rows:
        NH, esz = N // 2, 4 if fp32 else 8
        assert (TY + 2) * (2 * TXH + 2) <= lds and TXH == min(w, NH), (N, fp32)
        large = 10 * N ** 3 * esz > 2 ** 29
        assert unit == (64 if large and not fp32 else 128), (N, fp32)
        if large and NH * esz % 64 == 0:
            assert w * esz % 64 == 0, (N, fp32, w)


def test_ideal_chunks_alternate_where_neighbours_run_together(rule):
    rows = rule("""
  for (int N = 4; N <= kMaxN; N += 2)
    for (int f = 0; f < 2; f++) {
      const int w = ideal_width(N, f);
      printf("%d %d %lld %d %d\\n", N, f, (long long)ideal_plane_blocks(N, w), ideal_slots(f),
             ideal_alternates(N, w, f));
    }""")
    for N, fp32, plane, slots, alternate in rows:
        assert alternate == (2 * plane <= slots), (N, fp32)
        assert alternate or N > 256, (N, fp32)
        assert not alternate or N < 512, (N, fp32)


def test_euler_maruyama_tiles(rule):
    """Rows of whole 64-byte units are split into such tiles; every tile fits the
    kernels' plane and its ring the block's threads; a step of a side up to 256
    fits the 8192 slots of the call without a handle."""
    rows = rule("""
  for (int N = 4; N <= 1024; N++) {
    int TX, TY, TZ;
    em_tile(N, TX, TY, TZ);
    printf("%d %d %d %d %d %d\\n", N, TX, TY, TZ, em_blocks(N), em_alternates(N, TX, TY));
  }""")
    for N, TX, TY, TZ, blocks, alternate in rows:
        assert (TY + 2) * (TX + 2) <= 400 and TX * TY <= 256 and 2 * (TX + TY) <= 256, N
        assert 1 <= TZ <= N and TX <= N and TY <= N, N
        even = -(-N // -(-N // 64))
        lanes = min(N, 256 // TX) / -(-N // TX)
        if N >= 100 and N % 8 == 0:
            assert TX in (48, 64) or (TX == even and lanes > 1.1 * max(5 / -(-N // 48),
                                                                      4 / -(-N // 64))), N
            assert lanes >= 0.9 * (256 // even) / -(-N // even), N
        else:
            assert TX == even, N
        plane = -(-N // TX) * -(-N // TY)
        assert blocks == plane * -(-N // TZ), N
        assert N > 256 or blocks <= 8192, N
        assert alternate == (2 * plane <= 1024), N


def test_half_sweeps_of_one_fp64_lattice_march_from_196_on(rule):
    rows = rule("""
  printf("%lld %lld %lld\\n", (long long)phi_march_sites(false, 1),
         (long long)phi_march_sites(true, 1), (long long)phi_march_sites(false, 60));""")
    one64, one32, batch64 = rows[0]
    assert 194 ** 3 < one64 <= 200 ** 3
    assert 180 ** 3 < one32 <= 192 ** 3
    assert batch64 == one32


def test_charge_factor_is_a_float_or_nan(rule):
    """-log2(e) / 2 chi: NaN outside 2^-100 .. 2^100, else within a float's
    rounding (relative error in units of 2^-26)."""
    rows = rule("""
  for (int e = -1000; e <= 1000; e++)
    for (int m = 8; m < 16; m++) {
      const double chi = __builtin_ldexp((double)m, e - 4), l2 = charge_l2(chi);
      const double ref = -1.4426950408889634 / (2. * chi);
      printf("%d %d %d %d\\n", e, m, l2 != l2,
             l2 != l2 ? 0 : (int)(67108864. * __builtin_fabs(l2 / ref - 1.)));
    }""")
    for e, m, nan, err in rows:
        d = m * 2.0 ** (e - 3)
        assert nan == (not 2.0 ** -100 <= d <= 2.0 ** 100), (e, m)
        assert err <= 4, (e, m)
