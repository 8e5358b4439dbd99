"""The library's own tiles (no request) on sides where their rules split rows
and chunks differently, against fixed tiles: a tile does not change a bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    import langevina_amd
    langevina_amd.lib()
    return langevina_amd


# 6: one tile wraps onto itself; 22, 50, 90: one x tile, a last row tile or
# chunk that is short; 66, 104: rows of 33 and 52 half-columns; 130, 150: rows
# split in two; FP32 holds narrower ideal tiles
@pytest.mark.parametrize("N,prec", [(6, 0), (22, 1), (50, 0), (66, 1), (90, 0), (104, 1),
                                    (130, 0), (150, 1)])
def test_default_tiles_keep_results(L, N, prec):
    print(f"[gpu-test] default tiles {N} {prec}", flush=True)
    from langevina_amd.autotune import set_ideal_tile, set_sweep_tiles
    u = np.random.default_rng(N).normal(size=(N, N, N, 10)) * 0.5
    out = []
    for fixed in (False, True):
        ctx = L.Context(L.model_params(N, seed=3), precision=prec)
        if fixed:
            set_ideal_tile(ctx, 0, 16, 8)
            set_sweep_tiles(ctx, 0, 0, 0, 16, 8 if N >= 8 else 2)
        ctx.set_field(u)
        ctx.run(0.04, 3)  # three shuffles of the sweep directions
        out.append((ctx.get_field(), ctx.monitors()))
        ctx.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    for kind in ("phi", "charge"):
        for k in ("down_counts", "up_counts", "up_yes", "up_no"):
            assert out[0][1][kind][k] == out[1][1][kind][k], (kind, k)


def test_default_tiles_of_a_mixed_batch_keep_results(L):
    """Replicas of several sides share one launch and one choice of depths:
    each gives the bits it gives alone."""
    print("[gpu-test] default tiles, batch", flush=True)
    sizes = [8, 22, 64, 34]
    reps = [L.model_params(N, seed=7 + i) for i, N in enumerate(sizes)]
    us = [np.random.default_rng(N).normal(size=(N, N, N, 10)) * 0.5 for N in sizes]
    ctx = L.Context(reps)
    for r, u in enumerate(us):
        ctx.set_field(u, r)
    ctx.run(0.04, 2)
    for r, u in enumerate(us):
        one = L.Context(reps[r])
        one.set_field(u)
        one.run(0.04, 2)
        np.testing.assert_array_equal(ctx.get_field(r), one.get_field(), err_msg=str(sizes[r]))
        one.close()
    ctx.close()


# The phi march's own tiles against the per-site kernel: 34: one row of 17
# half-columns in tiles of 15 rows; 66, 90: rows of 33 and 45, not a multiple
# of eight blocks per plane; 140: two tiles of 35; 208: two of 64, the second
# 40 wide, and (FP64) large enough for non-temporal stores
@pytest.mark.parametrize("N,prec", [(34, 0), (66, 1), (90, 0), (140, 1), (208, 0)])
def test_phi_kernels_agree_on_default_tiles(L, N, prec):
    print(f"[gpu-test] phi kernels {N} {prec}", flush=True)
    u = np.random.default_rng(N).normal(size=(N, N, N, 10)) * 0.5
    ref = None
    for kernel in (L.PHI_SITE, L.PHI_MARCH, L.PHI_AUTO):
        ctx = L.Context(L.model_params(N, seed=5), precision=prec)
        ctx.set_phi_kernel(kernel)
        ctx.set_field(u)
        ctx.run(0.04, 1)
        got, mon = ctx.get_field(), ctx.monitors()["phi"]
        ctx.close()
        ref = ref or (got, mon)
        np.testing.assert_array_equal(ref[0], got)
        for k in ("down_counts", "up_counts", "up_yes", "up_no"):
            assert ref[1][k] == mon[k], k


def test_phi_march_of_a_mixed_batch_keeps_results(L):
    """Replicas that go to one XCD as a whole and replicas that are cut into
    bands in one launch."""
    print("[gpu-test] phi march, batch", flush=True)
    sizes = [66] + [12] * 30 + [34]
    us = [np.random.default_rng(i).normal(size=(N, N, N, 10)) * 0.5 for i, N in enumerate(sizes)]
    out = []
    for kernel in (L.PHI_SITE, L.PHI_MARCH):
        ctx = L.Context([L.model_params(N, seed=7 + i) for i, N in enumerate(sizes)])
        ctx.set_phi_kernel(kernel)
        for r, u in enumerate(us):
            ctx.set_field(u, r)
        ctx.run(0.04, 1)
        out.append([ctx.get_field(r) for r in range(len(sizes))])
        ctx.close()
    for r, N in enumerate(sizes):
        np.testing.assert_array_equal(out[0][r], out[1][r], err_msg=f"{r}: {N}")
    for r in (0, 5, 31):
        one = L.Context(L.model_params(sizes[r], seed=7 + r))
        one.set_field(us[r])
        one.run(0.04, 1)
        np.testing.assert_array_equal(out[1][r], one.get_field(), err_msg=str(r))
        one.close()


# Launches of both parities (1: bricks, 2: the march) against half-sweeps.  6:
# the block's rows are the lattice, so its facing rows are its own; 22, 34, 50:
# short last blocks and wavefronts with lanes that have no site or straddle
# rows; 64: one brick per CU; 130: rows of 65, 13 of them a block
@pytest.mark.parametrize("N,prec", [(6, 0), (6, 1), (22, 0), (34, 1), (50, 0), (64, 0), (64, 1),
                                    (130, 0)])
@pytest.mark.parametrize("scounts", [(2, 3), (3, 1)])  # 3: a pair and one in place
def test_two_parity_launches_keep_results(L, monkeypatch, N, prec, scounts):
    print(f"[gpu-test] both parities {N} {prec} {scounts}", flush=True)
    u = np.random.default_rng(N).normal(size=(N, N, N, 10)) * 0.5
    out = []
    for pairs, wide in (("0", "0"), ("1", "0"), ("1", "1"), ("2", "0"), ("2", "1")):
        monkeypatch.setenv("LGV_PHI_PAIRS", pairs)
        monkeypatch.setenv("LGV_FORCE_WIDE", wide)
        ctx = L.Context(L.model_params(N, seed=5), precision=prec, scounts=scounts)
        ctx.set_field(u)
        ctx.run(0.04, 2)
        ctx.set_phi_kernel(L.PHI_SITE)  # folds the counts, no pairs
        ctx.hb_phi_step(0.01)
        ctx.set_phi_kernel(L.PHI_AUTO)
        ctx.run(0.04, 1)
        out.append((ctx.get_field(), ctx.monitors(), ctx.rng_state().sweep_ctr))
        ctx.close()
    for got in out[1:]:
        np.testing.assert_array_equal(out[0][0], got[0])
        assert out[0][2] == got[2]
        for k in ("down_counts", "up_counts", "up_yes", "up_no"):
            assert out[0][1]["phi"][k] == got[1]["phi"][k], k


def test_two_parity_launches_of_a_batch_keep_results(L, monkeypatch):
    print("[gpu-test] both parities, batch", flush=True)
    sizes = [34, 8, 8, 8, 22]
    out = []
    for pairs in ("0", "1", "2"):
        monkeypatch.setenv("LGV_PHI_PAIRS", pairs)
        ctx = L.Context([L.model_params(N, seed=7 + i) for i, N in enumerate(sizes)])
        for r, N in enumerate(sizes):
            ctx.set_field(np.random.default_rng(r).normal(size=(N, N, N, 10)) * 0.5, r)
        ctx.run(0.04, 2)
        out.append([(ctx.get_field(r), ctx.monitors(r)["phi"]["up_yes"]) for r in range(5)])
        ctx.close()
    for got in out[1:]:
        for r in range(5):
            np.testing.assert_array_equal(out[0][r][0], got[r][0], err_msg=str(r))
            assert out[0][r][1] == got[r][1]


def test_sweep_counters_of_mixed_calls(L):
    """Each call takes its streams from the counter that the calls before it
    left, whether the host or the replicas hold it: the same call alone, on a
    new context with that counter set, gives the same field."""
    print("[gpu-test] sweep counters", flush=True)
    N, dt = 12, 0.03
    calls = ["phi", "phi", "ideal", "phi", "charge", "phi", "step", "phi", "run", "graph",
             "phi", "set", "phi", "graph"]
    takes = {"phi": 2, "ideal": 1, "charge": 7, "step": 22, "run": 44, "graph": 66, "set": 0}

    def call(ctx, what):
        if what == "phi":
            ctx.hb_phi_step(dt)
        elif what == "ideal":
            ctx.ideal_step(dt)
        elif what == "charge":
            ctx.charge_step(dt)
        elif what == "step":
            ctx.step(dt)
        elif what == "set":
            ctx.set_rng_state(ctx.rng_state())
        else:
            ctx.use_graph(2 if what == "graph" else 0)
            ctx.run(dt, 3 if what == "graph" else 2)
            ctx.use_graph(0)

    ctx = L.Context(L.model_params(N, seed=8))
    ctx.set_field(np.random.default_rng(2).normal(size=(N, N, N, 10)) * 0.5)
    counter = ctx.rng_state().sweep_ctr
    for what in calls:
        before, state = ctx.get_field(), ctx.rng_state()
        assert state.sweep_ctr == counter, what
        call(ctx, what)
        one = L.Context(L.model_params(N, seed=8))
        one.set_field(before)
        one.set_rng_state(state)
        call(one, what)
        np.testing.assert_array_equal(ctx.get_field(), one.get_field(), err_msg=what)
        one.close()
        counter += takes[what]
    assert ctx.rng_state().sweep_ctr == counter
    # and all of them with nothing read in between
    one = L.Context(L.model_params(N, seed=8))
    one.set_field(np.random.default_rng(2).normal(size=(N, N, N, 10)) * 0.5)
    for what in calls:
        call(one, what)
    oavg = one.measure()[2]
    np.testing.assert_array_equal(oavg, ctx.measure()[2])
    np.testing.assert_array_equal(ctx.get_field(), one.get_field())
    one.close()
    ctx.close()


# Lattices large enough for tiles of whole 64-byte units, against tiles of 16: 176:
# charge tiles of 48 and 40; 208: charge 64 and 40, ideal 56 and 48 stored past the
# caches; 224 FP32: charge 64 and 48; 272: ideal and charge 48, 48, 40; 288 FP32:
# ideal four of 32 and 16; 336: against ideal tiles of 40, whose chunks do not
# alternate
@pytest.mark.parametrize("N,prec,tile", [(176, 0, (16, 8)), (208, 0, (16, 8)), (224, 1, (16, 8)),
                                         (272, 0, (16, 8)), (288, 1, (16, 8)), (336, 0, (40, 8))])
def test_tiles_of_whole_units_keep_results(L, N, prec, tile):
    print(f"[gpu-test] whole-unit tiles {N} {prec}", flush=True)
    from langevina_amd.autotune import set_ideal_tile, set_sweep_tiles
    u = np.random.default_rng(N).normal(size=(N, N, N, 10)) * 0.5
    out = []
    for fixed in (False, True):
        ctx = L.Context(L.model_params(N, seed=3), precision=prec)
        if fixed:
            set_ideal_tile(ctx, 0, *tile)
            set_sweep_tiles(ctx, 0, 0, 0, 16, 8)
        ctx.set_field(u)
        ctx.run(0.04, 2)
        out.append((ctx.get_field(), ctx.monitors()["charge"], ctx.ideal_tile()))
        ctx.close()
    assert out[0][2] != out[1][2] == tile
    np.testing.assert_array_equal(out[0][0], out[1][0])
    for k in ("down_counts", "up_counts", "up_yes", "up_no"):
        assert out[0][1][k] == out[1][1][k], k
