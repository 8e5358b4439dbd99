"""The library's own tiles (no request) on sides where their rules split rows
and chunks differently, against fixed tiles: a tile does not change a bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def L():
    import torch
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    import langevina_amd
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
    out = []
    for kernel in (L.PHI_SITE, L.PHI_MARCH):
        ctx = L.Context(L.model_params(N, seed=5), precision=prec)
        ctx.set_phi_kernel(kernel)
        ctx.set_field(u)
        ctx.run(0.04, 1)
        out.append((ctx.get_field(), ctx.monitors()["phi"]))
        ctx.close()
    np.testing.assert_array_equal(out[0][0], out[1][0])
    for k in ("down_counts", "up_counts", "up_yes", "up_no"):
        assert out[0][1][k] == out[1][1][k], k


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
