"""The Euler--Maruyama marches on sides where their tiles, depths and march
directions differ, against the recursion in torch, and the reverse pass with
the last segment's states kept from the forward run and recomputed."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu
PAR = dict(m2=-1.2, lam=1.1, H=0.02, gamma=0.9, dt=0.01, seed=11)


@pytest.fixture(scope="module")
def torch():
    torch = pytest.importorskip("torch")
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    return torch


def stepper(N, nsteps, ckpt, noise):
    from langevina_amd.em import EulerMaruyama
    return EulerMaruyama(N, PAR["m2"], PAR["lam"], PAR["H"], PAR["gamma"], PAR["dt"], PAR["seed"],
                         nsteps, ckpt, noise_kind=noise)


def drift_step(torch, phi):
    """One step without its noise."""
    nb = sum(torch.roll(phi, s, d) for d in (1, 2, 3) for s in (1, -1))
    out = phi - PAR["gamma"] * PAR["dt"] * (-(nb - 6 * phi) + PAR["m2"] * phi +
                                            PAR["lam"] * (phi ** 2).sum(0) * phi)
    out[0] += PAR["gamma"] * PAR["dt"] * PAR["H"]
    return out


# 4, 5: one tile wraps onto itself; 33, 64: one-plane chunks; 66: rows of 33, chunks
# of two; 80, 97: chunks of four, the last one short; 130: chunks of eight, the
# last of two planes, marched in either direction
@pytest.mark.parametrize("noise", [0, 1])
@pytest.mark.parametrize("N", [4, 5, 33, 64, 66, 80, 97, 130])
def test_the_difference_of_two_runs_is_the_drift(torch, N, noise):
    """Two states stepped with the same noise differ by the difference of
    their drift steps, whatever the noise: rounding of a dozen operations on
    values of a few units."""
    print(f"[gpu-test] em tiles {N} {noise}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(N)
    a, b = (torch.randn((4, N, N, N), generator=g, device="cuda", dtype=torch.float64)
            for _ in range(2))
    outs = []
    h = stepper(N, 4, 2, noise)  # steps on its own stream
    for phi in (a, b):
        out = torch.empty_like(phi)
        obs = torch.empty(6, device="cuda", dtype=torch.float64)
        torch.cuda.synchronize()
        h.step(phi.data_ptr(), out.data_ptr(), 3, obs.data_ptr())
        torch.cuda.synchronize()
        mean = out.mean((1, 2, 3))
        assert (obs[:4] - mean).abs().max().item() <= 1e-14
        outs.append(out)
    h.close()
    diff = (outs[0] - outs[1]) - (drift_step(torch, a) - drift_step(torch, b))
    assert diff.abs().max().item() <= 64 * np.finfo(float).eps * max(a.abs().max().item(), 1) ** 3


@pytest.mark.parametrize("nsteps,ckpt", [(7, 3), (6, 3), (5, 8), (4, 1)])
def test_kept_and_recomputed_states_give_the_same_gradients(torch, nsteps, ckpt):
    """The first backward call after a forward run uses the states that run
    left, the second recomputes every segment but the first; a series in
    between takes the room of the kept states."""
    print(f"[gpu-test] em segments {nsteps} {ckpt}", flush=True)
    N = 12
    phi = torch.randn((4, N, N, N), device="cuda", dtype=torch.float64)
    torch.cuda.synchronize()
    h = stepper(N, nsteps, ckpt, 0)  # runs on its own stream and waits for it
    got = []
    for between in (False, True, False):
        if not got or between:
            h.forward(phi.data_ptr(), nsteps)
        if between:
            h.series(phi.data_ptr(), 2)
        grad = torch.zeros_like(phi)
        torch.cuda.synchronize()
        par = h.backward(grad.data_ptr())
        got.append((grad.cpu().numpy(), par))
    h.close()
    for grad, par in got[1:]:
        np.testing.assert_array_equal(grad, got[0][0])
        np.testing.assert_array_equal(par, got[0][1])


# Rows of whole 64-byte units in tiles of 64 and 48 sites: 104: 64 and 40; 136: 48,
# 48, 40; 240: five of 48; 352: six of 64, the last of 32, every chunk marched upwards
WHOLE = [104, 136, 240, 352]


@pytest.mark.parametrize("N", WHOLE)
def test_tiles_of_whole_units_give_the_drift(torch, N):
    test_the_difference_of_two_runs_is_the_drift(torch, N, 0)


@pytest.mark.parametrize("N", WHOLE)
def test_tiles_of_whole_units_give_the_adjoint(torch, N):
    """Two steps, the loss phibar_0 of the last state: the gradient is
    J(phi_0) J(phi_1) e_0 / V with the one-step Jacobian J, which is symmetric."""
    print(f"[gpu-test] em adjoint tiles {N}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(N)
    phi0 = torch.randn((4, N, N, N), generator=g, device="cuda", dtype=torch.float64)
    phi1, grad = torch.empty_like(phi0), torch.empty_like(phi0)
    torch.cuda.synchronize()
    h = stepper(N, 2, 2, 0)
    h.forward(phi0.data_ptr(), 1)
    h.backward(grad.data_ptr())
    h.step(phi0.data_ptr(), phi1.data_ptr(), 0)
    torch.cuda.synchronize()
    h.close()
    gdt, big = PAR["gamma"] * PAR["dt"], 0.
    lam = torch.zeros_like(phi0)
    lam[0] = 1. / N ** 3
    for phi in (phi1, phi0):
        lap = sum(torch.roll(lam, s, d) for d in (1, 2, 3) for s in (1, -1)) - 6 * lam
        lam = lam - gdt * (-lap + PAR["m2"] * lam + PAR["lam"] * (
            (phi ** 2).sum(0) * lam + 2 * phi * (phi * lam).sum(0)))
        big = max(big, (phi ** 2).sum(0).max().item())
    # a dozen operations a step on terms of up to (1 + gdt 3 lambda |phi|^2) / V
    tol = 64 * np.finfo(float).eps * (1 + 3 * gdt * PAR["lam"] * big) ** 2 / N ** 3
    assert (grad - lam).abs().max().item() <= tol
