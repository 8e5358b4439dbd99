"""The workloads this framework is timed on, each through its public entry
points: the ModelG run loop on one lattice and on a batch of lattices, its
single sweeps, the measurement pass, and the Model A Euler--Maruyama stepper
with its adjoint.

    listed()            the fixed cases
    draw(rng)           one more case of the same ranges
    prepare(case, seed) inputs and contexts on the GPU
    run(state)          one pass, its outputs
    work(case)          bytes and operations a pass cannot do without
    exact(case, seed)   the outputs in FP64 from plain torch and numpy

Contexts run with the library's own choices of tiles and kernels, which is how
the run driver uses them.  A context's field storage is handed out as a tensor
over its device address: ten component planes (phi_0..3, A_1..3, V_1..3), each
split into its two checkerboard halves [z][y][x / 2].  That address names the
first of a replica's two buffers, which holds the live planes after an even
number of out-of-place sweeps, so the cases take even numbers of them.
"""
import math

import numpy as np
import torch

import langevina_amd as L
from langevina_amd import em as EM
from langevina_amd.autograd import modela_em_loss

# the reference's default couplings (the critical region of the O(4) model)
COUPLINGS = dict(mass0=-4.70052, lam=4.0, H=0.003, chi=5.0, gamma=1.0)
DT = 0.04
# Model A Euler--Maruyama: a quench from small fields, as bench.py --em
EM_COUPLINGS = dict(m2=-4.813, lam=1.0, H=0.01, gamma=1.0, dt=0.02)


# ------------------------------------------------------------------ cases

def listed():
    return [
        # the production run of a small lattice: 2000 steps from graphs with a
        # measurement every 20; one pass is the stretch between two of them
        dict(name="evolve_64", kind="evolve", N=64, fp32=False, steps=20, graph=10, measure=True),
        # a lattice side that is no power of two, launched step by step
        dict(name="evolve_100", kind="evolve", N=100, fp32=False, steps=4, graph=0,
             measure=False),
        # a middle-sized lattice in FP32 storage
        dict(name="evolve_128_fp32", kind="evolve", N=128, fp32=True, steps=4, graph=0,
             measure=False),
        # the headline lattice, in both storage types
        dict(name="evolve_256", kind="evolve", N=256, fp32=False, steps=2, graph=0,
             measure=False),
        dict(name="evolve_256_fp32", kind="evolve", N=256, fp32=True, steps=2, graph=0,
             measure=False),
        # the finite-size-scaling ensemble: 96 lattices stepped together, each
        # measured after ten steps
        dict(name="ensemble_96", kind="ensemble", n32=48, n48=32, n64=16, steps=10, graph=10),
        # one time step of the thermalization on the heat-bath lattice: six
        # phi sweeps (twelve half-sweeps) and nothing else
        dict(name="thermalize_32", kind="thermalize", N=32, fp32=False),
        # the sub-steppers on their own, sides that are no power of two
        dict(name="ideal_150", kind="ideal", N=150, fp32=False),
        dict(name="charge_90", kind="charge", N=90, fp32=False),
        # the measurement pass of the headline lattice
        dict(name="measure_256", kind="measure", N=256, fp32=False),
        # a training step through the Euler--Maruyama trajectory: loss and
        # gradients of 500 steps, checkpoints every 50
        dict(name="em_loss_128", kind="em_loss", N=128, nsteps=500, window=250, ckpt=50,
             gaussian=False),
        # a measurement series of a small odd lattice with Gaussian noise
        dict(name="em_series_33", kind="em_series", N=33, nsteps=100, every=10, gaussian=True),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _even(rng, lo, hi):
    return min(hi, max(lo, 2 * (_log_int(rng, lo, hi) // 2)))


def draw(rng):
    kind = rng.choice(["evolve", "evolve", "evolve", "ensemble", "thermalize", "ideal", "charge",
                       "measure", "em_loss", "em_series"])
    fp32 = rng.random() < 0.5
    if kind == "evolve":
        N = _even(rng, 24, 224)
        steps = 2 * rng.randint(1, max(1, min(10, (1 << 24) // N ** 3)))
        return dict(kind=kind, N=N, fp32=fp32, steps=steps, graph=rng.choice([0, 2]),
                    measure=rng.random() < 0.5)
    if kind == "ensemble":
        return dict(kind=kind, n32=rng.randint(4, 48), n48=rng.randint(2, 32),
                    n64=rng.randint(1, 16), steps=2 * rng.randint(1, 5), graph=rng.choice([0, 2]))
    if kind == "em_loss":
        nsteps = _log_int(rng, 40, 250)
        return dict(kind=kind, N=_log_int(rng, 16, 112), nsteps=nsteps, window=nsteps // 2,
                    ckpt=rng.randint(8, 40), gaussian=rng.random() < 0.5)
    if kind == "em_series":
        return dict(kind=kind, N=_log_int(rng, 16, 128), nsteps=_log_int(rng, 40, 250),
                    every=rng.randint(1, 20), gaussian=rng.random() < 0.5)
    return dict(kind=kind, N=_even(rng, 24, 224), fp32=fp32)


# ------------------------------------------------------------------ inputs

def _generator(seed, k=0):
    return torch.Generator(device="cuda").manual_seed((int(seed) * 1009 + k) % (1 << 62))


def _model_seed(seed, k=0):
    return (int(seed) * 101 + k) % (1 << 30)


def _fields(N, gen, chi):
    """(10, N, N, N) [component, z, y, x]: phi near the critical point (<phi^2>
    about one, nearest neighbours correlated) around a small condensate, and
    Gaussian charges of variance chi without their zero mode."""
    u = torch.randn((10, N, N, N), generator=gen, device="cuda", dtype=torch.float64)
    w = u[:4]
    nn = sum(torch.roll(w, s, d) for d in (1, 2, 3) for s in (1, -1))
    u[:4] = 0.44 * (w + 0.22 * nn)
    u[0] += 0.3
    u[4:] *= math.sqrt(chi)
    u[4:] -= u[4:].mean(dim=(1, 2, 3), keepdim=True)
    return u


def _sizes(case):
    return [32] * case["n32"] + [48] * case["n48"] + [64] * case["n64"]


def _ensemble(case, seed):
    return L.lgv.ensemble_params(_sizes(case), seed0=_model_seed(seed), **_without(COUPLINGS, "H"))


def _without(d, *keys):
    return {k: v for k, v in d.items() if k not in keys}


class _DeviceArray:
    """A context's field storage, for torch.as_tensor."""

    def __init__(self, ctx, N, fp32):
        ptr, _ = ctx.field_device_ptr()
        self.ctx = ctx
        self.__cuda_array_interface__ = {"shape": (10, 2, N, N, N // 2), "version": 2,
                                         "typestr": "<f4" if fp32 else "<f8",
                                         "data": (ptr, False)}


def prepare(case, seed):
    kind = case["kind"]
    if kind in ("em_loss", "em_series"):
        N = case["N"]
        phi0 = 0.1 * torch.randn((4, N, N, N), generator=_generator(seed), device="cuda",
                                 dtype=torch.float64)
        noise = EM.NOISE_GAUSSIAN if case["gaussian"] else EM.NOISE_UNIFORM
        state = dict(case=case, phi0=phi0, noise=noise, seed=_model_seed(seed))
        if kind == "em_loss":
            state["phi0"].requires_grad_(True)
            state["couplings"] = [torch.tensor(EM_COUPLINGS[k], dtype=torch.float64,
                                               requires_grad=True) for k in ("m2", "H", "lam")]
        else:
            c = EM_COUPLINGS
            state["stepper"] = EM.EulerMaruyama(N, c["m2"], c["lam"], c["H"], c["gamma"], c["dt"],
                                                state["seed"], case["nsteps"],
                                                math.isqrt(case["nsteps"]), noise_kind=noise)
            state["stepper"].set_stream(torch.cuda.current_stream().cuda_stream)
            state["final"] = torch.empty_like(phi0)
        return state
    if kind == "ensemble":
        ctx = L.Context(_ensemble(case, seed), precision=L.FP32)
        for r, N in enumerate(ctx.N):
            u = _fields(N, _generator(seed, r), COUPLINGS["chi"])
            ctx.set_field(u.permute(1, 2, 3, 0).contiguous().cpu().numpy(), r)
        ctx.use_graph(case["graph"])
        return dict(case=case, ctx=ctx)
    N = case["N"]
    ctx = L.Context(L.model_params(N, seed=_model_seed(seed), **COUPLINGS),
                    precision=L.FP32 if case["fp32"] else L.FP64)
    u = _fields(N, _generator(seed), COUPLINGS["chi"])
    ctx.set_field(u.permute(1, 2, 3, 0).contiguous().cpu().numpy())
    if case.get("graph"):
        ctx.use_graph(case["graph"])
    fields = torch.as_tensor(_DeviceArray(ctx, N, case["fp32"]), device="cuda")
    return dict(case=case, ctx=ctx, fields=fields)


# ------------------------------------------------------------------ a pass

def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "em_loss":
        leaves = [*state["couplings"], state["phi0"]]
        for t in leaves:
            t.grad = None
        m2, H, lam, phi0 = leaves
        loss = modela_em_loss(m2, H, lam, phi0, gamma=EM_COUPLINGS["gamma"],
                              dt=EM_COUPLINGS["dt"], nsteps=case["nsteps"],
                              window=case["window"], ckpt_every=case["ckpt"],
                              seed=state["seed"], noise_kind=state["noise"])
        loss.backward()
        return dict(loss=loss.detach(), m2=m2.grad, H=H.grad, lam=lam.grad, phi0=phi0.grad)
    if kind == "em_series":
        rows = state["stepper"].series(state["phi0"].data_ptr(), case["every"],
                                       state["final"].data_ptr())
        return dict(rows=rows, final=state["final"])
    ctx = state["ctx"]
    if kind == "evolve":
        ctx.run(DT, case["steps"])
        out = dict(fields=state["fields"])
        if case["measure"]:
            out["measured"] = ctx.measure_full()
        return out
    if kind == "ensemble":
        ctx.run(DT, case["steps"])
        return _by_size(ctx.N, [ctx.measure(r) for r in range(ctx.nrep)])
    if kind == "measure":
        return ctx.measure_full()
    if kind == "thermalize":
        for _ in range(6):
            ctx.hb_phi_step(DT / 6)
    elif kind == "ideal":
        for _ in range(2):
            ctx.ideal_step(DT / 3)
    else:
        for _ in range(2):
            ctx.charge_step(DT)
    return dict(fields=state["fields"])


def _by_size(sizes, measured):
    """Walls, phase walls and averages of the lattices, those of one size in one array."""
    out = {}
    for N in sorted(set(sizes)):
        rows = [m for n, m in zip(sizes, measured) if n == N]
        out[str(N)] = dict(zip(("wall", "wallphase", "oavg"),
                               (np.stack([r[i] for r in rows]) for i in range(3))))
    return out


# ------------------------------------------------------------------ work

# Per site of one launch-independent pass, FP64 fields: an ideal substep reads
# and writes ten values, a phi half-sweep reads four and writes the four of
# every second site, the two parities of a charge direction read and write six.
_IDEAL, _HALF_SWEEP, _CHARGE = 160, 48, 96
# Floating-point operations and, beside them, the integer operations of the
# random streams (about eleven per draw and forty per stream).
_IDEAL_OPS, _HALF_SWEEP_OPS, _CHARGE_OPS = 260, 110, 330
_STEP = 3 * _IDEAL + 12 * _HALF_SWEEP + 3 * _CHARGE
_STEP_OPS = 3 * _IDEAL_OPS + 12 * _HALF_SWEEP_OPS + 3 * _CHARGE_OPS


def work(case):
    kind = case["kind"]
    if kind == "ensemble":
        V = sum(N ** 3 for N in _sizes(case))
        return {"bytes": V * (case["steps"] * _STEP + 80) / 2,
                "flops": V * (case["steps"] * _STEP_OPS + 160)}
    V = case["N"] ** 3
    if kind == "em_loss":
        # forward 64 bytes a step; reverse: the recomputed step and the adjoint
        return {"bytes": V * case["nsteps"] * (64 + 64 + 96), "flops": V * case["nsteps"] * 520}
    if kind == "em_series":
        return {"bytes": V * case["nsteps"] * 64, "flops": V * case["nsteps"] * 180}
    size = 0.5 if case["fp32"] else 1
    if kind == "evolve":
        m = 1 if case["measure"] else 0
        return {"bytes": size * V * (case["steps"] * _STEP + m * 80),
                "flops": V * (case["steps"] * _STEP_OPS + m * 160)}
    nbytes, ops = {"measure": (80, 160), "thermalize": (12 * _HALF_SWEEP, 12 * _HALF_SWEEP_OPS),
                   "ideal": (2 * _IDEAL, 2 * _IDEAL_OPS),
                   "charge": (6 * _CHARGE, 6 * _CHARGE_OPS)}[kind]
    return {"bytes": size * V * nbytes, "flops": V * ops}


# ------------------------------------------------------------------ exact
#
# The same inputs through the algorithm in FP64 with plain torch: per-site
# xoroshiro128+ streams in int64 arithmetic (which wraps), sweeps over whole
# arrays with checkerboard masks.  Arrays are (batch, component, z, y, x).

_M64 = (1 << 64) - 1


def _s64(x):
    x &= _M64
    return x - (1 << 64) if x >> 63 else x


def _shr(x, k):
    return (x >> k) & ((1 << (64 - k)) - 1)


def _rotl(x, k):
    return (x << k) | _shr(x, 64 - k)


def _mix(z):
    """splitmix64's output function, on Python integers or int64 tensors."""
    if isinstance(z, int):
        z = ((z ^ (z >> 30)) * 0xbf58476d1ce4e5b9) & _M64
        z = ((z ^ (z >> 27)) * 0x94d049bb133111eb) & _M64
        return z ^ (z >> 31)
    z = (z ^ _shr(z, 30)) * _s64(0xbf58476d1ce4e5b9)
    z = (z ^ _shr(z, 27)) * _s64(0x94d049bb133111eb)
    return z ^ _shr(z, 31)


def _seed_word(seed):
    """The first 32-bit word of std::seed_seq{seed}."""
    m = 0xffffffff

    def T(x):
        return x ^ (x >> 27)

    r = (1664525 * T(0x8b8b8b8b) + 1) & m
    b = (1664525 * T(r) + seed) & m
    return (1566083941 * T((3 * b) & m)) & m


def _base_key(seed):
    return _mix(_seed_word(seed) ^ 0x6a09e667f3bcc909)


def _stream_key(base, counter):
    return _mix((base + _mix((counter + 0x9e3779b97f4a7c15) & _M64)) & _M64)


class _Streams:
    """One xoroshiro128+ engine per site, seeded from stream keys (batch)."""

    def __init__(self, keys, sites):
        k = torch.tensor([_s64(x) for x in keys], device="cuda").view(-1, *[1] * sites.dim())
        key = _mix(k ^ _mix(sites + _s64(0x3c6ef372fe94f82b)))
        self.s0 = key + _s64(0x01d353e5f3993bb0)
        self.s1 = (key + 1) * _s64(0x7b9c0df6cb193b20)

    def next(self, mask=None):
        """canonical doubles of the next outputs; engines outside mask stay."""
        a, b = self.s0, self.s1
        x = a + b
        b = b ^ a
        n0, n1 = _rotl(a, 55) ^ b ^ (b << 14), _rotl(b, 36)
        if mask is None:
            self.s0, self.s1 = n0, n1
        else:
            self.s0, self.s1 = torch.where(mask, n0, a), torch.where(mask, n1, self.s1)
        d = _shr(x, 32).double() * 2.0 ** 32 + (x & 0xffffffff).double()
        return (d * 2.0 ** -64).clamp(max=1 - 2.0 ** -53)

    def variance1(self):
        r3 = math.sqrt(3.0)
        return self.next() * (r3 + r3) - r3


def _lattice(N):
    """Linear site indices and parities of the lattice."""
    s = torch.arange(N ** 3, device="cuda").view(N, N, N)
    z, y, x = s // (N * N), s // N % N, s % N
    return s, (x + y + z) & 1


class _ModelG:
    """Lattices of one size in FP64: u (batch, 10, N, N, N), seeds and H per lattice."""

    def __init__(self, u, seeds, H, c=COUPLINGS):
        self.u, self.c = u, c
        self.N = u.shape[-1]
        self.H = torch.tensor(H, device="cuda", dtype=torch.float64).view(-1, 1, 1, 1)
        self.base = [_base_key(s) for s in seeds]
        self.counter = 0
        self.sites, self.parity = _lattice(self.N)

    def keys(self):
        k = [_stream_key(b, self.counter) for b in self.base]
        self.counter += 1
        return k

    def phi_step(self, dt):
        c = self.c
        lambda2, amp = 0.5 * (6.0 + c["mass0"]), math.sqrt(2.0 * dt * c["gamma"])
        for parity in (0, 1):
            g = _Streams(self.keys(), self.sites)
            phi = self.u[:, :4]
            heff = sum(torch.roll(phi, 1, d) + torch.roll(phi, -1, d) for d in (4, 3, 2))
            heff[:, 0] += self.H
            new = torch.stack([phi[:, a] + amp * g.variance1() for a in range(4)], 1)
            s0, s1 = (phi * phi).sum(1), (new * new).sum(1)
            dS = (-(heff * (new - phi)).sum(1) + lambda2 * (s1 - s0) +
                  c["lam"] / 4.0 * (s1 * s1 - s0 * s0))
            accept = ((dS < 0) | (g.next() < torch.exp(-dS))) & (self.parity == parity)
            self.u[:, :4] = torch.where(accept[:, None], new, phi)

    def rotate(self, tau):
        phi, A, V = self.u[:, :4], self.u[:, 4:7], self.u[:, 7:]
        h = 0.5 * tau / self.c["chi"]

        def quaternion(v):
            r = v.square().sum(1, keepdim=True).sqrt()
            return torch.cat([torch.cos(r), -torch.sinc(r / math.pi) * v], 1)

        def product(a, b):
            return torch.stack([
                a[:, 0] * b[:, 0] - a[:, 1] * b[:, 1] - a[:, 2] * b[:, 2] - a[:, 3] * b[:, 3],
                a[:, 0] * b[:, 1] + b[:, 0] * a[:, 1] + a[:, 2] * b[:, 3] - a[:, 3] * b[:, 2],
                a[:, 0] * b[:, 2] + b[:, 0] * a[:, 2] + a[:, 3] * b[:, 1] - a[:, 1] * b[:, 3],
                a[:, 0] * b[:, 3] + b[:, 0] * a[:, 3] + a[:, 1] * b[:, 2] - a[:, 2] * b[:, 1]], 1)

        right, left = quaternion(h * (V - A)), quaternion(-h * (V + A))
        self.u[:, :4] = product(left, product(phi, right))

    def ideal_step(self, dt):
        self.counter += 1  # the counter of the energy comparison
        self.rotate(dt / 2)
        phi = self.u[:, :4]
        S = sum(torch.roll(phi, 1, d) + torch.roll(phi, -1, d) for d in (4, 3, 2))
        for k in range(3):
            a, b = 1 + (k + 1) % 3, 1 + (k + 2) % 3
            self.u[:, 4 + k] += dt * (phi[:, 0] * S[:, k + 1] - phi[:, k + 1] * S[:, 0] -
                                      self.H * phi[:, k + 1])
            self.u[:, 7 + k] += dt * (phi[:, a] * S[:, b] - phi[:, b] * S[:, a])
        self.rotate(dt / 2)

    def orders(self):
        """Per lattice, the shuffled directions and parities of a charge sweep."""
        out = []
        for k in self.keys():
            key = _mix(k ^ _mix(0x3c6ef372fe94f82b))
            s0 = (0x01d353e5f3993bb0 + key) & _M64
            s1 = (0x7b9c0df6cb193b20 * (key + 1)) & _M64
            x = (s0 + s1) & _M64
            t = s1 ^ s0
            r0 = (((s0 << 55) | (s0 >> 9)) ^ t ^ (t << 14)) & _M64
            r1 = ((t << 36) | (t >> 28)) & _M64
            dirs, n = [0, 1, 2], x * 6 >> 64
            p = n // 3
            dirs[1], dirs[p] = dirs[p], dirs[1]
            p = n % 3
            dirs[2], dirs[p] = dirs[p], dirs[2]
            first = (r0 + r1) & _M64
            out.append((dirs, [1, 0] if first * 2 >> 64 == 0 else [0, 1]))
        return out

    def charge_step(self, dt):
        c = self.c
        rms = math.sqrt(2.0 * dt * (c["gamma"] / 3.0 * c["chi"]))
        orders = self.orders()
        for i in range(3):
            for j in range(2):
                keys = self.keys()
                for d, e in sorted({(o[0][i], o[1][j]) for o in orders}):
                    which = [b for b, o in enumerate(orders) if (o[0][i], o[1][j]) == (d, e)]
                    self.exchange(which, [keys[b] for b in which], d, e, rms)

    def exchange(self, which, keys, d, e, rms):
        g = _Streams(keys, self.sites)
        lower = self.parity == e
        dim = 3 - d  # of (batch, z, y, x)
        for comp in range(4, 10):
            a = self.u[which, comp]
            b = torch.roll(a, -1, dim)
            q = rms * g.variance1()
            dS = ((a - q) * (a - q) + (b + q) * (b + q) - a * a - b * b) / (2.0 * self.c["chi"])
            up = ~(dS < 0)
            q = torch.where(lower & (~up | (g.next(up) < torch.exp(-dS))), q, 0.0)
            self.u[which, comp] = a - q + torch.roll(q, 1, dim)

    def step(self, dt):
        for _ in range(3):
            self.ideal_step(dt / 3)
            for _ in range(2):
                self.phi_step(dt / 6)
        self.charge_step(dt)

    def planes(self):
        """The first lattice as (component, parity, z, y, x / 2)."""
        N = self.N
        z = torch.arange(N, device="cuda").view(N, 1, 1)
        y = torch.arange(N, device="cuda").view(1, N, 1)
        h = torch.arange(N // 2, device="cuda").view(1, 1, N // 2)
        out = [self.u[0].gather(3, (2 * h + ((p + y + z) & 1)).expand(10, N, N, N // 2))
               for p in (0, 1)]
        return torch.stack(out, 1)

    def walls(self, b=0):
        """Slice means: wall (3, 11, N), wallphase (3, 14, N), averages (11)."""
        u = self.u[b]
        phi, rho = u[:4], u[4:]
        phi2 = phi.square().sum(0)
        sigma = phi2.sqrt()
        n = phi / sigma

        def contract(A, V):
            return torch.stack([-(n[1] * A[0]) - n[2] * A[1] - n[3] * A[2],
                                n[0] * A[0] + n[3] * V[1] - n[2] * V[2],
                                n[0] * A[1] - n[3] * V[0] + n[1] * V[2],
                                n[0] * A[2] + n[2] * V[0] - n[1] * V[1]])

        obs = torch.cat([phi, rho, phi2[None], sigma[None], n, contract(rho[:3], rho[3:]),
                         contract(rho[3:], rho[:3]), phi2[None]])
        w = torch.stack([obs.mean((1, 2)), obs.mean((1, 3)), obs.mean((2, 3))]).cpu().numpy()
        return w[:, :11], w[:, 11:], w[0, :11].mean(1)

    def measured(self):
        wall, phase, oavg = self.walls()
        wall_k, phase_k = (np.fft.rfft(w, axis=-1) / self.N for w in (wall, phase))
        rotated = np.empty((3, 14, wall_k.shape[-1]), complex)
        for d in range(3):
            phi, A, V, phi2 = (wall_k[d, s] for s in (slice(0, 4), slice(4, 7), slice(7, 10), 10))
            n = phi[:, 0] / np.sqrt((np.abs(phi[:, 0]) ** 2).sum())

            def contract(a, v):
                return [-(n[1] * a[0]) - n[2] * a[1] - n[3] * a[2],
                        n[0] * a[0] + n[3] * v[1] - n[2] * v[2],
                        n[0] * a[1] - n[3] * v[0] + n[1] * v[2],
                        n[0] * a[2] + n[2] * v[0] - n[1] * v[1]]

            along = (n[:, None] * phi).sum(0)
            rotated[d, 0] = along
            rotated[d, 1:5] = phi - n[:, None] * along
            rotated[d, 5:9], rotated[d, 9:13], rotated[d, 13] = contract(A, V), contract(V, A), phi2
        return dict(wall=wall, wallphase=phase, oavg=oavg, wall_k=wall_k, wall_k_rotated=rotated,
                    wallphase_k=phase_k)


class _EulerMaruyama:
    """The Euler--Maruyama recursion and its adjoint on whole arrays."""

    def __init__(self, case, seed):
        self.N = case["N"]
        self.gaussian = case["gaussian"]
        self.base = _base_key(_model_seed(seed))
        self.sites = torch.arange(self.N ** 3, device="cuda").view((self.N,) * 3)
        c = EM_COUPLINGS
        self.m2, self.H, self.lam, self.gdt = c["m2"], c["H"], c["lam"], c["gamma"] * c["dt"]

    def noise(self, n):
        g = _Streams([_stream_key(self.base, (1 << 62) | n)], self.sites)
        if not self.gaussian:
            return torch.cat([g.variance1() for _ in range(4)])
        out = []
        for _ in range(2):
            u, v = g.next(), g.next()
            r, a = torch.sqrt(-2.0 * torch.log(1.0 - u)), 2.0 * math.pi * v
            out += [r * torch.cos(a), r * torch.sin(a)]
        return torch.cat(out)

    @staticmethod
    def laplacian(f):
        return sum(torch.roll(f, s, d) for d in (1, 2, 3) for s in (1, -1)) - 6.0 * f

    def step(self, phi, n):
        drift = -self.laplacian(phi) + (self.m2 + self.lam * phi.square().sum(0)) * phi
        drift[0] -= self.H
        return phi - self.gdt * drift + math.sqrt(2.0 * self.gdt) * self.noise(n)

    def adjoint(self, phi, l):
        """J^T l and the step's contributions to d/d(m2, H, lambda)."""
        s, p = phi.square().sum(0), (phi * l).sum(0)
        out = l - self.gdt * (-self.laplacian(l) + self.m2 * l +
                              self.lam * (s * l + 2.0 * phi * p))
        return out, torch.stack([-self.gdt * p.sum(), self.gdt * l[0].sum(),
                                 -self.gdt * (s * p).sum()])


def _exact_em(case, seed):
    em = _EulerMaruyama(case, seed)
    N, n = case["N"], case["nsteps"]
    V = N ** 3
    phi = 0.1 * torch.randn((4, N, N, N), generator=_generator(seed), device="cuda",
                            dtype=torch.float64)
    if case["kind"] == "em_series":
        rows = []
        for k in range(n):
            if k % case["every"] == 0:
                bar = phi.mean((1, 2, 3))
                rows.append(torch.cat([bar, phi.square().sum(0).mean()[None],
                                       V * bar.square().sum()[None]]))
            phi = em.step(phi, k)
        return dict(rows=torch.stack(rows), final=phi)
    states, bars = [], []
    for k in range(n):
        states.append(phi)
        phi = em.step(phi, k)
        bars.append(phi[0].mean())
    w = torch.stack(bars[n - case["window"]:])
    loss = w.mean() + V * (w - w.mean()).square().mean()
    l, grads = torch.zeros_like(phi), torch.zeros(3, device="cuda", dtype=torch.float64)
    for k in range(n - 1, -1, -1):
        at = k - (n - case["window"])
        if at >= 0:
            l[0] += (1.0 / V + 2.0 * (w[at] - w.mean())) / case["window"]
        l, g = em.adjoint(states.pop(), l)
        grads += g
    return dict(loss=loss, m2=grads[0], H=grads[1], lam=grads[2], phi0=l)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("em_loss", "em_series"):
        return _exact_em(case, seed)
    if kind == "ensemble":
        sizes, params = _sizes(case), _ensemble(case, seed)
        measured = [None] * len(sizes)
        for N in sorted(set(sizes)):
            which = [r for r, n in enumerate(sizes) if n == N]
            u = torch.stack([_fields(N, _generator(seed, r), COUPLINGS["chi"]) for r in which])
            m = _ModelG(u.float().double(), [params[r].seed for r in which],
                        [params[r].H for r in which])
            for _ in range(case["steps"]):
                m.step(DT)
            for b, r in enumerate(which):
                measured[r] = m.walls(b)
        return _by_size(sizes, measured)
    u = _fields(case["N"], _generator(seed), COUPLINGS["chi"])
    u = u.float().double() if case["fp32"] else u
    m = _ModelG(u[None], [_model_seed(seed)], [COUPLINGS["H"]])
    if kind == "measure":
        return m.measured()
    if kind == "evolve":
        for _ in range(case["steps"]):
            m.step(DT)
        out = dict(fields=m.planes())
        if case["measure"]:
            out["measured"] = m.measured()
        return out
    for _ in range({"thermalize": 6, "ideal": 2, "charge": 2}[kind]):
        {"thermalize": m.phi_step, "ideal": m.ideal_step,
         "charge": m.charge_step}[kind]({"thermalize": DT / 6, "ideal": DT / 3, "charge": DT}[kind])
    return dict(fields=m.planes())
