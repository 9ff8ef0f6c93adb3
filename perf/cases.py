"""The work this library is used for, as cases that can be timed and compared.

A case is a dict of plain values. `prepare` makes what a user's program has in hand before the call (a
context loaded with a mid-run state, a trained network), `run` is one pass through the public entry
points, `exact` is the same pass in float64 with plain torch, `work` what a pass cannot do without.

Kinds of cases:
  particles  `steps` fixed-step substeps of one scene, then its state read back (a frame of a simulation)
  batch      the same for several independent scenes in one context
  cloth      the same for a sand block and a cloth in one context, the mesh read back as well
  solve      one 1/60 s frame of the adaptive loop, then the state
  gradient   loss gradient of the return-map network from and to device memory
  train      one epoch of the network's training on logged (trial, projected) pairs

The initial states are those of a running simulation, not of a fresh lattice: jittered particles, a
smooth velocity field with its affine momenta, strains that grow with the depth below the surface (so
that sand has elastic, cone, tip and near-apex particles), accumulated plastic amounts.
"""
import ctypes
import functools
import math

import numpy as np
import torch

from anisotropicelastoplasticity_amd import Solver, _lib, scenes
from anisotropicelastoplasticity_amd.api import levelset

GRAVITY = 9.8
STATE = (("x", 3), ("v", 3), ("B", 9), ("F", 9), ("plastic", 1), ("volume", 1))


def listed():
    return [
        # A user trying a scene out in the reference's own mode: cubic splines, stress at the predicted
        # F, the reference's friction, hardening angle, z up. Launches and host time count.
        dict(name="tiny_reference", kind="particles", material="sand", order=3, predicted=True, friction="reference",
             phi="hardening", res="24x24x24", cells="6x6x5", fill=1.0, dt=2e-4, steps=20, z_up=True),
        # The plain snow block on 64^3 (32,768 particles).
        dict(name="snow_block", kind="particles", material="snow", order=2, predicted=False, friction="sticky",
             phi="constant", res="64x64x64", cells="16x16x16", fill=1.0, dt=1e-4, steps=30),
        # The sand column on 128^3: 2^20 particles, about 21 per cell, the ordinary production run.
        dict(name="sand_column", kind="particles", material="sand", order=2, predicted=False, friction="coulomb",
             phi="constant", res="128x128x128", cells="32x128x32", fill=0.727, dt=5e-5, steps=30),
        # The largest scene: 2^22 sand particles with their own friction angles on 256^3, launch shapes
        # from the autotuner.
        dict(name="sand_phi", kind="particles", material="sand", order=2, predicted=False, friction="coulomb",
             phi="particle", res="256x256x256", cells="64x128x64", fill=1.0, dt=5e-5, steps=20, tuned=True),
        # The same scene with the learned return map (BF16 network, gate, exact fallback).
        dict(name="sand_phi_surrogate", kind="particles", material="sand", order=2, predicted=False, friction="coulomb",
             phi="particle", res="256x256x256", cells="64x128x64", fill=1.0, dt=5e-5, steps=8, tuned=True,
             surrogate=True),
        # The reference's mode at a production size, odd resolutions and a ragged lattice.
        dict(name="reference_mode", kind="particles", material="sand", order=3, predicted=True, friction="reference",
             phi="hardening", res="97x89x103", cells="37x35x31", fill=0.93, dt=1e-4, steps=16, z_up=True),
        # Sand falling on a cloth: about 500k particles and a 256 x 256-vertex mesh on 128^3.
        dict(name="cloth_sand", kind="cloth", res="128x128x128", cells="40x39x40", n_side=256, dt=2e-5, steps=30),
        # Many small scenes in one context: snow and sand, 64^3 to 112^3.
        dict(name="batch", kind="batch", scenes=16, n_min=20000, n_max=300000, dt=5e-5, steps=20),
        # One frame of the adaptive loop, as the reference's solve(), on a spinning block of soft snow in free flight.
        dict(name="solve_frame", kind="solve", material="snow", order=2, predicted=False, friction="coulomb",
             phi="constant", res="64x64x64", cells="21x23x22", fill=1.0, cfl=0.05),
        # Online training: the allocation-free gradient of a small batch in device memory.
        dict(name="gradient_2048", kind="gradient", rows=2048),
        # The surrogate's training: an epoch of 4096-row batches.
        dict(name="train_epoch", kind="train", rows=65536, batch=4096),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case of the same ranges."""
    kind = rng.choice(["particles"] * 6 + ["batch", "cloth", "solve", "gradient", "train"])
    if kind == "gradient":
        return dict(kind=kind, rows=_log_int(rng, 17, 2048))
    if kind == "train":
        return dict(kind=kind, rows=_log_int(rng, 2000, 131072), batch=rng.choice([777, 1024, 4096]))
    if kind == "batch":
        return dict(kind=kind, scenes=rng.randint(3, 20), n_min=_log_int(rng, 2000, 20000),
                    n_max=_log_int(rng, 40000, 300000), dt=5e-5, steps=rng.randint(8, 20))
    if kind == "cloth":
        c = _log_int(rng, 8, 40)
        res = rng.choice([64, 81, 96, 128])
        c = min(c, int(0.3 * res))
        return dict(kind=kind, res="%dx%dx%d" % (res, res, res), cells="%dx%dx%d" % (c, max(4, c - rng.randint(0, 5)), c),
                    n_side=rng.randint(20, 256), dt=2e-5, steps=rng.randint(10, 40))
    n = _log_int(rng, 1000, 2000000 if kind == "particles" else 150000)
    c = max(4, int(round((n / 8.0) ** (1.0 / 3.0))))
    cells = [max(3, int(round(c * rng.uniform(0.7, 1.4)))) for _ in range(3)]
    fill = rng.choice([1.0, 1.0, rng.uniform(0.6, 1.3)])
    edge = max(cells) * fill / rng.uniform(0.35, 0.8)
    res = max(16, min(256, int(round(edge))))
    res = [min(256, res + rng.choice([0, 0, -1, 1, 3])) for _ in range(3)]
    cells = [max(3, min(cc, int((0.4 if kind == "solve" else 0.8) * min(res) / fill))) for cc in cells]
    material = rng.choice(["sand", "sand", "snow"])
    cubic = rng.random() < 0.25
    case = dict(kind=kind, material=material, order=3 if cubic else 2, predicted=cubic and rng.random() < 0.7,
                friction=rng.choice(["coulomb", "coulomb", "sticky", "reference"]),
                phi=rng.choice(["constant", "hardening", "particle"]) if material == "sand" else "constant",
                res="x".join(str(r) for r in res), cells="x".join(str(cc) for cc in cells), fill=round(fill, 3))
    if kind == "solve":
        case.update(cfl=0.05, material="snow", phi="constant", predicted=False, order=2)
    else:
        case.update(dt=min(1e-4, 0.2 / max(res) / 20.0), steps=rng.randint(10, 40))
    if rng.random() < 0.3:
        case["z_up"] = True
    if kind == "particles" and material == "sand" and not cubic and rng.random() < 0.25:
        case["surrogate"] = True
    return case


def _ints(text):
    return tuple(int(t) for t in text.split("x"))


def _device():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


# ------------------------------------------------------------------ inputs
class _Inputs:
    """One scene's parameters and its mid-run particle state (float32 torch tensors, planes x particles)."""

    def __init__(self, seed, material, order, predicted, friction, phi, res, cells, fill, z_up=False, E=None, nu=None,
                 angle=30.0, floor=0.06, speed=0.8):
        dev = _device()
        gen = torch.Generator(device=dev).manual_seed(int(seed))

        def uniform(*shape):
            return torch.rand(*shape, generator=gen, device=dev, dtype=torch.float64)

        self.material, self.order, self.predicted, self.friction, self.phi = material, order, predicted, friction, phi
        self.res, self.up, self.weight = res, 2 if z_up else 1, GRAVITY
        self.rho = 400.0 if material == "snow" else 2200.0
        self.E = E if E else (1.4e5 if material == "snow" else 3.5e5)
        self.nu = nu if nu else (0.2 if material == "snow" else 0.3)
        self.dp_h = (35.0, 9.0, 0.2, 10.0) if phi == "hardening" else (angle, 0.0, 0.0, 0.0)
        self.mu = 0.2 if friction == "reference" else 0.4
        # cubic grid cells; the longest axis of the domain is 1
        self.h = 1.0 / max(res)
        self.size = [r * self.h for r in res]
        # a lattice of cells with 8 jittered particles each, `fill` grid cells wide, standing on the floor
        edge = [c * fill * self.h for c in cells]
        lo = [(s - e) / 2 for s, e in zip(self.size, edge)]
        if floor is not None:
            lo[self.up] = floor
        c = torch.tensor(cells, dtype=torch.float64, device=dev)
        n = 8 * cells[0] * cells[1] * cells[2]
        k = torch.arange(n, device=dev)
        cell, sub = k // 8, k % 8
        idx = torch.stack([cell % cells[0], cell // cells[0] % cells[1], cell // (cells[0] * cells[1])])
        corner = torch.stack([sub % 2, sub // 2 % 2, sub // 4])
        t = (idx + (corner + uniform(3, n)) / 2) / c[:, None]
        x = torch.tensor(lo, device=dev, dtype=torch.float64)[:, None] + torch.tensor(edge, device=dev, dtype=torch.float64)[:, None] * t
        self.n = n
        # a smooth velocity field, its gradient in the affine momenta, and some noise
        h = self.h
        wave = 2 * math.pi * (1 + 2 * uniform(3, 3))
        shift = 2 * math.pi * uniform(3, 1)
        arg = wave @ x + shift
        v = speed * torch.sin(arg) + 0.01 * (uniform(3, n) - 0.5)
        v[self.up] -= 1.0
        grad = speed * torch.cos(arg)[:, None, :] * wave[:, :, None]  # (a, b, n): d v_a / d x_b
        B = grad * (h * h / (4.0 if order == 2 else 3.0))
        # strains: compression by the weight above, a deviatoric part in proportion, a small rotation
        lam = self.E * self.nu / (1 + self.nu) / (1 - 2 * self.nu)
        shear = self.E / 2 / (1 + self.nu)
        depth = (lo[self.up] + edge[self.up] - x[self.up]).clamp_min(0.0)
        press = -(self.rho * GRAVITY * depth / (lam + 2 * shear / 3)).clamp_max(0.02)
        dev_amp = press.abs() * (0.05 + 0.4 * uniform(n)) + 2e-5
        S = uniform(3, 3, n) - 0.5
        S = (S + S.transpose(0, 1)) / 2
        eye = torch.eye(3, device=dev, dtype=torch.float64)
        S = S - (S[0, 0] + S[1, 1] + S[2, 2]) / 3 * eye[:, :, None]
        strain = press / 3 * eye[:, :, None] + dev_amp * S
        W = 0.05 * torch.sin(arg)
        skew = torch.zeros(3, 3, n, device=dev, dtype=torch.float64)
        skew[0, 1], skew[0, 2], skew[1, 2] = W[0], W[1], W[2]
        skew = skew - skew.transpose(0, 1)
        F = torch.einsum("ijn,jkn->ikn", eye[:, :, None] + strain, eye[:, :, None] + skew + 0.5 * torch.einsum("ijn,jkn->ikn", skew, skew))
        plastic = 0.1 + 0.5 * uniform(n) if material == "sand" else 1.0 + 0.02 * (uniform(n) - 0.5)
        vol = edge[0] * edge[1] * edge[2] / n
        f32 = torch.float32
        self.x, self.v, self.B, self.F = x.to(f32), v.to(f32), B.reshape(9, n).to(f32), F.reshape(9, n).to(f32)
        self.plastic = plastic.to(f32)
        self.volume = torch.full((n,), vol, device=dev, dtype=f32)
        self.mass = torch.full((n,), self.rho * vol, device=dev, dtype=f32)
        self.angles = (25 + 15 * uniform(n)).to(f32) if phi == "particle" else None
        self.boxes = [("box", (0.05, 0.05, 0.05), tuple(s - 0.05 for s in self.size)), ("sphere", (0.5, 0.15, 0.75), 0.1)]

    def in_flight(self):
        """The block spinning in free flight (no gravity in its frame), unstrained and soft. The speed of
        the fastest node sets the adaptive step: with strained free surfaces or an impact that would
        be a matter of the last bits of nearly empty nodes."""
        f64, n = torch.float64, self.n
        x = self.x.to(f64)
        spin = torch.tensor([[0.0, -0.9, 0.4], [0.9, 0.0, -0.6], [-0.4, 0.6, 0.0]], device=x.device, dtype=f64)
        v = spin @ (x - x.mean(1, keepdim=True)) + 0.1 * torch.tensor([[1.0], [-0.6], [0.5]], device=x.device, dtype=f64)
        h = self.h
        self.v = v.to(torch.float32)
        self.B = (spin * (h * h / (4.0 if self.order == 2 else 3.0))).reshape(9, 1).expand(9, n).to(torch.float32).contiguous()
        self.F = torch.eye(3, device=x.device, dtype=torch.float32).reshape(9, 1).expand(9, n).contiguous()
        self.E, self.weight = 1e3, 0.0
        return self

    @staticmethod
    def of(case, seed):
        inp = _Inputs._plain(case, seed)
        return inp.in_flight() if case["kind"] == "solve" else inp

    @staticmethod
    def _plain(case, seed):
        return _Inputs(seed, case["material"], case["order"], case["predicted"], case["friction"], case["phi"],
                       _ints(case["res"]), _ints(case["cells"]), case["fill"], bool(case.get("z_up")),
                       floor=None if case["kind"] == "solve" else 0.06, speed=0.4 if case.get("surrogate") else 0.8)

    def gravity(self):
        g = [0.0, 0.0, 0.0]
        g[self.up] = -self.weight
        return g

    def scene(self, name="case"):
        """The library's description of the scene."""
        g = self.gravity()
        if self.material == "snow":
            p = scenes.snow_params(self.order, g)
        else:
            p = scenes.sand_params(self.order, gravity=g)
            for i, hv in enumerate(self.dp_h):
                p.dp_h[i] = hv
            p.per_particle_phi = int(self.angles is not None)
        p.youngs_modulus, p.poisson_ratio, p.friction = self.E, self.nu, self.mu
        p.stress_at_predicted_F = int(self.predicted)
        p.friction_model = {"reference": _lib.FRICTION_REFERENCE, "coulomb": _lib.FRICTION_COULOMB,
                            "sticky": _lib.FRICTION_STICKY}[self.friction]
        prims = [levelset(_lib.LS_BOX, b[1] + (0.0,), b[2] + (0.0,)) if b[0] == "box" else
                 levelset(_lib.LS_SPHERE, b[1] + (b[2],)) for b in self.boxes]
        host = {k: None if t is None else t.cpu().numpy() for k, t in
                dict(x=self.x, v=self.v, B=self.B, F=self.F, plastic=self.plastic, mass=self.mass, volume=self.volume,
                     phi=self.angles).items()}
        return scenes.Scene(name, p, (0.0, 0.0, 0.0), tuple(self.size), self.res, prims, host, 0.0, 1)


def _batch_inputs(case, seed):
    """Independent snow and sand cubes, particle counts log-uniform, moduli and angles spread."""
    rng = np.random.default_rng(int(seed))
    layout = np.random.default_rng(11)  # the same sizes for every seed: a batch is one launch shape
    got = []
    for k in range(case["scenes"]):
        want = math.exp(layout.uniform(math.log(case["n_min"]), math.log(case["n_max"])))
        c = max(4, int(round((want / 8) ** (1.0 / 3.0))))
        res = max(int(layout.choice([64, 80, 96, 112])), int(c / 0.8))
        got.append(_Inputs(int(rng.integers(1 << 40)), "sand" if k % 2 else "snow", 2, False, "coulomb", "constant",
                           (res,) * 3, (c, c, c), 1.0, E=float(math.exp(rng.uniform(math.log(1e5), math.log(1e6)))),
                           nu=float(rng.uniform(0.2, 0.35)), angle=float(rng.uniform(25, 40))))
    return got


# (the in-plane force grows with the inverse edge length: this modulus is what 1/300 edges carry at dt = 2e-5)
CLOTH = dict(youngs_modulus=1.0, poisson_ratio=0.3, shear_stiffness=1e3, stiffness=1e4, friction_angle=20.0,
             density=2e3, thickness=0.04)


def _cloth_inputs(case, seed):
    """A sand block just above a falling, slightly wavy cloth over a sphere."""
    res, cells = _ints(case["res"]), _ints(case["cells"])
    sand = _Inputs(seed, "sand", 2, False, "coulomb", "constant", res, cells, 0.96, floor=0.62)
    sand.boxes = [sand.boxes[0], ("sphere", (0.5, 0.4, 0.5), 0.15)]
    side = case["n_side"]
    edge = min(1.0 / 300.0, 0.8 / side) if side > 128 else 0.4 / side
    mx, faces = scenes.grid_mesh(side, side, edge, (0.5 - edge * (side - 1) / 2,) * 2, 0.605)
    rng = np.random.default_rng(int(seed))
    mx = mx.astype(np.float64)
    mx[1] += 0.002 * np.sin(9 * mx[0] + rng.uniform(0, 6)) * np.cos(7 * mx[2] + rng.uniform(0, 6))
    mv = np.stack([0.1 * np.sin(5 * mx[1] + 3 * mx[2]), -1.5 + 0.2 * np.cos(4 * mx[0] + rng.uniform(0, 6)), 0.1 * np.cos(6 * mx[0])])
    return sand, mx.astype(np.float32), mv.astype(np.float32), np.asarray(faces, np.int32)


def _uniform_pairs(rows, seed):
    """(trial strains, angle, K/mu) rows and their Drucker-Prager cone returns, as the pair log holds."""
    g = np.random.default_rng(int(seed))
    lam_over_mu = g.uniform(0.67, 2.33, rows)
    angle = g.uniform(25.0, 40.0, rows)
    tr = -np.exp(g.uniform(np.log(3e-4), np.log(2e-2), rows))
    dev = g.normal(size=(rows, 3))
    dev -= dev.mean(axis=1, keepdims=True)
    dev = -np.sort(-dev, axis=1)
    dev /= np.linalg.norm(dev, axis=1, keepdims=True)
    sf = np.sin(np.deg2rad(angle))
    cone = -(3 * lam_over_mu + 2) / 2 * tr * (math.sqrt(2.0 / 3.0) * 2 * sf / (3 - sf))
    over = np.exp(g.uniform(np.log(1e-6), np.log(6e-4), rows))
    eps = tr[:, None] / 3 + (cone + over)[:, None] * dev
    H = tr[:, None] / 3 + cone[:, None] * dev
    return (np.concatenate([eps, angle[:, None], (lam_over_mu + 2.0 / 3.0)[:, None]], axis=1).astype(np.float32),
            H.astype(np.float32))


@functools.lru_cache(maxsize=1)
def _trained_weights():
    """The network a program with the surrogate keeps: trained once on the GPU."""
    pairs, H = _uniform_pairs(1 << 20, 77)
    with Solver(0) as s:
        s.surrogate_init(1)
        for epochs, lr in ((4, 3e-3), (4, 1e-3), (4, 3e-4)):
            s.surrogate_train(pairs, H, epochs=epochs, batch=4096, lr=lr, seed=2)
        return s.surrogate_get_weights()


LAYERS = ((128, 32, 5, 128), (128, 128, 128, 128), (128, 128, 128, 128), (128, 128, 128, 128), (16, 128, 128, 3))


def _fresh_weights(seed):
    """A network at the start of its training, in the library's flat layout (padding at zero)."""
    g = np.random.default_rng(int(seed))
    flat = []
    for layer, (rows, cols, fan_in, outs) in enumerate(LAYERS):
        a = math.sqrt(3.0 / fan_in) * (0.1 if layer == 4 else 1.0)
        w = np.zeros((rows, cols), np.float32)
        w[:outs, :fan_in] = g.uniform(-a, a, (outs, fan_in))
        flat += [w.reshape(-1), np.zeros(rows, np.float32)]
    return np.concatenate(flat)


# ------------------------------------------------------------------ prepare and run
class _State:
    pass


def _pinned(n, rows):
    """Page-locked host memory that a frame is read into, as numpy planes."""
    t = torch.empty((rows, n) if rows > 1 else (n,), dtype=torch.float32, pin_memory=torch.cuda.is_available())
    return t.numpy()


def _pointer(a):
    return a.ctypes.data_as(ctypes.POINTER(ctypes.c_float))


def _particle_buffers(n):
    return {name: _pinned(n, rows) for name, rows in STATE}


def prepare(case, seed):
    kind = case["kind"]
    s = _State()
    s.case = dict(case)
    s.solver = Solver(0)
    if kind in ("particles", "solve"):
        scene = _Inputs.of(case, seed).scene()
        scene.load_into(s.solver)
        s.out = _particle_buffers(scene.n)
        if case.get("tuned"):
            s.solver.autotune(case["dt"], reps=5)
        if case.get("surrogate"):
            s.solver.surrogate_set_weights(_trained_weights())
            s.solver.set_surrogate(True, 1e-5)
    elif kind == "batch":
        batch = [inp.scene("scene%d" % k) for k, inp in enumerate(_batch_inputs(case, seed))]
        s.solver.load_batch(batch)
        s.out = _particle_buffers(sum(sc.n for sc in batch))
    elif kind == "cloth":
        sand, mx, mv, faces = _cloth_inputs(case, seed)
        scene = sand.scene()
        scene.load_into(s.solver)
        s.solver.set_mesh(mx, faces, v=mv, **CLOTH)
        s.out = _particle_buffers(scene.n)
        s.mesh = dict(vx=_pinned(mx.shape[1], 3), vv=_pinned(mx.shape[1], 3), D=_pinned(len(faces), 9))
    elif kind == "gradient":
        s.solver.surrogate_set_weights(_fresh_weights(seed))
        pairs, H = _uniform_pairs(case["rows"], seed)
        s.pairs, s.H = torch.from_numpy(pairs).cuda(), torch.from_numpy(H).cuda()
        s.grad = torch.empty(s.solver.surrogate_nparam(), device="cuda")
        s.loss = torch.empty(1, device="cuda")
        torch.cuda.synchronize()
    elif kind == "train":
        s.solver.surrogate_set_weights(_fresh_weights(seed))
        s.pairs, s.H = _uniform_pairs(case["rows"], seed)
    return s


def _check(s, rc, what):
    if rc != _lib.MPM_OK:
        raise RuntimeError("%s: %s" % (what, s.lib.mpm_last_error(s.h).decode()))


def _read_particles(s):
    solver = s.solver
    _check(solver, solver.lib.mpm_get_particles(solver.h, *[_pointer(s.out[name]) for name, _ in STATE]), "mpm_get_particles")
    return s.out


def run(s):
    case, solver = s.case, s.solver
    kind = case["kind"]
    if kind in ("particles", "batch"):
        solver.run(case["dt"], case["steps"])
        return _read_particles(s)
    if kind == "cloth":
        solver.run(case["dt"], case["steps"])
        out = dict(_read_particles(s))
        m = s.mesh
        _check(solver, solver.lib.mpm_get_mesh(solver.h, _pointer(m["vx"]), _pointer(m["vv"]), _pointer(m["D"])), "mpm_get_mesh")
        out.update(m)
        return out
    if kind == "solve":
        solver.solve(case["cfl"], 0.0)  # ends after the frame that takes t past 0
        return _read_particles(s)
    if kind == "gradient":
        rc = solver.lib.mpm_surrogate_gradient_noalloc(solver.h, s.pairs.data_ptr(), s.H.data_ptr(), case["rows"],
                                                       s.grad.data_ptr(), s.loss.data_ptr())
        _check(solver, rc, "mpm_surrogate_gradient_noalloc")
        solver.synchronize()  # the gradient is ready for the caller's own stream from here on
        return dict(grad=s.grad, loss=s.loss)
    losses = solver.surrogate_train(s.pairs, s.H, epochs=1, batch=case["batch"], lr=1e-3, seed=5)
    return dict(losses=losses, weights=solver.surrogate_get_weights())


# ------------------------------------------------------------------ work
# Per particle and substep: 208 B of state (P2G reads x v B F m V, G2P reads x F plastic and writes x v B F
# plastic) and per active node 56 B; about 38 flops per node of the stencil in P2G, 48 in G2P and 600 in
# the singular value decomposition and the return map. The state read back: 26 floats in and out.
def _particle_work(n, order, steps, nodes, phi):
    stencil = (order + 1) ** 3
    return dict(bytes=float(steps * ((208 + (4 if phi else 0)) * n + 56 * nodes) + 208 * n),
                flops=float(steps * n * (stencil * 86 + 600)))


def _nodes(cells, fill):
    return float(np.prod([c * fill + 3 for c in cells]))


def work(case):
    kind = case["kind"]
    if kind in ("gradient", "train"):
        rows = case["rows"]
        macs = 5 * 128 + 3 * 128 * 128 + 128 * 3
        weights = sum(r * c + r for r, c, _, _ in LAYERS)
        steps = 1 if kind == "gradient" else -(-rows // case["batch"])
        return dict(bytes=float(32 * rows + steps * weights * (8 if kind == "gradient" else 32)), flops=6.0 * macs * rows)
    if kind == "batch":
        total = dict(bytes=0.0, flops=0.0)
        layout = np.random.default_rng(11)
        for _ in range(case["scenes"]):
            want = math.exp(layout.uniform(math.log(case["n_min"]), math.log(case["n_max"])))
            layout.choice([64, 80, 96, 112])
            c = max(4, int(round((want / 8) ** (1.0 / 3.0))))
            w = _particle_work(8 * c ** 3, 2, case["steps"], _nodes((c, c, c), 1.0), False)
            total = {k: total[k] + w[k] for k in total}
        return total
    cells = _ints(case["cells"])
    n = 8 * cells[0] * cells[1] * cells[2]
    if kind == "cloth":
        points = n + case["n_side"] ** 2 + 2 * (case["n_side"] - 1) ** 2
        return _particle_work(points, 2, case["steps"], _nodes(cells, 0.96), False)
    steps = case["steps"] if kind == "particles" else int(1.0 / 60.0 / (case["cfl"] / 300.0))
    w = _particle_work(n, case["order"], steps, _nodes(cells, case["fill"]), case["phi"] == "particle")
    if case.get("surrogate"):
        w["flops"] += 0.4 * steps * n * 2 * (5 * 128 + 3 * 128 * 128 + 128 * 3)
    return w


# ------------------------------------------------------------------ float64
def _f32(v):
    return float(np.float32(v))


def _weights64(order, r):
    """B-spline value and derivative (per cell) at r cells from the node."""
    a = r.abs()
    sg = torch.where(r < 0, -1.0, 1.0)
    if order == 3:
        near, far = 0.5 * a ** 3 - a * a + 2.0 / 3.0, (2 - a) ** 3 / 6
        dnear, dfar = sg * (1.5 * a * a - 2 * a), -sg * 0.5 * (2 - a) ** 2
        zero = torch.zeros_like(a)
        return torch.where(a < 1, near, torch.where(a < 2, far, zero)), torch.where(a < 1, dnear, torch.where(a < 2, dfar, zero))
    near, far = 0.75 - a * a, 0.5 * (1.5 - a) ** 2
    dnear, dfar = -2 * r, -sg * (1.5 - a)
    zero = torch.zeros_like(a)
    return torch.where(a < 0.5, near, torch.where(a < 1.5, far, zero)), torch.where(a < 0.5, dnear, torch.where(a < 1.5, dfar, zero))


def _mm(A, B):
    return torch.einsum("ijn,jkn->ikn", A, B)


def _svd64(F):
    """One-sided Jacobi SVD of n 3x3 matrices (3, 3, n): U, S in decreasing order, V."""
    w = [F[:, c].clone() for c in range(3)]  # columns (3, n)
    eye = torch.eye(3, device=F.device, dtype=F.dtype)
    v = [eye[:, c:c + 1].expand(3, F.shape[2]).clone() for c in range(3)]
    for _ in range(12):
        for p, q in ((0, 1), (0, 2), (1, 2)):
            al, be, ga = (w[p] ** 2).sum(0), (w[q] ** 2).sum(0), (w[p] * w[q]).sum(0)
            on = ga.abs() > 1e-17 * torch.sqrt(al * be)
            zeta = (be - al) / torch.where(on, 2 * ga, torch.ones_like(ga))
            t = torch.where(zeta >= 0, 1.0, -1.0) / (zeta.abs() + torch.sqrt(1 + zeta * zeta))
            t = torch.where(on, t, torch.zeros_like(t))
            c = 1 / torch.sqrt(1 + t * t)
            s = c * t
            w[p], w[q] = c * w[p] - s * w[q], s * w[p] + c * w[q]
            v[p], v[q] = c * v[p] - s * v[q], s * v[p] + c * v[q]
    W, V = torch.stack(w, 1), torch.stack(v, 1)
    S = torch.sqrt((W ** 2).sum(0))
    S, order = torch.sort(S, dim=0, descending=True)
    take = order[None].expand(3, 3, -1)
    W, V = W.gather(1, take), V.gather(1, take)
    return W / S, S, V


class _Exact:
    """The explicit MPM substep in float64."""

    def __init__(self, inp, mesh=None):
        f64 = torch.float64
        self.inp = inp
        self.res = inp.res
        dev = inp.x.device
        self.dev = dev
        self.h = torch.tensor([s / r for s, r in zip(inp.size, inp.res)], device=dev, dtype=f64)
        self.dinv = (3.0 if inp.order == 3 else 4.0) / float(self.h.min()) ** 2
        n = inp.n
        self.x, self.v = inp.x.to(f64), inp.v.to(f64)
        self.B, self.F = inp.B.to(f64).reshape(3, 3, n), inp.F.to(f64).reshape(3, 3, n)
        self.q, self.m, self.vol = inp.plastic.to(f64), inp.mass.to(f64), inp.volume.to(f64)
        E, nu = _f32(inp.E), _f32(inp.nu)
        self.lam, self.shear = E * nu / (1 + nu) / (1 - 2 * nu), E / 2 / (1 + nu)
        self.g = torch.tensor([_f32(g) for g in inp.gravity()], device=dev, dtype=f64)
        self.n = n
        self.mesh = mesh
        if mesh is not None:
            mesh.attach(self)

    # stencil: for every offset the node index, the weight, its gradient and the node's position
    def stencil(self):
        k = self.inp.order
        gx = self.x / self.h[:, None]
        base = torch.floor(gx - 0.5) if k == 2 else torch.floor(gx) - 1
        base = base.clamp(-8, 1 << 20).to(torch.int64)
        w, dw, ok = [], [], []
        for d in range(3):
            node = [base[d] + o for o in range(k + 1)]
            pair = [_weights64(k, gx[d] - nd) for nd in node]
            inside = [(nd >= 0) & (nd < self.res[d]) for nd in node]
            w.append([torch.where(i, p[0], torch.zeros_like(p[0])) for p, i in zip(pair, inside)])
            dw.append([torch.where(i, p[1], torch.zeros_like(p[1])) / self.h[d] for p, i in zip(pair, inside)])
            ok.append([nd.clamp(0, self.res[d] - 1) for nd in node])
        for oz in range(k + 1):
            for oy in range(k + 1):
                wyz = w[1][oy] * w[2][oz]
                for ox in range(k + 1):
                    idx = (ok[2][oz] * self.res[1] + ok[1][oy]) * self.res[0] + ok[0][ox]
                    pos = torch.stack([(base[0] + ox) * self.h[0], (base[1] + oy) * self.h[1], (base[2] + oz) * self.h[2]])
                    gw = torch.stack([dw[0][ox] * wyz, w[0][ox] * dw[1][oy] * w[2][oz], w[0][ox] * w[1][oy] * dw[2][oz]])
                    yield idx, w[0][ox] * wyz, gw, pos

    def moduli(self):
        if self.inp.material == "snow":
            sc = torch.exp(10.0 * (1 - self.q))
            return self.lam * sc, self.shear * sc
        return self.lam, self.shear

    def kirchhoff(self, F, Fn):
        """V P(F) Fn^T of the material particles."""
        U, S, V = _svd64(F)
        if self.inp.material == "snow":
            lam, mu = self.moduli()
            J = torch.linalg.det(F.permute(2, 0, 1))
            inv_t = torch.linalg.inv(F.permute(2, 0, 1)).permute(2, 1, 0)
            P = 2 * mu * (F - torch.einsum("ikn,jkn->ijn", U, V)) + lam * (J - 1) * J * inv_t
        else:
            ln = torch.log(S)
            d = (2 * self.shear * ln + self.lam * ln.sum(0)) / S
            P = torch.einsum("ikn,kn,jkn->ijn", U, d, V)
        return self.vol[: P.shape[2]] * torch.einsum("ikn,jkn->ijn", P, Fn)

    def scatter(self, impulse, stress, momentum=True):
        """Node mass and sum of w (m v + m Dinv B (x_i - x_p)) + w impulse - stress grad w."""
        ng = self.res[0] * self.res[1] * self.res[2]
        acc = torch.zeros(ng, 4, device=self.dev, dtype=torch.float64)
        mB = self.m * self.dinv * self.B if momentum else None
        mv = self.m * self.v if momentum else None
        for idx, w, gw, pos in self.stencil():
            val = torch.zeros_like(self.v)
            if momentum:
                val = val + w * (mv + torch.einsum("ijn,jn->in", mB, pos - self.x))
            if stress is not None:
                val = val - torch.einsum("ijn,jn->in", stress, gw)
            if impulse is not None:
                val = val + w * impulse
            acc.index_add_(0, idx, torch.cat([(w * self.m)[None], val]).T.contiguous())
        return acc[:, 0], acc[:, 1:].T

    def collide(self, v):
        """Post-friction and pre-friction node velocities."""
        inp, dev = self.inp, self.dev
        ax = [torch.arange(r, device=dev, dtype=torch.float64) * h for r, h in zip(self.res, self.h)]
        z, y, x = torch.meshgrid(ax[2], ax[1], ax[0], indexing="ij")
        X = torch.stack([x.reshape(-1), y.reshape(-1), z.reshape(-1)])
        phi = torch.full_like(X[0], 3e38)
        nrm = torch.zeros_like(X)
        for b in inp.boxes:
            if b[0] == "box":
                dist = [X[d] - _f32(b[1][d]) for d in range(3)] + [_f32(b[2][d]) - X[d] for d in range(3)]
                order = [dist[0], dist[3], dist[1], dist[4], dist[2], dist[5]]
                p = torch.stack(order)
                at = p.argmin(0)
                p = p.gather(0, at[None])[0]
                nn = torch.zeros_like(X)
                for d in range(3):
                    nn[d] = torch.where(at == 2 * d, 1.0, torch.where(at == 2 * d + 1, -1.0, 0.0))
            else:
                c = torch.tensor([_f32(t) for t in b[1]], device=dev, dtype=torch.float64)[:, None]
                length = torch.sqrt(((X - c) ** 2).sum(0))
                p, nn = length - _f32(b[2]), (X - c) / length.clamp_min(1e-300)
            near = p < phi
            phi, nrm = torch.where(near, p, phi), torch.where(near, nn, nrm)
        inside = phi <= 0
        if inp.friction == "sticky":
            v = torch.where(inside, torch.zeros_like(v), v)
            return v, v
        vn = (v * nrm).sum(0)
        hit = inside & (vn < 0)
        vt = v - vn * nrm
        length = torch.sqrt((vt ** 2).sum(0))
        mu = _f32(inp.mu)
        if inp.friction == "reference":
            after = torch.where(length < -mu * vn, torch.zeros_like(vt), vt)
        else:
            after = torch.where(length <= -mu * vn, torch.zeros_like(vt), vt * (1 + mu * vn / length.clamp_min(1e-300)))
        return torch.where(hit, after, v), torch.where(hit, vt, v)

    def gather_gradient(self, v):
        G = torch.zeros(3, 3, self.x.shape[1], device=self.dev, dtype=torch.float64)
        for idx, _, gw, _ in self.stencil():
            G += v[:, idx][:, None] * gw[None]
        return G

    def grid_velocity(self, mass, mom):
        return torch.where(mass > 0, mom / torch.where(mass > 0, mass, torch.ones_like(mass)), torch.zeros_like(mom))

    def particle_stress(self, F, Fn):
        K = self.kirchhoff(F[:, :, : self.n], Fn[:, :, : self.n])
        return K if self.mesh is None else self.mesh.stress(self, K)

    def substep(self, dt, dt_after=None):
        """One substep; dt_after(vmax): the step that the second half uses (adaptive runs)."""
        inp = self.inp
        impulse = None if self.mesh is None else self.mesh.impulse(self, dt)
        if inp.predicted:
            mass, mom = self.scatter(None, None)
            v0 = self.grid_velocity(mass, mom)
            Fh = self.F + dt * _mm(self.gather_gradient(v0), self.F)
            _, force = self.scatter(None, self.particle_stress(Fh, self.F), momentum=False)
            v = torch.where(mass > 0, v0 + dt * (self.grid_velocity(mass, force) + self.g[:, None]), v0)
        else:
            mass, mom = self.scatter(impulse, dt * self.particle_stress(self.F, self.F))
            v = self.grid_velocity(mass, mom)
            v = torch.where(mass > 0, v + dt * self.g[:, None], v)
        if dt_after is not None:
            dt = dt_after(float(torch.sqrt((v ** 2).sum(0)).max()))
        v, vbf = self.collide(v)
        vp, vb = torch.zeros_like(self.v), torch.zeros_like(self.v)
        B, G = torch.zeros_like(self.B), torch.zeros_like(self.B)
        for idx, w, gw, pos in self.stencil():
            vi, bi = v[:, idx], vbf[:, idx]
            vp += w * vi
            vb += w * bi
            B += (w * vi)[:, None] * (pos - self.x)[None]
            G += bi[:, None] * gw[None]
        self.v, self.B = vp, B
        self.x = self.x + dt * vb
        self.F = self.F + dt * _mm(G, self.F)
        self.return_map()
        if self.mesh is not None:
            self.mesh.follow(self)

    def return_map(self):
        inp, n = self.inp, self.n
        F = self.F[:, :, :n]
        U, S, V = _svd64(F)
        if inp.material == "snow":
            Sn = S.clamp(1 - _f32(2.5e-2), 1 + _f32(7.5e-3))
            self.q = self.q * (S / Sn).prod(0)
        else:
            h = [_f32(t) for t in inp.dp_h]
            phi = (inp.angles.to(torch.float64) if inp.angles is not None else h[0]) + (h[1] * self.q - h[3]) * torch.exp(-h[2] * self.q)
            sf = torch.sin(phi * math.pi / 180)
            alpha = math.sqrt(2.0 / 3.0) * 2 * sf / (3 - sf)
            ln = torch.log(S)
            tr = ln.sum(0)
            e = ln - tr / 3
            en = torch.sqrt((e ** 2).sum(0))
            dg = en + (3 * self.lam + 2 * self.shear) / 2 / self.shear * tr * alpha
            elastic, tip = dg <= 0, (en == 0) | (tr > 0)
            H = ln - dg / en.clamp_min(1e-300) * e
            H = torch.where(elastic, ln, torch.where(tip, torch.zeros_like(ln), H))
            zero = torch.zeros_like(dg)
            self.q = self.q + torch.where(elastic, zero, torch.where(tip, torch.sqrt((ln ** 2).sum(0)), dg))
            Sn = torch.exp(H)
        self.F = torch.cat([torch.einsum("ikn,kn,jkn->ijn", U, Sn, V), self.F[:, :, n:]], 2)

    def outputs(self):
        n = self.n
        return dict(x=self.x[:, :n], v=self.v[:, :n], B=self.B[:, :, :n].reshape(9, n), F=self.F[:, :, :n].reshape(9, n),
                    plastic=self.q, volume=self.vol[:n])


class _Mesh64:
    """A triangle cloth whose vertices and elements follow the particles as material points."""

    def __init__(self, x, v, faces):
        self.x0, self.v0, self.faces = x, v, faces

    @staticmethod
    def _qr(D):
        q1 = D[:, 0]
        r11 = torch.sqrt((q1 ** 2).sum(0))
        q1 = q1 / r11
        r12 = (D[:, 1] * q1).sum(0)
        q2 = D[:, 1] - r12 * q1
        r22 = torch.sqrt((q2 ** 2).sum(0))
        q2 = q2 / r22
        r13, r23 = (D[:, 2] * q1).sum(0), (D[:, 2] * q2).sum(0)
        q3 = D[:, 2] - r13 * q1 - r23 * q2
        r33 = torch.sqrt((q3 ** 2).sum(0))
        return torch.stack([q1, q2, q3 / r33], 1), r11, r12, r13, r22, r23, r33

    def attach(self, sim):
        f64, dev = torch.float64, sim.dev
        X, Vv = torch.from_numpy(self.x0).to(dev, f64), torch.from_numpy(self.v0).to(dev, f64)
        f = torch.from_numpy(self.faces).to(dev, torch.int64)
        p = [X[:, f[:, c]] for c in range(3)]
        d1, d2 = p[1] - p[0], p[2] - p[0]
        nrm = torch.linalg.cross(d1.T, d2.T).T
        size = torch.sqrt((nrm ** 2).sum(0))
        vol = 0.25 * 0.5 * size * _f32(CLOTH["thickness"])
        nv, ne = X.shape[1], f.shape[0]
        vvol = torch.zeros(nv, device=dev, dtype=f64)
        for c in range(3):
            vvol.index_add_(0, f[:, c], vol)
        D = torch.stack([d1, d2, nrm / size], 1)
        self.f, self.nv, self.ne, self.evol = f, nv, ne, vol
        _, r11, r12, _, r22, _, _ = self._qr(D)
        self.i11, self.i12, self.i22 = 1 / r11, -r12 / r11 / r22, 1 / r22
        self.cn = torch.linalg.inv(D.permute(2, 0, 1))[:, 2, :].T  # D^-T e3
        eye = torch.eye(3, device=dev, dtype=f64)[:, :, None].expand(3, 3, nv)
        zero = torch.zeros(3, 3, nv + ne, device=dev, dtype=f64)
        rho = _f32(CLOTH["density"])
        sim.x = torch.cat([sim.x, X, (p[0] + p[1] + p[2]) / 3], 1)
        sim.v = torch.cat([sim.v, Vv, (Vv[:, f[:, 0]] + Vv[:, f[:, 1]] + Vv[:, f[:, 2]]) / 3], 1)
        sim.B, sim.F = torch.cat([sim.B, zero], 2), torch.cat([sim.F, eye, D], 2)
        sim.m, sim.vol = torch.cat([sim.m, rho * vvol, rho * vol]), torch.cat([sim.vol, vvol, vol])

    def impulse(self, sim, dt):
        """dt x the in-plane vertex forces; the element stresses are kept for `stress`."""
        n, nv = sim.n, self.nv
        E, nu = _f32(CLOTH["youngs_modulus"]), _f32(CLOTH["poisson_ratio"])
        lam, mu = E * nu / (1 + nu) / (1 - 2 * nu), E / 2 / (1 + nu)
        D = sim.F[:, :, n + nv:]
        Q, r11, r12, r13, r22, r23, r33 = self._qr(D)
        a00, a01, a11 = self.i11 * r11, self.i11 * r12 + self.i12 * r22, self.i22 * r22
        size = torch.sqrt((a00 + a11) ** 2 + a01 ** 2)
        c, s = (a00 + a11) / size, -a01 / size
        J = a00 * a11
        p00 = 2 * mu * (a00 - c) + lam * (J - 1) * a11
        p01, p10 = 2 * mu * (a01 + s), -2 * mu * s - lam * (J - 1) * a01
        p11 = 2 * mu * (a11 - c) + lam * (J - 1) * a00
        f2 = -(p00 * self.i11 + p01 * self.i12) * Q[:, 0]
        f3 = -p01 * self.i22 * Q[:, 0] - p11 * self.i22 * Q[:, 1]
        force = torch.zeros(nv, 3, device=sim.dev, dtype=torch.float64)
        for corner, f in ((0, -(f2 + f3)), (1, f2), (2, f3)):
            force.index_add_(0, self.f[:, corner], f.T.contiguous())
        zero = torch.zeros_like(r11)
        s11, s12, s22 = self.i11 * p00 + self.i12 * p10, self.i11 * p01 + self.i12 * p11, self.i22 * p11
        gam, k = _f32(CLOTH["shear_stiffness"]), _f32(CLOTH["stiffness"])
        n33 = torch.where(r33 > 1, zero, -k * (1 - r33) ** 2)
        dR = torch.stack([torch.stack([s11, s12, gam * r13]), torch.stack([zero, s22, gam * r23]), torch.stack([zero, zero, n33])])
        R = torch.stack([torch.stack([r11, r12, r13]), torch.stack([zero, r22, r23]), torch.stack([zero, zero, r33])])
        K = torch.einsum("ikn,jkn->ijn", dR, R)
        up = torch.triu(torch.ones(3, 3, device=sim.dev, dtype=torch.float64))[:, :, None]
        K = K * up + (K * up).transpose(0, 1) * (1 - up)
        y0 = self.cn[0] / r11
        y1 = (self.cn[1] - r12 * y0) / r22
        y2 = (self.cn[2] - r13 * y0 - r23 * y1) / r33
        dF3 = torch.einsum("ijn,jn->in", Q, torch.einsum("ijn,jn->in", K, torch.stack([y0, y1, y2])))
        self.element = self.evol * dF3[:, None] * D[:, 2][None]
        out = torch.zeros_like(sim.v)
        out[:, n:n + nv] = dt * force.T
        return out

    def stress(self, sim, K):
        return torch.cat([K, torch.zeros(3, 3, self.nv, device=sim.dev, dtype=torch.float64), self.element], 2)

    def follow(self, sim):
        """Skew affine momenta, element points at their centroids, directions return-mapped."""
        n, nv = sim.n, self.nv
        Bm = sim.B[:, :, n:]
        sim.B = torch.cat([sim.B[:, :, :n], (Bm - Bm.transpose(0, 1)) / 2], 2)
        X, Vv = sim.x[:, n:n + nv], sim.v[:, n:n + nv]
        p = [X[:, self.f[:, c]] for c in range(3)]
        sim.x = torch.cat([sim.x[:, :n + nv], (p[0] + p[1] + p[2]) / 3], 1)
        sim.v = torch.cat([sim.v[:, :n + nv], sum(Vv[:, self.f[:, c]] for c in range(3)) / 3], 1)
        D = torch.stack([p[1] - p[0], p[2] - p[0], sim.F[:, 2, n + nv:]], 1)
        Q, _, _, r13, _, r23, r33 = self._qr(D)
        fn = _f32(CLOTH["stiffness"]) * (r33 - 1) ** 2
        ft = _f32(CLOTH["shear_stiffness"]) * torch.sqrt(r13 ** 2 + r23 ** 2)
        limit = math.tan(math.radians(_f32(CLOTH["friction_angle"]))) * fn
        scale = torch.where(ft > limit, limit / ft.clamp_min(1e-300), torch.ones_like(ft))
        apart = r33 > 1
        zero, one = torch.zeros_like(r33), torch.ones_like(r33)
        r13, r23 = torch.where(apart, zero, r13 * scale), torch.where(apart, zero, r23 * scale)
        D[:, 2] = Q[:, 0] * r13 + Q[:, 1] * r23 + Q[:, 2] * torch.where(apart, one, r33)
        sim.F = torch.cat([sim.F[:, :, :n + nv], D], 2)

    def outputs(self, sim):
        n, nv = sim.n, self.nv
        return dict(vx=sim.x[:, n:n + nv], vv=sim.v[:, n:n + nv], D=sim.F[:, :, n + nv:].reshape(9, -1))


def _solve64(sim, cfl):
    """One frame of the adaptive loop: Dt = cfl / max(300, vmax / h_min), clamped to the frame's end."""
    hmin = float(sim.h.min())

    def step(vmax):
        return cfl / max(300.0, vmax / hmin)

    mass, mom = sim.scatter(None, None)
    dt = step(float(torch.sqrt((sim.grid_velocity(mass, mom) ** 2).sum(0)).max()))
    inner, done = 0.0, False

    def after(vmax):
        nonlocal dt, inner, done
        dt = step(vmax)
        if inner + dt >= 1.0 / 60.0:
            dt, done = 1.0 / 60.0 - inner, True
        inner += dt
        return _f32(dt)

    while not done:
        sim.substep(_f32(dt), after)


def _network64(flat):
    """The network's layers as float64 leaves: (weight, bias) per layer over the flat vector."""
    t = torch.from_numpy(np.asarray(flat, np.float64)).to(_device()).requires_grad_(True)
    at, layers = 0, []
    for rows, cols, _, _ in LAYERS:
        layers.append((t[at:at + rows * cols].view(rows, cols), t[at + rows * cols:at + rows * cols + rows]))
        at += rows * cols + rows
    return t, layers


def _loss64(layers, pairs, H):
    """Sum over rows and outputs of (y - t)^2, with y, t the corrections in units of 1e-3."""
    x = torch.cat([pairs[:, :3] / 0.02, (pairs[:, 3:4] - 32.5) / 7.5, pairs[:, 4:5] - 2.5], 1)
    x = torch.nn.functional.pad(x, (0, 27))
    for k, (w, b) in enumerate(layers):
        x = x @ w.T + b
        if k < 4:
            x = torch.nn.functional.silu(x)
    return ((x[:, :3] - (H - pairs[:, :3]) / 1e-3) ** 2).sum()


def _mix64(z):
    m = (1 << 64) - 1
    z = (z + 0x9E3779B97F4A7C15) & m
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & m
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
    return z ^ (z >> 31)


def _train64(case, seed):
    """One epoch of Adam in the trainer's seeded row order."""
    rows, batch = case["rows"], min(case["batch"], case["rows"])
    pairs, H = _uniform_pairs(rows, seed)
    order = list(range(rows))
    for i in range(rows - 1, 0, -1):
        j = _mix64(5 ^ ((0xD1B54A32D192ED03 * (i + 1)) & ((1 << 64) - 1))) % (i + 1)
        order[i], order[j] = order[j], order[i]
    pairs, H = (torch.from_numpy(a[order].astype(np.float64)).to(_device()) for a in (pairs, H))
    flat = _fresh_weights(seed).astype(np.float64)
    active = torch.zeros(flat.size, device=_device(), dtype=torch.float64)
    at = 0
    for r, c, fan_in, outs in LAYERS:
        active[at:at + r * c].view(r, c)[:outs, :fan_in] = 1
        active[at + r * c:at + r * c + outs] = 1
        at += r * c + r
    m1 = m2 = 0.0
    total, step = 0.0, 0
    lr, b1, b2 = _f32(1e-3), _f32(0.9), _f32(0.999)
    for r0 in range(0, rows, batch):
        nb = min(batch, rows - r0)
        t, layers = _network64(flat)
        loss = _loss64(layers, pairs[r0:r0 + nb], H[r0:r0 + nb])
        total += float(loss.detach())
        g, = torch.autograd.grad(loss / nb, t)
        g = g * active
        step += 1
        m1 = b1 * m1 + (1 - b1) * g
        m2 = b2 * m2 + (1 - b2) * g * g
        move = lr * (m1 / (1 - b1 ** step)) / (torch.sqrt(m2 / (1 - b2 ** step)) + 1e-8)
        flat = (t.detach() - move * active).cpu().numpy()
    return dict(losses=np.array([total / rows]), weights=flat)


def exact(case, seed):
    kind = case["kind"]
    if kind == "train":
        return _train64(case, seed)
    if kind == "gradient":
        t, layers = _network64(_fresh_weights(seed))
        pairs, H = (torch.from_numpy(a.astype(np.float64)).to(_device()) for a in _uniform_pairs(case["rows"], seed))
        loss = _loss64(layers, pairs, H) / case["rows"]
        g, = torch.autograd.grad(loss, t)
        return dict(grad=g, loss=loss.detach().reshape(1))
    if case.get("surrogate"):
        return None  # a BF16 network behind a gate: its outputs have no float64 value
    if kind == "batch":
        sims = [_Exact(inp) for inp in _batch_inputs(case, seed)]
    elif kind == "cloth":
        sand, mx, mv, faces = _cloth_inputs(case, seed)
        sims = [_Exact(sand, _Mesh64(mx, mv, faces))]
    else:
        sims = [_Exact(_Inputs.of(case, seed))]
    for sim in sims:
        if kind == "solve":
            _solve64(sim, case["cfl"])
        else:
            for _ in range(case["steps"]):
                sim.substep(_f32(case["dt"]))
    outs = [sim.outputs() for sim in sims]
    got = {name: torch.cat([o[name] for o in outs], -1) for name, _ in STATE}
    if kind == "cloth":
        got.update(sims[0].mesh.outputs(sims[0]))
    return got
