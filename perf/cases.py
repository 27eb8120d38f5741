"""The work that users of the library run on one GPU, as measurable cases.

A case is a dict of plain values.  `listed()` names the fixed ones, `draw()`
makes more of the same kinds and ranges, `prepare()` builds what a program
holds before the call (inputs from a seed, the film or trainer it keeps),
`run()` is one pass through the public entry points, `work()` the bytes and
operations a pass cannot do without and `exact()` the same outputs in 64 bits
by plain PyTorch.

Kinds
  exact       calc_potential_exact on host arrays
  reforder    calc_potential_exact_gpu on host arrays (the reference kernel's
              summation order)
  march       time_marching: the adaptive time loop with its output files
  film        Film.steps + Film.get_m: a resident film (direct sum or FMM)
  rk4         Hfield + rk4_step on host arrays: one step of a program that
              keeps its state on the host
  infer       Film.surrogate_potential: the learned surrogate on one film
  grad        SurrogateTrainer.gradient: loss and gradient of one batch
"""
import math
import os
import sys
import tempfile

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "mms-gpu_amd"))
import mms_gpu as mg  # noqa: E402

F = np.float32
MU_0, MS, AEXCH = F(4 * np.pi * 1e-7), F(8.6e5), F(1.3e-11)
ALFA, GAMMA, CELL = F(0.5), F(2.211e5), F(5e-9)
FORMS = {"fp32": mg.M2L_FP32, "bf16x3": mg.M2L_BF16X3, "fp16x2_f16x2near": mg.M2L_FP16X2_FP16X2NEAR}
CH = 64  # channels of the surrogate
NM = 32  # its Fourier modes per axis


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # the smallest call: a potential of the 32 x 32 x 3 film by the direct
        # sum on host arrays; launches, copies and latency
        dict(name="exact_32x32x3", kind="exact", xd=32, yd=32, zd=3, dz=1.0),
        # the same call on the 256 x 256 x 3 film, the size up to which a
        # program checks the FMM against the direct sum
        dict(name="exact_256x256x3", kind="exact", xd=256, yd=256, zd=3, dz=1.0),
        # the reference GPU kernel's order on a ragged film with flat cells
        dict(name="reforder_100x75x3", kind="reforder", xd=100, yd=75, zd=3, dz=0.6),
        # the reference program's own use: adaptive marching of a small film
        # from a random state with its text output of every accepted step
        dict(name="march_64x64x3", kind="march", xd=64, yd=64, zd=3, dz=1.0, P=3, finaltime=3e-14),
        # the smallest resident film, direct sum, 1e-13 s steps in between two
        # looks at the state
        dict(name="film_32x32x3_direct", kind="film", xd=32, yd=32, zd=3, dz=1.0, solver="direct", P=0, form="fp32",
             leaf=4, state="random", steps=100, dt=1e-13, hx=0.0),
        # an odd-sized direct-sum film of round dots (non-magnetic cells)
        dict(name="film_161x117x3_direct", kind="film", xd=161, yd=117, zd=3, dz=0.6, solver="direct", P=0,
             form="fp32", leaf=4, state="dots", steps=10, dt=1e-13, hx=7958.0),
        # the 256 x 256 x 3 dot film, FMM of order 4 in the default form
        dict(name="film_256x256x3_fmm4", kind="film", xd=256, yd=256, zd=3, dz=1.0, solver="fmm", P=4, form="fp32",
             leaf=4, state="dots", steps=100, dt=1e-13, hx=7958.0),
        # the largest film: 1024 x 1024 x 4 domains, FMM of order 6, 16-bit
        # split operands on the matrix cores
        dict(name="film_1024x1024x4_fmm6", kind="film", xd=1024, yd=1024, zd=4, dz=1.0, solver="fmm", P=6,
             form="fp16x2_f16x2near", leaf=8, state="domains", steps=50, dt=5e-14, hx=0.0),
        # one step from host arrays, a ragged film with the FMM of order 6 in
        # FP32, fields and slopes copied back
        dict(name="rk4_250x190x4_fmm6", kind="rk4", xd=250, yd=190, zd=4, dz=1.0, P=6, dt=1e-13),
        # a large ragged film with the BF16 split on the matrix cores
        dict(name="film_705x498x4_fmm6", kind="film", xd=705, yd=498, zd=4, dz=1.0, solver="fmm", P=6, form="bf16x3",
             leaf=8, state="dots", steps=20, dt=1e-13, hx=7958.0),
        # the surrogate's potential of the 1024 x 1024 x 4 film
        dict(name="infer_1024x1024x4", kind="infer", xd=1024, yd=1024, zd=4),
        # a training batch of eight 128 x 128 x 3 films, forward and backward
        dict(name="grad_8x128x128x3", kind="grad", xd=128, yd=128, zd=3, batch=8),
    ]


def draw(rng):
    def side(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    dz = rng.choice([1.0, 0.6, 0.5])
    kind = rng.choice(["exact", "exact", "reforder", "march", "film", "film", "film", "film", "rk4", "infer", "grad"])
    if kind == "exact":
        return dict(kind=kind, xd=side(20, 256), yd=side(20, 256), zd=rng.randint(1, 4), dz=dz)
    if kind == "reforder":
        return dict(kind=kind, xd=side(20, 128), yd=side(20, 128), zd=rng.randint(1, 3), dz=dz)
    if kind == "march":
        return dict(kind=kind, xd=side(24, 80), yd=side(24, 80), zd=3, dz=1.0, P=rng.randint(3, 4), finaltime=2e-14)
    if kind == "film":
        solver = rng.choice(["direct", "fmm", "fmm"])
        out = dict(kind=kind, dz=dz, solver=solver, state=rng.choice(["random", "domains", "dots"]),
                   hx=rng.choice([0.0, 7958.0]))
        if solver == "direct":
            out.update(xd=side(24, 180), yd=side(24, 180), zd=rng.randint(1, 4), P=0, form="fp32", leaf=4,
                       steps=rng.randint(5, 20), dt=1e-13 if dz == 1.0 else 4e-14)
        else:
            out.update(xd=side(96, 1024), yd=side(96, 1024), zd=rng.randint(2, 4), P=rng.randint(3, 6),
                       form=rng.choice(sorted(FORMS)), leaf=rng.choice([4, 8]), steps=rng.randint(5, 15),
                       dt=1e-13 if dz == 1.0 else 4e-14)
        return out
    if kind == "rk4":
        return dict(kind=kind, xd=side(64, 400), yd=side(64, 400), zd=rng.randint(2, 4), dz=dz, P=rng.randint(3, 6),
                    dt=4e-14)
    if kind == "infer":
        return dict(kind=kind, xd=side(128, 1000), yd=side(128, 1000), zd=rng.randint(2, 4))
    return dict(kind=kind, xd=side(64, 128), yd=side(64, 128), zd=rng.randint(2, 3), batch=rng.randint(2, 8))


# ----------------------------------------------------------------- inputs --
def _unit(rng, n):
    v = rng.standard_normal((n, 3))
    return v / np.linalg.norm(v, axis=1, keepdims=True)


def _film_state(xd, yd, zd, state, seed):
    """(material uint8 [n], M float32 [3n]) of one film: 'random' unit vectors,
    32-cell in-plane 'domains' (both all magnetic), or round 'dots' on a
    64-cell pitch, each with a vortex and 1% noise."""
    rng = np.random.default_rng(seed)
    n = xd * yd * zd
    mat = np.ones((zd, yd, xd), np.uint8)
    if state == "random":
        m = _unit(rng, n)
    elif state == "domains":
        ang = rng.uniform(0, 2 * np.pi, ((yd + 31) // 32, (xd + 31) // 32))
        a = np.repeat(np.repeat(ang, 32, 0), 32, 1)[:yd, :xd]
        m = np.broadcast_to(np.stack([np.cos(a), np.sin(a), 0 * a], -1), (zd, yd, xd, 3)).reshape(-1, 3)
    else:
        pitch = min(64, xd, yd)
        y, x = np.mgrid[0:yd, 0:xd]
        cx, cy = (x // pitch + 0.5) * pitch, (y // pitch + 0.5) * pitch
        px, py = x + 0.5 - cx, y + 0.5 - cy
        r = np.hypot(px, py)
        sign = rng.integers(0, 2, ((yd + pitch - 1) // pitch, (xd + pitch - 1) // pitch, 2)) * 2.0 - 1.0
        sg = sign[y // pitch, x // pitch]
        mz = sg[..., 0] * np.exp(-(r / 2.0) ** 2)
        ip = np.sqrt(1 - mz * mz) * sg[..., 1] / np.maximum(r, 1e-9)
        m = np.broadcast_to(np.stack([-py * ip, px * ip, mz], -1), (zd, yd, xd, 3)).reshape(-1, 3)
        m = m + 0.01 * _unit(rng, n)
        m = m / np.linalg.norm(m, axis=1, keepdims=True)
        mat[:, r > 0.33 * pitch] = 0
    M = (m * float(MS)).astype(F)
    M[mat.ravel() == 0] = 0
    return mat.ravel(), np.ascontiguousarray(M).ravel()


def _charge(xd, yd, zd, state, seed):
    """Charge density of a film state (central differences, zero outside)."""
    _, M = _film_state(xd, yd, zd, state, seed)
    m = np.pad(M.reshape(zd, yd, xd, 3), ((1, 1), (1, 1), (1, 1), (0, 0)))
    d = (m[1:-1, 1:-1, 2:, 0] - m[1:-1, 1:-1, :-2, 0]) + (m[1:-1, 2:, 1:-1, 1] - m[1:-1, :-2, 1:-1, 1]) \
        + (m[2:, 1:-1, 1:-1, 2] - m[:-2, 1:-1, 1:-1, 2])
    return np.ascontiguousarray(d / (2 * CELL), F).ravel()


def _march_state(case, seed):
    """Random state of the reference program: a one-cell non-magnetic border
    and the inner layers magnetic, in-plane angles."""
    xd, yd, zd = case["xd"], case["yd"], case["zd"]
    mat = np.zeros((zd, yd, xd), np.uint8)
    mat[1:zd - 1, 1:yd - 1, 1:xd - 1] = 1
    a = np.random.default_rng(seed).uniform(0, 2 * np.pi, (zd, yd, xd))
    M = (np.stack([np.cos(a), np.sin(a), 0 * a], -1) * float(MS)).astype(F)
    M[mat == 0] = 0
    return mat.ravel(), M.ravel()


def _weights(seed):
    """Network weights of the spread that training starts from."""
    rng = np.random.default_rng(seed + 77)

    def nrm(count, fan):
        return rng.standard_normal(count, dtype=F) * F(math.sqrt(2.0 / fan))
    z = np.zeros(CH, F)
    return np.concatenate([nrm(CH * 27, 27), z, nrm(CH * CH * 9, CH * 9), z, nrm(CH * CH * 9, CH * 9), z,
                           nrm(NM * NM * CH * CH, 16 * CH), nrm(CH * CH * 9, CH * 9), z, nrm(CH, CH), z[:1]])


def _pairs(case, seed):
    """Charges and (unit-scale, smooth) target potentials of a training batch."""
    xd, yd, zd = case["xd"], case["yd"], case["zd"]
    rho, phi = [], []
    for f in range(case["batch"]):
        q = _charge(xd, yd, zd, ("random", "domains", "dots")[f % 3], seed * 31 + f)
        rho.append(q)
        t = q.astype(np.float64).reshape(zd, yd, xd)
        for ax in (1, 2):
            t = sum(np.roll(t, k, ax) for k in range(-4, 5)) / 9
        phi.append((t * float(CELL) ** 2).astype(F).ravel())
    return np.stack(rho), np.stack(phi)


def _d(case):
    return CELL, CELL, F(CELL * F(case["dz"]))


def prepare(case, seed):
    k = case["kind"]
    if k in ("exact", "reforder"):
        dims = (case["xd"], case["yd"], case["zd"])
        return dict(kind=k, dims=dims, d=_d(case), q=_charge(*dims, "random", seed))
    if k == "march":
        mat, M = _march_state(case, seed)
        return dict(kind=k, case=case, mat=mat, M=M, d=_d(case), dir=tempfile.TemporaryDirectory(prefix="march_"))
    if k == "film":
        mat, M = _film_state(case["xd"], case["yd"], case["zd"], case["state"], seed)
        f = mg.Film(case["xd"], case["yd"], case["zd"], *_d(case),
                    solver=mg.SOLVER_FMM if case["solver"] == "fmm" else mg.SOLVER_DIRECT, P=case["P"],
                    m2l_precision=FORMS[case["form"]], leaf_width=case["leaf"], mu_0=MU_0, Ms=MS, Aexch=AEXCH,
                    alfa=ALFA, gamma=GAMMA, external=mg.EXT_CONST, hext=(case["hx"], 0.0, 0.0), material=mat)
        f.set_m(M)
        return dict(kind=k, film=f, steps=case["steps"], dt=case["dt"])
    if k == "rk4":
        mat, M = _film_state(case["xd"], case["yd"], case["zd"], "dots", seed)
        n = mat.size
        return dict(kind=k, case=case, d=_d(case), mat=mat, M=M,
                    out={v: np.zeros(3 * n, F) for v in ("M2", "H", "slope", "this_slope")},
                    charge=np.zeros(n, F), potential=np.zeros(n, F))
    if k == "infer":
        dims = (case["xd"], case["yd"], case["zd"])
        f = mg.Film(*dims, CELL, CELL, CELL, mu_0=MU_0, Ms=MS, Aexch=AEXCH, alfa=ALFA, gamma=GAMMA)
        f.surrogate_init(_weights(seed))
        return dict(kind=k, film=f, q=_charge(*dims, "domains", seed))
    rho, phi = _pairs(case, seed)
    t = mg.SurrogateTrainer(case["xd"], case["yd"], case["zd"], CELL, MS, case["batch"], _weights(seed))
    t.add(rho, phi)
    return dict(kind=k, trainer=t, idx=np.arange(case["batch"]))


def run(s):
    k = s["kind"]
    if k == "exact":
        pot = np.empty_like(s["q"])
        _ok(mg.calc_potential_exact(s["q"], *s["dims"], *s["d"], pot))
        return pot
    if k == "reforder":
        pot = np.empty_like(s["q"])
        _ok(mg.calc_potential_exact_gpu(s["q"], *s["dims"], *s["d"], pot))
        return pot
    if k == "march":
        c, M = s["case"], s["M"].copy()
        _ok(mg.time_marching(s["mat"], M, c["finaltime"], 1e-15, c["xd"], c["yd"], c["zd"], *s["d"], c["P"], MU_0, MS,
                             AEXCH, ALFA, GAMMA, 1, 1, 0, 1, sim_name=s["dir"].name))
        with open(os.path.join(s["dir"].name, "dynamics.dat")) as f:
            steps = sum(1 for _ in f)
        return {"M": M, "steps": steps}
    if k == "film":
        f = s["film"]
        f.steps(s["steps"], s["dt"])
        return f.get_m()
    if k == "rk4":
        c, o = s["case"], s["out"]
        g = (c["xd"], c["yd"], c["zd"], *s["d"], c["P"], MU_0, MS, AEXCH)
        _ok(mg.Hfield(s["M"], o["H"], s["charge"], s["potential"], 0.0, *g, 1, 1, 1, 1))
        st, _ = mg.rk4_step(0.0, c["dt"], s["mat"], s["M"], o["M2"], o["H"], o["slope"], o["this_slope"], s["charge"],
                            s["potential"], *g, ALFA, GAMMA, 1, 1, 1, 1)
        _ok(st)
        return {**o, "charge": s["charge"], "potential": s["potential"]}
    if k == "infer":
        return s["film"].surrogate_potential(s["q"])
    g, loss = s["trainer"].gradient(s["idx"])
    return {"gradient": g, "loss": F(loss)}


def _ok(status):
    if status != 0:
        raise mg.MmsError(mg.last_error())


# ------------------------------------------------------------------- work --
def work(case):
    """Bytes: a call's host arrays once; for steps on a resident film its
    state read and written once a pass.  Operations: a convolution by
    transforms for the direct sums, the order-P operators (near field 2
    operations a pair, M2L 2 K^2 a box pair) for the FMM, the network's
    products for the surrogate."""
    k = case["kind"]

    def fft(xd, yd, zd):
        return 2 * 2.5 * 8 * xd * yd * zd * math.log2(max(2, 8 * xd * yd * zd))

    def fmm(xd, yd, zd, P, leaf):
        K = (P + 1) * (P + 2) / 2
        return xd * yd * zd * (2 * 9 * leaf * leaf * zd + 4 / 3 * 27 * zd * 2 * K * K / (leaf * leaf) + 4 * K)

    dims = (case["xd"], case["yd"], case["zd"])
    n = dims[0] * dims[1] * dims[2]
    if k in ("exact", "reforder"):
        return {"bytes": 8 * n, "flops": fft(*dims) if k == "exact" else 3.0 * n * n}
    if k == "march":
        # about one accepted step per 1.2e-15 s, five evaluations each
        steps = case["finaltime"] / 1.2e-15
        return {"bytes": 25 * n, "flops": fmm(*dims, case["P"], 4) * 5 * steps}
    if k == "film":
        one = fft(*dims) if case["solver"] == "direct" else fmm(*dims, case["P"], case["leaf"])
        return {"bytes": 25 * n, "flops": 4 * case["steps"] * (one + 100.0 * n)}
    if k == "rk4":
        return {"bytes": n * (12 * 6 + 8 + 1), "flops": 4 * (fmm(*dims, case["P"], 4) + 100.0 * n)}
    conv = 2.0 * (27 * CH + 3 * 9 * CH * CH + CH + 4 * NM * CH)
    if k == "infer":
        return {"bytes": 8 * n + 4 * 4306945, "flops": conv * n}
    return {"bytes": 8 * n * case["batch"] + 2 * 4 * 4306945, "flops": 3 * conv * n * case["batch"]}


# ------------------------------------------------------------ 64-bit values --
def _dev():
    return torch.device("cuda" if torch.cuda.is_available() else "cpu")


def _good(n):
    """Smallest 2^a 3^b 5^c >= n."""
    while True:
        m = n
        for p in (2, 3, 5):
            while m % p == 0:
                m //= p
        if m == 1:
            return n
        n += 1


class _Field:
    """Demag, exchange and uniform field of films [B, 3, z, y, x] in 64 bits."""

    def __init__(self, dims, d, hext, exchange=True):
        xd, yd, zd = dims
        self.dims, self.d, self.exchange, self.hext = dims, [float(v) for v in d], exchange, hext
        self.pad = (_good(2 * zd - 1) if zd > 1 else 1, _good(2 * yd - 1), _good(2 * xd - 1))
        axes = []
        for n, p, h in zip((zd, yd, xd), self.pad, self.d[::-1]):
            i = torch.arange(p, device=_dev(), dtype=torch.float64)
            axes.append((torch.minimum(i, p - i) * h) ** 2)
        r = (axes[0][:, None, None] + axes[1][None, :, None] + axes[2][None, None, :]).sqrt()
        g = torch.where(r > 0, self.d[0] * self.d[1] * self.d[2] / r, torch.zeros_like(r))
        self.G = torch.fft.rfftn(g, dim=(-3, -2, -1)).real.contiguous()

    def potential(self, rho):
        xd, yd, zd = self.dims
        f = torch.fft.rfftn(rho, s=self.pad, dim=(-3, -2, -1)) * self.G
        return torch.fft.irfftn(f, s=self.pad, dim=(-3, -2, -1))[..., :zd, :yd, :xd]

    @staticmethod
    def _nb(a, axis, step):
        out = torch.zeros_like(a)
        n = a.shape[axis]
        if n > 1:
            src, dst = (1, 0) if step > 0 else (0, 1)
            out.narrow(axis, dst, n - 1).copy_(a.narrow(axis, src, n - 1))
        return out

    def charge(self, m):
        dx, dy, dz = self.d
        return sum((self._nb(m[:, c], ax, 1) - self._nb(m[:, c], ax, -1)) / (2 * h)
                   for c, ax, h in ((0, -1, dx), (1, -2, dy), (2, -3, dz)))

    def __call__(self, m):
        """(H, charge, potential) at state m."""
        rho = self.charge(m)
        phi = self.potential(rho)
        H = torch.stack([(self._nb(phi, ax, 1) - self._nb(phi, ax, -1)) / (8 * math.pi * h)
                         for ax, h in ((-1, self.d[0]), (-2, self.d[1]), (-3, self.d[2]))], 1)
        if self.exchange:
            cm = 2 * float(AEXCH) / (float(MU_0) * float(MS) ** 2)
            for ax, h in ((-1, self.d[0]), (-2, self.d[1]), (-3, self.d[2])):
                H += cm / h ** 2 * (self._nb(m, ax, 1) + self._nb(m, ax, -1) - 2 * m)
        return H + self.hext, rho, phi


def _slope(m, H):
    c = torch.cross(m, H, dim=1)
    return -float(GAMMA) * c - float(ALFA) * float(GAMMA) / float(MS) * torch.cross(m, c, dim=1)


def _rk4(field, m, mat, dt, H=None):
    """One step of the magnetic cells; returns (M2, last H, slope, last slope, charge, potential)."""
    H = field(m)[0] if H is None else H
    k = _slope(m, H) * mat
    slope = k.clone()
    for h, w in ((0.5, 2.0), (0.5, 2.0), (1.0, 1.0)):
        H, rho, phi = field(m + h * dt * k)
        k = _slope(m + h * dt * k, H) * mat
        slope += w * k
    out = m + dt / 6 * slope
    out = torch.where(mat > 0, out * (float(MS) / out.norm(dim=1, keepdim=True).clamp_min(1e-300)), out)
    return out, H, slope, k, rho, phi


def _to_film(M, dims):
    xd, yd, zd = dims
    return torch.from_numpy(M.reshape(-1, zd, yd, xd, 3)).to(_dev(), torch.float64).permute(0, 4, 1, 2, 3).contiguous()


def _to_host(m):
    return m.permute(0, 2, 3, 4, 1).reshape(-1).cpu().numpy()


def _mat(mat, dims):
    xd, yd, zd = dims
    return torch.from_numpy(mat.reshape(-1, 1, zd, yd, xd)).to(_dev(), torch.float64)


def _uniform(h):
    return torch.tensor(h, dtype=torch.float64, device=_dev()).reshape(-1, 3, 1, 1, 1)


def _exact_march(case, seed):
    dims = (case["xd"], case["yd"], case["zd"])
    mat, M = _march_state(case, seed)
    d = _d(case)
    field, m, mt = _Field(dims, d, _uniform([0.0, 0, 0])), _to_film(M, dims), _mat(mat, dims)
    scale = -0.5 * float(MU_0) * float(d[0] * d[1] * d[2]) / 1.6e-19
    H = field(m)[0]
    t, dt, steps = 0.0, float(F(1e-15)), 0
    while t <= float(F(case["finaltime"])):
        E = float((m * H * mt).sum()) * scale
        m2 = _rk4(field, m, mt, dt, H)[0]
        H2 = field(m2)[0]
        if float((m2 * H2 * mt).sum()) * scale - E > 0.1:
            dt /= 2.5
            continue
        torque = float((torch.cross(m2, H2, dim=1) * mt).norm(dim=1).max()) / float(MS) ** 2
        t, dt, m, H, steps = t + dt, 1e-14 / torque / 2, m2, H2, steps + 1
        if torque < 1e-3:
            break
    return {"M": _to_host(m), "steps": steps}


def _network(w, q, batch, dims):
    """The surrogate in 64 bits: charge [batch * z, y, x] in units of Ms / dx
    -> potential in units of Ms dx (w: the weight vector, a tensor)."""
    xd, yd, zd = dims
    at = [0]

    def take(*shape):
        n = math.prod(shape)
        at[0] += n
        return w[at[0] - n:at[0]].reshape(shape)
    lift, bl = take(CH, 3, 3, 3), take(CH)
    w1, b1, w2, b2 = take(CH, CH, 3, 3), take(CH), take(CH, CH, 3, 3), take(CH)
    mode, w3, b3, wp, bp = take(NM, NM, CH, CH), take(CH, CH, 3, 3), take(CH), take(CH), take(1)

    def conv(a, k):  # [B, y, x, ci] by taps [co, ci, 3, 3]
        p = torch.nn.functional.pad(a, (0, 0, 1, 1, 1, 1))
        return sum(p[:, i:i + yd, j:j + xd] @ k[:, :, i, j].T for i in range(3) for j in range(3))

    def gelu(a):
        return 0.5 * a * (1 + torch.tanh(0.7978845608 * (a + 0.044715 * a * a * a)))

    def basis(n):
        x = torch.arange(n, dtype=torch.float64, device=q.device)
        rows = [torch.ones_like(x)]
        for k in range(1, NM):
            a = 2 * math.pi * ((k + 1) // 2) * x / n
            rows.append(torch.cos(a) if k % 2 else torch.sin(a))
        return math.sqrt(2.0 / n) * torch.stack(rows)

    f = q.reshape(batch, zd, yd, xd)
    near = torch.zeros_like(f)
    near[:, 1:] += f[:, :-1]
    near[:, :-1] += f[:, 1:]
    planes = torch.stack([f, near, f.sum(1, keepdim=True) - f - near], -1).reshape(batch * zd, yd, xd, 3)
    h1 = gelu(conv(gelu(conv(planes, lift) + bl), w1) + b1)
    Bx, By = basis(xd), basis(yd)
    X = (h1.transpose(2, 3).reshape(-1, xd) @ Bx.T).reshape(batch * zd, yd, CH, NM)       # [B, y, c, kx]
    H = (X.permute(0, 2, 3, 1).reshape(-1, yd) @ By.T).reshape(batch * zd, CH, NM, NM)     # [B, c, kx, ky]
    H = H.permute(3, 2, 0, 1).contiguous()                                                 # [ky, kx, B, c]
    G = torch.stack([H[i] @ mode[i].transpose(1, 2).contiguous() for i in range(NM)])
    X2 = (G.permute(1, 2, 3, 0).reshape(-1, NM) @ By).reshape(NM, batch * zd, CH, yd)      # [kx, B, c, y]
    S = (X2.permute(1, 3, 2, 0).reshape(-1, NM) @ Bx).reshape(batch * zd, yd, CH, xd).transpose(2, 3)
    h3 = gelu(conv(gelu(conv(h1, w2) + b2 + S), w3) + b3)
    return h3 @ wp + bp


def exact(case, seed):
    k = case["kind"]
    if k == "march":
        return _exact_march(case, seed)
    dims = (case["xd"], case["yd"], case["zd"])
    if k in ("exact", "reforder"):
        q = torch.from_numpy(_charge(*dims, "random", seed)).to(_dev(), torch.float64)
        return _Field(dims, _d(case), 0.0).potential(q.reshape(1, *dims[::-1])).reshape(-1).cpu().numpy()
    if k == "film":
        mat, M = _film_state(*dims, case["state"], seed)
        field = _Field(dims, _d(case), _uniform([float(F(case["hx"])), 0.0, 0.0]))
        m, mt = _to_film(M, dims), _mat(mat, dims)
        for _ in range(case["steps"]):
            m = _rk4(field, m, mt, float(F(case["dt"])))[0]
        return _to_host(m)
    if k == "rk4":
        mat, M = _film_state(*dims, "dots", seed)
        field = _Field(dims, _d(case), _uniform([0.3 * float(F(1) / MU_0), 0.0, 0.0]))
        got = _rk4(field, _to_film(M, dims), _mat(mat, dims), float(F(case["dt"])))
        return {**{n: _to_host(v) for n, v in zip(("M2", "H", "slope", "this_slope"), got)},
                "charge": got[4].reshape(-1).cpu().numpy(), "potential": got[5].reshape(-1).cpu().numpy()}
    w = torch.from_numpy(_weights(seed)).to(_dev(), torch.float64)
    unit_q, unit_p = float(CELL / MS), float(MS * CELL)
    if k == "infer":
        q = torch.from_numpy(_charge(*dims, "domains", seed)).to(_dev(), torch.float64) * unit_q
        with torch.no_grad():
            return (_network(w, q, 1, dims) * unit_p).reshape(-1).cpu().numpy()
    rho, phi = (torch.from_numpy(a).to(_dev(), torch.float64) for a in _pairs(case, seed))
    w.requires_grad_(True)
    out = (_network(w, rho.reshape(-1) * unit_q, case["batch"], dims) * unit_p).reshape(case["batch"], -1)
    loss = (((out - phi) ** 2).sum(1) / (phi ** 2).sum(1)).mean()
    loss.backward()
    return {"gradient": w.grad.cpu().numpy(), "loss": np.float64(loss.detach().cpu().item())}
