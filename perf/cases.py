"""The calls by which the speed of this repository is judged, over the sizes,
directions, precision modes and options that its users run.

listed() gives them, draw() more of the same ranges, prepare() the inputs and
handles that a user's program holds before the call, run() one call (or, for
the resident contexts, one run() of `inner` SD steps and the read-back of what
it computes), work() what a call cannot do without and exact() the same
results from plain torch in 64 bits.

Kinds of case:
  sd     DeviceSD.run(): `inner` steepest-descent steps and the energy
         evaluation on orbitals that stay on the GPU, `nmol` water molecules
         in an `edge`-bohr cell on a `grid`^3 FFT grid with `ne` orbitals.
         The density and the Hamiltonian and Lagrange matrices are read back;
         with `orbitals` the updated orbitals too.  A run of hundreds of calls
         reads large orbitals back once, at its end, so the large cells leave
         them on the device.
  batch  Batch.run(): `count` independent small cells, one call.
  dropin cpsd(): the reference's own entry point on host arrays, which it
         reads and fills on every call.
  fft    the allocation-free FFT entry point on device arrays: `nbatch`
         half-complex fields to real space, and as many real fields back.
  train  cpsd_mlp_train(): `iters` Adam steps of the per-G network over `n`
         samples (a forward and a backward pass each).
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "simple-cpsd_amd"))
import cpsd_amd  # noqa: E402
import learned  # noqa: E402

DT, FMASS = 5.8, 400000.0      # the time step and fictitious mass of every workload
DTE = DT / math.sqrt(FMASS)
KMAX = 8.0                     # largest factor of the kinetic preconditioner
LR = 3e-3                      # Adam step of the training case


# ----------------------------------------------------------------- the cases

def _sd(name, nmol, edge, grid, ne, inner=10, mode=0, precond=False, move=False, graphs=False, orbitals=False):
    return dict(name=name, kind="sd", nmol=nmol, edge=edge, grid=grid, ne=ne, inner=inner, mode=mode,
                precond=precond, move=move, graphs=graphs, orbitals=orbitals)


def listed():
    return [
        # one water molecule, the smallest workload of the benchmark: launches and latency
        _sd("water1-32", 1, 20.0, 32, 4, orbitals=True),
        # a small cell with an odd number of orbitals, replayed from a HIP graph
        _sd("water5-48-odd", 5, 17.6, 48, 21, graphs=True, orbitals=True),
        # ions that move every step, so projectors and forces are formed in each (molecular dynamics of a cluster)
        _sd("water8-64-move", 8, 14.8, 64, 32, move=True),
        # a medium cell in single-precision steps with a preconditioner: geometry scans, training cells
        _sd("water16-80-mode1-K", 16, 16.0, 80, 64, mode=1, precond=True),
        # the 32-water liquid cell, the reference's step
        _sd("water32-96", 32, 18.6, 96, 128),
        # the same cell as it is converged fastest: split-BF16 products and a preconditioner
        _sd("water32-96-mode3-K", 32, 18.6, 96, 128, mode=3, precond=True),
        # the 64-water liquid cell, the largest workload of the benchmark, the reference's step
        _sd("water64-128", 64, 23.5, 128, 256),
        # and as it is converged fastest
        _sd("water64-128-mode3-K", 64, 23.5, 128, 256, mode=3, precond=True),
        # many small cells of uneven size at once (screening of clusters), one call for all
        dict(name="batch16-mode1", kind="batch", count=16, sizes_seed=0, inner=10, mode=1),
        # a program of the reference relinked: host arrays in and out of every call
        dict(name="dropin-water4-48", kind="dropin", nmol=4, edge=16.3, grid=48, ne=16, inner=10),
        # the FFT layer on its own, both directions
        dict(name="fft-96x8", kind="fft", grid=96, nbatch=8),
        # training of the learned preconditioner on one 32-water cell's G vectors
        dict(name="train-235k", kind="train", n=234980, iters=50),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _water(rng, top):
    """molecules, cell edge, grid and orbitals: clusters of up to 8 molecules in 12-22 bohr cells, liquid
    density above; orbital counts with and without empty states above the four per molecule"""
    nmol = _log_int(rng, 1, top)
    if nmol <= 8:
        edge = round(12.0 + 10.0 * (nmol - 1) / 7.0 + rng.uniform(-0.4, 0.4), 2)
        grid = rng.choice([g for g in (24, 32, 40, 48, 64) if g >= 24 + 2 * nmol])
    else:
        edge = round(18.6 * (nmol / 32.0) ** (1.0 / 3.0) + rng.uniform(-0.3, 0.3), 2)
        grid = rng.choice([64, 80, 96] if nmol <= 24 else [80, 96])
    ne = 4 * nmol + rng.choice([0, 0, 0, 0, 1, 2, 5])
    return nmol, edge, grid, ne


def draw(rng):
    kind = rng.choice(["sd"] * 6 + ["batch", "dropin", "fft", "train"])
    if kind == "sd":
        nmol, edge, grid, ne = _water(rng, 40)
        mode = rng.choice([0, 0, 0, 1, 3 if ne in (128, 256) else 1])
        move = mode < 2 and nmol <= 24 and rng.random() < 0.2
        c = _sd(None, nmol, edge, grid, ne, inner=rng.choice([5, 10, 10]), mode=mode, move=move,
                precond=not move and rng.random() < 0.4, graphs=not move and rng.random() < 0.3,
                orbitals=ne <= 20)
        del c["name"]
        return c
    if kind == "batch":
        return dict(kind="batch", count=rng.randint(3, 24), sizes_seed=rng.randrange(1000), inner=rng.choice([5, 10]),
                    mode=rng.choice([0, 1]))
    if kind == "dropin":
        nmol, edge, grid, ne = _water(rng, 8)
        return dict(kind="dropin", nmol=nmol, edge=edge, grid=grid, ne=ne, inner=rng.choice([1, 5, 10]))
    if kind == "fft":
        grid = rng.choice([8, 12, 16, 20, 24, 32, 40, 48, 64, 80, 96, 128])
        return dict(kind="fft", grid=grid, nbatch=_log_int(rng, 1, max(1, min(200, 7000000 // grid ** 3))))
    return dict(kind="train", n=_log_int(rng, 5000, 700000), iters=rng.randint(10, 60))


# ---------------------------------------------------------------- the inputs

def _gen(seed):
    g = torch.Generator(device=_dev())
    g.manual_seed(int(seed))
    return g


def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def _weights(n):
    """of the half-complex G-space inner product, per kx"""
    w = torch.full((n // 2 + 1,), 2.0, dtype=torch.float64, device=_dev())
    w[0] = 1.0
    return w


def _orbitals(cell, ne, seed):
    """complex Gaussian coefficients on the masked G vectors, orthonormalised, in the reference's layout"""
    idx = torch.from_numpy(np.flatnonzero(cell.masker[0::2])).to(_dev())
    w = _weights(cell.nfft)[idx % (cell.nfft // 2 + 1)]
    c = torch.randn((ne, idx.numel(), 2), dtype=torch.float64, device=_dev(), generator=_gen(seed))
    a = c.reshape(ne, -1)
    L = torch.linalg.cholesky((a * w.repeat_interleave(2)) @ a.T)
    a = torch.linalg.inv(L) @ a
    full = torch.zeros((ne, cell.nfft3d, 2), dtype=torch.float64, device=_dev())
    full[:, idx] = a.reshape(ne, -1, 2)
    return full.reshape(-1).cpu().numpy()


def _factors(cell):
    return learned.kinetic_factor(cell.tg, KMAX, 1.0)


def _batch_cells(case, seed):
    return [(cpsd_amd.water_cell(m, L, n, seed=seed * 100 + i), 4 * m, seed * 100 + i)
            for i, (m, L, n) in enumerate(cpsd_amd.water_batch_specs(case["sizes_seed"], case["count"]))]


def _fields(case, seed):
    """half-complex fields with the decay of a pseudo-density's spectrum, and real fields"""
    n, nb = case["grid"], case["nbatch"]
    g = _gen(seed)
    k = torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64, device=_dev())
    k2 = (k[:, None, None] ** 2 + k[None, :, None] ** 2
          + torch.arange(n // 2 + 1, device=_dev(), dtype=torch.float64)[None, None, :] ** 2)
    x = torch.randn((nb, n, n, n // 2 + 1, 2), dtype=torch.float64, device=_dev(), generator=g)
    x *= torch.exp(-8.0 * k2 / n ** 2)[None, ..., None]
    r = torch.zeros((nb, n, n, n + 2), dtype=torch.float64, device=_dev())
    r[..., :n] = torch.randn((nb, n, n, n), dtype=torch.float64, device=_dev(), generator=g)
    return x, r


def _samples(case, seed):
    """features, weights and targets distributed as those of a water cell's G vectors"""
    rng = np.random.default_rng(seed)
    n = case["n"]
    t = 130.0 * rng.random(n) ** (2.0 / 3.0)        # |G|^2/2 over the cutoff sphere
    X = np.stack([np.log1p(t) / 5.0, t / (1.0 + t), np.arcsinh(-3.0 * np.exp(-0.1 * t) * rng.random(n)),
                  np.arcsinh(2.0 * np.exp(-0.2 * t) * rng.random(n))], axis=1).astype(np.float32)
    target = learned.kinetic_factor(t, KMAX, 1.0) * np.exp(0.1 * rng.standard_normal(n))
    w = (np.exp(-0.05 * t) / np.exp(-0.05 * t).sum() + 1.0 / n) / target ** 2
    return X, w, w * target, learned.init_params(seed)


def prepare(case, seed):
    if case["kind"] == "sd":
        cell = cpsd_amd.water_cell(case["nmol"], case["edge"], case["grid"], seed=seed)
        dev = cpsd_amd.DeviceSD(cell, case["ne"])
        dev.set_graphs(case["graphs"])
        if case["move"]:
            dev.set_ions(1)
        dev.set_precision(case["mode"])
        if case["precond"]:
            dev.set_preconditioner(_factors(cell))
        dev.set_orbitals(_orbitals(cell, case["ne"], seed))
        if case["precond"]:
            dev.run(case["inner"], DT, FMASS)      # the preconditioned steps start with the second call
        return dict(case=case, dev=dev)
    if case["kind"] == "batch":
        devs = []
        for cell, ne, s in _batch_cells(case, seed):
            d = cpsd_amd.DeviceSD(cell, ne)
            d.set_precision(case["mode"])
            d.set_orbitals(_orbitals(cell, ne, s))
            devs.append(d)
        return dict(case=case, devs=devs, batch=cpsd_amd.Batch(devs))
    if case["kind"] == "dropin":
        cell = cpsd_amd.water_cell(case["nmol"], case["edge"], case["grid"], seed=seed)
        return dict(case=case, cell=cell, c2=_orbitals(cell, case["ne"], seed), E=np.zeros(10))
    if case["kind"] == "fft":
        x, r = _fields(case, seed)
        return dict(case=case, x=x, r=r, a=torch.empty_like(x), b=torch.empty_like(r))
    X, A, B, p = _samples(case, seed)
    return dict(case=case, X=X, A=A, B=B, p=p)


# ------------------------------------------------------------------ the calls

def _read(dev, orbitals):
    return dev.get(c2=orbitals, dn=True, hml=True, lmd=True)


def _batch_out(cells):
    """energies and deltas of all cells, then every cell's density and Hamiltonian matrix"""
    return dict(E=np.array([c["E"] for c in cells]), delta=np.array([(c["deltae"], c["deltac"]) for c in cells]),
                dn=[c["dn"] for c in cells], hml=[c["hml"] for c in cells])


def run(state):
    case = state["case"]
    if case["kind"] == "sd":
        dev = state["dev"]
        E, de, dc = dev.run(case["inner"], DT, FMASS)
        out = dict(E=E, deltae=de, deltac=dc, **_read(dev, case["orbitals"]))
        if case["move"]:
            out.update(dev.get_ions())
        return out
    if case["kind"] == "batch":
        res = state["batch"].run(case["inner"], DT, FMASS)
        return _batch_out([dict(E=E, deltae=de, deltac=dc, **d.get(dn=True, hml=True))
                           for (E, de, dc), d in zip(res, state["devs"])])
    if case["kind"] == "dropin":
        out = cpsd_amd.cpsd_dropin(state["cell"], case["ne"], case["inner"], state["c2"], state["E"], DT, FMASS)
        state["c2"], state["E"] = out["c2"], out["E"]
        return {k: out[k] for k in ("c1", "c2", "cpsi", "dn", "hml", "lmd", "E", "deltae", "deltac")}
    if case["kind"] == "fft":
        # the transforms are in place and the program keeps its fields
        stream = torch.cuda.current_stream().cuda_stream
        for way, src, dst in ((+1, state["x"], state["a"]), (-1, state["r"], state["b"])):
            dst.copy_(src)
            if cpsd_amd.hip_lib().cpsd_fft3d_batch_noalloc(way, case["grid"], case["nbatch"], dst.data_ptr(), stream):
                raise RuntimeError(cpsd_amd.hip_lib().cpsd_last_error().decode())
        return state["a"], state["b"]
    p, hist = cpsd_amd.mlp_train(state["X"], state["A"], state["B"], state["p"], case["iters"], LR)
    return p, hist


# ------------------------------------------------------------------- the work

def _step_work(nmol, n, ne, precond, move):
    """one SD step: orbitals in and out, projectors and potentials read; a forward and an inverse FFT of
    every orbital, the KB projection and apply, the overlaps and the constraint"""
    ng = math.pi / 12.0 * n ** 3
    nproj = 6 * nmol
    b = 16.0 * ng * (2 * ne + nproj) + 8.0 * 4 * n ** 3
    f = ne * 2 * 2.5 * n ** 3 * math.log2(n ** 3) + 8.0 * ng * ne * (nproj + 1.5 * ne)
    if precond:
        f += 4.0 * ng * ne * ne
    if move:
        f += 4.0 * ng * ne * nproj
    return b, f


def work(case):
    if case["kind"] in ("sd", "dropin", "batch"):
        if case["kind"] == "batch":
            cells = [(m, n, 4 * m) for m, _, n in cpsd_amd.water_batch_specs(case["sizes_seed"], case["count"])]
        else:
            cells = [(case["nmol"], case["grid"], case["ne"])]
        tot = [_step_work(m, n, ne, case.get("precond", False), case.get("move", False)) for m, n, ne in cells]
        b, f = (case["inner"] * sum(t[k] for t in tot) for k in (0, 1))
        return {"bytes": b, "flops": f}
    if case["kind"] == "fft":
        n, nb = case["grid"], case["nbatch"]
        return {"bytes": 2.0 * nb * 2 * 8 * n * n * (n + 2), "flops": 2.0 * nb * 2.5 * n ** 3 * math.log2(n ** 3)}
    return {"bytes": 24.0 * case["n"], "flops": 6.0 * (4 * 32 + 32 * 32 + 32) * case["n"] * case["iters"]}


# ------------------------------------------------- the same results in 64 bits

class _Plain:
    """the SD step in plain torch, FP64, on the masked G vectors"""

    def __init__(self, cell, ne, c):
        n, d = cell.nfft, _dev()
        nh = n // 2 + 1
        t = lambda v: torch.from_numpy(np.ascontiguousarray(v)).to(d)  # noqa: E731
        self.cell, self.n, self.ne = cell, n, ne
        self.idx = t(np.flatnonzero(cell.masker[0::2]))
        self.kx, self.ky, self.kz = self.idx % nh, self.idx // nh % n, self.idx // (nh * n)
        self.w = _weights(n)[self.kx]
        self.wr = self.w.repeat_interleave(2)
        self.tg, self.vc, self.vg = (t(v)[self.idx] for v in (cell.tg, cell.vc, cell.vg))
        self.G = t(cell.G).reshape(3, -1)[:, self.idx]
        self.vl = t(cell.vl).reshape(cell.nkind, -1)[:, self.idx]
        self.vnl = t(cell.vnl).reshape(cell.nkind, 9, -1)[:, :, self.idx]
        self.c = torch.view_as_complex(t(c).reshape(ne, cell.nfft3d, 2)[:, self.idx].contiguous())
        self.r = t(cell.r).reshape(-1, 3)
        self.structure()

    def structure(self):
        cell, n = self.cell, self.n
        ub = torch.from_numpy(cell.unitg).to(_dev()).reshape(3, 3)
        self.s = torch.zeros_like(self.c[0])
        self.vall = torch.zeros_like(self.c[0])
        self.exi, beta, nrm, ion = [], [], [], []
        sg = [k - n * (k > n // 2).to(k.dtype) for k in (self.kx, self.ky, self.kz)]
        for i, ia in enumerate(cell.katm):
            ph = ub @ self.r[i] + math.pi
            a = ph[0] * sg[0] + ph[1] * sg[1] + ph[2] * sg[2]
            e = torch.complex(torch.cos(a), -torch.sin(a))
            self.exi.append(e)
            self.s += cell.zv[ia] * e
            self.vall += self.vl[ia] * e
            for lm in range(cell.lmmax[ia]):
                beta.append(e * self.vnl[ia, lm] * (1j if 1 <= lm <= 3 else 1.0))
                nrm.append(cell.vnlnrm[9 * ia + lm])
                ion.append(i)
        self.B = torch.stack(beta)
        self.nrm = torch.tensor(nrm, dtype=torch.float64, device=_dev())
        self.pion = torch.tensor(ion, device=_dev())

    def dot(self, a, b):
        return (torch.view_as_real(a).flatten(1) * self.wr) @ torch.view_as_real(b.resolve_conj()).flatten(1).T

    def up(self, g):
        """masked G to real space, unnormalised"""
        f = torch.zeros((g.shape[0], self.n ** 2 * (self.n // 2 + 1)), dtype=g.dtype, device=g.device)
        f[:, self.idx] = g
        f = torch.fft.ifftn(f.reshape(-1, self.n, self.n, self.n // 2 + 1), dim=(1, 2), norm="forward")
        f[..., 0].imag.zero_()
        f[..., -1].imag.zero_()
        return torch.fft.irfft(f, n=self.n, norm="forward")

    def down(self, r):
        return torch.fft.rfftn(r, dim=(1, 2, 3)).flatten(1)[:, self.idx]

    @staticmethod
    def lda(d):
        """Slater exchange and Vosko-Wilk-Nusair correlation, the reference's parameters"""
        n13 = (6.0 * d / math.pi) ** (1.0 / 3.0)
        rs = 0.620350490899400 / (2.0 * (d + 1e-30)) ** 0.333333333333333
        x = rs.sqrt()
        xx = rs + 3.72744 * x + 12.9352
        ec = (3.10907e-2 * torch.log(rs / xx) + 9.690228e-4 * torch.log((x + 0.10498) ** 2 / xx)
              + 3.878329e-2 * torch.atan(3.075995 / (x + 1.86372)))
        uc = ec - 0.166666666666667 * x * (6.21814e-2 / x + 1.938045e-3 / (x + 0.10498)
                                           - 3.205972e-2 * (2.0 * x + 3.72744) / xx
                                           - 0.1192972 / ((x + 1.86372) ** 2 + 9.461748))
        return -n13 + uc, -0.75 * n13 + ec

    def pairs(self):
        """real-space Ewald pairs: displacements of every image, their lengths and charge products"""
        c = self.cell
        i, j = np.triu_indices(c.nion, 1)
        img = torch.from_numpy(c.rcell.reshape(3, 27)).to(_dev()).T
        x = (self.r[i] - self.r[j])[:, None, :] + img[None]
        zz = torch.from_numpy(c.zv[c.katm[i]] * c.zv[c.katm[j]]).to(_dev())
        r = x.norm(dim=-1)
        w = r / c.rcut
        p = 1.0 + w * (0.0705230784 + w * (0.0422820123 + w * (0.0092705272 + w * (
            0.0001520143 + w * (0.0002765672 + w * 0.0000430638)))))
        return i, j, x, r, w, p ** -16.0, zz[:, None]

    def forces(self, c1, dng, sw):
        c, om = self.cell, self.cell.omega
        f = torch.zeros_like(self.r)
        for i, ia in enumerate(c.katm):
            v = self.exi[i] * self.vl[ia]
            f[i] += self.G @ (self.w * (dng.imag * v.real - dng.real * v.imag))
            e = self.exi[i]
            f[i] += self.G @ (self.w * self.vg * (e.real * self.s.imag - e.imag * self.s.real)) * c.zv[ia] / om
        z = sw.to(c1.dtype) @ c1
        f.index_add_(0, self.pion, -4.0 * (self.w * (z.imag * self.B.real - z.real * self.B.imag)) @ self.G.T)
        i, j, x, r, w, erfc, zz = self.pairs()
        g = (x * (zz * (erfc + 1.128379167 * w * torch.exp(-w * w)) / r ** 3)[..., None]).sum(1)
        f.index_add_(0, torch.from_numpy(i).to(_dev()), g)
        f.index_add_(0, torch.from_numpy(j).to(_dev()), -g)
        return f

    def lagrange(self, c1, c2, project):
        eye = torch.eye(self.ne, dtype=torch.float64, device=_dev())
        a11, a12, a22, d = self.dot(c1, c1), self.dot(c1, c2), self.dot(c2, c2), 0.0
        if project:
            d = a12 - eye
            a22 = a22 - d.T @ a12 - a12.T @ d + d.T @ a11 @ d
            a12 = a12 - a11 @ d
            s12 = (eye - a12) / 2
            s21 = s12.T
        else:
            up = torch.triu(a12), torch.triu(a12.T)
            s12, s21 = ((eye - (u + u.T - torch.diag(torch.diag(u)))) / 2 for u in up)
        s22, s11 = (eye - a22) / (2 * DTE), -a11 * DTE / 2
        X = s22
        for _ in range(30):
            Y = s22 + s21 @ X + X @ s12 + X @ (s11 @ X)
            done = (Y - X).abs().max() < 1e-15
            X = Y
            if done:
                break
        return X - d / DTE

    def steps(self, inner, Eold, K=None, h=None, move=False):
        """`inner` steps and the energy evaluation: everything a call returns"""
        c, n, om = self.cell, self.n, self.cell.omega
        scal1, scal2 = 1.0 / n ** 3, 1.0 / om
        for _ in range(inner):
            if move:
                self.structure()
            c1 = self.c
            dn = torch.zeros((n, n, n), dtype=torch.float64, device=_dev())
            step = max(1, 2 ** 25 // n ** 3)
            for b in range(0, self.ne, step):
                dn += scal2 * (self.up(c1[b:b + step]) ** 2).sum(0)
            dng = self.down(2.0 * scal1 * dn[None])[0]
            xcp, xce = self.lda(dn)
            V = self.up((self.vall * scal2 + dng * self.vc)[None])[0] + xcp
            P = self.dot(self.B, c1)
            sw = -P * scal2 / self.nrm[:, None]
            cp = -self.tg * c1 + sw.T.to(c1.dtype) @ self.B
            for b in range(0, self.ne, step):
                cp[b:b + step] -= scal1 * self.down(self.up(c1[b:b + step]) * V)
            c2 = c1 + DTE * cp
            if K is not None:
                c2 = c1 + K * DTE * (cp + h.T.to(c1.dtype) @ c1)
            lmd = self.lagrange(c1, c2, K is not None)
            self.c = c2 + DTE * (lmd.T.to(c1.dtype) @ c1)
            r1, f = self.r, None
            if move:
                f = self.forces(c1, dng, sw)
                m = torch.from_numpy(c.amass[c.katm]).to(_dev())[:, None]
                self.r = r1 + DT / m.sqrt() * f
        u = torch.triu(-self.dot(c1, cp))
        hml = u + u.T - torch.diag(torch.diag(u))
        save, self.r = self.r, r1
        _, _, _, r, _, erfc, zz = self.pairs()
        self.r = save
        dot1 = lambda a, b: (self.w * (a.real * b.real + a.imag * b.imag)).sum().item()  # noqa: E731
        E = np.zeros(10)
        E[1] = 2.0 * torch.diag(hml).sum().item()
        E[4] = dot1(self.s, self.s * self.vg) * 0.5 * scal2 + c.cewald + (zz * erfc / r).sum().item()
        E[2] = dot1(dng, dng * self.vc) * om * 0.5
        E[3] = 2.0 * (dn * xce).sum().item() * om * scal1
        E[9] = 2.0 * (dn * xcp).sum().item() * om * scal1
        E[5] = 2.0 * torch.diag(self.dot(c1, c1 * self.tg)).sum().item()
        E[6] = dot1(self.vall, dng)
        E[7] = 2.0 * (P ** 2 * scal2 / self.nrm[:, None]).sum().item()
        E[8] = 2.0 * E[2]
        E[0] = E[1] + E[4] + E[3] - E[2] - E[9]
        d = self.c - c1
        pad = torch.zeros((n, n, n + 2), dtype=torch.float64, device=_dev())
        pad[..., :n] = dn
        flat = lambda m: m.T.reshape(-1).cpu().numpy()  # noqa: E731
        out = dict(E=E, deltae=float(E[0] - Eold) / (DT * inner),
                   deltac=torch.diag(self.dot(d, d)).max().item() / DTE, dn=pad.reshape(-1).cpu().numpy(),
                   hml=flat(hml), lmd=flat(lmd))
        if move:
            out.update(r1=r1.reshape(-1).cpu().numpy(), r2=self.r.reshape(-1).cpu().numpy(),
                       fion=f.reshape(-1).cpu().numpy())
        self.h, self.c1, self.cp = hml, c1, d
        return out

    def full(self, c):
        f = torch.zeros((self.ne, self.cell.nfft3d), dtype=c.dtype, device=c.device)
        f[:, self.idx] = c
        return torch.view_as_real(f).reshape(-1).cpu().numpy()


def _exact_train(case, seed):
    X, A, B, p = _samples(case, seed)
    t = lambda v: torch.from_numpy(np.asarray(v, dtype=np.float32)).to(_dev()).double()  # noqa: E731
    X, A, B = t(X), t(A), t(B)
    p = t(p).requires_grad_(True)
    m, v, hist = torch.zeros_like(p), torch.zeros_like(p), []
    for it in range(1, case["iters"] + 1):
        w1, b1, w2, b2, w3, b3 = torch.split(p, [128, 32, 1024, 32, 32, 1])
        h = torch.tanh(X @ w1.reshape(4, 32) + b1)
        y = torch.tanh(h @ w2.reshape(32, 32) + b2) @ w3 + b3
        K = torch.exp(torch.clamp(y, max=12.0))
        loss = (A * K * K - 2.0 * B * K).sum()
        g, = torch.autograd.grad(loss, p)
        hist.append(loss.item())
        with torch.no_grad():
            m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
            p -= LR * (m / (1 - 0.9 ** it)) / ((v / (1 - 0.999 ** it)).sqrt() + 1e-8)
    return p.detach().cpu().numpy(), np.array(hist)


def exact(case, seed):
    if case["kind"] == "sd":
        cell = cpsd_amd.water_cell(case["nmol"], case["edge"], case["grid"], seed=seed)
        s = _Plain(cell, case["ne"], _orbitals(cell, case["ne"], seed))
        E, K, h = 0.0, None, None
        if case["precond"]:
            E = s.steps(case["inner"], E)["E"][0]
            K, h = torch.from_numpy(_factors(cell)).to(_dev())[s.idx], s.h
        out = s.steps(case["inner"], E, K, h, case["move"])
        if case["orbitals"]:
            out["c2"] = s.full(s.c)
        return out
    if case["kind"] == "batch":
        return _batch_out([_Plain(cell, ne, _orbitals(cell, ne, s)).steps(case["inner"], 0.0)
                           for cell, ne, s in _batch_cells(case, seed)])
    if case["kind"] == "dropin":
        cell = cpsd_amd.water_cell(case["nmol"], case["edge"], case["grid"], seed=seed)
        s = _Plain(cell, case["ne"], _orbitals(cell, case["ne"], seed))
        out = s.steps(case["inner"], 0.0)
        out.update(c1=s.full(s.c1), c2=s.full(s.c), cpsi=s.full(s.cp))
        return out
    if case["kind"] == "fft":
        x, r = _fields(case, seed)
        n = case["grid"]
        f = torch.fft.ifftn(torch.view_as_complex(x), dim=(1, 2), norm="forward")
        f[..., 0].imag.zero_()
        f[..., -1].imag.zero_()
        a = torch.zeros_like(r)
        a[..., :n] = torch.fft.irfft(f, n=n, norm="forward")
        b = torch.fft.rfftn(r[..., :n], dim=(1, 2, 3))
        return a.reshape(x.shape), torch.view_as_real(b).reshape(r.shape)
    return _exact_train(case, seed)
