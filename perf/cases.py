"""Performance cases of the multislice framework.

Each case is work that a user's program hands to namsa_amd through its public
entry points: probe scans over the compiled grid sizes (one probe position to
over a thousand, thin and thick specimens, CBEDs, fused detectors, exit
waves), the preparation of a new specimen, a batch of materials as one graph,
a training-set sample with its records, detector integrals of stored CBEDs,
and the learned coarse-slice corrector in inference and in training.

`exact` restates each result in 64 bits with plain torch and numpy.
"""
import math

import numpy as np
import torch

import namsa_amd._lib as L
from namsa_amd import DEFAULT_PROBE, MSAGPU, corrector, records
from namsa_amd.batch import MaterialBatch
from namsa_amd.msa import KIRKLAND_PATH

DEV = "cuda" if torch.cuda.is_available() else "cpu"
SIZES = (128, 192, 256, 384, 512, 768, 1024, 2048)
WEIGHTS = KIRKLAND_PATH.parent / "corrector_c4_f8.npz"
KV, SEMI, PIX = 200.0, 0.025, 0.125
DENSITY = 0.06          # atoms per cubic Angstrom of the specimens
PROBE = dict(DEFAULT_PROBE, scherzer=False, aberration_dict={"C1": 60.0, "C3": 1.0e4, "C5": 0.0})


# ------------------------------------------------------------------ the cases
def listed():
    return [
        # one CBED of a 104-slice crystal slab: the smallest call, latency and launches
        dict(name="probe-256", work="scan", n=256, scan=1, scan_y=1, slices=104, dz=2.0, output="cbed", detectors=0),
        # a fast low-resolution 4D-STEM map, odd raster
        dict(name="scan-128", work="scan", n=128, scan=33, scan_y=33, slices=60, dz=2.0, output="cbed", detectors=0),
        # the 4D-STEM workload of the benchmark, part of its raster: CBEDs with BF and ADF images
        dict(name="scan-512", work="scan", n=512, scan=16, scan_y=12, slices=150, dz=2.0, output="cbed", detectors=2),
        # exit waves for holography or for a solver that goes on from them
        dict(name="exit-384", work="scan", n=384, scan=11, scan_y=11, slices=40, dz=2.0, output="exit_wave", detectors=0),
        # a specimen thick enough for the schedules that hold every twiddle
        dict(name="thick-768", work="scan", n=768, scan=5, scan_y=5, slices=204, dz=2.0, output="cbed", detectors=0),
        # the largest grid, thick: a few positions of a polycrystal-sized cell
        dict(name="thick-2048", work="scan", n=2048, scan=4, scan_y=2, slices=304, dz=1.0, output="cbed", detectors=0),
        # several materials, each with its own grid, slices and raster, replayed as one graph
        dict(name="materials", work="materials", grids="128x25x40 192x16x32 256x36x48 512x16x40 768x9x24 1024x4x32",
             dz=2.0),
        # one sample of a training set: CBEDs with their sums, float16 records, the potential record
        dict(name="dataset-256", work="dataset", n=256, scan=8, scan_y=8, slices=64, dz=2.0),
        # a new specimen: tables, transmission slices, probe (before every simulation)
        dict(name="specimen-512", work="specimen", n=512, slices=150, dz=2.0),
        # virtual detectors on stored CBEDs
        dict(name="detectors-512", work="detectors", n=512, probes=250, detectors=2),
        # the learned coarse-slice path, 64 probes through 400 A
        dict(name="learned-256", work="learned", probes=64, thickness=400),
        # one minibatch of the corrector's training: loss and every gradient
        dict(name="train-256", work="train", batch=16, pool=40),
    ]


def _cost(case):
    """Rough time of a pass in arbitrary units (grid points x slices)."""
    k = case["work"]
    if k == "scan":
        return case["scan"] * case["scan_y"] * (case["slices"] + 2) * case["n"] ** 2
    if k == "materials":
        return sum(b * s * n * n for n, b, s in _grids(case))
    if k == "dataset":
        return case["scan"] * case["scan_y"] * (case["slices"] + 4) * case["n"] ** 2
    if k == "specimen":
        return 20 * case["slices"] * case["n"] ** 2
    if k == "detectors":
        return case["probes"] * case["detectors"] * case["n"] ** 2
    if k == "learned":
        return case["probes"] * (case["thickness"] // 8 + 80) * 256 ** 2
    return 1000 * case["batch"] * 256 ** 2


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    top = max(_cost(c) for c in listed())
    while True:
        k = rng.choice(["scan", "scan", "scan", "scan", "materials", "dataset", "specimen", "detectors", "learned", "train"])
        if k == "scan":
            n = rng.choice(SIZES)
            thick = 210 if n % 3 == 0 else 310
            case = dict(work=k, n=n, scan=_log(rng, 1, 36), scan_y=_log(rng, 1, 36), slices=_log(rng, 4, thick),
                        dz=rng.choice([1.0, 2.0]), output=rng.choice(["cbed", "cbed", "exit_wave"]), detectors=0)
            if case["output"] == "cbed":
                case["detectors"] = rng.choice([0, 1, 2])
        elif k == "materials":
            parts = ["%dx%dx%d" % (rng.choice(SIZES[:-1]), _log(rng, 2, 30), _log(rng, 8, 60)) for _ in range(rng.randint(2, 6))]
            case = dict(work=k, grids=" ".join(parts), dz=2.0)
        elif k == "dataset":
            case = dict(work=k, n=rng.choice(SIZES[:5]), scan=_log(rng, 2, 16), scan_y=_log(rng, 2, 16),
                        slices=_log(rng, 10, 120), dz=2.0)
        elif k == "specimen":
            case = dict(work=k, n=rng.choice(SIZES), slices=_log(rng, 10, 200), dz=rng.choice([1.0, 2.0]))
        elif k == "detectors":
            case = dict(work=k, n=rng.choice(SIZES), probes=_log(rng, 1, 1200), detectors=rng.randint(1, 4))
        elif k == "learned":
            case = dict(work=k, probes=rng.randint(5, 96), thickness=8 * rng.randint(5, 50))
        else:
            case = dict(work=k, batch=rng.randint(4, 24), pool=rng.randint(24, 48))
        out = case.get("n", 0) ** 2 * (case.get("probes", 0) or case.get("scan", 0) * case.get("scan_y", 0))
        if _cost(case) <= top and out <= 1 << 27 and case.get("n", 0) ** 2 * case.get("slices", 0) <= 310 * 2048 ** 2:
            return case


# ------------------------------------------------------------------ inputs
def _grids(case):
    return [tuple(int(v) for v in p.split("x")) for p in case["grids"].split()]


def _atoms(seed, n, depth):
    """A film of n * PIX A square and `depth` A thick: half of it a crystal
    with thermal displacements, half amorphous; light to heavy elements."""
    rng = np.random.default_rng(seed)
    side = n * PIX
    total = max(64, int(DENSITY * side * side * depth))
    xyz = rng.uniform(0.0, 1.0, (total, 3)) * np.array([side, side, depth])
    half = xyz[:, 2] < depth / 2
    a = 2.55                                      # one site per a^3: the crystal half keeps the density
    xyz[half] = (np.floor(xyz[half] / a) + 0.5) * a + rng.normal(0.0, 0.08, (int(half.sum()), 3))
    xyz = np.clip(xyz, 0.0, np.array([side, side, depth]))
    xyz[0], xyz[1] = 0.0, [side, side, depth]
    z = rng.choice([6, 14, 29, 79], total)
    rec = np.zeros(total, dtype=[("atomic_number", "i"), ("x", "f"), ("y", "f"), ("z", "f"), ("occ", "f"), ("DW", "f")])
    rec["atomic_number"], rec["occ"], rec["DW"] = z, 1.0, 0.08
    rec["x"], rec["y"], rec["z"] = xyz[:, 0], xyz[:, 1], xyz[:, 2]
    return rec


def _depth(case):
    return case["slices"] * case["dz"] + 0.25


def _sim(rec, n, dz):
    sim = MSAGPU(KV, SEMI, rec, sampling=np.array([n, n]), debye_waller=False)
    sim.setup_device(0)
    sim.calc_atomic_potentials()
    sim.build_potential_slices(dz)
    sim.build_probe(PROBE)
    return sim


def _annuli(n, count):
    """Detector weights [count][n][n]: bright field first, then annuli."""
    k = np.arange(n) * (1.0 / PIX) / (n - 1) - 0.5 / PIX
    r = np.sqrt(k[:, None] ** 2 + k[None, :] ** 2)
    edges = [0.0, 0.9, 1.8, 2.4, 3.2]
    return np.stack([((r >= a) & (r < b)).astype(np.float32) for a, b in zip(edges[:count], edges[1:count + 1])])


def _patterns(case, seed, dtype):
    """Stored CBEDs: a bright disc with speckle on a decaying background."""
    n, p = case["n"], case["probes"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    k = torch.linspace(-0.5 / PIX, 0.5 / PIX, n, device=DEV, dtype=torch.float64)
    r = (k[:, None] ** 2 + k[None, :] ** 2).sqrt()
    env = (1.0 / (1.0 + torch.exp(20.0 * (r - 1.0))) + 0.02 * torch.exp(-r)).to(torch.float32) / (n * n)
    noise = torch.rand((p, n, n), device=DEV, generator=g, dtype=torch.float32)
    return (env * noise).to(dtype)


def _train_pool(case, seed):
    """Exit spectra, vacuum spectra and target CBEDs of probes through random
    projected potentials, as the pair pool holds them: plain torch."""
    n, p = 256, case["pool"]
    g = torch.Generator(device=DEV).manual_seed(seed)
    f = dict(device=DEV, dtype=torch.float64)
    kmax = 1.0 / PIX
    k = torch.arange(n, **f) * kmax / (n - 1) - kmax / 2
    k2 = k[:, None] ** 2 + k[None, :] ** 2
    lam = _lam()
    mask = (k2.sqrt() < kmax / 3).to(torch.float64)
    psi_k = 1.0 / (1.0 + torch.exp(160.0 * (k2.sqrt() - SEMI / lam))) * torch.exp(-1j * math.pi * lam * 60.0 * k2)
    pos = (torch.rand((p, 2), generator=g, **f) - 0.5) * 16.0
    ramp = torch.exp(-2j * math.pi * (pos[:, 0, None, None] * k[:, None] + pos[:, 1, None, None] * k[None, :]))
    th = 8.0 * torch.randint(5, 51, (p,), generator=g, device=DEV).to(torch.float64)
    psi0 = psi_k * ramp * torch.exp(-1j * math.pi * lam * k2 * th[:, None, None]) * mask
    psi0 = psi0 / (psi0.abs() ** 2).sum((1, 2), keepdim=True).sqrt()
    nv = 4
    v = torch.randn((nv, n, n), generator=g, **f)
    damp = torch.exp(-k2 / 4.0)
    spec = torch.fft.fftshift(torch.fft.fft2(v), dim=(1, 2)) * damp
    v = torch.fft.ifft2(torch.fft.ifftshift(spec, dim=(1, 2))).real
    v = v / v.std()
    vi = torch.arange(p, device=DEV) % nv
    wave = torch.fft.ifft2(torch.fft.ifftshift(psi0, dim=(1, 2)))

    def through(strength):
        w = wave * torch.exp(1j * strength * v[vi])
        return torch.fft.fftshift(torch.fft.fft2(w), dim=(1, 2)) * mask

    vh = torch.fft.fftshift(torch.fft.fft2(v), dim=(1, 2))
    return dict(pc=through(0.5).to(torch.complex64), p0=psi0.to(torch.complex64),
                f=(through(0.55).abs() ** 2).to(torch.float32), vh=vh.to(torch.complex64), th=th.to(torch.float32),
                vi=vi.to(torch.int32), km=torch.full((p,), kmax, device=DEV, dtype=torch.float32))


def prepare(case, seed):
    k = case["work"]
    if k in ("scan", "dataset"):
        sim = _sim(_atoms(seed, case["n"], _depth(case)), case["n"], case["dz"])
        sim.generate_probe_positions(grid_steps=np.array([case["scan"], case["scan_y"]]))
        sim.plan_simulation()
        det = _annuli(case["n"], case["detectors"]) if case.get("detectors") else None
        return dict(case=case, sim=sim, det=det)
    if k == "materials":
        specs = [dict(records=_atoms(seed * 16 + i, n, s * case["dz"] + 0.25), N=n, dz=case["dz"], kv=KV, semi=SEMI,
                      grid_steps=np.array([b, 1]), probe=PROBE) for i, (n, b, s) in enumerate(_grids(case))]
        batch = MaterialBatch(specs)
        batch.capture()
        return dict(case=case, batch=batch)
    if k == "specimen":
        return dict(case=case, records=_atoms(seed, case["n"], _depth(case)))
    if k == "detectors":
        n = case["n"]
        return dict(case=case, cbed=_patterns(case, seed, torch.float32),
                    det=torch.from_numpy(_annuli(n, case["detectors"])).to(DEV))
    if k == "learned":
        sim = _sim(_atoms(seed, 256, case["thickness"] + 0.5), 256, 1.0)
        mat = corrector.SpectralMaterial(sim, dz=1.0, factors=(8,))
        corr = corrector.SpectralCorrector.load(WEIGHTS)
        return dict(case=case, mat=mat, corr=corr, pos=torch.from_numpy(_positions(case, seed)).to(DEV))
    pool = corrector.SpectralPairPool((8,))
    d = _train_pool(case, seed)
    pool.PC, pool.P0, pool.F, pool.VH, pool.TH, pool.VI, pool.KM = {8: d["pc"]}, d["p0"], d["f"], d["vh"], d["th"], d["vi"], d["km"]
    corr = corrector.SpectralCorrector.load(WEIGHTS)
    corr.net.ensure(case["batch"])
    return dict(case=case, pool=pool, corr=corr, idx=_minibatch(case, seed))


def _positions(case, seed):
    return np.random.default_rng(seed + 1).uniform(-8.0, 8.0, (case["probes"], 2)).astype(np.float32)


def _minibatch(case, seed):
    return np.random.default_rng(seed + 2).choice(case["pool"], size=case["batch"], replace=False)


# ------------------------------------------------------------------ one pass
def run(state):
    case = state["case"]
    k = case["work"]
    if k == "scan":
        sim = state["sim"]
        sim.multislice(detectors=state["det"], output="exit_wave" if case["output"] == "exit_wave" else "auto")
        if state["det"] is not None:
            return {"cbed": sim.probes_device, "images": sim.detector_signals.astype(np.float32)}
        return {"cbed": sim.probes_device}
    if k == "dataset":
        sim = state["sim"]
        sim.multislice(moments=True)
        return {"cbed": records.process_cbed(sim.probes_device, moments=sim.cbed_moments_device, as_tensor=True),
                "potential": records.process_potential(sim.potential_slices_device, as_tensor=True)}
    if k == "materials":
        batch = state["batch"]
        batch.replay()
        return [batch.cbed(i) for i in range(len(batch.mats))]
    if k == "specimen":
        sim = _sim(state["records"], case["n"], case["dz"])
        return {"tables": sim.tables_device, "slices": sim.potential_slices_device, "psi_k": sim.psi_k, "psi": sim.psi,
                "normalization": sim.normalization}
    if k == "detectors":
        n, p, d = case["n"], case["probes"], case["detectors"]
        out = torch.empty((p, d), dtype=torch.float64, device=DEV)
        L.call("namsa_integrate", L.ptr(state["cbed"]), p, n, n, L.ptr(state["det"]), d, L.ptr(out), L.stream_handle())
        return out
    if k == "learned":
        return corrector.run_spectral(state["corr"], state["mat"], state["pos"], case["thickness"], tau=None)
    corr = state["corr"]
    corrector.spectral_batch_loss(corr, state["pool"], state["idx"], grad=True)
    _, _, h, w = corr.window
    return {"grad": corr.net.grad, "out": corr.net.out.reshape(-1)[:2 * case["batch"] * h * w]}


def work(case):
    """What a pass cannot do without: inputs read once, outputs written once;
    the transforms of every probe and slice (5 N log2 N each) and the products."""
    k = case["work"]

    def scan(n, p, s, out):
        fft = 5.0 * n * n * math.log2(n * n)
        return dict(bytes=8.0 * n * n * (s + 2) + out * n * n * p, flops=p * (s * (2 * fft + 12.0 * n * n) + 2 * fft))

    if k == "scan":
        w = scan(case["n"], case["scan"] * case["scan_y"], case["slices"], 8 if case["output"] == "exit_wave" else 4)
        w["bytes"] += 4.0 * case["detectors"] * case["n"] ** 2
        return w
    if k == "dataset":
        return scan(case["n"], case["scan"] * case["scan_y"], case["slices"], 2)
    if k == "materials":
        parts = [scan(n, b, s, 4) for n, b, s in _grids(case)]
        return {key: sum(p[key] for p in parts) for key in ("bytes", "flops")}
    if k == "specimen":
        atoms = DENSITY * (case["n"] * PIX) ** 2 * _depth(case)
        return dict(bytes=8.0 * case["n"] ** 2 * (case["slices"] + 3) + 24.0 * atoms, flops=atoms * 64.0 * 64.0)
    if k == "detectors":
        return dict(bytes=4.0 * case["n"] ** 2 * (case["probes"] + case["detectors"]) + 8.0 * case["probes"] * case["detectors"],
                    flops=2.0 * case["n"] ** 2 * case["probes"] * case["detectors"])
    px = 170.0 * 170.0
    net = 2.0 * px * 32 * 7 + 4 * (2.0 * px * 32 * 32 + 2.0 * 2.0 * 32 * px * 32 * 1.2) + 2.0 * px * 66 * 64
    weights = 4.0 * 4 * 256 * 64 * 64
    if k == "learned":
        p = case["probes"]
        w = scan(256, p, case["thickness"] // 8, 4)
        return dict(bytes=w["bytes"] + weights, flops=w["flops"] + p * net)
    b = case["batch"]
    return dict(bytes=b * 256.0 * 256.0 * 20 + 2 * weights, flops=3.0 * b * net)


# ------------------------------------------------------------------ 64-bit results
def _f32(x):
    return float(np.float32(x))


def _lam():
    v = KV * 1e3
    return 12.2643 / math.sqrt(v + 0.97845e-6 * v * v)


def _sigma():
    e, m, c = 1.602176634e-19, 9.1093837139e-31, 299792458.0
    v = KV * 1e3
    return 2 * math.pi * (m * c * c + e * v) / (2 * m * c * c + e * v) / (_lam() * v)


def _tables(z_list, pix, reach=8.0, over=2):
    """Projected atomic potentials (Kirkland) on the pixel grid, minimum 0."""
    params = np.load(KIRKLAND_PATH)
    p = int(math.floor(reach / pix))
    g = torch.linspace(-reach / 2, reach / 2, over * p, dtype=torch.float64)
    r = (g[:, None] ** 2 + g[None, :] ** 2).sqrt()
    pref = 4 * math.pi ** 2 * 0.529 * 14.4
    out = []
    for z in z_list:
        v = torch.zeros_like(r)
        for a, b, c, d in zip(*params[z - 1]):
            v += pref * a * torch.special.modified_bessel_k0(2 * math.pi * r * math.sqrt(b) + 0.1)
            v += pref / 2 * (c / d) * torch.exp(-math.pi ** 2 * r ** 2 / d)
        v = v.reshape(p, over, p, over).mean((1, 3))
        out.append(v - v.min())
    return torch.stack(out).to(DEV)


class _Specimen:
    """Site lists and tables of a structure; potential(i) sums one slice."""

    def __init__(self, rec, n, dz):
        xyz = np.stack([rec["x"], rec["y"], rec["z"]], 1).astype(np.float32)
        self.n, dims = n, (xyz.max(0) - xyz.min(0)).astype(np.float64)
        self.pix = dims[0] / n
        self.kmax = n / dims[0]
        zs = np.unique(rec["atomic_number"])
        self.tables = _tables(zs, self.pix)
        self.S = int(math.floor(dims[2] / dz))
        bounds = (np.arange(self.S + 1) * dz).astype(np.float32)
        sl = np.searchsorted(bounds, xyz[:, 2], side="right") - 1
        keep = np.nonzero((sl >= 0) & (sl < self.S))[0]
        order = keep[np.argsort(sl[keep], kind="stable")]
        px = (xyz[order, :2].astype(np.float64) / self.pix).astype(np.int64)
        self.site = torch.from_numpy(np.stack([np.searchsorted(zs, rec["atomic_number"][order]), px[:, 1], px[:, 0]], 1)).to(DEV)
        self.offs = np.concatenate([[0], np.cumsum(np.bincount(sl[order], minlength=self.S))])

    def potential(self, i, j=None):
        """Sum of the tables of the sites of slices [i, j)."""
        n, p = self.n, self.tables.shape[1]
        v = torch.zeros(n * n, dtype=torch.float64, device=DEV)
        flat = self.tables.reshape(len(self.tables), -1)
        d = torch.arange(p, device=DEV)
        b, e = int(self.offs[i]), int(self.offs[i + 1 if j is None else j])
        for s in range(b, e, 2048):
            z, y, x = self.site[s:min(e, s + 2048)].unbind(1)

            def span(c):
                lo = torch.round(c.double() - p * 0.5).long()
                at = lo[:, None] + d
                return at, (at >= 0) & (at < n) & (at < torch.round(c.double() + p * 0.5).long()[:, None])

            (yy, oky), (xx, okx) = span(y), span(x)
            ok = (oky[:, :, None] & okx[:, None, :]).reshape(len(z), -1)
            at = (yy.clamp(0, n - 1)[:, :, None] * n + xx.clamp(0, n - 1)[:, None, :]).reshape(len(z), -1)
            v.index_add_(0, at.reshape(-1), (flat[z] * ok).reshape(-1))
        return v.reshape(n, n)

    def slice(self, i):
        ph = self.potential(i) * _f32(_sigma())
        return torch.complex(torch.cos(ph), torch.sin(ph))


def _k_axis(n, kmax):
    return torch.arange(n, dtype=torch.float64, device=DEV) * _f32(kmax) / (n - 1) - _f32(kmax) / 2


def _probe_k(n, kmax):
    k = _k_axis(n, kmax)
    kr = (k[:, None] ** 2 + k[None, :] ** 2).sqrt()
    lam = _f32(_lam())
    ap = 1.0 / (1.0 + torch.exp(-160.0 * (_f32(SEMI / _lam()) - kr.float().double())))
    a = PROBE["aberration_dict"]
    q = kr * lam
    chi = 2 * _f32(math.pi) / lam * (-0.5 * a["C1"] * q ** 2 + 0.25 * a["C3"] * q ** 4)
    return ap * torch.exp(-1j * chi)


def _propagator(n, kmax, dz):
    k = _k_axis(n, kmax)
    kf = (k[:, None] ** 2 + k[None, :] ** 2).sqrt().float().double()
    mask = (kf < _f32(kmax / 3)).double()
    return torch.exp(-1j * math.pi * kf * kf * _f32(_lam()) * _f32(dz)) * mask


def _probes(psi_k, pos, kmax):
    n = psi_k.shape[0]
    k = _k_axis(n, kmax)
    y, x = pos.double().unbind(1)
    ramp = torch.exp(-2j * math.pi * y[:, None] * k)[:, :, None] * torch.exp(-2j * math.pi * x[:, None] * k)[:, None, :]
    return torch.fft.fftshift(torch.fft.ifft2(psi_k * ramp, norm="forward"), dim=(1, 2))


def _norm(psi_k):
    return float((torch.fft.ifft2(psi_k, norm="forward").abs() ** 2).sum())


def _raster(n, gx, gy):
    side = n * PIX
    lo, hi = (0.5 - side * 0.5) / 2, (0.5 + side * 0.5) / 2
    ys, xs = np.linspace(lo, hi, gy), np.linspace(lo, hi, gx)
    return torch.from_numpy(np.stack([np.tile(ys, gx), np.repeat(xs, gy)], 1).astype(np.float32)).to(DEV)


def _exit(spec, psi, pm, slices):
    n2 = psi.shape[-1] ** 2
    for t in slices:
        psi = psi * (t / n2)
        psi = torch.fft.ifft2(torch.fft.fft2(psi) * pm, norm="forward")
    return psi


def _cbeds(rec, n, dz, pos):
    spec = _Specimen(rec, n, dz)
    psi_k = _probe_k(n, spec.kmax)
    psi = _exit(spec, _probes(psi_k, pos, spec.kmax), _propagator(n, spec.kmax, dz), (spec.slice(i) for i in range(spec.S)))
    out = (torch.fft.fft2(psi) / n).abs() ** 2 / _norm(psi_k)
    return out, psi / math.sqrt(_norm(psi_k)), spec


def _potential_record(spec):
    n = spec.n
    m = sum(spec.slice(i).imag for i in range(spec.S)).cpu().numpy() / spec.S
    radius = int(4.0 * 1.2 + 0.5)
    x = np.arange(-radius, radius + 1)
    w = np.exp(-0.5 / 1.44 * x * x)
    w /= w.sum()
    p = np.pad(m, radius, mode="symmetric")
    p = sum(w[i] * p[i:i + n, :] for i in range(2 * radius + 1))
    p = sum(w[i] * p[:, i:i + n] for i in range(2 * radius + 1))
    p = p[n // 4:3 * n // 4, n // 4:3 * n // 4]
    return torch.from_numpy(((p - p.mean()) / max(p.std(), 1.0 / math.sqrt(p.size)))[None])


def _gelu(x):
    return 0.5 * x * (1.0 + torch.tanh(math.sqrt(2.0 / math.pi) * (x + 0.044715 * x ** 3)))


_SHAPES = {"Wl": (32, 7), "bl": (32,), "G": (4, 16, 16, 64, 64), "W": (4, 32, 32), "b": (4, 32), "Q1": (64, 32),
           "bq1": (64,), "Q2": (2, 64), "bq2": (2,)}


def _weights():
    """The shipped weights, one flat vector with each group padded to 64 values."""
    bits = np.load(WEIGHTS, allow_pickle=False)["theta_bf16"].astype(np.uint32) << 16
    return torch.from_numpy(bits.view(np.float32).astype(np.float64)).to(DEV)


def _named(flat):
    views, at = {}, 0
    for name, shape in _SHAPES.items():
        size = int(np.prod(shape))
        views[name] = flat[at:at + size].reshape(shape)
        at += -(-size // 64) * 64
    return views


def _network(p, u):
    b, _, h, w = u.shape
    k = torch.arange(16, dtype=torch.float64, device=DEV) - 8
    fy = torch.exp(-2j * math.pi * torch.arange(h, device=DEV, dtype=torch.float64)[:, None] * k / h)
    fx = torch.exp(-2j * math.pi * torch.arange(w, device=DEV, dtype=torch.float64)[:, None] * k / w)
    mix = lambda m, x: (m @ x.reshape(b, x.shape[1], h * w)).reshape(b, m.shape[0], h, w)  # noqa: E731
    x = mix(p["Wl"], u) + p["bl"][:, None, None]
    for i in range(4):
        modes = fy.T @ (x.to(torch.complex128) @ fx)                       # [b][c][p][q]
        both = torch.cat([modes.real, modes.imag], 1).permute(2, 3, 1, 0)   # [p][q][2c][b]
        y = (p["G"][i].contiguous() @ both.contiguous()).permute(3, 2, 0, 1)
        y = torch.complex(y[:, :32].contiguous(), y[:, 32:].contiguous())
        pre = ((fy.conj() @ y) @ fx.conj().T.contiguous()).real / (h * w) + mix(p["W"][i], x) + p["b"][i][:, None, None]
        x = _gelu(pre) if i < 3 else pre
    hid = _gelu(mix(p["Q1"], x) + p["bq1"][:, None, None])
    return mix(p["Q2"], hid) + p["bq2"][:, None, None]


def _window(n, kmax):
    k = _k_axis(n, kmax)
    kf = (k[:, None] ** 2 + k[None, :] ** 2).sqrt().float()
    at = torch.nonzero((kf < np.float32(kmax / 3)).any(1)).reshape(-1)
    return slice(int(at[0]), int(at[-1]) + 1)


def _net_inputs(pc, p0, vh, th, n, kmax):
    """Channels of the network over the band window, from centred spectra."""
    s = _window(n, kmax)
    k = _k_axis(n, kmax)
    k2 = (k[:, None] ** 2 + k[None, :] ** 2)[s, s]
    c, z = pc[:, s, s] * n, p0[:, s, s] * n
    one = torch.ones_like(c.real)
    return torch.stack([c.real, c.imag, z.real, z.imag, math.pi * _lam() * 8.0 / 10.0 * k2 * one,
                        one * th[:, None, None] / 400.0, torch.log1p(100.0 / (n * n) * vh[:, s, s].abs())], 1)


def _exact_learned(case, seed):
    n, thick = 256, case["thickness"]
    rec = _atoms(seed, n, thick + 0.5)
    pos = torch.from_numpy(_positions(case, seed)).to(DEV)
    spec = _Specimen(rec, n, 8.0)
    psi_k = _probe_k(n, spec.kmax)
    psi = _probes(psi_k, pos, spec.kmax)
    scale = n * math.sqrt(_norm(psi_k))
    pc = torch.fft.fft2(_exit(spec, psi, _propagator(n, spec.kmax, 8.0), (spec.slice(i) for i in range(thick // 8)))) / scale
    p0 = torch.fft.fft2(_exit(spec, psi, _propagator(n, spec.kmax, float(thick)), [torch.ones((), device=DEV)])) / scale
    sign = 1.0 - 2.0 * ((torch.arange(n, device=DEV)[:, None] + torch.arange(n, device=DEV)) % 2)
    vh = torch.fft.fft2(spec.potential(0, thick // 8) * _sigma() * sign)
    th = torch.full((len(pos),), float(thick), device=DEV, dtype=torch.float64)
    s = _window(n, spec.kmax)
    p = _named(_weights())
    for b in range(0, len(pos), 8):
        o = _network(p, _net_inputs(pc[b:b + 8], p0[b:b + 8], vh[None].expand(len(pc[b:b + 8]), n, n), th[b:b + 8], n, spec.kmax))
        pc[b:b + 8, s, s] *= 1.0 + torch.complex(o[:, 0].contiguous(), o[:, 1].contiguous())
    return pc.abs() ** 2


def _exact_train(case, seed):
    n, kmax, d = 256, 1.0 / PIX, _train_pool(case, seed)
    idx = torch.from_numpy(_minibatch(case, seed)).to(DEV)
    pc, p0, f = d["pc"][idx].to(torch.complex128), d["p0"][idx].to(torch.complex128), d["f"][idx].double()
    vh, th = d["vh"][d["vi"][idx].long()].to(torch.complex128), d["th"][idx].double()
    flat = _weights().requires_grad_(True)
    s, b = _window(n, kmax), len(idx)
    outs, total = [], torch.zeros_like(flat)
    for i in range(0, b, 4):
        j = slice(i, min(b, i + 4))
        o = _network(_named(flat), _net_inputs(pc[j], p0[j], vh[j], th[j], n, kmax))
        psi = pc[j, s, s] * (1.0 + torch.complex(o[:, 0].contiguous(), o[:, 1].contiguous()))
        i1, i2 = psi.real ** 2 + psi.imag ** 2, f[j, s, s]
        loss = (((i1 - i2) ** 2).sum((1, 2)) / (i2 ** 2).sum((1, 2))).sum() / b
        total += torch.autograd.grad(loss, flat)[0]
        outs.append(o.detach())
    out = torch.cat(outs).permute(1, 0, 2, 3).reshape(-1)
    return {"grad": total, "out": out}


def exact(case, seed):
    k = case["work"]
    if k == "scan":
        n = case["n"]
        cb, ex, _ = _cbeds(_atoms(seed, n, _depth(case)), n, case["dz"], _raster(n, case["scan"], case["scan_y"]))
        if case["output"] == "exit_wave":
            return {"cbed": ex}
        if not case["detectors"]:
            return {"cbed": cb}
        det = torch.from_numpy(_annuli(n, case["detectors"])).to(DEV).double()
        return {"cbed": cb, "images": torch.stack([(cb * d).sum((1, 2)) for d in det], 1)}
    if k == "dataset":
        n = case["n"]
        cb, _, spec = _cbeds(_atoms(seed, n, _depth(case)), n, case["dz"], _raster(n, case["scan"], case["scan_y"]))
        mean, std = cb.mean((1, 2), keepdim=True), cb.std((1, 2), keepdim=True, correction=0)
        return {"cbed": (cb - mean) / std, "potential": _potential_record(spec)}
    if k == "materials":
        return [_cbeds(_atoms(seed * 16 + i, n, s * case["dz"] + 0.25), n, case["dz"], _raster(n, b, 1))[0]
                for i, (n, b, s) in enumerate(_grids(case))]
    if k == "specimen":
        spec = _Specimen(_atoms(seed, case["n"], _depth(case)), case["n"], case["dz"])
        psi_k = _probe_k(case["n"], spec.kmax)
        psi = torch.fft.fftshift(torch.fft.ifft2(psi_k, norm="forward"))
        norm = _norm(psi_k)
        slices = torch.stack([spec.slice(i).to(torch.complex128) for i in range(spec.S)])
        return {"tables": spec.tables, "slices": slices, "psi_k": psi_k, "psi": psi / math.sqrt(norm), "normalization": norm}
    if k == "detectors":
        cb = _patterns(case, seed, torch.float32)
        det = torch.from_numpy(_annuli(case["n"], case["detectors"])).to(DEV).double()
        return torch.stack([torch.stack([(c.double() * d).sum() for d in det]) for c in cb])
    if k == "learned":
        return _exact_learned(case, seed)
    return _exact_train(case, seed)
