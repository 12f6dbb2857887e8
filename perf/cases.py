"""What this framework is timed on: the sampler, the kriging build and the covariance summaries, as programs call them.

A pass of a "fit" case is what a fit does between two saved samples: `thin`
HMC iterations (L = 25 leapfrog steps each: momentum draw, 26 gradients,
energies, accept), then the saved sample itself.  L = 25 and thin = 3 are the
command-line tools' defaults, as is the power-of-two embedding ("pow2").  A
"batch" case runs the same iteration for several chains of uneven size at
once.  A "kriging" case builds W for a pair of images, and the "mce" cases are
the two covariance summaries the parameter estimation starts from; these take
host images and return host arrays.

The step size is a small power of two, as early in the burn-in, and the accept
draw is 0 (every proposal is accepted): a draw close to the accept ratio would
let the last digit of an energy decide what the pass returns.  For the same reason the accept ratio itself, exp of a
small difference of two large energies, is left out of the outputs; the
energies it is made of are all there.
"""
import functools
import math

import numpy as np
import torch

from dualres_amd import Chain, mce, problem
from dualres_amd.batch import Batch
from dualres_amd.kriging import kriging_build

L, THIN, EPS = 25, 3, 1.0 / 128
SIGMA = (1.0, 4.0)  # noise precisions of the highres and stdres images (sd 1 and 0.5)
RADIUS = 6.9        # kriging neighbourhood, mm
ENERGIES = ("log_prior0", "log_lik0", "e0", "log_prior1", "log_lik1", "k1", "sse_h", "sse_s")


def _fit(name, dims, vox, precision, dual, embed, state="compat", psi=0.132, nu=1.5):
    return {"name": name, "what": "fit", "nx": dims[0], "ny": dims[1], "nz": dims[2], "vox": vox, "dual": dual,
            "precision": precision, "state": state, "embed": embed, "tau2": 0.806, "psi": psi, "nu": nu}


def _image(name, what, dims, vox, psi=0.132, nu=1.5):
    return {"name": name, "what": what, "nx": dims[0], "ny": dims[1], "nz": dims[2], "vox": vox, "tau2": 0.806,
            "psi": psi, "nu": nu}


def listed():
    return [
        # a small region of interest, single resolution: the shortest kernels, so launches and latency
        _fit("fit_roi_fp32", (20, 24, 18), 3.0, "fp32", False, "pow2"),
        # a whole 2 mm image, single resolution, in the precision of dualgpm
        _fit("fit_2mm_fp64", (40, 48, 40), 2.0, "fp64", False, "smooth", nu=1.0),
        # a 1.5 mm dual-resolution fit in dualgpm's precision, default embedding
        _fit("fit_dual_1.5mm_fp64", (64, 80, 64), 1.5, "fp64", True, "pow2"),
        # an uneven 1.5 mm dual-resolution image of the serving mix, in dualgpmf's precision; the smooth
        # embedding has lengths with factors 3, 5 and 7
        _fit("fit_dual_1.5mm_fp32", (95, 113, 97), 1.5, "fp32", True, "smooth", psi=0.12, nu=1.3),
        # the 1 mm dual-resolution fit of bench.py, on twice the image's size
        _fit("fit_dual_1mm_fp32", (128, 160, 128), 1.0, "fp32", True, "2x"),
        # the same image alone in double precision with the default embedding: the largest torus
        _fit("fit_1mm_fp64", (128, 160, 128), 1.0, "fp64", False, "pow2"),
        # one iteration of several subjects' dual-resolution chains together
        {"name": "batch_dual_fp32", "what": "batch", "chains": 8, "lo": 32, "hi": 80, "vox": 1.5, "dual": True,
         "precision": "fp32", "state": "compat", "embed": "smooth", "tau2": 1.0, "psi": 0.12, "nu": 1.3,
         "mode": "streams", "sizes": 7},
        # kriging weights at the start of a fit: many systems of about 370 unknowns, few of about 1,300
        _image("kriging_1.5mm", "kriging", (64, 80, 64), 1.5),
        _image("kriging_1mm", "kriging", (48, 60, 48), 1.0),
        # parameter estimation before a fit: estimate_rbf's per-offset summary and the binned one
        _image("mce_offsets_1mm", "mce", (128, 160, 128), 1.0),
        _image("mce_offsets_roi", "mce", (33, 41, 29), 2.0),
        _image("mce_binned_1mm", "mce_binned", (128, 160, 128), 1.0),
    ]


def draw(rng):
    def between(a, b):  # spread over the logarithm, odd sizes among them
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    what = rng.choice(["fit", "fit", "fit", "dual", "dual", "batch", "kriging", "mce", "mce_binned"])
    c = {"tau2": 0.806, "psi": round(rng.uniform(0.08, 0.2), 4), "nu": round(rng.uniform(0.8, 1.8), 3)}
    if what in ("fit", "dual", "batch"):
        c.update(precision=rng.choice(["fp32", "fp64"]), state=rng.choice(["compat", "compat", "real"]),
                 embed=rng.choice(["pow2", "smooth"]), dual=what != "fit", what="fit")
    if what == "batch":
        lo = between(20, 32)
        c.update(what="batch", chains=rng.randint(3, 8), lo=lo, hi=lo + rng.randint(8, 40), vox=1.5,
                 dual=rng.random() < 0.5, mode=rng.choice(["graph", "streams", "eager"]), sizes=rng.randrange(1000))
        return c
    lo, hi, vox = {"fit": (16, 128, (1.0, 3.0)), "dual": (24, 100, (1.4, 2.2)), "kriging": (28, 64, (1.3, 2.2)),
                   "mce": (24, 128, (1.0, 3.0)), "mce_binned": (24, 128, (1.0, 3.0))}[what]
    c.setdefault("what", what)
    c.update(nx=between(lo, hi), ny=between(lo, int(1.2 * hi)), nz=between(lo, hi), vox=round(rng.uniform(*vox), 2))
    return c


# ---------------------------------------------------------------- inputs
def _dims(case):
    return case["nx"], case["ny"], case["nz"]


def _theta(case):
    return case["tau2"], case["psi"], case["nu"]


@functools.lru_cache(maxsize=64)
def _geometry(dims, dual):
    """Masks and indices of an ellipsoid-masked image (and of its 2x2x2 block means)."""
    m = problem.ellipsoid_mask(dims, 0.45)
    ijk = problem.nonzero_ijk(m)
    sm = problem.ellipsoid_mask(tuple(d // 2 for d in dims), 0.45) if dual else None
    return m, ijk - ijk.min(axis=0), sm


def _qforms(dims, vox):
    q = problem.qform_axis(vox, dims)
    return q, problem.qform_axis(2 * vox, tuple(d // 2 for d in dims), origin=[q[a, 3] + 0.5 * vox for a in range(3)])


def _torus_sq(M, vox):
    """Squared Euclidean distance on the torus, shape (M2, M1, M0)."""
    d = []
    for a in range(3):
        t = torch.arange(M[a], device="cuda", dtype=torch.float64)
        d.append((torch.minimum(t, M[a] - t) * vox) ** 2)
    return d[2][:, None, None] + d[1][None, :, None] + d[0][None, None, :]


def _images(dims, vox, theta, seed, dual):
    """A GP draw plus unit noise on the mask (and its block means plus noise of sd 0.5), float32 values."""
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1000003 + 17 * dims[0] + 5 * dims[1] + dims[2])
    M = tuple(2 * d for d in dims)
    c = theta[0] * torch.exp(-theta[1] * _torus_sq(M, vox).sqrt() ** theta[2])
    lam = torch.fft.fftn(c).real.clamp_min(0.0)
    e = torch.complex(*(torch.randn(lam.shape, generator=g, device="cuda", dtype=torch.float64) for _ in range(2)))
    f = torch.fft.fftn((lam / lam.numel()).sqrt() * e).real[:dims[2], :dims[1], :dims[0]]
    m, _, sm = _geometry(dims, dual)

    def noisy(v, sd, mask):
        y = v + sd * torch.randn(v.shape, generator=g, device="cuda", dtype=torch.float64)
        y = y.float().double().cpu().numpy()
        y[y == 0] = 1e-30
        return np.where(mask, y, 0.0)

    hr = noisy(f, 1.0, m)
    if not dual:
        return hr, None
    h = [d // 2 for d in dims]
    b = f[:2 * h[2], :2 * h[1], :2 * h[0]].reshape(h[2], 2, h[1], 2, h[0], 2).mean(dim=(1, 3, 5))
    return hr, noisy(b, 0.5, sm)


@functools.lru_cache(maxsize=24)
def _weights(dims, vox, theta):
    """W depends on the masks, the grids and theta, not on the data: programs that fit several images of one geometry
    build it once."""
    m, _, sm = _geometry(dims, True)
    q, qs = _qforms(dims, vox)
    return kriging_build(m.astype(np.float64), q, sm.astype(np.float64), qs, theta, RADIUS)


def _embedding(ijk, dims, rule):
    if rule == "2x":
        return tuple(2 * d for d in dims)
    mx = [int(v) for v in ijk.max(axis=0)]
    return tuple(problem.smooth_even(2 * v) for v in mx) if rule == "smooth" else tuple(
        1 << max(1, (2 * v - 1).bit_length()) for v in mx)


def _members(case):
    """The chains of a fit (one) or a batch: a fit case each."""
    if case["what"] == "fit":
        return [case]
    sizes = np.random.default_rng(case["sizes"])
    out = []
    for _ in range(case["chains"]):
        n = [int(sizes.integers(case["lo"], case["hi"] + 1)) for _ in range(3)]
        out.append(dict(case, nx=n[0], ny=n[1], nz=n[2], psi=round(case["psi"] * float(sizes.uniform(0.7, 1.4)), 4)))
    return out


def _fit_inputs(m, seed):
    dims, th = _dims(m), _theta(m)
    mask, ijk, smask = _geometry(dims, m["dual"])
    hr, std = _images(dims, m["vox"], th, seed, m["dual"])
    W = _weights(dims, m["vox"], th) if m["dual"] else None
    return {"ijk": ijk, "theta": th, "q": _qforms(dims, m["vox"])[0], "Yh": hr[mask], "W": W,
            "Ys": std[smask] if m["dual"] else None, "embed": _embedding(ijk, dims, m["embed"]), "seed": 77 + 13 * int(seed)}


def _chain(m, p):
    c = Chain(p["ijk"], p["theta"], p["q"], n_datasets=2 if m["dual"] else 1, precision=m["precision"],
              state_mode=m["state"], embed=None if m["embed"] == "pow2" else p["embed"], seed=p["seed"])
    c.set_data(p["Yh"], p["Ys"], p["W"])
    c.add_data_to_mu()
    c.set_output_indices(p["ijk"])
    c.set_sigma_sq_inv(SIGMA[:c.n_datasets])
    return c


def prepare(case, seed):
    what = case["what"]
    if what in ("fit", "batch"):
        chains = [_chain(m, _fit_inputs(m, seed + 101 * i)) for i, m in enumerate(_members(case))]
        s = {"what": what, "chains": chains, "dtype": np.float32 if case["precision"] == "fp32" else np.float64}
        if what == "batch":
            s["batch"] = Batch(chains, case["mode"])
        return s
    dims, th = _dims(case), _theta(case)
    q, qs = _qforms(dims, case["vox"])
    hr, std = _images(dims, case["vox"], th, seed, what == "kriging")
    if what == "kriging":  # another subject has another scale of its covariance
        th = (th[0], th[1] * (1.0 + 0.01 * (int(seed) % 17)), th[2])
    return {"what": what, "hr": hr, "std": std, "q": q, "qs": qs, "theta": th}


# ---------------------------------------------------------------- one pass
def _energies(results, dtype):
    return np.array([[r[k] for k in ENERGIES] for r in results], dtype=dtype)


def run(s):
    what = s["what"]
    if what == "fit":
        c = s["chains"][0]
        r = [c.update(EPS, L, 0.0) for _ in range(THIN)]
        return {"energies": _energies(r, s["dtype"]), "mu": c.mu_().astype(s["dtype"], copy=False)}
    if what == "batch":
        r = s["batch"].update(EPS, L, 0.0)
        return {"energies": _energies(r, s["dtype"]),
                "mu": [c.mu_().astype(s["dtype"], copy=False) for c in s["chains"]]}
    if what == "kriging":
        W = kriging_build(s["hr"], s["q"], s["std"], s["qs"], s["theta"], RADIUS)
        return {"indptr": W.indptr, "indices": W.indices, "data": W.data}
    if what == "mce":
        cov, dist, npairs = mce.mce_summary(s["hr"], s["q"])
        return {"covariance": cov, "distance": dist, "npairs": npairs}
    cov, dist, npairs = mce.mce_binned(s["hr"], s["q"], nbins=64, maxdist=20.0)
    return {"covariance": cov, "distance": dist, "npairs": npairs}


# ---------------------------------------------------------------- what a pass cannot do without
def _ball(vox):
    """Offsets (x, y, z) within the neighbourhood, z slowest."""
    n = int(np.float32(RADIUS) / np.float32(vox))
    r = np.arange(-n, n + 1)
    z, y, x = np.meshgrid(r, r, r, indexing="ij")
    P = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    f = P.astype(np.float32) * np.float32(vox)
    sq = f * f
    return P[np.sqrt(sq[:, 0] + sq[:, 1] + sq[:, 2], dtype=np.float32) <= np.float32(RADIUS)]


@functools.lru_cache(maxsize=64)
def _neighbours(dims, vox):
    """(rows, entries, rows whose ball leaves the mask, their entries) of W."""
    m, _, sm = _geometry(dims, True)
    pad = 16
    mt = torch.nn.functional.pad(torch.from_numpy(m).cuda().to(torch.int32), (pad,) * 6)
    at = torch.from_numpy(2 * problem.nonzero_ijk(sm) + pad).cuda()
    n = torch.zeros(at.shape[0], dtype=torch.int64, device="cuda")
    P = _ball(vox)
    for x, y, z in P.tolist():
        n += mt[at[:, 2] + z, at[:, 1] + y, at[:, 0] + x]
    b = n < len(P)
    return at.shape[0], int(n.sum()), int(b.sum()), int(n[b].sum())


def work(case):
    what = case["what"]
    if what in ("fit", "batch"):
        total, flops, s = 0.0, 0.0, 4 if case["precision"] == "fp32" else 8
        for m in _members(case):
            _, ijk, _ = _geometry(_dims(m), m["dual"])
            M = _embedding(ijk, _dims(m), m["embed"])
            N, Nh, nh = M[0] * M[1] * M[2], (M[0] // 2 + 1) * M[1] * M[2], len(ijk)
            # a step reads and writes mu and p and reads 1 / lambda once per mode, reads the data and mu at the
            # voxels, and reads each entry of W that no two rows share once
            step, ops = Nh * 9 * s + 2 * nh * s, 5.0 * N * math.log2(N) + 14.0 * Nh
            if m["dual"]:
                rows, nnz, _, own = _neighbours(_dims(m), m["vox"])
                step, ops = step + own * s + 2 * rows * s, ops + 4.0 * nnz
            n = THIN if what == "fit" else 1
            # an iteration draws p (and the imaginary chain's), moves that chain once, and returns the sample
            total += n * (L * step + Nh * s * (3 + (10 if m["state"] == "compat" else 0))) + 8 * nh
            flops += n * (L + 1) * ops
        return {"bytes": total, "flops": flops}
    dims = _dims(case)
    nvox = dims[0] * dims[1] * dims[2]
    if what == "kriging":
        rows, nnz, brows, own = _neighbours(dims, case["vox"])
        return {"bytes": 8.0 * (nvox + nvox // 8) + 12.0 * nnz + 8.0 * rows, "flops": (own / brows) ** 3 / 3 * brows}
    reach = 25 if what == "mce" else math.ceil(20.0 / case["vox"])
    N = 1.0
    for d in dims:
        N *= d + reach
    return {"bytes": 8.0 * nvox + 12.0 * 25348, "flops": 5 * 2.5 * N * math.log2(N)}


# ---------------------------------------------------------------- the same in 64 bits, plain torch and numpy
def _philox(seed, stream, block):
    """Philox4x32-10 (Salmon et al., SC'11): four 32-bit words of each counter (block, stream), as int64."""
    lo = 0xFFFFFFFF
    a, b = block & lo, block >> 32
    c, d = torch.full_like(block, stream & lo), torch.full_like(block, stream >> 32)
    k0, k1 = seed & lo, seed >> 32
    for _ in range(10):
        p0, p1 = a * 0xD2511F53, c * 0xCD9E8D57
        a, b, c, d = ((p1 >> 32) & lo) ^ b ^ k0, p1 & lo, ((p0 >> 32) & lo) ^ d ^ k1, p0 & lo
        k0, k1 = (k0 + 0x9E3779B9) & lo, (k1 + 0xBB67AE85) & lo
    return a, b, c, d


def _box_muller(u1, u2):
    r, t = (-2.0 * u1.log()).sqrt(), 2.0 * math.pi * u2
    return r * t.cos(), r * t.sin()


def _normals(seed, stream, key, fp32, split):
    """The normal pair of each key: 24-bit uniforms of two words of a block in single precision (`split`: two keys
    share a block, words a, c and b, d), 53-bit ones of all four words in double."""
    if fp32:
        a, b, c, d = _philox(seed, stream, key >> 1 if split else key)
        if split:
            odd = (key & 1).bool()
            a, c = torch.where(odd, b, a), torch.where(odd, d, c)
        return _box_muller(*(((w >> 8).double() + 0.5) / 2.0 ** 24 for w in (a, c)))
    a, b, c, d = _philox(seed, stream, key)
    return _box_muller(*((((h >> 5) << 26 | l >> 6).double() + 0.5) / 2.0 ** 53 for h, l in ((a, b), (c, d))))


def _lambda(M, vox, theta):
    """Eigenvalues of the circulant covariance; distances rounded to single precision, as the model defines them."""
    ax = [torch.arange(M[a], device="cuda") for a in range(3)]
    sq = [(torch.minimum(t, M[a] - t).float() * np.float32(vox).item()) ** 2 for a, t in enumerate(ax)]
    d = (sq[0][None, None, :] + sq[1][None, :, None]) + sq[2][:, None, None]
    d = d.double().sqrt().float().double()
    return torch.fft.rfftn(theta[0] * torch.exp(-theta[1] * d ** theta[2])).real


class _Exact:
    """One chain in float64, state kept as half spectra [M2][M1][M0 / 2 + 1]."""

    def __init__(self, m, p):
        self.M, self.fp32, self.seed = p["embed"], m["precision"] == "fp32", p["seed"]
        M0, M1, M2 = self.M
        self.N, self.it = M0 * M1 * M2, 0
        lam = _lambda(self.M, m["vox"], p["theta"])
        self.pos = lam > 0
        self.il = torch.where(self.pos, 1.0 / lam, torch.zeros_like(lam))
        self.w = torch.full((M0 // 2 + 1,), 2.0, device="cuda", dtype=torch.float64)
        self.w[0] = self.w[-1] = 1.0
        self.ilm = torch.where(self.pos, 1.0 / (self.il + SIGMA[0]), torch.zeros_like(lam))
        ijk = torch.from_numpy(p["ijk"]).cuda()
        self.at = ijk[:, 0] + M0 * (ijk[:, 1] + M1 * ijk[:, 2])
        self.Yh = torch.from_numpy(p["Yh"]).cuda()
        if m["dual"]:
            W = p["W"]
            self.Ys = torch.from_numpy(p["Ys"]).cuda()
            self.vals, self.cols = torch.from_numpy(W.data).cuda(), torch.from_numpy(W.indices).cuda().long()
            rp = torch.from_numpy(W.indptr.astype(np.int64)).cuda()
            self.rows = torch.repeat_interleave(torch.arange(len(p["Ys"]), device="cuda"), rp.diff())
            self.W = torch.sparse_csr_tensor(rp, self.cols, self.vals, size=W.shape)
        self.dual = m["dual"]
        sq = lam.clamp_min(0.0).sqrt() / 10.0
        self.x = self._noise(2) * sq + self._forward(self.Yh)
        self.xi = self._noise(3) * sq if m["state"] == "compat" else None

    def _noise(self, stream):
        M0, M1, M2 = self.M
        pair = torch.arange(self.N // 2, device="cuda")
        a, b = _normals(self.seed, stream, pair, self.fp32, False)
        return torch.fft.rfftn(torch.stack([a, b], dim=1).reshape(M2, M1, M0))

    def _forward(self, r):
        f = torch.zeros(self.N, device="cuda", dtype=torch.float64)
        f[self.at] = r
        return torch.fft.rfftn(f.reshape(self.M[::-1]))

    def _mu(self, x):
        return torch.fft.irfftn(x, s=self.M[::-1]).reshape(-1)[self.at]

    def _white(self, stream):
        """Hermitian white noise of variance N per mode: the spectrum of a white field."""
        M0, M1, M2 = self.M
        H = M0 // 2 + 1
        i = torch.arange(H * M1 * M2, device="cuda")
        kx, row = i % H, i // H
        partner = ((M2 - row // M1) % M2 * M1 + (M1 - row % M1) % M1) * H + kx
        edge = (kx == 0) | (kx == H - 1)
        own, conj = edge & (partner == i), edge & (partner < i)
        a, b = _normals(self.seed, stream, torch.where(conj, partner, i), self.fp32, True)
        sd = math.sqrt(0.5 * self.N)
        re = torch.where(own, a * math.sqrt(self.N), a * sd)
        im = torch.where(own, torch.zeros_like(b), torch.where(conj, -b, b) * sd)
        return torch.complex(re, im).reshape(M2, M1, H)

    def _momentum(self, stream):
        z = self._white(stream)
        e0 = self._quad(z, torch.ones_like(self.il))
        return torch.where(self.pos, z * (self.il + SIGMA[0]).sqrt(), torch.zeros_like(z)), e0

    def _quad(self, x, a):
        return float((self.w * a * (x.real ** 2 + x.imag ** 2)).sum())

    def _force(self, x):
        mu = self._mu(x)
        d = self.Yh - mu
        r, sse = SIGMA[0] * d, [float(d @ d), 0.0]
        if self.dual:
            e = self.Ys - self.W @ mu
            sse[1] = float(e @ e)
            r = r + SIGMA[1] * torch.zeros_like(r).index_add_(0, self.cols, self.vals * e[self.rows])
        return self._forward(r) - x * self.il, sse

    def update(self):
        x, xi, N = self.x, self.xi, self.N
        p, e0 = self._momentum(4 * self.it)
        pri0 = self._quad(x, self.il)
        g, sse0 = self._force(x)
        p = p + 0.5 * EPS * g
        for s in range(L):
            x = x + EPS * p * self.ilm
            g, sse = self._force(x)
            p = p + (0.5 if s == L - 1 else 1.0) * EPS * g
        pri1, k1 = self._quad(x, self.il), self._quad(p, self.ilm)
        if xi is not None:  # the imaginary part sees no data
            q, e = self._momentum(4 * self.it + 1)
            e0, pri0 = e0 + e, pri0 + self._quad(xi, self.il)
            q = q - 0.5 * EPS * self.il * xi
            for s in range(L):
                xi = xi + EPS * q * self.ilm
                q = q - (0.5 if s == L - 1 else 1.0) * EPS * self.il * xi
            pri1, k1 = pri1 + self._quad(xi, self.il), k1 + self._quad(q, self.ilm)
        lik = [-0.5 * (SIGMA[0] * v[0] + (SIGMA[1] * v[1] if self.dual else 0.0)) for v in (sse0, sse)]
        self.x, self.xi, self.it = x, xi, self.it + 1
        return [-0.5 * pri0 / N, lik[0], -0.5 * e0 / N, -0.5 * pri1 / N, lik[1], -0.5 * k1 / N, sse[0], sse[1]]


def _exact_weights(s, vox):
    """Each row's neighbours in the mask, in the ball's order, and the solution of its kriging system, scaled to sum 1;
    distances and kernel values rounded to single precision, as the model defines them."""
    f32 = np.float32
    tau2, psi, nu = (float(f32(t)) for t in s["theta"])

    def kern(d):  # float32 distances
        return (tau2 * torch.exp(-psi * d.double() ** nu)).float()

    def root(v):
        return v.double().sqrt().float()

    P = _ball(vox)
    X = torch.from_numpy(P.astype(f32) * f32(vox)).cuda()
    D = X[:, None, :] - X[None, :, :]
    D = D * D
    K = kern(root((D[..., 0] + D[..., 1]) + D[..., 2])).double()
    K.fill_diagonal_(1.0)
    at = problem.nonzero_ijk(s["std"])
    m = np.linalg.inv(s["q"].astype(np.float64)) @ s["qs"].astype(np.float64)

    def map4(q, v):  # q [v, 1], each product and sum rounded to float32
        q = np.asarray(q, dtype=f32)
        acc = np.zeros(v.shape, f32)
        for c in range(3):
            acc = acc + q[:3, c] * v[..., c:c + 1].astype(f32)
        return acc + q[:3, 3]

    base = np.trunc(map4(m, at)).astype(np.int64)
    nb = base[:, None, :] + P[None]
    # a neighbour counts when its flat offset is a voxel of the image that is present, and so is its place in the
    # bounding box of the present voxels
    present = s["hr"] != 0
    sizes, found = present.shape, problem.nonzero_ijk(s["hr"])
    lo, box = found.min(axis=0), np.ptp(found, axis=0) + 1
    off = (nb[..., 2] * sizes[1] + nb[..., 1]) * sizes[2] + nb[..., 0]
    inside = (off >= 0) & (off < present.size)
    inside &= present.reshape(-1)[np.where(inside, off, 0)]
    r = nb - lo
    off = (r[..., 2] * box[1] + r[..., 1]) * box[0] + r[..., 0]
    boxed = present[lo[2]:lo[2] + box[2], lo[1]:lo[1] + box[1], lo[0]:lo[0] + box[0]].reshape(-1)
    inside &= (off >= 0) & (off < boxed.size)
    inside &= boxed[np.where(inside, off, 0)]
    d = torch.from_numpy(map4(s["qs"], at)).cuda()[:, None, :] - torch.from_numpy(map4(s["q"], nb)).cuda()
    d = d * d
    kp = kern(root((d[..., 0] + d[..., 1]) + d[..., 2]) + f32(1e-5).item()).double()
    inside = torch.from_numpy(inside).cuda()
    rule = torch.cat([inside.double(), torch.where(inside, kp, torch.zeros_like(kp))], dim=1)
    uniq, of = torch.unique(rule, dim=0, return_inverse=True)
    n = len(P)
    # conjugate gradients on all systems together: they share K, an absent neighbour's unknown stays 0
    on, b = uniq[:, :n], uniq[:, n:]
    sol, res = torch.zeros_like(b), b.clone()
    p, rr = res.clone(), (res * res).sum(dim=1)
    floor = 1e-30 * rr
    for _ in range(1500):
        if bool((rr <= floor).all()):
            break
        Ap = (p @ K) * on
        a = rr / (p * Ap).sum(dim=1).clamp_min(1e-300)
        sol, res = sol + a[:, None] * p, res - a[:, None] * Ap
        r2 = (res * res).sum(dim=1)
        p, rr = res + (r2 / rr.clamp_min(1e-300))[:, None] * p, r2
    sol = sol / sol.sum(dim=1, keepdim=True)
    return sol[of][inside].cpu().numpy()


def _exact_sums(img, off):
    """Over the voxel pairs (u, u + p) present in the image: sum x(u) x(u + p), sum x(u), sum x(u + p), their number."""
    x = torch.from_numpy(img).cuda()
    reach = np.abs(off).max(axis=0)
    M = [problem.smooth_even(int(n + r)) for n, r in zip(x.shape, reach[::-1])]
    X, B = torch.fft.rfftn(x, s=M), torch.fft.rfftn((x != 0).double(), s=M)
    o = torch.from_numpy(off.astype(np.int64)).cuda()
    at = (o[:, 2] % M[0], o[:, 1] % M[1], o[:, 0] % M[2])
    got = [torch.fft.irfftn(p.conj() * q, s=M)[at].cpu().numpy() for p, q in ((X, X), (X, B), (B, X), (B, B))]
    return got[0], got[1], got[2], np.rint(got[3])


def _distance(q, off):
    """||Q p|| with products and sums rounded to float32."""
    v = off.astype(np.float32) * np.diag(q)[:3].astype(np.float32)
    sq = v * v
    return np.sqrt((sq[:, 0] + sq[:, 1]) + sq[:, 2], dtype=np.float32)


def exact(case, seed):
    what = case["what"]
    if what in ("fit", "batch"):
        energies, mu = [], []
        for i, m in enumerate(_members(case)):
            c = _Exact(m, _fit_inputs(m, seed + 101 * i))
            for _ in range(THIN if what == "fit" else 1):
                energies.append(c.update())
            mu.append(c._mu(c.x).cpu().numpy())
            del c
        return {"energies": np.array(energies), "mu": mu[0] if what == "fit" else mu}
    s = prepare(case, seed)
    if what == "kriging":
        return {"indptr": None, "indices": None, "data": _exact_weights(s, case["vox"])}
    if what == "mce":
        off = mce.mce_offsets()
        sxy, sx, sy, n = _exact_sums(s["hr"], off)
        cov = np.where(n > 1, (sxy - sx * sy / np.maximum(n, 1)) / np.maximum(n - 1, 1), 0.0)
        return {"covariance": cov, "distance": np.sqrt(((off * np.diag(s["q"])[:3]) ** 2).sum(axis=1)), "npairs": None}
    r = math.ceil(20.0 / case["vox"])
    z, y, x = np.meshgrid(np.arange(0, r + 1), np.arange(-r, r + 1), np.arange(-r, r + 1), indexing="ij")
    off = np.stack([x.ravel(), y.ravel(), z.ravel()], axis=1)
    off = off[(off[:, 2] > 0) | (off[:, 1] > 0) | ((off[:, 1] == 0) & (off[:, 0] >= 0))]  # one of each +-p
    d = _distance(s["q"], off)
    off, d = off[d <= 20.0], d[d <= 20.0].astype(np.float64)
    sxy, sx, sy, n = _exact_sums(s["hr"], off)
    w = 20.0 / 64
    b = np.minimum(63, (d / w).astype(np.int64))
    Sxy, Sx, Sy, Sn, Sd = (np.bincount(b, weights=v, minlength=64) for v in (sxy, sx, sy, n, d * n))
    cov = np.where(Sn > 1, (Sxy - Sx * Sy / np.maximum(Sn, 1)) / np.maximum(Sn - 1, 1), 0.0)
    dist = np.where(Sn > 0, Sd / np.maximum(Sn, 1), (np.arange(64) + 0.5) * w)
    return {"covariance": cov, "distance": dist, "npairs": None}
