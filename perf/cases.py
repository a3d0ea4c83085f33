"""Timing cases of the common-lines engine: what its users have it do.

Each case is one call (or one short sequence of calls) of a public entry
point on inputs resident where the user has them, with the sizes of the
framework's own workloads (``aspire_amd/workloads.py``, ``bench.py``) cut so
that a pass stays under a second, the smallest stacks users start with, and
odd sizes between.  ``listed`` gives the fixed cases, ``draw`` one more of the
same ranges, ``prepare`` makes a case's inputs from a seed, ``run`` makes one
pass, ``work`` says what a pass cannot do without, and ``exact`` evaluates the
outputs in FP64 with torch alone.

Families:

* ``search``    per-pair records of ``cryo_clmatrix``: noisy projections of a
  blob phantom, all pairs, every precision, with and without the map filter;
* ``pft``       the polar Fourier transform before it, both methods;
* ``rotlines``  common lines and 1-D shifts of known rotations;
* ``lsqr``      the least squares for the 2-D shifts;
* ``vote``      the voting synchronization matrix;
* ``sync3n``    the triangle scores, the pair probabilities and one step of
  the J-synchronization power method on one set of relative rotations.
"""
import math

import numpy as np
import torch

import aspire_amd
from aspire_amd import clmatrix, shifts, sync3n, vote

DEV = "cuda"
PROBS = (0.5, 1.0, 2.2, 1.0, 2.5, 0.78)  # P2, A, a, B, b, x0


def _search(name, K, n_r, n_theta, max_shift, step, precision, snr, dtype="complex128", radius=0):
    return dict(name=name, family="search", K=K, n_r=n_r, n_theta=n_theta, max_shift=max_shift, step=step,
                precision=precision, snr=snr, dtype=dtype, radius=radius)


def listed():
    return [
        # a few class averages looked at interactively: latency of one call
        _search("search_small_fp16", 40, 33, 360, 0.0, 1.0, "fp16", 1.0),
        # 1000 images, 13 shifts, SNR 1/8 with BF16 operands
        _search("search_mid_bf16", 1000, 45, 360, 6.0, 1.0, "bf16", 0.125),
        # the headline's per-pair shape (n_r=65, 41 shifts, SNR 1/16) in the default precision
        _search("search_large_fp16", 2000, 65, 360, 10.0, 0.5, "fp16", 0.0625),
        # the plain FP32 path, an odd ray count and single-precision rays
        _search("search_fp32", 251, 44, 300, 4.0, 1.0, "fp32", 0.125, "complex64"),
        # the FP64 reference arithmetic on a small stack, a user's check of the fast paths
        _search("search_fp64", 100, 45, 360, 6.0, 1.0, "fp64", 0.125),
        # argument 6 of cryo_clmatrix, the 3 x 3 map filter, on the 100-image workload
        _search("search_filtered", 100, 33, 360, 0.0, 1.0, "fp16", 1.0, radius=1),
        # polar Fourier transform of the headline's images, exact sums (the default)
        dict(name="pft_exact", family="pft", K=1000, n=129, n_r=65, n_theta=360, method="exact", dtype="float64"),
        # large single-precision images through the NUFFT
        dict(name="pft_nufft", family="pft", K=100, n=359, n_r=180, n_theta=360, method="nufft", dtype="float32"),
        # cryo_estimate_shifts' pair loop over every pair
        dict(name="rotlines", family="rotlines", K=1500, n_r=65, n_theta=360, max_shift=10.0, step=0.5, share=1.0),
        # its least squares, 4.5 million equations with outlier lines
        dict(name="lsqr", family="lsqr", K=3000, n_theta=360, wrong=0.3),
        # the voting synchronization matrix of 1000 images
        dict(name="vote", family="vote", K=1000, n_theta=360, wrong=0.3),
        # the sync3n triangle kernels of 1000 images, 4 vectors in the power step
        dict(name="sync3n", family="sync3n", N=1000, bins=100, vectors=4, entries=0),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


# contraction work (8 S L^2 R per pair) a drawn search may have, by precision
_MOST = {"bf16": 6e14, "fp16": 6e14, "fp32": 1.2e13, "fp64": 2e12, "filtered": 1e11}


def draw(rng):
    family = rng.choice(["search", "search", "search", "search", "filtered", "pft", "pft", "rotlines", "lsqr",
                         "vote", "sync3n"])
    n_theta = rng.choice([72, 150, 180, 300, 360, 360])
    if family in ("search", "filtered"):
        precision = "fp64" if family == "filtered" else rng.choice(["fp16", "fp16", "bf16", "fp32", "fp64"])
        K, n_r = _log_uniform(rng, 8, 1500), rng.randint(17, 97)
        step = rng.choice([1.0, 1.0, 0.5])
        max_shift = step * rng.choice([0, 2, 4, 7, 12])
        if family == "filtered":
            max_shift = step * rng.choice([0, 0, 1])
        snr = rng.choice([0.125, 0.0625] if precision == "bf16" else [1.0, 0.125, 0.0625])
        c = _search("", K, n_r, n_theta, max_shift, step, precision, snr, rng.choice(["complex128", "complex64"]),
                    rng.randint(1, 3) if family == "filtered" else 0)
        while c["K"] > 4 and _contraction(c) > _MOST["filtered" if c["radius"] else precision]:
            c["K"] = c["K"] * 9 // 10
    elif family == "pft":
        n = rng.randint(33, 259)
        c = dict(family="pft", K=_log_uniform(rng, 1, 900), n=n, n_r=(n + 1) // 2, n_theta=n_theta,
                 method=rng.choice(["exact", "nufft"]), dtype=rng.choice(["float64", "float32"]))
        while c["K"] > 1 and c["K"] * c["n"] ** 2 * c["n_r"] * n_theta > 6e11:
            c["K"] = c["K"] * 9 // 10
    elif family == "rotlines":
        c = dict(family="rotlines", K=_log_uniform(rng, 10, 1400), n_r=rng.randint(17, 65), n_theta=n_theta,
                 max_shift=float(rng.choice([0, 3, 6, 10])), step=rng.choice([1.0, 0.5]),
                 share=rng.choice([1.0, 1.0, 0.1]))
    elif family == "sync3n":
        c = dict(family="sync3n", N=_log_uniform(rng, 20, 900), bins=rng.choice([10, 100, 256]),
                 vectors=rng.randint(1, 5), entries=rng.choice([0, 0, 1, 2]))
    else:
        c = dict(family=family, K=_log_uniform(rng, 20, 2800 if family == "lsqr" else 900), n_theta=n_theta,
                 wrong=rng.choice([0.0, 0.3, 0.8]))
    c.pop("name", None)
    return c


# ------------------------------------------------------------------ inputs
def _rotations(gen, K):
    """K Haar rotations, K x 3 x 3 float64 on the CPU."""
    q = torch.randn((K, 4), generator=gen, dtype=torch.float64)
    a, b, c, d = (q / q.norm(dim=1, keepdim=True)).T
    return torch.stack([a * a + b * b - c * c - d * d, 2 * b * c - 2 * a * d, 2 * a * c + 2 * b * d,
                        2 * b * c + 2 * a * d, a * a - b * b + c * c - d * d, -2 * a * b + 2 * c * d,
                        -2 * a * c + 2 * b * d, 2 * a * b + 2 * c * d, a * a - b * b - c * c + d * d],
                       dim=1).reshape(K, 3, 3)


def _images(gen, rots, n, snr, shift):
    """K x n x n noisy projections of a 20-blob phantom, shifted up to
    `shift` px, index order [image, x, y] (x along the rotation's second row)."""
    K = rots.shape[0]
    centers = torch.randn((20, 3), generator=gen, dtype=torch.float64)
    centers = centers / centers.norm(dim=1, keepdim=True) * 0.5 * torch.rand((20, 1), generator=gen, dtype=torch.float64) ** (1 / 3)
    width = 0.05 + 0.1 * torch.rand(20, generator=gen, dtype=torch.float64)
    amp = 0.5 + 0.5 * torch.rand(20, generator=gen, dtype=torch.float64)
    px = 2.0 / (n - 1) * shift * (2 * torch.rand((K, 2), generator=gen, dtype=torch.float64) - 1)
    x0 = (rots[:, 1] @ centers.T + px[:, :1]).to(DEV)
    y0 = (rots[:, 0] @ centers.T + px[:, 1:]).to(DEV)
    w2, coef = (width ** 2).to(DEV), (amp * width * math.sqrt(math.pi)).to(DEV)
    t = (torch.arange(n, dtype=torch.float64, device=DEV) - (n - 1) / 2) / ((n - 1) / 2)
    ex = torch.exp(-((t[None, :, None] - x0[:, None, :]) ** 2) / w2) * coef
    ey = torch.exp(-((t[None, None, :] - y0[:, :, None]) ** 2) / w2[:, None])
    img = torch.bmm(ex, ey)
    noise = torch.Generator(device=DEV).manual_seed(int(torch.randint(1 << 40, (1,), generator=gen)))
    img += torch.sqrt(img[0].var() / snr) * torch.randn(img.shape, generator=noise, dtype=torch.float64, device=DEV)
    return img


def _polar(img, n_r, n_theta):
    """The polar Fourier transform's sums, K x n_theta x n_r complex128 (img:
    K x n x n, [image, x, y])."""
    K, n, _ = img.shape
    L = n_theta // 2
    g = torch.ceil(torch.arange(n, dtype=torch.float64, device=DEV) - n / 2)
    r = torch.arange(n_r, dtype=torch.float64, device=DEV) * (2 * math.pi / (2 * n_r - 1))
    th = torch.arange(L, dtype=torch.float64, device=DEV) * (2 * math.pi / n_theta)
    fx, fy = (torch.outer(torch.sin(th), r).ravel(), torch.outer(torch.cos(th), r).ravel())
    x = img.reshape(K, n * n).T.to(torch.complex128)
    out = torch.empty((L * n_r, K), dtype=torch.complex128, device=DEV)
    step = max(64, (1 << 25) // (n * n))
    for m in range(0, L * n_r, step):
        ph = fx[m:m + step, None, None] * g[:, None] + fy[m:m + step, None, None] * g
        out[m:m + step] = torch.polar(torch.ones_like(ph), ph).reshape(-1, n * n) @ x
    pf = torch.empty((K, n_theta, n_r), dtype=torch.complex128, device=DEV)
    pf[:, :L] = out.reshape(L, n_r, K).permute(2, 0, 1)
    pf[:, L:] = pf[:, :L].conj()
    return pf


def _pairs(K):
    return torch.triu_indices(K, K, 1)


def _true_lines(rots, n_theta):
    """1-based common lines of every pair k1 < k2, cl1 <= n_theta/2."""
    r, (i, j) = rots.to(DEV), _pairs(rots.shape[0]).to(DEV)
    # U = R_j^T R_i
    ut = lambda a, b: (r[j, 0, a] * r[i, 0, b] + r[j, 1, a] * r[i, 1, b]) + r[j, 2, a] * r[i, 2, b]  # noqa: E731
    line = lambda y, x: torch.floor((torch.atan2(y, x) + math.pi) / (2 * math.pi) * n_theta + 0.5).long() % n_theta  # noqa: E731
    c1, c2 = line(ut(2, 0), -ut(2, 1)), line(-ut(0, 2), ut(1, 2))
    fold = c1 >= n_theta // 2
    c1, c2 = torch.where(fold, c1 - n_theta // 2, c1), torch.where(fold, c2 - n_theta // 2, c2)
    return c1 + 1, torch.where(c2 < 0, c2 + n_theta, c2) + 1


def _estimated_lines(gen, K, n_theta, wrong):
    """(cl1, cl2) as a search leaves them: the true lines, a share replaced by
    random ones; and the generator of the rest."""
    c1, c2 = _true_lines(_rotations(gen, K), n_theta)
    g = torch.Generator(device=DEV).manual_seed(int(torch.randint(1 << 40, (1,), generator=gen)))
    bad = torch.rand(c1.shape, generator=g, device=DEV) < wrong
    c1 = torch.where(bad, torch.randint(1, n_theta // 2 + 1, c1.shape, generator=g, device=DEV), c1)
    c2 = torch.where(bad, torch.randint(1, n_theta + 1, c2.shape, generator=g, device=DEV), c2)
    return c1.int(), c2.int(), g


def _angles(cl1, cl2, n_theta):
    """Line angles (a, b) and the orientation sign of every equation."""
    L = n_theta // 2
    a, b = (cl1.double() - 1) * math.pi / L, (cl2.double() - 1) * math.pi / L
    flip = b >= math.pi
    return a, torch.where(flip, b - math.pi, b), torch.where(flip, -1.0, 1.0).double()


def _coefficients(cl1, cl2, n_theta):
    a, b, s = _angles(cl1, cl2, n_theta)
    return s * torch.sin(a), s * torch.cos(a), -torch.sin(b), -torch.cos(b)


def prepare(case, seed):
    gen = torch.Generator().manual_seed(int(seed))
    family, st = case["family"], dict(case=case)
    if family in ("search", "rotlines"):
        rots = _rotations(gen, case["K"])
        img = _images(gen, rots, 2 * case["n_r"] - 1, case.get("snr", 0.25), 5.0 if case["max_shift"] else 0.0)
        pf = _polar(img, case["n_r"], case["n_theta"])
        if case.get("dtype") == "complex64":
            pf = pf.to(torch.complex64)
        st["pf"] = pf.permute(2, 1, 0)  # n_r x n_theta x K, column-major
        if family == "rotlines":
            st["rots"] = rots.permute(1, 2, 0).contiguous().to(DEV)
            P = case["K"] * (case["K"] - 1) // 2
            if case["share"] < 1:
                st["sel"] = (torch.rand(P, generator=gen) < case["share"]).to(torch.uint8).to(DEV)
    elif family == "pft":
        img = _images(gen, _rotations(gen, case["K"]), case["n"], 0.0625, 5.0).to(getattr(torch, case["dtype"]))
        st["img"] = img.transpose(1, 2).contiguous().permute(2, 1, 0)  # n x n x K, column-major
    elif family in ("lsqr", "vote"):
        K, T = case["K"], case["n_theta"]
        st["cl1"], st["cl2"], g = _estimated_lines(gen, K, T, case["wrong"])
        if family == "lsqr":
            xy = 10 * torch.rand((K, 2), generator=g, dtype=torch.float64, device=DEV) - 5
            (i, j), c = _pairs(K).to(DEV), _coefficients(st["cl1"], st["cl2"], T)
            s = c[0] * xy[i, 0] + c[1] * xy[i, 1] + c[2] * xy[j, 0] + c[3] * xy[j, 1]
            s += 0.5 * torch.randn(s.shape, generator=g, dtype=torch.float64, device=DEV)
            st["shift"] = (torch.round(2 * s) / 2).clamp(-10, 10)  # on the search's half-pixel grid
    else:
        N = case["N"]
        i, j = _pairs(N)
        r = _rotations(gen, N)
        m = torch.bmm(r[i].transpose(1, 2).contiguous(), r[j].contiguous())
        out = torch.rand(len(i), generator=gen) < 0.3
        m[out] = _rotations(gen, int(out.sum()))
        J = torch.tensor([1.0, 1.0, -1.0], dtype=torch.float64)
        flip = (torch.rand(len(i), generator=gen) < 0.4)[:, None, None]
        m = torch.where(flip, J[:, None] * m * J, m)
        st["R"] = m.transpose(1, 2).contiguous().to(DEV)  # each matrix column-major
        st["v"] = torch.rand((len(i), case["vectors"]), generator=gen, dtype=torch.float64).to(DEV)
        st["w"] = torch.rand(len(i), generator=gen, dtype=torch.float64).to(DEV)
    return st


def run(st):
    c = st["case"]
    if c["family"] == "search":
        rec, _ = clmatrix.clmatrix_records(st["pf"], c["max_shift"], c["step"], c["precision"],
                                           map_filter_radius=c["radius"])
        return rec
    if c["family"] == "pft":
        pf, freqs = aspire_amd.cryo_pft(st["img"], c["n_r"], c["n_theta"], method=c["method"])
        return dict(pf=pf, freqs=freqs)
    if c["family"] == "rotlines":
        cl1, cl2, s = shifts.common_lines_from_rotations(st["pf"], st["rots"], c["max_shift"], c["step"], st.get("sel"))
        return dict(cl1=cl1, cl2=cl2, shift=s)
    if c["family"] == "lsqr":
        return shifts.estimate_shifts(st["cl1"], st["cl2"], st["shift"], c["K"], c["n_theta"], 1e-8, 100)[0]
    if c["family"] == "vote":
        return vote.syncmatrix_vote_records(st["cl1"], st["cl2"], c["K"], c["n_theta"])[0]
    cum, hist, _ = sync3n.triangles_scores_mex(st["R"], c["bins"])
    ind, arb, _ = sync3n.pairs_probabilities_mex(st["R"], *PROBS)
    v2, _ = sync3n.signs_times_v_mex(st["R"], st["v"], c["entries"], st["w"] if c["entries"] == 2 else None)
    return dict(cum=cum, hist=hist, ind=ind, arb=arb, v2=v2)


# -------------------------------------------------------------------- work
def _n_shifts(case):
    return int(math.ceil(2 * case["max_shift"] / case["step"] + 1))


def _contraction(case):
    """Flops of both correlation maps of every pair and shift."""
    P, L = case["K"] * (case["K"] - 1) // 2, case["n_theta"] // 2
    return 8.0 * _n_shifts(case) * L * L * (case["n_r"] - 1) * P


def work(case):
    family = case["family"]
    K = case.get("K", case.get("N"))
    P = K * (K - 1) // 2
    if family == "search":
        rays = K * case["n_theta"] * case["n_r"] * (8 if case["dtype"] == "complex64" else 16)
        # both maps come from one set of products on a symmetric shift grid
        flops = _contraction(case) / 2
        if case["radius"]:
            flops += 4.0 * (2 * case["radius"] + 1) * 2 * (case["n_theta"] // 2) ** 2 * _n_shifts(case) * P
        return dict(bytes=rays + 28.0 * P, flops=flops)
    if family == "pft":
        single = case["dtype"] == "float32"
        points = case["n_r"] * case["n_theta"] // 2
        b = K * (case["n"] ** 2 * (4 if single else 8) + 2 * points * (8 if single else 16))
        if case["method"] == "exact":
            return dict(bytes=float(b), flops=4.0 * points * case["n"] ** 2 * K)
        side = 2 * case["n"]
        return dict(bytes=float(b), flops=K * (2.5 * side * side * math.log2(side * side) + 4.0 * 256 * points))
    if family == "rotlines":
        return dict(bytes=K * case["n_theta"] * case["n_r"] * 16 + 16.0 * P,
                    flops=2.0 * _n_shifts(case) * (case["n_r"] - 1) * 4 * P * case["share"])
    if family == "lsqr":
        return dict(bytes=16.0 * P + 16 * K, flops=30 * 16.0 * P)
    if family == "vote":
        return dict(bytes=8.0 * P + 32.0 * K * K, flops=60 * 8.0 * P * K)
    return dict(bytes=P * (3 * 72 + 24 + 16.0 * case["vectors"]), flops=3 * 297.0 * K * (K - 1) * (K - 2) / 6)


# ------------------------------------------------------- the outputs in FP64
def _half_rays(pf):
    """Filtered, normalized half rays, K x L x R complex128 (pf: K x T x n_r)."""
    K, T, n_r = pf.shape
    L, R = T // 2, n_r - 1
    full = torch.cat([pf[:, L:, 1:].flip(2), pf[:, :L]], dim=2).to(torch.complex128)
    k = torch.arange(-R, R + 1, dtype=torch.float64, device=DEV)
    h = torch.sqrt(k.abs()) * torch.exp(-k ** 2 / (2 * (R / 4.0) ** 2))
    h[R - 1:R + 2] = 0
    full = full * h
    return (full / torch.linalg.vector_norm(full, dim=2, keepdim=True))[:, :, :R]


def _phases(case):
    R = case["n_r"] - 1
    s = -case["max_shift"] + torch.arange(_n_shifts(case), dtype=torch.float64, device=DEV) * case["step"]
    th = -2 * math.pi * torch.outer(s, torch.arange(-R, 0, dtype=torch.float64, device=DEV)) / (2 * R + 1)
    return s, torch.polar(torch.ones_like(th), th)


def _filtered(maps, d):
    """cryo_average_clmap of n x L x 2L maps."""
    L = maps.shape[1]
    ext = torch.cat([maps, maps.roll(L, 2)], dim=1)
    w = 1.25 ** -torch.arange(-d, d + 1, dtype=torch.float64, device=DEV).abs()
    rows = sum(float(w[i]) * ext.roll(d - i, 1) for i in range(2 * d + 1))
    return 1.25 ** 21 * sum(float(w[i]) * rows.roll(d - i, 2) for i in range(2 * d + 1))[:, :L]


def _exact_search(case, seed):
    if _contraction(case) * (3 if case["radius"] else 1) > 1.2e14:
        return None
    rays = _half_rays(prepare(case, seed)["pf"].permute(2, 1, 0))
    s, ph = _phases(case)
    K, L, R = rays.shape
    corr, shift = [], []
    flat = torch.view_as_real(rays).reshape(K * L, 2 * R).T.contiguous()
    for k in range(K - 1):
        n = K - 1 - k
        best, bs = torch.zeros(n, dtype=torch.float64, device=DEV), torch.zeros(n, dtype=torch.float64, device=DEV)
        for j in range(len(s)):
            both = torch.stack([rays[k] * ph[j], rays[k].conj() * ph[j]])
            c = 2 * (torch.view_as_real(both).reshape(2 * L, 2 * R) @ flat[:, (k + 1) * L:])
            c = c.reshape(2, L, n, L)
            if case["radius"]:
                v = _filtered(c.permute(2, 1, 0, 3).reshape(n, L, 2 * L), case["radius"]).amax(dim=(1, 2))
            else:
                v = c.amax(dim=(0, 1, 3))
            bs = torch.where(v > best, s[j], bs)
            best = torch.maximum(v, best)
        corr.append(best)
        shift.append(bs)
    return dict(cl1=None, cl2=None, j=None, corr=torch.cat(corr), shift=torch.cat(shift))


def _exact_rotlines(case, seed):
    st = prepare(case, seed)
    rays = _half_rays(st["pf"].permute(2, 1, 0))
    s, ph = _phases(case)
    K, L, R = rays.shape
    i, j = _pairs(K).to(DEV)
    c1, c2 = _true_lines(st["rots"].permute(2, 0, 1), case["n_theta"])
    out = torch.empty(len(i), dtype=torch.float64, device=DEV)
    for a in range(0, len(i), 1 << 17):
        q = slice(a, a + (1 << 17))
        x, y = rays[i[q], c1[q] - 1], rays[j[q], (c2[q] - 1) % L]
        v1, v2 = (((z * y) @ ph.conj().T).real.max(dim=1) for z in (x.conj(), x))
        out[q] = s[torch.where(v1.values > v2.values, v1.indices, v2.indices)]
    if "sel" in st:
        out *= st["sel"]
    return dict(cl1=None, cl2=None, shift=out)


def _exact_lsqr(case, seed):
    """The minimum-norm least-squares solution, by CGLS run to convergence."""
    st = prepare(case, seed)
    K = case["K"]
    (i, j), c = _pairs(K).to(DEV), _coefficients(st["cl1"], st["cl2"], case["n_theta"])

    def forward(x):
        return c[0] * x[i, 0] + c[1] * x[i, 1] + c[2] * x[j, 0] + c[3] * x[j, 1]

    def adjoint(u):
        out = torch.zeros((K, 2), dtype=torch.float64, device=DEV)
        for at, cx, cy in ((i, c[0], c[1]), (j, c[2], c[3])):
            out.index_add_(0, at, torch.stack([cx * u, cy * u], dim=1))
        return out

    x = torch.zeros((K, 2), dtype=torch.float64, device=DEV)
    r = st["shift"].clone()
    g = adjoint(r)
    p, gg = g.clone(), (g * g).sum()
    stop = float(gg) * 1e-24
    for _ in range(100):
        if float(gg) <= stop:
            break
        q = forward(p)
        step = gg / (q * q).sum()
        x, r = x + step * p, r - step * q
        g = adjoint(r)
        new = (g * g).sum()
        p, gg = g + (new / gg) * p, new
    return x


def _exact_vote(case, seed):
    st = prepare(case, seed)
    K, T = case["K"], case["n_theta"]
    cl = torch.zeros((K, K), dtype=torch.float64, device=DEV)
    i, j = _pairs(K).to(DEV)
    cl[i, j], cl[j, i] = st["cl1"].double(), st["cl2"].double()
    S = torch.eye(2 * K, dtype=torch.float64, device=DEV)
    ticks = torch.linspace(0, 180, 60, dtype=torch.float64, device=DEV)
    for a in range(K - 1):
        b = torch.arange(a + 1, K, device=DEV)
        d1 = cl[a][None] - cl[a, b][:, None]
        d2 = cl[b, a][:, None] - cl[b]
        d3 = cl[:, b].T - cl[:, a][None]
        t1, t2, t3 = (d * 2 * math.pi / T for d in (d1, d2, d3))
        c1, c2, c3 = torch.cos(t1), torch.cos(t2), torch.cos(t3)
        ok = (1 + 2 * c1 * c2 * c3 - (c1 * c1 + c2 * c2 + c3 * c3) > 1e-5) & (cl[a] != 0) & (cl[b] != 0)
        cp = ((c3 - c1 * c2) / (torch.sin(t1) * torch.sin(t2))).clamp(-1, 1)
        ang = torch.where(ok, torch.acos(cp) * 180 / math.pi, 1e6)
        hist = torch.stack([torch.exp(-(ang - x) ** 2 / 18).sum(dim=1) for x in ticks], dim=1)
        keep = ok & ((ang - ticks[hist.argmax(dim=1)][:, None]).abs() < 6)
        # relative rotations of the kept triangles: the second angle's cosine from (c3, c2, c1)
        ca = (c3 - c2 * c1) / torch.sqrt(1 - c2 * c2) / torch.sqrt(1 - c1 * c1)
        far = lambda d: (d > T / 2 + 1e-12) | ((d < -1e-12) & (d > -T / 2))  # noqa: E731
        ca = torch.where(far(d1) != far(-d2), -ca, ca).clamp(-1, 1)
        n = keep.sum(dim=1).clamp(min=1)
        cb = torch.where(keep, ca, 0).sum(dim=1) / n
        some = (keep.sum(dim=1) > 0).double()
        t = math.pi - (cl[b, a] - 1) * 2 * math.pi / T
        u = (cl[a, b] - 1) * 2 * math.pi / T - math.pi
        sa, ca_, sc, cc = torch.sin(t), torch.cos(t), torch.sin(u), torch.cos(u)
        blk = [[(cc * ca_ - sc * cb * sa) * some, (-cc * sa - sc * cb * ca_) * some],
               [(sc * ca_ + cc * cb * sa) * some, (-sa * sc + cc * cb * ca_) * some]]
        for x in range(2):
            for y in range(2):
                S[2 * a + x, 2 * b + y] = blk[x][y]
                S[2 * b + y, 2 * a + x] = blk[x][y]
    return S


def _exact_sync3n(case, seed):
    st = prepare(case, seed)
    N = case["N"]
    i, j = _pairs(N).to(DEV)
    m = st["R"].transpose(1, 2)
    full = torch.zeros((N, N, 3, 3), dtype=torch.float64, device=DEV)
    full[i, j] = m
    J = torch.tensor([1.0, 1.0, -1.0], dtype=torch.float64, device=DEV)
    ne = case["vectors"]
    V = torch.zeros((N, N, ne), dtype=torch.float64, device=DEV)
    V[i, j] = st["v"]
    W = torch.zeros((N, N), dtype=torch.float64, device=DEV)
    W[i, j] = st["w"]
    cum, ind, arb = (torch.zeros((N, N), dtype=torch.float64, device=DEV) for _ in range(3))
    v2 = torch.zeros((N, N, ne), dtype=torch.float64, device=DEV)
    hist = torch.zeros(case["bins"], dtype=torch.float64, device=DEV)
    edges = torch.cumsum(torch.full((case["bins"] - 1,), 1.0 / case["bins"], dtype=torch.float64), 0).to(DEV)
    # signs of the side pairs (ij,jk), (ik,jk), (ij,ik) in the four configurations
    sign = torch.tensor([[1, 1, 1], [-1, 1, -1], [-1, -1, 1], [1, -1, -1]], dtype=torch.float64, device=DEV)
    P2, A, ea, B, eb, x0 = PROBS
    for a in range(N - 2):
        n = N - 1 - a
        jj, kk = torch.triu_indices(n, n, 1, device=DEV) + a + 1
        x, y, z = full[a, jj], full[jj, kk], full[a, kk]
        flip = lambda r: J[:, None] * r * J  # noqa: E731
        prod = lambda p, q: (p[:, :, :, None] * q[:, None]).sum(dim=2)  # noqa: E731
        xy = prod(x, y)
        c = torch.stack([((u - w) ** 2).sum(dim=(1, 2)) for u, w in
                         ((xy, z), (prod(flip(x), y), z), (prod(x, flip(y)), z), (xy, flip(z)))], dim=1)
        low, best = c.min(dim=1)
        sg = sign[best]
        sc = []
        for q in range(3):
            other = torch.where(sign[:, q][None] != sg[:, q:q + 1], c, torch.inf).min(dim=1).values
            sc.append(1 - torch.sqrt(low / other))
        hist += torch.bincount(torch.bucketize(torch.cat(sc), edges, right=True), minlength=case["bins"])
        pairs = ((torch.full_like(jj, a), jj), (jj, kk), (torch.full_like(jj, a), kk))
        u = [1 - q for q in sc]
        li = [torch.log(P2 * B * q ** eb * torch.exp(-eb / (1 - x0) * q) + (1 - P2) * A * q ** ea) for q in u]
        la = [torch.log(A * q ** ea) for q in u]
        if case["entries"] == 0:
            e = [sg[:, q] for q in range(3)]
        elif case["entries"] == 1:
            e = [sg[:, q] * sc[q] for q in range(3)]
        else:
            e = [sg[:, q] * (W[pairs[0]] * W[pairs[1]] * W[pairs[2]]) for q in range(3)]
        vij, vjk, vik = (V[p] for p in pairs)
        e = [q[:, None] for q in e]
        for p, (s, t), v in ((pairs[0], (0, 2), e[0] * vjk + e[2] * vik), (pairs[1], (0, 1), e[0] * vij + e[1] * vik),
                             (pairs[2], (1, 2), e[2] * vij + e[1] * vjk)):
            cum.index_put_(p, sc[s] + sc[t], accumulate=True)
            ind.index_put_(p, li[s] + li[t], accumulate=True)
            arb.index_put_(p, la[s] + la[t], accumulate=True)
            v2.index_put_(p, v, accumulate=True)
    return dict(cum=cum[i, j], hist=hist, ind=ind[i, j], arb=arb[i, j], v2=v2[i, j])


def exact(case, seed):
    family = case["family"]
    if family == "search":
        return _exact_search(case, seed)
    if family == "pft":
        if 8.0 * case["n"] ** 2 * case["n_r"] * case["n_theta"] / 2 * (case["K"] + 40) > 2e13:
            return None
        img = prepare(case, seed)["img"].double().permute(2, 0, 1)
        pf = _polar(img, case["n_r"], case["n_theta"]).permute(2, 1, 0)
        k, th = np.arange(case["n_r"]), np.arange(case["n_theta"] // 2) * (2 * np.pi / case["n_theta"])
        w = k * (2 * np.pi / (2 * case["n_r"] - 1))
        return dict(pf=pf, freqs=np.stack([np.outer(np.sin(th), w).ravel(), np.outer(np.cos(th), w).ravel()], axis=1))
    if family == "rotlines":
        return _exact_rotlines(case, seed)
    if family == "lsqr":
        return _exact_lsqr(case, seed)
    if family == "vote":
        return _exact_vote(case, seed)
    return _exact_sync3n(case, seed)
