"""The work that a program using paratt_amd has it do, as timed cases.

Families (key "kind" of a case):

  round     z = x + beta*y (formal sum) and its rounding: the step that every
            TT algorithm repeats.  Small trains are bound by latency and
            launches, the headline one by the matrix cores.
  rk4       one step-truncation RK4 step of the reaction-Burgers equation:
            seventeen roundings of low-rank, rank-deficient formal sums, four
            Hadamard products, eight stencil sums.
  modesum   S = sum_i D_i u for a periodic 3-point stencil: the core-wise
            finite-difference operator as an exact rank-2r train (streaming).
  flux      a copy of a train and the CDF Lax-Friedrichs flux along every mode
            of it: one dimension-split step of the CDF equation (streaming).
  dot       the grid-normalised inner product of two trains.
  marginal  all modes of a train but the first contracted against quadrature
            weights, then the cumulative distribution along the first.

Cores are handed out indexed (r_k, n_k, r_{k+1}) over the column-major core
memory, as views of the library's own device buffers or, after a rounding, as
their magnitudes: the signs of singular vectors are free, so a program that
compares or stores trains takes the magnitudes and an entry, which ties the
signs together.
"""
import ctypes as C
import math

import numpy as np
import torch

import paratt_amd as P


def listed():
    return [
        # the smallest rounding: a tiny correction added to a rank-6 train
        {"name": "round_d8_n16_r6", "kind": "round", "d": 8, "n": 16, "rx": 6, "ry": 6,
         "beta": 1e-10, "eps": 1e-8, "cap": 0, "mixed": False},
        # an ordinary sum whose ranks are all kept
        {"name": "round_d20_n32_r16", "kind": "round", "d": 20, "n": 32, "rx": 16, "ry": 16,
         "beta": 1.0, "eps": 1e-10, "cap": 0, "mixed": False},
        # sizes that are multiples of nothing, cut by the cap
        {"name": "round_d12_n301_r37_cap41", "kind": "round", "d": 12, "n": 301, "rx": 37,
         "ry": 22, "beta": 1.0, "eps": 1e-8, "cap": 41, "mixed": False},
        # the headline rounding
        {"name": "round_d40_n1024_r64_cap64", "kind": "round", "d": 40, "n": 1024, "rx": 64,
         "ry": 64, "beta": 1.0, "eps": 1e-8, "cap": 64, "mixed": False},
        # a small update of a large train: ill-conditioned sum, cut by the tolerance
        {"name": "round_d10_n1024_r64_update", "kind": "round", "d": 10, "n": 1024, "rx": 64,
         "ry": 64, "beta": 1e-10, "eps": 1e-8, "cap": 0, "mixed": False},
        # formal ranks above 128 (sums of several terms, products of trains)
        {"name": "round_d6_n96_r120_cap100", "kind": "round", "d": 6, "n": 96, "rx": 120,
         "ry": 72, "beta": 1.0, "eps": 1e-8, "cap": 100, "mixed": False},
        # the mixed-precision option of the left-to-right sweep
        {"name": "round_d12_n1024_r64_mixed", "kind": "round", "d": 12, "n": 1024, "rx": 64,
         "ry": 64, "beta": 1.0, "eps": 1e-8, "cap": 64, "mixed": True},
        # the time stepper at the size of its benchmark
        {"name": "rk4_d20_n256", "kind": "rk4", "d": 20, "n": 256, "terms": 2, "eps": 1e-8,
         "cap": 64},
        {"name": "modesum_d20_n1024_r32", "kind": "modesum", "d": 20, "n": 1024, "r": 32},
        {"name": "flux_d20_n256_r25", "kind": "flux", "d": 20, "n": 256, "r": 25},
        {"name": "dot_d40_n1024_r64", "kind": "dot", "d": 40, "n": 1024, "rx": 64, "ry": 64},
        # the CDF program's output step
        {"name": "marginal_d20_n64_r25", "kind": "marginal", "d": 20, "n": 64, "r": 25},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["round"] * 6 + ["rk4", "rk4", "modesum", "flux", "dot", "marginal"])
    if kind == "round":
        beta, eps = rng.choice([(1.0, 1e-6), (1.0, 1e-8), (1.0, 1e-10), (1e-3, 1e-8),
                                (1e-10, 1e-8)])
        size = rng.choice(["small", "small", "wide", "large"])
        if size == "small":
            d, n = rng.randint(4, 24), _log(rng, 12, 300)
            rx, ry = _log(rng, 2, 32), _log(rng, 2, 32)
        elif size == "wide":
            d, n = rng.randint(4, 16), _log(rng, 200, 1100)
            rx, ry = _log(rng, 16, 64), _log(rng, 16, 64)
        else:
            d, n = rng.randint(3, 6), _log(rng, 32, 100)
            rx, ry = _log(rng, 60, 100), _log(rng, 60, 100)
        r = rx + ry
        cap = rng.choice([0, max(2, int(0.6 * r))]) if beta == 1.0 else 0
        if size == "large":
            cap = max(rx, ry)
        return {"kind": "round", "d": d, "n": n, "rx": rx, "ry": ry, "beta": beta, "eps": eps,
                "cap": cap, "mixed": rng.random() < 0.15 and r <= 128}
    if kind == "rk4":
        return {"kind": "rk4", "d": rng.randint(4, 20), "n": _log(rng, 32, 256),
                "terms": rng.choice([1, 2]), "eps": 1e-8, "cap": 64}
    if kind == "modesum":
        return {"kind": "modesum", "d": rng.randint(3, 20), "n": _log(rng, 30, 1024),
                "r": _log(rng, 2, 32)}
    if kind == "flux":
        return {"kind": "flux", "d": rng.randint(3, 20), "n": _log(rng, 30, 1024),
                "r": _log(rng, 2, 48)}
    if kind == "dot":
        return {"kind": "dot", "d": rng.randint(3, 40), "n": _log(rng, 16, 1024),
                "rx": _log(rng, 3, 64), "ry": _log(rng, 3, 64)}
    return {"kind": "marginal", "d": rng.randint(3, 20), "n": _log(rng, 20, 300),
            "r": _log(rng, 2, 32)}


# ---------------------------------------------------------------- inputs

def _ranks(d, r):
    return [1] + [r] * (d - 1) + [1]


def _gen(seed, salt):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed) * 1009 + salt)
    return g


def _gaussian_cores(d, n, r, seed, salt):
    """N(0, 1/(n r_k)) cores, (r_{k+1}, n, r_k) each: trains of norm O(1)."""
    g, rr = _gen(seed, salt), _ranks(d, r)
    return [torch.randn(rr[k + 1], n, rr[k], generator=g, device="cuda", dtype=torch.float64)
            * (1.0 / math.sqrt(n * rr[k])) for k in range(d)]


def _density_cores(d, n, r, seed, salt):
    """Positive cores, as of a sum of r product densities with some mixing."""
    g, rr = _gen(seed, salt), _ranks(d, r)
    return [(torch.rand(rr[k + 1], n, rr[k], generator=g, device="cuda", dtype=torch.float64)
             + 0.1) * (1.0 / rr[k]) for k in range(d)]


def _bump_cores(d, n, terms, seed):
    """Sum of `terms` products of Gaussians on the periodic grid [0, 2 pi): centres about pi
    and widths about 0.5, both perturbed, as an exact rank-`terms` train."""
    rng = np.random.default_rng(int(seed))
    x = 2.0 * np.pi * np.arange(n) / n
    out = []
    for k in range(d):
        v = [np.exp(-((x - np.pi - 0.3 * rng.standard_normal()) ** 2)
                    / (0.5 * (1.0 + 0.3 * rng.uniform(-1.0, 1.0)))) for _ in range(terms)]
        r0, r1 = (1 if k == 0 else terms), (1 if k == d - 1 else terms)
        c = np.zeros((r1, n, r0))
        for t in range(terms):
            c[t if r1 > 1 else 0, :, t if r0 > 1 else 0] += v[t] * (1.0 if k else 1.0 / (1 + t))
        out.append(torch.from_numpy(c).cuda())
    return out


class _Array:
    """A core's device memory for torch; keeps the train that owns it."""

    def __init__(self, owner, ptr, shape):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": "<f8", "version": 2,
                                         "data": (int(ptr), False), "strides": None}


def _buffers(t):
    """The cores' memory as contiguous tensors (r_{k+1}, n_k, r_k)."""
    x = t.p.contents.x.contents
    d = x.numDim
    r, n, ptr = x.ttRank, x.dim, x.coreList
    return [torch.as_tensor(_Array(t, ptr[k], (r[k + 1], n[k], r[k])), device="cuda")
            for k in range(d)]


def _views(t):
    return [b.permute(2, 1, 0) for b in _buffers(t)]


def _train(cores):
    """The cores as a device train of the library."""
    d = len(cores)
    t = P.DevTT([c.shape[1] for c in cores], [1] + [c.shape[0] for c in cores])
    for v, c in zip(_buffers(t), cores):
        v.copy_(c)
    torch.cuda.synchronize()
    return t


def _stencil():
    return np.array([-0.5, 0.125, 0.5])


def _flux_coefficients(case, seed):
    """Wave speeds with both ghost values, sources, per mode."""
    rng = np.random.default_rng(int(seed))
    n = case["n"]
    return [(rng.standard_normal(n), rng.standard_normal(2), 0.1 * rng.standard_normal(n))
            for _ in range(case["d"])]


def _index(case, seed):
    rng = np.random.default_rng(int(seed))
    return [int(i) for i in rng.integers(0, case["n"], case["d"])]


DT_FLUX, DX_FLUX = 1.0e-4, 0.02


def _dp(a):
    return a.ctypes.data_as(C.POINTER(C.c_double))


def prepare(case, seed):
    kind, d, n = case["kind"], case["d"], case["n"]
    L = P.lib()
    s = {"case": case, "lib": L}
    if kind == "round":
        s["x"] = _train(_gaussian_cores(d, n, case["rx"], seed, 1))
        s["y"] = _train(_gaussian_cores(d, n, case["ry"], seed, 2))
        r = case["rx"] + case["ry"]
        s["z"] = P.DevTT([n] * d, _ranks(d, r))
        s["caps"] = _ranks(d, case["cap"] if case["cap"] else r)
        s["index"] = _index(case, seed)
    elif kind == "rk4":
        L.paratt_amd_rxn_burgers_setup.argtypes = [C.c_double, C.c_double, C.c_double, C.c_int]
        pp = C.POINTER(P.Paratt)
        L.paratt_amd_rk4_st.argtypes = [pp, pp, C.c_void_p, C.c_double, C.c_double, C.c_int]
        s["u"] = _train(_bump_cores(d, n, case["terms"], seed))
        s["new"] = P.DevTT([n] * d, [1] * (d + 1))
        s["field"] = C.cast(L.paratt_amd_rxn_burgers_field, C.c_void_p)
    elif kind == "modesum":
        L.paratt_amd_mode_sum.argtypes = [C.POINTER(P.Paratt), C.POINTER(C.c_double),
                                          C.POINTER(P.Paratt)]
        s["u"] = _train(_gaussian_cores(d, n, case["r"], seed, 1))
        s["s"] = P.DevTT([n] * d, _ranks(d, 2 * case["r"]))
        s["stencil"] = _stencil()
    elif kind == "flux":
        s["u"] = _train(_density_cores(d, n, case["r"], seed, 1))
        s["w"] = P.DevTT([n] * d, _ranks(d, case["r"]))
        s["coef"] = _flux_coefficients(case, seed)
    elif kind == "dot":
        s["x"] = _train(_density_cores(d, n, case["rx"], seed, 1))
        s["y"] = _train(_density_cores(d, n, case["ry"], seed, 2))
    else:
        s["x"] = _train(_density_cores(d, n, case["r"], seed, 1))
        s["w"] = np.full(n, 2.0 / n)
    return s


# ---------------------------------------------------------------- one pass

def _pair_marginals(t, n):
    """Marginals of the neighbouring pairs of modes (n x n each), the others summed with the
    grid's weights: what a program that steps a density looks at."""
    cores = _buffers(t)
    h = 1.0 / n
    sums = [c.sum(dim=1) * h for c in cores]                 # (r1, r0) per core
    left, right = [sums[0].new_ones(1)], [sums[0].new_ones(1)]
    for m in sums[:-1]:
        left.append(m @ left[-1])
    for m in reversed(sums[1:]):
        right.append(right[-1] @ m)
    right.reverse()
    out = []
    for k in range(len(cores) - 1):
        a = cores[k] @ left[k]                               # (r1, n)
        b = torch.tensordot(right[k + 1], cores[k + 1], dims=([0], [0]))  # (n, r1)
        out.append(b @ a)                                    # (n of mode k+1, n of mode k)
    # the library may reuse the cores from its next call on
    torch.cuda.current_stream().synchronize()
    return out


def run(s):
    case, L = s["case"], s["lib"]
    kind, d = case["kind"], case["d"]
    if kind == "round":
        x, y, z = s["x"], s["y"], s["z"]
        L.attac_tt_axpby(1.0, x.tt, case["beta"], y.tt, z.tt)
        if case["mixed"]:
            P.set_leaf_precision(1)
        P.truncate_rel(z, case["eps"], s["caps"])
        if case["mixed"]:
            P.set_leaf_precision(0)
        spec = P.last_round_spectra()[1:d]
        out = {"entry": P.entry(z, s["index"]), "ranks": np.array(z.r),
               "norm": P.last_round_stats().norm,
               "sigma": np.concatenate([spec[:, 16:17], spec[:, :13]], axis=1),
               "cores": [v.abs() for v in _views(z)]}
        # the library may reuse the cores from its next call on
        torch.cuda.current_stream().synchronize()
        return out
    if kind == "rk4":
        L.paratt_amd_rxn_burgers_setup(0.01, 2.0 * math.pi / case["n"], case["eps"], case["cap"])
        L.paratt_amd_rk4_st(s["u"].p, s["new"].p, s["field"], 1.0e-3, case["eps"], case["cap"])
        return {"ranks": np.array(s["new"].r), "pairs": _pair_marginals(s["new"], case["n"])}
    if kind == "modesum":
        L.paratt_amd_mode_sum(s["u"].p, _dp(s["stencil"]), s["s"].p)
        return _views(s["s"])
    if kind == "flux":
        L.copy_rank_change_tt(s["w"].tt, s["u"].tt)
        for k, (c, g, src) in enumerate(s["coef"]):
            L.pattac_apply_cdf_lf_flux(s["w"].p, k, _dp(c), _dp(g), _dp(src), DT_FLUX, DX_FLUX)
        return _views(s["w"])
    if kind == "dot":
        return P.dotprod(s["x"], s["y"])
    t = s["x"]
    for k in range(d - 1, 0, -1):
        t = P.apply_marginal(t, k, s["w"])
    P.marginal_cusum(t, 0, s["w"])
    return t.download_cores()[0]


# ---------------------------------------------------------------- what a pass cannot do without

def _sweep_ranks(d, n, r):
    """Bond ranks after the left-to-right sweep."""
    rr = _ranks(d, r)
    for k in range(1, d):
        rr[k] = min(rr[k], rr[k - 1] * n)
    return rr


def work(case):
    kind, d, n = case["kind"], case["d"], case["n"]

    def size(rr):
        return sum(rr[k] * n * rr[k + 1] for k in range(d))

    if kind == "round":
        r = case["rx"] + case["ry"]
        kept = case["cap"] or (case["rx"] if case["beta"] < case["eps"] else r)
        kept = min(kept, r)
        rr, out = _sweep_ranks(d, n, r), _ranks(d, kept)
        back = [1] * (d + 1)
        for k in range(d - 1, 0, -1):
            back[k] = min(kept, rr[k], back[k + 1] * n)
        fl = 0.0
        for k in range(d - 1):
            # R factor of a left unfolding, R times the next core
            fl += rr[k] * n * rr[k + 1] ** 2 + 2.0 * rr[k + 1] ** 2 * n * _ranks(d, r)[k + 2]
        for k in range(d - 1, 0, -1):
            # U Sigma into the core, its Gram, the new core
            fl += rr[k] ** 2 * n * back[k + 1] + 2.0 * rr[k] * back[k] * n * back[k + 1]
            fl += 2.0 * rr[k - 1] * n * rr[k] * back[k]
        by = 8.0 * (size(_ranks(d, case["rx"])) + size(_ranks(d, case["ry"])) + size(out))
        return {"bytes": by, "flops": fl}
    if kind == "rk4":
        # seventeen roundings of trains of formal ranks of about 20, each read and written once
        r = 12 * case["terms"]
        return {"bytes": 17 * 2 * 8.0 * size(_ranks(d, r)), "flops": 17.0 * 6 * size(_ranks(d, r)) * r}
    if kind == "modesum":
        by = 8.0 * (size(_ranks(d, case["r"])) + size(_ranks(d, 2 * case["r"])))
        return {"bytes": by, "flops": 5.0 * size(_ranks(d, case["r"]))}
    if kind == "flux":
        return {"bytes": 16.0 * size(_ranks(d, case["r"])), "flops": 10.0 * size(_ranks(d, case["r"]))}
    if kind == "dot":
        rx, ry = _ranks(d, case["rx"]), _ranks(d, case["ry"])
        fl = sum(2.0 * n * rx[k] * ry[k + 1] * (ry[k] + rx[k + 1]) for k in range(d))
        return {"bytes": 8.0 * (size(rx) + size(ry)), "flops": fl}
    return {"bytes": 8.0 * size(_ranks(d, case["r"])), "flops": 2.0 * size(_ranks(d, case["r"]))}


# ---------------------------------------------------------------- the same in 64 bits by torch

def _sum_cores(xs, ys, beta):
    d, out = len(xs), []
    for k in range(d):
        a, b = xs[k], ys[k]
        if k == 0:
            out.append(torch.cat([a, beta * b], dim=0))
        elif k == d - 1:
            out.append(torch.cat([a, b], dim=2))
        else:
            c = a.new_zeros(a.shape[0] + b.shape[0], a.shape[1], a.shape[2] + b.shape[2])
            c[: a.shape[0], :, : a.shape[2]] = a
            c[a.shape[0]:, :, a.shape[2]:] = b
            out.append(c)
    return out


def _exact_round(case, seed):
    """The rounding by QR and SVD sweeps on the host (LAPACK)."""
    d, n = case["d"], case["n"]
    r = case["rx"] + case["ry"]
    if sum(float(n) * r * r * r * 6.0 for _ in range(d)) > 3.0e11:
        return None  # more than about twenty seconds on the host
    xs = [c.cpu() for c in _gaussian_cores(d, n, case["rx"], seed, 1)]
    ys = [c.cpu() for c in _gaussian_cores(d, n, case["ry"], seed, 2)]
    # cores as (r0, n, r1), each over sqrt(n): the grid-normalised norm
    z = [c.permute(2, 1, 0).contiguous().numpy() / math.sqrt(n)
         for c in _sum_cores(xs, ys, case["beta"])]
    caps = _ranks(d, case["cap"] if case["cap"] else r)
    for k in range(d - 1):
        q, f = np.linalg.qr(z[k].reshape(-1, z[k].shape[2]))
        z[k] = q.reshape(z[k].shape[0], n, -1)
        z[k + 1] = np.tensordot(f, z[k + 1], axes=(1, 0))
    nrm = float(np.linalg.norm(z[-1]))
    delta = case["eps"] * nrm / math.sqrt(d - 1.0)
    ranks, sigma = _ranks(d, 1), np.zeros((d - 1, 14))
    for k in range(d - 1, 0, -1):
        m = z[k].reshape(z[k].shape[0], -1)
        u, sv, vt = np.linalg.svd(m, full_matrices=False)
        rho, tail = len(sv), 0.0
        for j in range(len(sv) - 1, -1, -1):
            tail += sv[j] ** 2
            if math.sqrt(tail) < delta:
                rho = j
            else:
                break
        rho = max(1, min(rho, caps[k]))
        ranks[k] = rho
        sigma[k - 1, 0] = sv[0]
        for q in range(13):
            if 0 <= rho - 13 + q < len(sv):
                sigma[k - 1, 1 + q] = sv[rho - 13 + q]
        z[k] = vt[:rho].reshape(rho, n, -1)
        z[k - 1] = np.tensordot(z[k - 1], u[:, :rho] * sv[:rho], axes=(2, 0))
    z = [c * math.sqrt(n) for c in z]
    entry = np.ones((1, 1))
    for c, j in zip(z, _index(case, seed)):
        entry = entry @ c[:, j, :]
    return {"cores": [np.abs(c) for c in z], "ranks": np.array(ranks), "norm": nrm,
            "sigma": sigma, "entry": float(entry[0, 0])}


def exact(case, seed):
    kind, d, n = case["kind"], case["d"], case["n"]
    if kind == "round":
        return _exact_round(case, seed)
    if kind == "modesum":
        us, (a, b, c) = _gaussian_cores(d, n, case["r"], seed, 1), _stencil()
        out = []
        for k, u in enumerate(us):
            du = a * torch.roll(u, 1, dims=1) + b * u + c * torch.roll(u, -1, dims=1)
            if k == 0:
                out.append(torch.cat([du, u], dim=0))
            elif k == d - 1:
                out.append(torch.cat([u, du], dim=2))
            else:
                top = torch.cat([u, du], dim=2)
                out.append(torch.cat([top, torch.cat([torch.zeros_like(u), u], dim=2)], dim=0))
        return [t.permute(2, 1, 0) for t in out]
    if kind == "flux":
        out = []
        for u, (c, g, src) in zip(_density_cores(d, n, case["r"], seed, 1),
                                  _flux_coefficients(case, seed)):
            # -c u with the ghosts' wave speeds on the boundary values, central difference, source
            v = torch.cat([-g[0] * u[:, :1], -torch.from_numpy(c).cuda()[:, None] * u,
                           -g[1] * u[:, -1:]], dim=1)
            out.append((v[:, 2:] - v[:, :-2]) * (0.5 / DX_FLUX)
                       + torch.from_numpy(src).cuda()[:, None] * u)
        return [t.permute(2, 1, 0) for t in out]
    if kind == "dot":
        xs = _density_cores(d, n, case["rx"], seed, 1)
        ys = _density_cores(d, n, case["ry"], seed, 2)
        a = xs[0].new_ones(1, 1)
        for x, y in zip(xs, ys):
            b = torch.tensordot(a, x, dims=([0], [2]))       # (ry0, rx1, n)
            a = torch.tensordot(b, y, dims=([0, 2], [2, 1])) / n
        return float(a)
    if kind == "marginal":
        xs = [c.cpu().numpy() for c in _density_cores(d, n, case["r"], seed, 1)]
        w = 2.0 / n
        v = np.ones(1)
        for c in reversed(xs[1:]):
            v = v @ (w * c.sum(axis=1))
        return np.cumsum(w * np.tensordot(v, xs[0], axes=(0, 0))[:, 0])
    return None
