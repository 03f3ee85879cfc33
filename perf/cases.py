"""What this package is used for, as single passes through its public entry points.

``listed()`` gives the fixed cases, ``draw(rng)`` one more of the same ranges.
``prepare`` makes the inputs a program holds before the call, ``run`` is the
call, ``work`` the bytes and operations no implementation can do without and
``exact`` the same outputs in 64 bits from plain torch.
"""

import math

import numpy as np
import torch

import gstools_amd as gsx
from gstools_amd import autograd as gsx_autograd
from gstools_amd import krige as gsx_krige
from gstools_amd import variogram as gsx_variogram
from gstools_amd.summate import summate_fourier_tensor_device, summate_incompr_grid_device

TWO_PI = 2.0 * math.pi


def listed():
    return [
        # the default call: a 100 x 100 map of a 2D Gaussian field, 1000 modes, FP64
        {"name": "sum-fp64-2d-1e4", "kind": "sum", "precision": "fp64", "dim": 2, "modes": 1000, "points": 10_000,
         "model": "gaussian", "len_scale": 10.0, "extent": 100.0},
        # FP64 values of a heavy-tailed 3D field at the nodes of an unstructured mesh
        {"name": "sum-fp64-3d-1e6", "kind": "sum", "precision": "fp64", "dim": 3, "modes": 1024, "points": 1_000_003,
         "model": "exponential", "len_scale": 20.0, "extent": 1000.0},
        # the same in FP32 at the largest mesh
        {"name": "sum-fp32-3d-4e6", "kind": "sum", "precision": "fp32", "dim": 3, "modes": 1024, "points": 4_000_000,
         "model": "exponential", "len_scale": 20.0, "extent": 1000.0},
        # calibration: misfit at a set of observation points and its gradients
        {"name": "grad-fp32-2d-2e3", "kind": "grad", "precision": "fp32", "dim": 2, "modes": 2048, "points": 2000,
         "len_scale": 15.0, "extent": 500.0},
        # calibration against a dense map
        {"name": "grad-fp32-2d-1e6", "kind": "grad", "precision": "fp32", "dim": 2, "modes": 2048,
         "points": 1_000_000, "len_scale": 15.0, "extent": 500.0},
        # one realization of a map on the matrix cores, as drawn many times in a Monte Carlo study
        {"name": "grid-bf16x3-2d-small", "kind": "grid", "precision": "bf16x3", "shape": "333x500", "modes": 1000,
         "model": "gaussian", "len_scale": 10.0, "spacing": 1.0},
        # the largest volume
        {"name": "grid-bf16x3-3d-512", "kind": "grid", "precision": "bf16x3", "shape": "512x512x512", "modes": 4096,
         "model": "matern15", "len_scale": 8.0, "spacing": 0.5},
        # an incompressible velocity field for transport
        {"name": "incompr-bf16x3-3d-128", "kind": "incompr", "precision": "bf16x3", "shape": "128x128x128",
         "modes": 4096, "model": "gaussian", "len_scale": 10.0, "spacing": 1.0},
        # a large periodic map by the Fourier method
        {"name": "fourier-2d-4096", "kind": "fourier", "shape": "4096x4096", "axis_modes": 256, "period": 4096.0,
         "len_scale": 200.0},
        # kriging of a few hundred measurements onto a map, estimate and variance
        {"name": "krige-300-4e4", "kind": "krige", "dim": 2, "cond": 300, "points": 40_000, "len_scale": 30.0,
         "extent": 200.0, "variance": True},
        # the variogram of a measurement campaign
        {"name": "vario-2d-5e3", "kind": "vario", "dim": 2, "points": 5000, "bins": 26, "estimator": "m",
         "directions": 0, "extent": 1000.0},
        # the variogram of a dense 3D data set
        {"name": "vario-3d-1e5", "kind": "vario", "dim": 3, "points": 100_000, "bins": 20, "estimator": "m",
         "directions": 0, "extent": 1000.0},
    ]


# ---------------------------------------------------------------- drawing ---
def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _spread(rng, count, total):
    """``count`` axis lengths whose product is about ``total``, uneven."""
    weights = [rng.uniform(0.6, 1.4) for _ in range(count)]
    mean = sum(weights) / count
    base = total ** (1.0 / count)
    return [max(2, int(round(base ** (w / mean)))) for w in weights]


def draw(rng):
    kind = rng.choice(["sum", "sum", "grad", "grid", "incompr", "fourier", "krige", "vario"])
    if kind == "sum":
        dim = rng.choice([1, 2, 3, 3])
        modes = _log_int(rng, 100, 8192)
        cap = 4.1e9 if rng.random() < 0.5 else 1.0e9
        return {"kind": kind, "precision": rng.choice(["fp64", "fp32"]), "dim": dim, "modes": modes,
                "points": _log_int(rng, 100, min(4.0e6, cap / modes)),
                "model": rng.choice(["gaussian", "exponential", "matern15"]), "len_scale": rng.uniform(5.0, 50.0),
                "extent": rng.uniform(50.0, 1000.0)}
    if kind == "grad":
        modes = _log_int(rng, 100, 4096)
        return {"kind": kind, "precision": rng.choice(["fp64", "fp32", "fp32"]), "dim": rng.choice([2, 3]),
                "modes": modes, "points": _log_int(rng, 200, min(1.0e6, 1.0e9 / modes)),
                "len_scale": rng.uniform(5.0, 30.0), "extent": rng.uniform(100.0, 500.0)}
    if kind == "grid":
        dim = rng.choice([2, 3])
        modes = _log_int(rng, 500, 8192)
        precision = rng.choice(["bf16x3", "bf16x3", "fp16x3", "fp64gemm"])
        shape = _spread(rng, dim, _log_int(rng, 4096, 16.0e6 if precision != "fp64gemm" else 2.0e10 / modes))
        return {"kind": kind, "precision": precision, "shape": "x".join(str(n) for n in shape), "modes": modes,
                "model": rng.choice(["gaussian", "matern15"]), "len_scale": rng.uniform(5.0, 30.0),
                "spacing": rng.choice([0.5, 1.0, 2.0])}
    if kind == "incompr":
        dim = rng.choice([2, 3])
        shape = _spread(rng, dim, _log_int(rng, 4096, 4_000_000))
        return {"kind": kind, "precision": rng.choice(["bf16x3", "fp16x3"]), "shape": "x".join(str(n) for n in shape),
                "modes": _log_int(rng, 500, 8192), "model": "gaussian", "len_scale": rng.uniform(5.0, 30.0),
                "spacing": 1.0}
    if kind == "fourier":
        dim = rng.choice([2, 2, 3])
        shape = _spread(rng, dim, _log_int(rng, 10_000, 16_000_000))
        return {"kind": kind, "shape": "x".join(str(n) for n in shape),
                "axis_modes": 2 * rng.randint(8, 128 if dim == 2 else 32), "period": float(max(shape)),
                "len_scale": rng.uniform(0.02, 0.2) * max(shape)}
    if kind == "krige":
        cond = _log_int(rng, 20, 1001)
        return {"kind": kind, "dim": rng.choice([2, 3]), "cond": cond,
                "points": _log_int(rng, 1000, min(1.0e6, 1.0e11 / cond ** 2)), "len_scale": rng.uniform(20.0, 80.0),
                "extent": rng.uniform(100.0, 1000.0), "variance": rng.random() < 0.75}
    points = _log_int(rng, 500, 100_000)
    dim = rng.choice([1, 2, 3])
    directions = rng.choice([0, 0, 0, 2]) if dim > 1 and points < 20_000 else 0
    return {"kind": "vario", "dim": dim, "points": points, "bins": rng.randint(10, 40),
            "estimator": rng.choice(["m", "m", "c"]), "directions": directions, "extent": 1000.0}


# ----------------------------------------------------------------- inputs ---
def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _normal(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float64)


def _uniform(g, *shape):
    return torch.rand(*shape, generator=g, device="cuda", dtype=torch.float64)


def _wavenumbers(g, model, dim, modes, len_scale):
    """Wave vectors of the models' spectral densities: normal for the Gaussian, multivariate
    t with 1 and 3 degrees of freedom for the Exponential and the Matern (nu 1.5)."""
    k = _normal(g, dim, modes)
    if model == "gaussian":
        return k * (math.sqrt(math.pi / 2.0) / len_scale)
    dof = 1 if model == "exponential" else 3
    chi = torch.sqrt((_normal(g, dof, modes) ** 2).mean(dim=0))
    return k / chi / len_scale


def _shape(case):
    return [int(n) for n in case["shape"].split("x")]


def prepare(case, seed):
    g = _generator(seed)
    kind = case["kind"]
    s = {"case": dict(case)}
    if kind in ("sum", "grad"):
        dim, modes, points = case["dim"], case["modes"], case["points"]
        s["z1"], s["z2"] = _normal(g, modes), _normal(g, modes)
        s["pos"] = _uniform(g, dim, points) * case["extent"]
        if kind == "sum":
            s["cov"] = _wavenumbers(g, case["model"], dim, modes, case["len_scale"])
        else:
            s["k"] = _wavenumbers(g, "matern15", dim, modes, 1.0).requires_grad_()
            s["len"] = torch.tensor(case["len_scale"], dtype=torch.float64, device="cuda", requires_grad=True)
            s["target"] = _normal(g, points)
            s["z1"].requires_grad_()
            s["z2"].requires_grad_()
    elif kind in ("grid", "incompr"):
        shape, modes = _shape(case), case["modes"]
        s["axes"] = [case["spacing"] * np.arange(n, dtype=np.float64) for n in shape]
        s["z1"], s["z2"] = _normal(g, modes), _normal(g, modes)
        s["cov"] = _wavenumbers(g, case["model"], len(shape), modes, case["len_scale"])
        s["alpha"] = math.sqrt(1.0 / modes)
    elif kind == "fourier":
        shape, m = _shape(case), case["axis_modes"]
        dk = TWO_PI / case["period"]
        ax = (torch.arange(m, dtype=torch.float64, device="cuda") - m // 2) * dk
        s["kaxes"] = [ax.clone() for _ in shape]
        s["axes"] = [np.arange(n, dtype=np.float64) for n in shape]
        k2 = sum(t ** 2 for t in torch.meshgrid(*s["kaxes"], indexing="ij")).reshape(-1)
        s["factor"] = torch.exp(-k2 * case["len_scale"] ** 2 / (2.0 * math.pi)) + 1.0e-9
        s["z1"], s["z2"] = _normal(g, k2.numel()), _normal(g, k2.numel())
    elif kind == "krige":
        dim, cond = case["dim"], case["cond"]
        s["model"] = gsx.Exponential(dim=dim, var=2.0, len_scale=case["len_scale"], nugget=0.1)
        s["cond_pos"] = _uniform(g, dim, cond) * case["extent"]
        s["pos"] = _uniform(g, dim, case["points"]) * case["extent"]
        s["cond"] = torch.cat([_normal(g, cond), torch.zeros(1, dtype=torch.float64, device="cuda")])
        x = s["cond_pos"].cpu().numpy()
        r = np.sqrt(((x[:, :, None] - x[:, None, :]) ** 2).sum(axis=0))
        a = np.zeros((cond + 1, cond + 1))
        a[:cond, :cond] = 2.0 * np.exp(-r / case["len_scale"]) + 0.1 * np.eye(cond)
        a[:cond, cond] = a[cond, :cond] = 1.0
        s["mat"] = torch.from_numpy(np.linalg.inv(a)).cuda()
    else:
        dim, points = case["dim"], case["points"]
        s["pos"] = _uniform(g, dim, points) * case["extent"]
        # a smooth field plus noise
        k = _normal(g, 32, dim) * (8.0 / case["extent"])
        phase = _uniform(g, 32, 1) * TWO_PI
        s["field"] = torch.cos(k @ s["pos"] + phase).sum(dim=0) / 4.0 + 0.3 * _normal(g, points)
        reach = case["extent"] * math.sqrt(dim) / 3.0
        s["edges"] = np.linspace(0.0, reach, case["bins"] + 1)
        if case["directions"]:
            s["dirs"] = np.eye(dim)[: case["directions"]]
    return s


# -------------------------------------------------------------------- run ---
def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "sum":
        return gsx.summate_device(s["cov"], s["z1"], s["z2"], s["pos"], case["precision"])
    if kind == "grad":
        u = gsx_autograd.randmeth_field(s["z1"], s["z2"], s["k"], s["pos"], len_scale=s["len"],
                                        precision=case["precision"])
        loss = torch.mean((u - s["target"]) ** 2)
        grads = torch.autograd.grad(loss, [s["z1"], s["z2"], s["k"], s["len"]])
        return (u.detach(),) + tuple(grads)
    if kind == "grid":
        alpha = 1.0 if case["precision"] == "fp64gemm" else s["alpha"]
        return gsx.summate_grid_device(s["cov"], s["z1"], s["z2"], s["axes"], case["precision"], alpha=alpha)
    if kind == "incompr":
        return summate_incompr_grid_device(s["cov"], s["z1"], s["z2"], s["axes"], case["precision"],
                                           alpha=s["alpha"])
    if kind == "fourier":
        return summate_fourier_tensor_device(s["factor"], s["kaxes"], s["z1"], s["z2"], s["axes"])
    if kind == "krige":
        cond = case["cond"]
        rhs = torch.empty((cond + 1, case["points"]), dtype=torch.float64, device="cuda")
        gsx_krige.krige_cov_device(s["model"], s["cond_pos"], s["pos"], out=rhs, row0=0)
        rhs[cond] = 1.0
        return gsx_krige.krige_sum_device(s["mat"], rhs, s["cond"], variance=case["variance"])
    if case["directions"]:
        return gsx_variogram.directional(s["field"], s["edges"], s["pos"], s["dirs"], estimator_type=case["estimator"],
                                         separate_dirs=True)
    return gsx_variogram.unstructured(s["field"], s["edges"], s["pos"], case["estimator"])


# ------------------------------------------------------------------- work ---
def work(case):
    kind = case["kind"]
    if kind in ("sum", "grad"):
        d, n, p = case["dim"], case["modes"], case["points"]
        word = 8 if case["precision"] == "fp64" else 4
        if kind == "sum":
            return {"bytes": 8 * (d + 2) * n + 8 * d * p + word * p, "flops": (2 * d + 6) * n * p}
        return {"bytes": 2 * 8 * (d + 2) * n + 8 * d * p + 16 * p, "flops": (6 * d + 16) * n * p}
    if kind in ("grid", "incompr"):
        shape = _shape(case)
        p, n, d = math.prod(shape), case["modes"], len(shape)
        comps = d if kind == "incompr" else 1
        word, per = (8, 4) if case["precision"] == "fp64gemm" else (4, 12)
        return {"bytes": 8 * (d + 2) * n + 8 * sum(shape) + word * comps * p, "flops": per * comps * n * p}
    if kind == "fourier":
        shape, m = _shape(case), case["axis_modes"]
        d = len(shape)
        # one complex contraction per axis, the last one for the real part only
        flops, lead = 0, 1
        for i in range(d):
            lead *= shape[i]
            flops += (4 if i == d - 1 else 8) * lead * m ** (d - i)
        return {"bytes": 3 * 8 * m ** d + 8 * math.prod(shape), "flops": flops}
    if kind == "krige":
        k, p = case["cond"] + 1, case["points"]
        flops = 2 * k * p + (k * k * p if case["variance"] else 0)
        return {"bytes": 8 * (k * k + k + (case["dim"] + (2 if case["variance"] else 1)) * p), "flops": flops}
    p, d = case["points"], case["dim"]
    return {"bytes": 8 * (d + 1) * p, "flops": (3 * d + 4) * p * (p - 1) // 2}


# ------------------------------------------------------------------ exact ---
def _chunk(columns):
    return max(1, int(2 ** 26 // max(columns, 1)))


def _phases(cov, pos):
    t = cov[0][None, :] * pos[0][:, None]
    for i in range(1, cov.shape[0]):
        t = t + cov[i][None, :] * pos[i][:, None]
    return t  # (points, modes)


def _exact_sum(cov, z1, z2, pos):
    out = torch.empty(pos.shape[1], dtype=torch.float64, device=pos.device)
    step = _chunk(cov.shape[1])
    for lo in range(0, pos.shape[1], step):
        t = _phases(cov, pos[:, lo:lo + step])
        out[lo:lo + step] = torch.cos(t) @ z1 + torch.sin(t) @ z2
    return out


def _exact_grad(s, case):
    z1, z2, kk, ln = (s[n].detach() for n in ("z1", "z2", "k", "len"))
    pos, n = s["pos"], case["modes"]
    cov = kk / ln
    scale = math.sqrt(1.0 / n)
    u = scale * _exact_sum(cov, z1, z2, pos)
    g = 2.0 * (u - s["target"]) / u.numel() * scale
    g1, g2, gk = torch.zeros_like(z1), torch.zeros_like(z2), torch.zeros_like(cov)
    step = _chunk(n)
    for lo in range(0, u.numel(), step):
        t = _phases(cov, pos[:, lo:lo + step])
        c, sn, gg = torch.cos(t), torch.sin(t), g[lo:lo + step]
        g1 += gg @ c
        g2 += gg @ sn
        for d in range(cov.shape[0]):
            gx = gg * pos[d, lo:lo + step]
            gk[d] += z2 * (gx @ c) - z1 * (gx @ sn)
    return u, g1, g2, gk / ln, -(gk * cov).sum() / ln


def _exact_grid(cov, z1, z2, axes, weight):
    """sum_j weight_j Re(c_j e^{i k_j x}) as one real product per first-axis slab."""
    axes = [torch.from_numpy(a).to(cov.device) for a in axes]
    ph = [k[:, None] * a[None, :] for k, a in zip(cov, axes)]
    b_re, b_im = (weight * z1)[:, None], -(weight * z2)[:, None]
    rest = [(torch.cos(t), torch.sin(t)) for t in ph[1:]]
    a_re, a_im = torch.cos(ph[0]).T.contiguous(), torch.sin(ph[0]).T.contiguous()
    c, sn = rest[0]
    e_re, e_im = b_re * c - b_im * sn, b_re * sn + b_im * c
    if len(rest) == 1:
        return (a_re @ e_re - a_im @ e_im).reshape(-1)
    c2, s2 = rest[1]
    n0, n1, n2 = (a.numel() for a in axes)
    out = torch.empty((n0, n1, n2), dtype=torch.float64, device=cov.device)
    for i in range(n1):
        re, im = e_re[:, i:i + 1], e_im[:, i:i + 1]
        out[:, i] = a_re @ (re * c2 - im * s2) - a_im @ (re * s2 + im * c2)
    return out.reshape(-1)


def _exact_fourier(s, case):
    shape, m = _shape(case), case["axis_modes"]
    e = [torch.exp(1j * k[:, None] * torch.from_numpy(a).to(k.device)[None, :]) for k, a in zip(s["kaxes"], s["axes"])]
    t = (s["factor"] * torch.complex(s["z1"], -s["z2"])).reshape([m] * len(shape))
    for i in range(len(shape) - 1):
        # contract the leading mode axis; the grid axis goes last
        t = torch.tensordot(t, e[i], dims=([0], [0]))
    # now (m_last, n_0, n_1, ...)
    lead = math.prod(shape[:-1])
    t = t.reshape(m, lead)
    out = t.real.T.contiguous() @ e[-1].real.contiguous() - t.imag.T.contiguous() @ e[-1].imag.contiguous()
    return out.reshape(-1)


def _exact_krige(s, case):
    cond, p = case["cond"], case["points"]
    field = torch.empty(p, dtype=torch.float64, device="cuda")
    error = torch.empty_like(field)
    step = 65536
    for lo in range(0, p, step):
        x = s["pos"][:, lo:lo + step]
        d2 = 0.0
        for a, b in zip(s["cond_pos"], x):
            d2 = d2 + (a[:, None] - b[None, :]) ** 2
        v = torch.ones((cond + 1, x.shape[1]), dtype=torch.float64, device="cuda")
        v[:cond] = 2.0 * torch.exp(-torch.sqrt(d2) / case["len_scale"])
        w = s["mat"] @ v
        field[lo:lo + step] = s["cond"] @ w
        error[lo:lo + step] = (v * w).sum(dim=0)
    return (field, error) if case["variance"] else field


def _exact_vario(s, case):
    pos, f = s["pos"], s["field"]
    p, nb = case["points"], case["bins"]
    edges = s["edges"].tolist()
    dirs = [None] if not case["directions"] else [int(np.argmax(v)) for v in s["dirs"]]
    below = torch.zeros((len(dirs), nb + 1), dtype=torch.float64, device="cuda")  # pairs nearer than each edge
    value = torch.zeros_like(below)
    step = max(1, 2 ** 25 // p)
    for lo in range(0, p, step):
        hi = min(p, lo + step)
        d2, diffs = 0.0, []
        for x in pos:
            diff = x[None, lo:] - x[lo:hi, None]
            diffs.append(diff)
            d2 = d2 + diff * diff
        dist = torch.sqrt(d2)
        later = torch.arange(lo, p, device="cuda")[None, :] > torch.arange(lo, hi, device="cuda")[:, None]
        x = f[None, lo:] - f[lo:hi, None]
        v = x * x if case["estimator"] == "m" else torch.sqrt(torch.abs(x))
        taken = torch.zeros_like(later)
        for n, axis in enumerate(dirs):
            ok = later
            if axis is not None:
                q = torch.abs(diffs[axis]) / dist
                near = (torch.arccos(torch.clamp(q, max=1.0)) < math.pi / 8) | ~(q < 1.0)
                ok = later & near & ~taken
                taken = taken | ok
            for i, e in enumerate(edges):
                hit = ok & (dist < e)
                below[n, i] += hit.sum()
                value[n, i] += torch.where(hit, v, 0.0).sum()
    cnt = below[:, 1:] - below[:, :-1]
    tot = value[:, 1:] - value[:, :-1]
    one = torch.clamp(cnt, min=1.0)
    if case["estimator"] == "m":
        gamma = tot / (2.0 * one)
    else:
        gamma = 0.5 * (tot / one) ** 4 / (0.457 + 0.494 / one + 0.045 / one ** 2)
    if not case["directions"]:
        gamma, cnt = gamma[0], cnt[0]
    return gamma.cpu().numpy(), cnt.to(torch.int64).cpu().numpy()


def exact(case, seed):
    s = prepare(case, seed)
    kind = case["kind"]
    if kind == "sum":
        return _exact_sum(s["cov"], s["z1"], s["z2"], s["pos"])
    if kind == "grad":
        return _exact_grad(s, case)
    if kind == "grid":
        out = _exact_grid(s["cov"], s["z1"], s["z2"], s["axes"], torch.ones_like(s["z1"]))
        return out if case["precision"] == "fp64gemm" else out * s["alpha"]
    if kind == "incompr":
        cov = s["cov"]
        k2 = (cov ** 2).sum(dim=0)
        rows = []
        for c in range(cov.shape[0]):
            w = (1.0 if c == 0 else 0.0) - cov[c] * cov[0] / k2
            rows.append(s["alpha"] * _exact_grid(cov, s["z1"], s["z2"], s["axes"], w))
        return torch.stack(rows)
    if kind == "fourier":
        return _exact_fourier(s, case)
    if kind == "krige":
        return _exact_krige(s, case)
    return _exact_vario(s, case)
