"""The workloads whose speed this repository looks after, each as a user's program runs it.

A case is a dict of plain values.  ``kind`` says which entry point it goes through:

* ``solve``  - one fused iSVD, ``Solver.solve`` on a matrix that is resident on the device;
* ``batch``  - several requests of different shapes in one ``solve_batch``;
* ``stages`` - the drivers' sequence: sketcher, orthogonalizer, integrator and former objects,
  with the collection of bases materialized between them;
* ``sketch`` - the sketching stage alone.

``listed()`` are the workloads by name, ``draw(rng)`` gives others of the same ranges.

The bases of a sketch come from Gram matrices, whose condition is the square of the decay of the
singular values over the kept directions, so the spectra here fall by a factor of 2.5 to 50 over
them: then every output is determined by the input to many more digits than the comparison of two
versions needs.  The Wen-Yin integrator is left out for the same reason: its step sizes amplify a
change in the last bit of its input to 1e-8 or more of its result.
"""
import ctypes
import math

import torch

import mcnla_amd as mc
from mcnla_amd import _lib

_PRECISION = {"f64": mc.PREC_F64, "bf16": mc.PREC_MIXED_BF16, "bf16x3": mc.PREC_MIXED_BF16X3,
              "f16": mc.PREC_MIXED_F16, "f16x2": mc.PREC_MIXED_F16X2,
              "f16x3": mc.PREC_MIXED_F16X3}
_FORMER = {"svd": mc.SvdFormer, "gramian": mc.RowBlockGramianFormer}
_SOLVE = {"kind": "solve", "dtype": "f64", "order": "col", "precision": "f64", "former": "svd"}


def listed():
    def case(name, **kw):
        return dict(_SOLVE, name=name, **kw)
    return [
        # the smallest configured problem: latency and launches count
        case("solve 2000x1000 f64", m=2000, n=1000, k=10, p=10, N=4, spectrum="slow"),
        # a request of ordinary size of the serving stream, in the serving precision
        case("request 6311x1703 bf16", m=6311, n=1703, k=27, p=10, N=20, spectrum="geometric",
             rho=0.95, dtype="f32", precision="bf16"),
        # an ordinary FP64 problem of odd sizes through the row-block classes: A row-major,
        # Gramian former
        case("solve 12347x1999 f64 row", m=12347, n=1999, k=21, p=10, N=17, spectrum="geometric",
             rho=0.93, order="row", former="gramian"),
        # a batch of serving requests on one stream
        {"name": "batch of 12 bf16", "kind": "batch", "count": 12, "dtype": "f32",
         "precision": "bf16"},
        # the largest serving shape in the two-product FP16 mode
        case("request 50000x5000 f16x2", m=50000, n=5000, k=50, p=10, N=32, spectrum="geometric",
             rho=0.95, dtype="f32", precision="f16x2"),
        # the headline problem, mixed precision
        case("solve 100000x10000 bf16", m=100000, n=10000, k=20, p=12, N=64, spectrum="decay",
             dtype="f32", precision="bf16"),
        # the headline problem, plain FP64
        case("solve 100000x10000 f64", m=100000, n=10000, k=20, p=12, N=64, spectrum="decay"),
        # the tall problem: few columns, many sketches, row-major FP32 A
        case("solve 500000x2000 f64 row", m=500000, n=2000, k=50, p=14, N=128, spectrum="stack",
             rho=0.96, dtype="f32", order="row", former="gramian"),
        # the drivers' stage sequence with their default sketch count and oversampling
        case("stages 20000x4000 f64", m=20000, n=4000, k=20, p=12, N=16, spectrum="decay")
        | {"kind": "stages"},
        # the sketching stage alone: the largest share of an FP64 solve, odd sizes
        case("sketch 30011x2503 f64", m=30011, n=2503, k=23, p=12, N=24, spectrum="decay")
        | {"kind": "sketch"},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))
    what = rng.choice(["solve", "solve", "solve", "solve", "request", "request", "batch", "stages",
                       "sketch", "tall"])
    if what == "batch":
        return {"kind": "batch", "count": rng.randint(2, 12), "dtype": "f32",
                "precision": rng.choice(["bf16", "bf16", "f16", "f64"]),
                "first": rng.randint(0, 10000)}
    c = dict(_SOLVE, spectrum="geometric", order=rng.choice(["col", "row"]),
             former=rng.choice(["svd", "gramian"]))
    last = rng.uniform(0.05, 0.4)  # the last kept singular value over the first
    if what == "tall":  # few columns and many sketches
        c.update(m=log_int(50000, 400000), n=log_int(500, 1500), k=rng.randint(10, 50),
                 p=rng.randint(10, 14), N=rng.randint(32, 96), spectrum="stack",
                 dtype=rng.choice(["f32", "f64"]))
        return c | {"rho": round(last ** (1 / (c["k"] + c["p"])), 4)}
    if what == "request":
        m = log_int(1000, 50000)
        c.update(m=m, n=min(m, log_int(500, 5000)), k=rng.randint(5, 50), p=10,
                 N=rng.randint(8, 32), dtype="f32", order="col", former="svd",
                 precision=rng.choice(["bf16", "bf16", "f16", "f16x2", "bf16x3", "f16x3"]))
        return c | {"rho": round(last ** (1 / (c["k"] + c["p"])), 4)}
    m = log_int(1000, 60000)
    c.update(m=m, n=min(m, log_int(500, 8000)), k=rng.randint(5, 40), p=rng.randint(8, 14),
             N=rng.randint(4, 40), dtype=rng.choice(["f64", "f64", "f32"]))
    if c["k"] <= 24 and rng.random() < 0.6:
        c["spectrum"] = "decay"
    else:
        c["rho"] = round(last ** (1 / (c["k"] + c["p"])), 4)
    if what != "solve":
        c["kind"] = what
    return c


# --------------------------------------------------------------------------------------------
# Inputs

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _sigma(case, device="cuda"):
    i = torch.arange(case["n"], dtype=torch.float64, device=device)
    if case["spectrum"] == "slow":
        return 0.95 ** i + 1e-6
    return case["rho"] ** i


def _cosines(n, gen):
    """An orthogonal n x n matrix: the cosine basis with its rows and columns' signs drawn."""
    i = torch.arange(n, dtype=torch.float64, device="cuda")
    q = torch.cos(math.pi / (2 * n) * (2 * i + 1)[:, None] * i[None, :]) * math.sqrt(2.0 / n)
    q[:, 0] *= math.sqrt(0.5)
    sign = torch.randint(0, 2, (2, n), device="cuda", generator=gen).double() * 2 - 1
    return sign[0][:, None] * q * sign[1][None, :]


def _matrix(case, seed):
    """A as a torch tensor of its logical shape, in the storage order of the case."""
    m, n = case["m"], case["n"]
    gen = _generator(seed)
    dtype = torch.float64 if case["dtype"] == "f64" else torch.float32

    def normal(*shape):
        return torch.randn(*shape, dtype=torch.float64, device="cuda", generator=gen)
    if case["spectrum"] == "decay":
        # 50 singular values 0.9^i over a noise floor of norm 1e-3
        u, v = normal(m, 50) / math.sqrt(m), normal(n, 50) / math.sqrt(n)
        u *= 0.9 ** torch.arange(50, dtype=torch.float64, device="cuda")
        noise = 1e-3 / (math.sqrt(m) + math.sqrt(n))
        if case["order"] == "col":
            a = torch.randn(n, m, dtype=dtype, device="cuda", generator=gen).mul_(noise)
            return a.addmm_(v.to(dtype), u.t().contiguous().to(dtype)).t()
        a = torch.randn(m, n, dtype=dtype, device="cuda", generator=gen).mul_(noise)
        return a.addmm_(u.to(dtype), v.t().contiguous().to(dtype))
    s = _sigma(case)
    if case["spectrum"] == "stack":
        # row blocks that are sign-flipped copies of one dense square block with these values
        block = ((_cosines(n, gen) * s) @ _cosines(n, gen).t().contiguous()).to(dtype)
        count = -(-m // n)
        sign = torch.randint(0, 2, (count, n), device="cuda", generator=gen).to(dtype) * 2 - 1
        a = (sign[:, :, None] * block[None]).reshape(count * n, n)[:m].contiguous()
    else:
        # (I - 2uu') [diag(s); 0] (I - 2vv') with random unit vectors
        u, v = normal(m), normal(n)
        u /= u.norm()
        v /= v.norm()
        a = torch.outer(u, 4 * torch.dot(u[:n], s * v) * v - 2 * u[:n] * s)
        a[:n] -= torch.outer(2 * s * v, v)
        a[:n].diagonal().add_(s)
        a = a.to(dtype)
    return a if case["order"] == "row" else a.t().contiguous().t()


def _view(a, order):
    """The framework's view of a device matrix that torch owns."""
    import numpy as np
    dtype = np.float64 if a.dtype == torch.float64 else np.float32
    return mc.DeviceArray.view(a.data_ptr(), a.shape, dtype, "F" if order == "col" else "C")


def _parameters(case):
    p = mc.Parameters().setSize(case["m"], case["n"]).setRank(case["k"])
    p.setOverRank(case["p"]).setNumSketch(case["N"]).sync()
    return p


def _omega_mode(case):
    return mc.OMEGA_PHILOX_F16 if case["precision"] == "f16x2" else mc.OMEGA_PHILOX


def _solver_state(case, seed):
    a = _matrix(case, seed)
    solver = mc.Solver(_parameters(case), former=_FORMER[case["former"]],
                       precision=_PRECISION[case["precision"]], seed=seed % 100003,
                       omega_mode=_omega_mode(case))
    return {"case": case, "a": a, "A": _view(a, case["order"]), "solver": solver}


def _requests(case, seed):
    """The serving stream's requests as solve cases, with one decay over the kept directions."""
    first = case.get("first", 0)
    out = []
    for r in mc.workloads.serving_stream(case["count"], seed=3 + first):
        out.append(dict(_SOLVE, m=r["m"], n=r["n"], k=r["k"], p=r["p"], N=r["N"],
                        spectrum="geometric", rho=0.1 ** (1 / (r["k"] + r["p"])),
                        dtype=case["dtype"], precision=case["precision"]))
    return [(c, seed + 7919 * i) for i, c in enumerate(out)]


def prepare(case, seed):
    if case["kind"] == "batch":
        return {"members": [_solver_state(c, s) for c, s in _requests(case, seed)]}
    if case["kind"] == "solve":
        return _solver_state(case, seed)
    P, prec = _parameters(case), _PRECISION[case["precision"]]
    a = _matrix(case, seed)
    state = {"case": case, "a": a, "A": _view(a, case["order"])}
    q = torch.empty(case["m"], P.dimSketchTotal(), dtype=torch.float64, device="cuda")
    state.update(q=q, Q=_view(q, "row"))
    sketcher = (mc.RowBlockGaussianProjectionSketcher if case["order"] == "row" else
                mc.ColBlockGaussianProjectionSketcher)
    state["sketcher"] = sketcher(P, seed=seed % 100003, precision=prec,
                                 omega_mode=_omega_mode(case)).initialize()
    if case["kind"] == "stages":
        qbar = torch.empty(case["m"], P.dimSketch(), dtype=torch.float64, device="cuda")
        state.update(qbar=qbar, Qbar=_view(qbar, "row"))
        state["orthogonalizer"] = mc.RowBlockGramianOrthogonalizer(P, precision=prec).initialize()
        state["integrator"] = mc.RowBlockKolmogorovNagumoIntegrator(P, precision=prec).initialize()
        state["former"] = _FORMER[case["former"]](P, precision=prec).initialize()
    return state


# --------------------------------------------------------------------------------------------
# A pass

class _Result:
    """Device memory of a solver or stage, for torch to view; it lives as long as the view."""

    def __init__(self, owner, ptr, shape, strides):
        self.owner = owner
        self.__cuda_array_interface__ = {"data": (ptr.value, False), "shape": shape,
                                         "strides": tuple(8 * s for s in strides),
                                         "typestr": "<f8", "version": 2}

    @classmethod
    def tensor(cls, *args):
        return torch.as_tensor(cls(*args), device="cuda")


def _factors(case, owner, s, u, v):
    m, n, k = case["m"], case["n"], case["k"]
    return {"S": _Result.tensor(owner, s, (k,), (1,)),
            "U": _Result.tensor(owner, u, (m, k), (1, m) if case["former"] == "svd" else (k, 1)),
            "V": _Result.tensor(owner, v, (n, k), (k, 1))}


def _solved(state):
    case, solver = state["case"], state["solver"]
    s, u, v, q = (ctypes.c_void_p() for _ in range(4))
    _lib.check(_lib.lib().mcnla_solver_results(solver._h, *(ctypes.byref(x) for x in (s, u, v, q))))
    out = _factors(case, solver, s, u, v)
    out["Qbar"] = _Result.tensor(solver, q, (case["m"], case["k"] + case["p"]), (case["k"] + case["p"], 1))
    out["iterations"] = solver.iteration()
    return out


def run(state):
    if "members" in state:
        members = state["members"]
        mc.solve_batch([x["solver"] for x in members], [x["A"] for x in members])
        return [_solved(x) for x in members]
    if "solver" in state:
        state["solver"].solve(state["A"])
        return _solved(state)
    state["sketcher"](state["A"], state["Q"])
    if "former" not in state:
        return state["q"]
    state["orthogonalizer"](state["Q"])
    state["integrator"](state["Q"], state["Qbar"])
    state["former"](state["A"], state["Qbar"])
    s, u, v = (ctypes.c_void_p() for _ in range(3))
    _lib.check(_lib.lib().mcnla_former_results(state["former"]._handle(),
                                               *(ctypes.byref(x) for x in (s, u, v))))
    out = _factors(state["case"], state["former"], s, u, v)
    out.update(Q=state["q"], Qbar=state["qbar"], iterations=state["integrator"].iteration())
    return out


# --------------------------------------------------------------------------------------------
# What a pass cannot do without

def work(case):
    if case["kind"] == "batch":
        every = [work(c) for c, _ in _requests(case, 0)]
        return {key: sum(w[key] for w in every) for key in ("bytes", "flops")}
    m, n, k, N = (float(case[x]) for x in "mnkN")
    l = k + case["p"]
    nl = l * N
    size = 8.0 if case["dtype"] == "f64" else 4.0
    if case["kind"] == "sketch":
        return {"bytes": size * m * n + 8 * m * nl, "flops": 2 * m * n * nl}
    # through Y = A Omega and Y'Y, or through A'A, whichever is less
    flops = min(2 * m * n * nl + m * nl * nl + 2 * m * nl * l,
                m * n * n + 2 * n * n * nl + n * nl * nl + 2 * m * n * l)
    out = m * k + n * k + m * l + (m * nl if case["kind"] == "stages" else 0)
    return {"bytes": size * m * n + 8 * out, "flops": flops + 2 * m * n * l + 2 * m * l * k}


# --------------------------------------------------------------------------------------------
# The same in 64 bits

def _mul_high(a, b):
    """High 32 bits of the product of 32-bit values (int64 tensors) with a 32-bit constant."""
    lo, hi = a & 0xFFFF, a >> 16
    return (hi * b + ((lo * b) >> 16)) >> 16 & 0xFFFFFFFF


def _omega(case, seed):
    """The n x Nl projection: Philox4x32-10 pairs through Box-Muller."""
    n, nl = case["n"], (case["k"] + case["p"]) * case["N"]
    pair = torch.arange((n * nl + 1) // 2, dtype=torch.int64, device="cuda")
    x, y = pair & 0xFFFFFFFF, pair >> 32
    z, w = torch.zeros_like(x), torch.zeros_like(x)
    k0, k1 = seed % 100003, 0
    for _ in range(10):
        h0, l0 = _mul_high(x, 0xD2511F53), (x * 0xD2511F53) & 0xFFFFFFFF
        h1, l1 = _mul_high(z, 0xCD9E8D57), (z * 0xCD9E8D57) & 0xFFFFFFFF
        x, y, z, w = h1 ^ y ^ k0, l1, h0 ^ w ^ k1, l0
        k0, k1 = (k0 + 0x9E3779B9) & 0xFFFFFFFF, (k1 + 0xBB67AE85) & 0xFFFFFFFF
    bits = (1 << 53) - 1
    u1 = ((((x << 21) ^ (y >> 11)) & bits).double() + 1) * 2.0 ** -53
    u2 = (((z << 21) ^ (w >> 11)) & bits).double() * 2.0 ** -53
    r, t = torch.sqrt(-2 * torch.log(u1)), 2 * math.pi * u2
    out = torch.stack([r * torch.cos(t), r * torch.sin(t)], 1).reshape(-1)[:n * nl]
    if _omega_mode(case) == mc.OMEGA_PHILOX_F16:
        out = out.float().half().double()
    return out.reshape(n, nl)


def _kolmogorov_nagumo(B, N, l, tol=1e-4):
    """Coefficients of the average of the N bases whose Gram matrix is B, from the first one."""
    X = torch.zeros(B.shape[0], l, dtype=B.dtype)
    X[:l] = torch.eye(l, dtype=B.dtype)
    for _ in range(256):
        Bc = B @ X
        Bg = B @ Bc / N
        Dc = Bc.t() @ Bc / N
        Z = Bc.t() @ Bg / N - Dc @ Dc
        lam, W = torch.linalg.eigh((Z + Z.t()) / 2)
        s = torch.sqrt(0.5 + torch.sqrt(0.25 - lam))
        C, Ci = (W * s) @ W.t(), (W / s) @ W.t()
        X = X @ (C - Dc @ Ci) + Bc @ Ci / N
        if not float((s - 1).norm()) >= tol:
            break
    return X


def _singular_values(case, seed):
    """S of one Kolmogorov-Nagumo solve, in 64 bits."""
    l, N = case["k"] + case["p"], case["N"]
    a = _matrix(case, seed)
    om = _omega(case, seed)
    step = max(1, (1 << 28) // case["n"])
    rows = range(0, case["m"], step)
    Y = torch.cat([a[i:i + step].double() @ om for i in rows])
    G = (Y.t() @ Y).cpu()
    T = torch.zeros_like(G)
    for i in range(N):
        b = slice(i * l, (i + 1) * l)
        L = torch.linalg.cholesky(G[b, b])
        T[b, b] = torch.linalg.inv(L).t()
    X = T @ _kolmogorov_nagumo(T.t() @ G @ T, N, l)
    Q, _ = torch.linalg.qr((Y @ X.cuda()).cpu())
    Q = Q.cuda()
    W = sum(Q[i:i + step].t() @ a[i:i + step].double() for i in rows)
    lam = torch.linalg.eigvalsh((W @ W.t()).cpu())
    return lam.flip(0)[:case["k"]].clamp(min=0).sqrt()


def exact(case, seed):
    if case["kind"] == "sketch":
        return _matrix(case, seed).double() @ _omega(case, seed)
    if case["kind"] == "batch":
        work_of = [(c, s) for c, s in _requests(case, seed)]
        return [dict.fromkeys(("S", "U", "V", "Qbar", "iterations")) |
                {"S": _singular_values(c, s)} for c, s in work_of]
    if case["N"] * (case["k"] + case["p"]) > 4096:
        return None  # the Gram matrix's iterations on the host would take too long
    # the singular vectors' signs and the bases' rotations are the implementation's own choice
    return {"S": _singular_values(case, seed)}
