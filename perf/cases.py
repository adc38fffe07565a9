"""The work whose speed counts: calls of the public entry points on the problem
family of the benchmark workloads and the tests, trilinear Q1 pencils (K, M) of
E^3 meshes with lognormal element coefficients, n = (E - 1)^3 rows.

kind "product"  Y = A X over a column block (GCGE_HIP_SpMM), by far the most
                frequent call of a solve.  numbering "grid": lexicographic, so
                the matrix has diagonal storage; "local": nodes shuffled within
                runs of 64, as an unstructured mesh numbered for locality has
                them (sliced ELLPACK, element gathers); "scattered": a random
                symmetric permutation (whole-row gathers).
kind "gram"     G = V^T W to the host (GCGE_HIP_Gram): projection and
                orthonormalisation blocks.
kind "combine"  Y = beta Y + V C (GCGE_HIP_LinearComb): Ritz vectors, the new P,
                and the projection W - V d.
kind "inner"    the right-hand sides M X and the block CG on K of a GCG
                iteration from starting vectors near the eigenvectors
                (GCGE_HIP_MultiLinearSolve, 20 iterations at most), float64 or
                with float32 directions and products ("mixed").
kind "gradient" dL/dkappa of an eigenvalue loss for every element
                (adjoint.q1_kappa_gradient), a host array as result.
kind "solve"    a whole differentiable solve: eigenvalues, and dL/dkappa of a
                loss on them through the eigenvectors (whose signs are free,
                so the gradient stands for them).
"""
import ctypes

import numpy as np
import torch

import gcge_old_amd as gcge
from gcge_old_amd import _native, adjoint

SOLVE_FLAGS = ["-gcge_conv_type", "RB", "-gcge_ev_tol", "1e-10", "-gcge_ev_max_it", "400",
               "-gcge_full_rr", "1", "-gcge_w_orth_type", "svqb", "-gcge_max_reorth_time", "2"]
CG_MAX_IT = 20


def listed():
    return [
        # one matrix-vector product on the small mesh: eigenvector adjoints, single-vector drivers
        dict(name="product_64_k1", kind="product", E=64, k=1, matrix="K", numbering="grid"),
        # the residual check and the inner solves of the 128^3 workload
        dict(name="product_128_k100", kind="product", E=128, k=100, matrix="K", numbering="grid"),
        # a matrix without grid structure, the block of a 50-pair solve
        dict(name="product_local_96_k50", kind="product", E=96, k=50, matrix="M", numbering="local"),
        # a matrix given in no useful order, a wide block
        dict(name="product_scattered_128_k100", kind="product", E=128, k=100, matrix="K",
             numbering="scattered"),
        # W against X and P in a 50-pair solve with the default block of 10
        dict(name="gram_64_60x10", kind="gram", E=64, m=60, k=10),
        # Rayleigh-Ritz projection of the 128^3 workload: [X, P, W]^T A W
        dict(name="gram_128_300x100", kind="gram", E=128, m=300, k=100),
        # projection W - V d of a partly converged block, ragged widths
        dict(name="combine_64_77x19", kind="combine", E=64, m=77, k=19, beta=1.0),
        # Ritz vectors of the 128^3 workload
        dict(name="combine_128_300x100", kind="combine", E=128, m=300, k=100, beta=0.0),
        # the inner solve of the 64^3 workload: many short launches
        dict(name="inner_64_k10", kind="inner", E=64, k=10, precision="fp64"),
        # the inner solve of the 128^3 workload in its mixed-precision form
        dict(name="inner_128_k100", kind="inner", E=128, k=100, precision="mixed"),
        # gradient of all 100 eigenvalues with respect to 128^3 coefficients
        dict(name="gradient_128_k100", kind="gradient", E=128, k=100),
        # the 64^3 gradient workload: 20 eigenpairs and the adjoint of their eigenvalues
        dict(name="solve_64_nev20", kind="solve", E=64, nev=20),
    ]


def _log_int(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def draw(rng):
    kind = rng.choice(["product"] * 5 + ["gram"] * 3 + ["combine"] * 3 + ["inner"] * 2 +
                      ["gradient", "solve"])
    E = _log_int(rng, 24, 128)
    if kind == "product":
        return dict(kind=kind, E=E, k=_log_int(rng, 1, 100), matrix=rng.choice("KM"),
                    numbering=rng.choice(["grid", "grid", "local", "scattered"]))
    if kind == "gram":
        return dict(kind=kind, E=E, m=_log_int(rng, 1, 300), k=_log_int(rng, 1, 100))
    if kind == "combine":
        return dict(kind=kind, E=E, m=_log_int(rng, 2, 300), k=_log_int(rng, 1, 100),
                    beta=rng.choice([0.0, 1.0]))
    if kind == "inner":
        # smaller meshes let columns reach the rate, and those that stop change what the others do
        return dict(kind=kind, E=_log_int(rng, 44, 128), k=_log_int(rng, 2, 100),
                    precision=rng.choice(["fp64", "mixed"]))
    if kind == "gradient":
        return dict(kind=kind, E=E, k=_log_int(rng, 1, 100))
    return dict(kind=kind, E=rng.randint(24, 56), nev=rng.randint(10, 24))


# ---- inputs, from the seed alone -------------------------------------------------------------


def _gen(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed(1000 * int(seed) + stream)
    return g


def _uniform_columns(n, cols, seed, stream):
    """cols columns uniform(-1, 1), a few at a time: (first column, (c, n) tensor)."""
    g = _gen(seed, stream)
    for c0 in range(0, cols, 16):
        c = min(16, cols - c0)
        yield c0, torch.rand((c, n), dtype=torch.float64, device="cuda", generator=g) * 2.0 - 1.0


def _mode_numbers(k):
    side = 1
    while side ** 3 < k:
        side += 1
    t = [(a * a + b * b + c * c, a, b, c) for a in range(1, side + 4) for b in range(1, side + 4)
         for c in range(1, side + 4)]
    return sorted(t)[:k]


def _ritz_columns(E, k, seed, stream):
    """Approximate eigenvectors: the sine modes of the cube, smallest first,
    with a hundredth of noise; columns of about unit 2-norm times (2/h)^(3/2)
    (so that x^T M x is about 1)."""
    N = E - 1
    s = torch.arange(1, E, dtype=torch.float64, device="cuda") * (np.pi / E)
    g = _gen(seed, stream)
    modes = _mode_numbers(k)
    for c0 in range(0, k, 16):
        part = modes[c0:c0 + 16]
        x = torch.stack([(torch.sin(c * s)[:, None, None] * torch.sin(b * s)[None, :, None] *
                          torch.sin(a * s)[None, None, :]).reshape(-1) for _, a, b, c in part])
        noise = torch.rand((len(part), N ** 3), dtype=torch.float64, device="cuda", generator=g)
        yield c0, 2.0 ** 1.5 * (x + 0.01 * (2.0 * noise - 1.0))


def _kappa(E, seed):
    return np.exp(np.random.default_rng([int(seed), 1]).standard_normal(E ** 3))


def _node_row(E, seed, numbering):
    n = (E - 1) ** 3
    rng = np.random.default_rng([int(seed), 2])
    if numbering == "grid":
        return None
    if numbering == "scattered":
        return rng.permutation(n).astype(np.int32)
    key = np.arange(n) // 64 + rng.random(n)
    node_row = np.empty(n, dtype=np.int32)
    node_row[np.argsort(key, kind="stable")] = np.arange(n, dtype=np.int32)
    return node_row


def _coefficients(m, k, seed):
    """Columns of about orthonormal coefficients, as eigenvectors of the projected matrix have."""
    return np.asfortranarray(np.random.default_rng([int(seed), 3]).standard_normal((m, k)) / np.sqrt(m))


def _weights(k, seed):
    return np.random.default_rng([int(seed), 4]).standard_normal(k)


# ---- multivecs as tensors --------------------------------------------------------------------


class _MultiVecHead(ctypes.Structure):
    _fields_ = [("magic", ctypes.c_uint32), ("n", ctypes.c_int), ("ncols", ctypes.c_int),
                ("ld", ctypes.c_long), ("data", ctypes.c_void_p)]


class _Strided:
    def __init__(self, mv, ptr, shape, strides):
        self.mv = mv
        self.__cuda_array_interface__ = dict(data=(ptr, False), shape=shape, strides=strides,
                                             typestr="<f8", version=3)


def _tensor(mv):
    """The column block of a DeviceMultiVec as a (columns, rows) tensor over
    the same memory, which it keeps allocated: outputs outlive their state."""
    h = _MultiVecHead.from_address(mv.handle)
    if h.magic != 0x4D564531 or h.n != mv.n or h.ncols != mv.ncols:
        raise RuntimeError("unexpected multivec layout")
    t = torch.as_tensor(_Strided(mv, h.data, (h.ncols, h.n), (8 * h.ld, 8)), device="cuda")
    t.owner = mv
    return t


def _multivec(n, cols, columns=()):
    mv = gcge.DeviceMultiVec(n, cols)
    torch.cuda.synchronize()
    t = _tensor(mv)
    for c0, block in columns:
        t[c0:c0 + block.shape[0]] = block
    torch.cuda.synchronize()
    return mv, t


def _matrix(case, seed):
    E, which = case["E"], case.get("matrix", "K")
    return gcge.DeviceMatrix.q1(E, _kappa(E, seed) if which == "K" else None,
                                "stiffness" if which == "K" else "mass",
                                _node_row(E, seed, case.get("numbering", "grid")))


def prepare(case, seed):
    torch.cuda.init()
    gcge.init()
    lib, kind, E = _native.hip(), case["kind"], case["E"]
    n = (E - 1) ** 3
    s = dict(kind=kind, lib=lib, case=case)
    if kind == "product":
        k = case["k"]
        s["A"] = _matrix(case, seed)
        s["X"], _ = _multivec(n, k, _uniform_columns(n, k, seed, 1))
        s["Y"], s["out"] = _multivec(n, k)
    elif kind == "gram":
        m, k = case["m"], case["k"]
        s["V"], _ = _multivec(n, m, _uniform_columns(n, m, seed, 1))
        s["W"], _ = _multivec(n, k, _uniform_columns(n, k, seed, 2))
        s["G"] = np.zeros((m, k), order="F")
    elif kind == "combine":
        m, k = case["m"], case["k"]
        s["V"], _ = _multivec(n, m, _uniform_columns(n, m, seed, 1))
        s["C"] = _coefficients(m, k, seed)
        if case["beta"] != 0.0:
            # W - V d on a block that the call overwrites: a pass starts from the block kept here
            s["W"], _ = _multivec(n, k, _uniform_columns(n, k, seed, 2))
        s["Y"], s["out"] = _multivec(n, k)
    elif kind == "inner":
        k = case["k"]
        s["K"] = _matrix(case, seed)
        s["M"] = gcge.DeviceMatrix.q1(E, None, "mass")
        mixed = case["precision"] == "mixed"
        s["K"].set_precision(mixed)
        s["M"].set_precision(mixed)
        s["X"], _ = _multivec(n, k, _ritz_columns(E, k, seed, 1))
        lam = [np.pi ** 2 * m[0] for m in _mode_numbers(k)]
        s["X0"], x0 = _multivec(n, k, _ritz_columns(E, k, seed, 1))
        x0 /= torch.tensor(lam, dtype=torch.float64, device="cuda")[:, None]
        s["R"], s["res"] = _multivec(n, k)
        s["Y"], s["out"] = _multivec(n, k)
        torch.cuda.synchronize()
    elif kind == "gradient":
        k = case["k"]
        s["X"], _ = _multivec(n, k, _ritz_columns(E, k, seed, 1))
        s["w"] = _weights(k, seed)
    else:
        s["K"] = _matrix(case, seed)
        s["M"] = gcge.DeviceMatrix.q1(E, None, "mass")
        s["w"] = _weights(case["nev"], seed)
        s["seed"] = int(seed) % 1000003 + 1
    return s


def run(s):
    kind, lib, case = s["kind"], s["lib"], s["case"]
    if kind == "product":
        lib.GCGE_HIP_SpMM(s["A"].handle, s["X"].handle, 0, s["Y"].handle, 0, case["k"])
        return s["out"]
    if kind == "gram":
        lib.GCGE_HIP_Gram(s["V"].handle, 0, case["m"], s["W"].handle, 0, case["k"],
                          _native.as_dptr(s["G"]), case["m"])
        return s["G"]
    if kind == "combine":
        if "W" in s:
            lib.GCGE_HIP_Axpby(1.0, s["W"].handle, 0, 0.0, s["Y"].handle, 0, case["k"])
        lib.GCGE_HIP_LinearComb(s["V"].handle, 0, case["m"], _native.as_dptr(s["C"]), case["m"],
                                case["beta"], s["Y"].handle, 0, case["k"])
        return s["out"]
    if kind == "inner":
        k = case["k"]
        lib.GCGE_HIP_SpMM(s["M"].handle, s["X"].handle, 0, s["R"].handle, 0, k)
        lib.GCGE_HIP_Axpby(1.0, s["X0"].handle, 0, 0.0, s["Y"].handle, 0, k)
        lib.GCGE_HIP_SetLinearSolverParams(CG_MAX_IT, 1e-2, 0, 0.0, None)
        lib.GCGE_HIP_MultiLinearSolve(s["K"].handle, s["R"].handle, 0, s["Y"].handle, 0, k)
        # with float32 directions the solution is the result; the residuals left in the
        # right-hand sides are float32 values that a program reads no further
        return [s["out"], s["res"]] if case["precision"] == "fp64" else [s["out"]]
    if kind == "gradient":
        return adjoint.q1_kappa_gradient(case["E"], s["X"], s["w"])
    out = gcge.solve(s["K"], s["M"], case["nev"], SOLVE_FLAGS, seed=s["seed"])
    return [out["eval"], adjoint.q1_kappa_gradient(case["E"], out["evec"], s["w"])]


# ---- what a pass cannot do without ----------------------------------------------------------


def _entries(E, matrix):
    """Stored entries: 27 couplings of M, 21 of K (none to the face neighbours), boundary cut off."""
    N = E - 1
    line, shift = N, N - 1  # one-dimensional pairs (i, i + d), d = 0 and d = +-1
    every = (line + 2 * shift) ** 3
    return every if matrix == "M" else every - 6 * shift * line * line


def work(case):
    kind, E = case["kind"], case["E"]
    n = (E - 1) ** 3
    if kind == "product":
        z = _entries(E, case["matrix"])
        index = 0 if case["numbering"] == "grid" else 4
        return dict(bytes=z * (8 + index) + 16.0 * n * case["k"], flops=2.0 * z * case["k"])
    if kind == "gram":
        return dict(bytes=8.0 * n * (case["m"] + case["k"]), flops=2.0 * n * case["m"] * case["k"])
    if kind == "combine":
        cols = case["m"] + case["k"] * (1 if case["beta"] == 0.0 else 2)
        return dict(bytes=8.0 * n * cols, flops=2.0 * n * case["m"] * case["k"])
    if kind == "inner":
        # per step the values once, and x, r and p read and written once
        b, k, steps = 8 if case["precision"] == "fp64" else 4, case["k"], CG_MAX_IT - 1
        zk, zm = _entries(E, "K"), _entries(E, "M")
        return dict(bytes=steps * (b * zk + 6.0 * b * n * k) + 8.0 * zm + 32.0 * n * k,
                    flops=steps * (2.0 * zk + 10.0 * n) * k + 2.0 * (zm + zk) * k)
    if kind == "gradient":
        return dict(bytes=8.0 * n * case["k"] + 8.0 * E ** 3, flops=2.0 * 72 * E ** 3 * case["k"])
    # about 40 iterations, each with the products, inner solve and projections of its block
    nev, block = case["nev"], max(min(case["nev"], 10), case["nev"] // 5)
    basis = 2 * nev + 2 * block
    per = (CG_MAX_IT + 2) * (8.0 * _entries(E, "K") + 48.0 * n * block) + 8.0 * n * 4 * basis
    return dict(bytes=40 * per, flops=40 * 2.0 * n * (4 * basis * block + 30 * CG_MAX_IT * block))


# ---- the same in plain torch, 64 bits -------------------------------------------------------


def _element(matrix, E):
    k1 = np.array([[1.0, -1.0], [-1.0, 1.0]])
    m1 = np.array([[2.0, 1.0], [1.0, 2.0]]) / 6.0
    h = 1.0 / E
    if matrix == "M":
        return h ** 3 * np.kron(np.kron(m1, m1), m1)
    return h * (np.kron(np.kron(k1, m1), m1) + np.kron(np.kron(m1, k1), m1) +
                np.kron(np.kron(m1, m1), k1))


CORNERS = [(z, y, x) for z in (0, 1) for y in (0, 1) for x in (0, 1)]  # as np.kron orders them


def _apply(matrix, E, kappa, X):
    """A X for X (columns, n) in lexicographic order, element by element."""
    N = E - 1
    el = _element(matrix, E)
    full = torch.zeros((X.shape[0], E + 1, E + 1, E + 1), dtype=torch.float64, device=X.device)
    full[:, 1:E, 1:E, 1:E] = X.reshape(-1, N, N, N)
    out = torch.zeros_like(full)
    for p, (pz, py, px) in enumerate(CORNERS):
        t = torch.zeros((X.shape[0], E, E, E), dtype=torch.float64, device=X.device)
        for q, (qz, qy, qx) in enumerate(CORNERS):
            if el[p, q] != 0.0:
                t.add_(full[:, qz:qz + E, qy:qy + E, qx:qx + E], alpha=float(el[p, q]))
        if kappa is not None:
            t *= kappa
        out[:, pz:pz + E, py:py + E, px:px + E] += t
    return out[:, 1:E, 1:E, 1:E].reshape(X.shape[0], -1)


def _kappa_grid(E, seed, matrix):
    return None if matrix == "M" else torch.from_numpy(_kappa(E, seed)).cuda().reshape(E, E, E)


def exact(case, seed):
    kind, E = case["kind"], case["E"]
    n = (E - 1) ** 3
    if kind == "product":
        kap = _kappa_grid(E, seed, case["matrix"])
        order = _node_row(E, seed, case["numbering"])
        order = None if order is None else torch.from_numpy(order.astype(np.int64)).cuda()
        out = []
        for _, x in _uniform_columns(n, case["k"], seed, 1):
            y = _apply(case["matrix"], E, kap, x if order is None else x[:, order])
            if order is not None:
                y = torch.empty_like(y).index_copy_(1, order, y)
            out.append(y)
        return torch.cat(out)
    if kind == "gram":
        W = torch.cat([x for _, x in _uniform_columns(n, case["k"], seed, 2)])
        return torch.cat([x @ W.T for _, x in _uniform_columns(n, case["m"], seed, 1)]).cpu().numpy()
    if kind == "combine":
        C = torch.from_numpy(np.ascontiguousarray(_coefficients(case["m"], case["k"], seed))).cuda()
        Y = torch.zeros((case["k"], n), dtype=torch.float64, device="cuda")
        for c0, x in _uniform_columns(n, case["m"], seed, 1):
            Y += C[c0:c0 + x.shape[0]].T.contiguous() @ x
        if case["beta"] != 0.0:
            for c0, x in _uniform_columns(n, case["k"], seed, 2):
                Y[c0:c0 + x.shape[0]] += case["beta"] * x
        return Y
    if kind == "inner":
        kap, xs, rs = _kappa_grid(E, seed, "K"), [], []
        lam = torch.tensor([np.pi ** 2 * m[0] for m in _mode_numbers(case["k"])],
                           dtype=torch.float64, device="cuda")[:, None]
        for c0, col in _ritz_columns(E, case["k"], seed, 1):
            x = col / lam[c0:c0 + col.shape[0]]
            r = _apply("M", E, None, col) - _apply("K", E, kap, x)
            rho = (r * r).sum(1, keepdim=True)
            start, p = rho.sqrt(), r.clone()
            for it in range(1, CG_MAX_IT):
                w = _apply("K", E, kap, p)
                alpha = rho / (p * w).sum(1, keepdim=True)
                x += alpha * p
                r -= alpha * w
                new = (r * r).sum(1, keepdim=True)
                if it < CG_MAX_IT - 1 and bool((new.sqrt() < 1.01e-2 * start).any()):
                    return None  # a column that stops early changes what the others do
                p = r + (new / rho) * p
                rho = new
            xs.append(x)
            rs.append(r)
        return [torch.cat(xs), torch.cat(rs)] if case["precision"] == "fp64" else [torch.cat(xs)]
    if kind == "gradient":
        el, N = _element("K", E), E - 1
        w = _weights(case["k"], seed)
        out = torch.zeros((E, E, E), dtype=torch.float64, device="cuda")
        for c0, x in _ritz_columns(E, case["k"], seed, 1):
            full = torch.zeros((x.shape[0], E + 1, E + 1, E + 1), dtype=torch.float64, device="cuda")
            full[:, 1:E, 1:E, 1:E] = x.reshape(-1, N, N, N)
            wc = torch.from_numpy(w[c0:c0 + x.shape[0]].copy()).cuda()[:, None, None, None]
            for p, (pz, py, px) in enumerate(CORNERS):
                t = torch.zeros((x.shape[0], E, E, E), dtype=torch.float64, device="cuda")
                for q, (qz, qy, qx) in enumerate(CORNERS):
                    t.add_(full[:, qz:qz + E, qy:qy + E, qx:qx + E], alpha=float(el[p, q]))
                out += (wc * t * full[:, pz:pz + E, py:py + E, px:px + E]).sum(0)
        return out.reshape(-1).cpu().numpy()
    return None  # no independent solver is quick enough at these sizes
