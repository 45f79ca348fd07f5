"""The work that users of this library have it do, as measurable cases.

Each case goes through the public entry points (hypre's C API as wrapped by
``hypre_amd.api``): products and residuals with a ParCSR matrix, assembly
through the IJ interface, one V-cycle as a preconditioner, PCG with a kept
hierarchy, and the whole of PCG setup + solve.  ``prepare`` makes what a
program has in hand before the call, ``run`` is one pass, ``exact`` the same
outputs from plain torch in 64 bits.
"""
import math

import numpy as np
import torch

from hypre_amd import api as hx

# PCG iterations to 1e-8 with l1-Jacobi V(1,1) and PMIS on these problems,
# and with the other options: the passes over the operator that work() counts
ITERATIONS = {"lap7": 13, "lap27": 16, "var7": 17, "jump27": 19}
ITERATIONS_GS, ITERATIONS_AGG = 8, 24


def listed():
    return [
        # the residual b - A x of a small grid: a convergence check inside a
        # user's own loop, where the call itself is most of the cost
        {"name": "residual_small", "kind": "residual", "problem": "lap7", "nx": 23, "ny": 19, "nz": 21},
        # y = A x on a large 27-point operator without a hierarchy
        {"name": "matvec_27pt", "kind": "matvec", "problem": "lap27", "nx": 161, "ny": 150, "nz": 170},
        # assembly of an irregular matrix (finite elements, any numbering)
        # from host arrays through the IJ interface: how data enters hypre
        {"name": "assemble_irregular", "kind": "assemble", "problem": "irregular", "nx": 47, "ny": 45, "nz": 52},
        # one V-cycle on such a matrix: the preconditioner of a user's own
        # Krylov method
        {"name": "cycle_irregular", "kind": "cycle", "problem": "irregular", "nx": 75, "ny": 64, "nz": 70},
        # setup + solve of the smallest benchmark problem (30^3 7-point):
        # launches and host round trips
        {"name": "step_7pt_30", "kind": "step", "problem": "lap7", "nx": 30, "ny": 30, "nz": 30},
        # an ordinary grid whose edges are no multiple of anything
        {"name": "step_7pt_ragged", "kind": "step", "problem": "lap7", "nx": 117, "ny": 131, "nz": 109},
        # the headline problem: 27-point 200^3, setup + solve in FP64
        {"name": "step_27pt_200", "kind": "step", "problem": "lap27", "nx": 200, "ny": 200, "nz": 200},
        # 256^3 7-point with a kept hierarchy: one more right-hand side, as in
        # time stepping
        {"name": "solve_7pt_256", "kind": "solve", "problem": "lap7", "nx": 256, "ny": 256, "nz": 256},
        # variable coefficients over six decades on 8^3-node cells
        {"name": "step_var7", "kind": "step", "problem": "var7", "nx": 150, "ny": 150, "nz": 150},
        # the largest: 27-point jumping coefficients on 320^3, FP32 V-cycle
        # inside FP64 PCG
        {"name": "step_jump27_320_fp32", "kind": "step", "problem": "jump27", "nx": 320, "ny": 320, "nz": 320,
         "fp32": True},
        # hypre's own host defaults: HMIS coarsening, hybrid l1 Gauss-Seidel
        # (13 down, 14 up)
        {"name": "step_hmis_gs", "kind": "step", "problem": "lap27", "nx": 64, "ny": 64, "nz": 64,
         "coarsen": 10, "gs": True},
        # one aggressive level with modified multipass interpolation, the
        # usual choice where memory counts on 7-point problems
        {"name": "step_agg_7pt", "kind": "step", "problem": "lap7", "nx": 140, "ny": 128, "nz": 151, "agg": 1},
    ]


def draw(rng):
    """One more case of the same families; edges spread over their logarithm."""
    def edges(lo, hi):
        return [int(round(math.exp(rng.uniform(math.log(lo), math.log(hi))))) for _ in range(3)]

    kind = rng.choice(["residual", "matvec", "assemble", "cycle", "solve", "step", "step", "step"])
    c = {"kind": kind}
    if kind in ("assemble", "cycle"):
        lo, hi = (12, 60) if kind == "assemble" else (14, 100)
        c["problem"] = "irregular"
        c["nx"], c["ny"], c["nz"] = edges(lo, hi)
        return c
    if kind in ("residual", "matvec"):
        c["problem"] = rng.choice(["lap7", "lap27"])
        c["nx"], c["ny"], c["nz"] = edges(12, 180)
        return c
    c["problem"] = rng.choice(["lap7", "lap27", "var7", "jump27"])
    hi = 256 if c["problem"] in ("lap7", "var7") else 200
    if c["problem"] in ("var7", "jump27"):
        c["nx"] = c["ny"] = c["nz"] = edges(24, hi)[0]
    else:
        c["nx"], c["ny"], c["nz"] = edges(24, hi)
    option = rng.choice(["", "", "fp32", "gs", "agg", "hmis"])
    if option == "fp32":
        c["fp32"] = True
    elif option == "gs":
        c["gs"] = True
    elif option == "agg" and c["problem"] == "lap7":
        c["agg"] = 1
    elif option == "hmis" and kind == "step":
        # the first pass is serial: HMIS is run on moderate grids
        c["coarsen"] = 10
        c["nx"], c["ny"], c["nz"] = (min(c[k], 64) for k in ("nx", "ny", "nz"))
    return c


# ------------------------------------------------------------------ inputs
class _Device:
    """A device array of the library as torch sees it; keeps its owner alive."""

    def __init__(self, ptr, n, typestr, owner):
        self.owner = owner
        self.__cuda_array_interface__ = {"shape": (n,), "typestr": typestr, "data": (int(ptr or 0), False),
                                         "version": 2}


def _tensor(ptr, n, dtype, owner):
    if n == 0 or not ptr:
        return torch.empty(0, dtype=dtype, device="cuda")
    return torch.as_tensor(_Device(ptr, n, "<f8" if dtype is torch.float64 else "<i4", owner), device="cuda")


def _vector_tensor(v):
    import ctypes
    n, d = ctypes.c_int(), ctypes.c_void_p()
    hx.call("HYPRE_MI355X_ParVectorGetDevice", v.h, ctypes.byref(n), ctypes.byref(d))
    return _tensor(d.value, n.value, torch.float64, v)


def _matrix_tensors(A):
    import ctypes
    n, nnz = ctypes.c_int(), ctypes.c_int()
    ia, ja, a = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    hx.call("HYPRE_MI355X_ParCSRMatrixGetDevice", A.h, ctypes.byref(n), ctypes.byref(nnz),
            ctypes.byref(ia), ctypes.byref(ja), ctypes.byref(a))
    return (_tensor(ia.value, n.value + 1, torch.int32, A), _tensor(ja.value, nnz.value, torch.int32, A),
            _tensor(a.value, nnz.value, torch.float64, A))


def _uniform(n, seed):
    """n values, uniform on [-1, 1]: the benchmark's right-hand sides."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    return 2.0 * torch.rand(n, dtype=torch.float64, device="cuda", generator=g) - 1.0


def _kappa_seed(seed):
    return 1 + seed % 1000003


def _cells(case):
    """(nodes a cell edge, log10 range) of the variable coefficients."""
    return (8, -3.0, 3.0) if case["problem"] == "var7" else (16, -4.0, 4.0)


def _irregular(case, seed):
    """(ncols, cols, values) on the host, rows in ascending column order: the
    graph of a 27-point grid with two edges of five missing, log-uniform
    couplings over two decades, numbered at random inside stretches of 512
    nodes, with a weak reaction term; symmetric, diagonally dominant."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    g = torch.Generator(device="cuda").manual_seed(seed)
    at = torch.arange(n, device="cuda")
    label = torch.argsort((at // 512).double() + torch.rand(n, device="cuda", dtype=torch.float64, generator=g))
    label = label.reshape(nz, ny, nx)
    i, j = [], []
    for dz in (0, 1):
        for dy in (-1, 0, 1):
            for dx in (-1, 0, 1):
                if (dz, dy, dx) <= (0, 0, 0):
                    continue
                p = label[:nz - dz, max(0, -dy):ny - max(0, dy), max(0, -dx):nx - max(0, dx)]
                q = label[dz:, max(0, dy):ny + min(0, dy), max(0, dx):nx + min(0, dx)]
                i.append(p.reshape(-1))
                j.append(q.reshape(-1))
    i, j = torch.cat(i), torch.cat(j)
    keep = torch.randperm(i.numel(), device="cuda", generator=g)[:3 * i.numel() // 5]
    i, j = i[keep], j[keep]
    w = 10.0 ** (2.0 * torch.rand(i.numel(), dtype=torch.float64, device="cuda", generator=g) - 2.0)
    # summed on the host, in one order
    ends, ww = torch.cat([i, j]).cpu().numpy(), torch.cat([w, w]).cpu().numpy()
    diag = torch.from_numpy(np.bincount(ends, ww, n) + 1e-3).cuda()
    row, col = torch.cat([i, j, at]), torch.cat([j, i, at])
    val = torch.cat([-w, -w, diag])
    order = torch.argsort(row * n + col)
    ncols = torch.bincount(row, minlength=n)
    return (ncols.cpu().numpy().astype(np.int32), col[order].cpu().numpy().astype(np.int32),
            val[order].cpu().numpy())


def _assemble(ncols, cols, values):
    n = len(ncols)
    m = hx.IJMatrix(0, n - 1)
    m.initialize()
    m.set_values(np.arange(n, dtype=np.int32), ncols, cols, values)
    m.assemble()
    return m.get_object()


def _matrix(case, seed):
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["problem"] == "lap7":
        return hx.ParCSRMatrix.laplacian7(nx, ny, nz)
    if case["problem"] == "lap27":
        return hx.ParCSRMatrix.laplacian27(nx, ny, nz)
    if case["problem"] == "irregular":
        return _assemble(*_irregular(case, seed))
    cell, lo, hi = _cells(case)
    return hx.ParCSRMatrix.var_diffusion(nx, 7 if case["problem"] == "var7" else 27, cell, lo, hi, _kappa_seed(seed))


def _amg(case):
    amg = hx.BoomerAMG(coarsen_type=case.get("coarsen", 8), fp32_cycle=1 if case.get("fp32") else 0)
    if case.get("gs"):
        amg.set(relax_type=13)
        amg.set(relax_up=14)
    if case.get("agg"):
        amg.set(agg_num_levels=case["agg"], agg_interp_type=8)
    return amg


def prepare(case, seed):
    hx.initialize()
    kind = case["kind"]
    if kind == "assemble":
        return {"kind": kind, "host": _irregular(case, seed)}
    A = _matrix(case, seed)
    n, _ = A.dims()
    s = {"kind": kind, "A": A, "b": hx.ParVector(n), "x": hx.ParVector(n)}
    _vector_tensor(s["b"]).copy_(_uniform(n, seed))
    if kind in ("residual", "matvec"):
        s["y"] = hx.ParVector(n)
        s["out"] = _vector_tensor(s["y"])
        _vector_tensor(s["x"]).copy_(_uniform(n, seed + 1))
    else:
        s["out"] = _vector_tensor(s["x"])
        s["amg"] = _amg(case)
        if kind == "cycle":
            s["amg"].set(max_iter=1, tol=0.0)
            s["amg"].setup(A, s["b"], s["x"])
        else:
            s["pcg"] = hx.PCG(s["amg"], tol=1e-8)
            if kind == "solve":
                s["pcg"].setup(A, s["b"], s["x"])
    torch.cuda.synchronize()    # torch's stream and the library's meet here
    return s


def run(s):
    kind = s["kind"]
    if kind == "assemble":
        return _matrix_tensors(_assemble(*s["host"]))
    A, b, x = s["A"], s["b"], s["x"]
    if kind == "matvec":
        A.matvec(1.0, x, 0.0, s["y"])
    elif kind == "residual":
        b.copy_to(s["y"])
        A.matvec(-1.0, x, 1.0, s["y"])
    else:
        x.fill(0.0)
        if kind == "cycle":
            s["amg"].solve(A, b, x)
        else:
            if kind == "step":
                s["pcg"].setup(A, b, x)
            s["pcg"].solve(A, b, x)
    return s["out"]


# ------------------------------------------------------------------ what a pass needs
def _size(case):
    """Rows and stored entries of the operator."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    n = nx * ny * nz
    if case["problem"] in ("lap7", "var7"):
        return n, 7 * n - 2 * (nx * ny + ny * nz + nx * nz)
    full = (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)
    return n, n + 2 * (3 * ((full - n) // 2) // 5) if case["problem"] == "irregular" else full


def work(case):
    """Each input read once and each output written once; for the iterations
    of a solve, three passes over the operator (the product, the residual
    after the first sweep, which starts from zero, and the last sweep) and
    the vectors they read and write, on all levels (a quarter more)."""
    n, nnz = _size(case)
    matrix, kind = 12.0 * nnz + 4.0 * (n + 1), case["kind"]
    if kind == "assemble":
        # in host memory and out in device memory
        return {"bytes": 2.0 * (12.0 * nnz + 4.0 * n), "flops": 0.0}
    if kind in ("matvec", "residual"):
        return {"bytes": matrix + 8.0 * n * (2 if kind == "matvec" else 3), "flops": 2.0 * nnz}
    inner = (8.0 * nnz + 4.0 * (n + 1) + 4.0 * 8 * n) if case.get("fp32") else matrix + 8.0 * 8 * n
    cycle = {"bytes": 1.25 * (2 * inner), "flops": 1.25 * 4.0 * nnz}
    if kind == "cycle":
        return cycle
    its = ITERATIONS_GS if case.get("gs") else ITERATIONS_AGG if case.get("agg") else ITERATIONS[case["problem"]]
    setup = 0.0 if kind == "solve" else 1.25 * matrix
    return {"bytes": setup + its * (cycle["bytes"] + matrix + 8.0 * 10 * n),
            "flops": its * (cycle["flops"] + 2.0 * nnz)}


def tolerance(case):
    kind = case["kind"]
    if kind == "assemble":
        return "exact"
    if kind in ("matvec", "residual"):
        # sums of at most 27 doubles in another order
        return {"rel": 2e-15, "max": 2e-14}
    if kind == "cycle":
        # four times what another order of the diagonals' sums changes
        return {"rel": 4e-14}
    # two solves that both end below a relative residual of 1e-8 differ by
    # what is left of the error (up to 8.4e-8 of the solution here): the last
    # iteration may fall to either side
    return {"rel": 4e-7}


# ------------------------------------------------------------------ the same in 64 bits
def _park_miller(seed, count):
    """hypre_Rand's stream: s <- 16807 s mod 2^31 - 1, values s / (2^31 - 1)."""
    out, s = np.empty(count), seed
    for k in range(count):
        s = 16807 * s % 2147483647
        out[k] = s / 2147483647
    return out


def _operator(case, seed):
    """A as a function of a (nz, ny, nx) grid, and its diagonal."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    if case["problem"] == "lap27":
        def box(x):
            for d in range(3):
                y = x.clone()
                y.narrow(d, 1, x.shape[d] - 1).add_(x.narrow(d, 0, x.shape[d] - 1))
                y.narrow(d, 0, x.shape[d] - 1).add_(x.narrow(d, 1, x.shape[d] - 1))
                x = y
            return x
        return (lambda x: 27.0 * x - box(x)), 26.0
    if case["problem"] == "lap7":
        faces, diag = [1.0, 1.0, 1.0], 6.0
    else:
        cell, lo, hi = _cells(case)
        nc = -(-nx // cell)
        u = torch.from_numpy(_park_miller(_kappa_seed(seed), nc ** 3)).reshape(nc, nc, nc).cuda()
        kappa = 10.0 ** (lo + (hi - lo) * u)
        for d in range(3):
            kappa = kappa.repeat_interleave(cell, d).narrow(d, 0, nx)
        faces, diag = [], torch.zeros_like(kappa)
        for d in range(3):
            m = nx - 1
            p, q = kappa.narrow(d, 0, m), kappa.narrow(d, 1, m)
            c = 2.0 * p * q / (p + q)
            faces.append(c)
            diag.narrow(d, 0, m).add_(c)
            diag.narrow(d, 1, m).add_(c)
            # a missing neighbour adds the node's own coefficient
            diag.select(d, 0).add_(kappa.select(d, 0))
            diag.select(d, m).add_(kappa.select(d, m))

    def apply(x):
        y = diag * x
        for d, c in enumerate(faces):
            m = x.shape[d] - 1
            y.narrow(d, 0, m).sub_(c * x.narrow(d, 1, m))
            y.narrow(d, 1, m).sub_(c * x.narrow(d, 0, m))
        return y
    return apply, diag


def _conjugate_gradients(apply, diag, b, tol, most):
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p, rz, end = z.clone(), torch.sum(r * z), tol * tol * float(torch.sum(b * b))
    for k in range(most):
        q = apply(p)
        alpha = rz / torch.sum(p * q)
        x += alpha * p
        r -= alpha * q
        if k % 16 == 15 and float(torch.sum(r * r)) < end:
            return x
        z = r / diag
        new = torch.sum(r * z)
        p = z + (new / rz) * p
        rz = new
    return None


def exact(case, seed):
    kind, n = case["kind"], _size(case)[0]
    if kind == "assemble":
        ncols, cols, values = _irregular(case, seed)
        row = np.repeat(np.arange(n), ncols)
        order = np.lexsort((np.arange(len(cols)), cols != row, row))    # the diagonal first
        ia = np.concatenate([[0], np.cumsum(ncols)]).astype(np.int32)
        return ia, cols[order], values[order]
    if case["problem"] not in ("lap7", "lap27", "var7") or min(case["nx"], case["ny"], case["nz"]) < 2:
        return None     # a V-cycle has no closed form; the jumps take plain CG too long
    if kind in ("solve", "step") and case["problem"] == "var7" and n > 5_000_000:
        return None     # thousands of iterations
    apply, diag = _operator(case, seed)
    shape = (case["nz"], case["ny"], case["nx"])
    b = _uniform(n, seed).reshape(shape)
    if kind in ("matvec", "residual"):
        y = apply(_uniform(n, seed + 1).reshape(shape))
        return (y if kind == "matvec" else b - y).reshape(-1)
    x = _conjugate_gradients(apply, diag, b, 1e-12, 2000 if case["problem"] != "var7" else 12000)
    return None if x is None else x.reshape(-1)
