"""What the speed of this library is measured on: calls a program makes through
lu2_amd's public entry points, over the sizes, precisions and options in use.

Kinds of case
  lu        Context.lumcolumn_dev: FP64 factorization and solve of lu2's
            augmented matrix (n x (n+16), b in column n), matrix in HBM,
            standard partial pivoting (the rule every measured configuration
            uses; lu2's own odd-column rule is unstable, so that no two orders
            of summation agree on its solutions)
  mixed     Context.solve_mixed: low-precision factors, FP64 refinement
  batch     Batch.solve: many small systems of uneven size in one launch
  dgemm     Context.dgemm_dev: lu2's mydgemm on blocks of one matrix
  residual  Context.residual_dev: the check of a solution

The factorization works in place, so a pass first restores the matrix from the
pristine copy that a program keeps for the residual check; that is one
device-to-device copy, under 2% of any large case.
"""
import math

import numpy as np
import torch

import lu2_amd as L

_ctx = None


def _context():
    """One context per process, as a program has it."""
    global _ctx
    if _ctx is None:
        _ctx = L.Context(0)
        _ctx.set_option(L.OPT_PIVMODE, L.PIV_GEPP)
    return _ctx


class _Buffer(L.DeviceBuffer):
    """A library allocation that torch can look at, freed with its last user."""

    def __init__(self, count, dtype):
        self.dtype, self.count = np.dtype(dtype), int(count)
        super().__init__(_context(), max(1, self.count) * self.dtype.itemsize)

    @property
    def __cuda_array_interface__(self):
        return {"shape": (self.count,), "typestr": self.dtype.str, "data": (self.ptr, False), "version": 3,
                "strides": None}

    def tensor(self):
        return torch.as_tensor(self, device="cuda")

    def __del__(self):
        if getattr(self, "ptr", None) and L and L._lib:   # not while the interpreter ends
            self.free()


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


# ---------------------------------------------------------------------------
def listed():
    return [
        # the smallest systems: launches and waits, no arithmetic to speak of
        {"name": "lu_n512", "kind": "lu", "n": 512, "nb": 64},
        # lu2's own example run (n=2048, block 256)
        {"name": "lu_n2048", "kind": "lu", "n": 2048, "nb": 256},
        # an ordinary size that is no power of two
        {"name": "lu_n9984", "kind": "lu", "n": 9984, "nb": 256},
        # lu2's drop-in configuration (n=32768, block 512)
        {"name": "lu_n32768", "kind": "lu", "n": 32768, "nb": 512},
        # the large end, with the block size of the n=65536 benchmark
        {"name": "lu_n49152", "kind": "lu", "n": 49152, "nb": 1024},
        # FP16x2 updates and refinement to the residual an FP64 factorization leaves
        {"name": "mixed_fp16x2_n32768", "kind": "mixed", "n": 32768, "nb": 2048, "prec": "fp16x2", "dominant": False,
         "target": 0.01},
        # FP32 factors, an ordinary size
        {"name": "mixed_fp32_n12288", "kind": "mixed", "n": 12288, "nb": 1024, "prec": "fp32", "dominant": False,
         "target": 0.01},
        # 16-bit updates of a diagonally dominant matrix
        {"name": "mixed_fp16_n32768", "kind": "mixed", "n": 32768, "nb": 2048, "prec": "fp16", "dominant": True,
         "target": 1.0},
        # the batched configuration: 4096 uneven systems, 1-4 right-hand sides
        {"name": "batch_fp64_4096", "kind": "batch", "systems": 4096, "nmin": 32, "nmax": 512, "rhs": 4,
         "prec": "fp64"},
        # a few small systems with FP32 factors and refinement
        {"name": "batch_fp32_300", "kind": "batch", "systems": 300, "nmin": 8, "nmax": 160, "rhs": 8, "prec": "fp32"},
        # lu2's update of a block of its matrix, odd width, the matrix's own row stride
        {"name": "dgemm_6000", "kind": "dgemm", "m": 6000, "n": 6001, "k": 512, "ld": 6544},
        # the check of a solution, no multiple of anything
        {"name": "residual_n20001", "kind": "residual", "n": 20001},
    ]


def _between(rng, lo, hi):
    """An integer spread evenly over the logarithm of [lo, hi]."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["lu", "lu", "mixed", "batch", "dgemm", "residual"])
    if kind == "lu":
        n = _between(rng, 300, 40000)
        nb = rng.choice([32, 64, 128]) if n < 2000 else rng.choice([128, 256, 512]) if n < 16000 else \
            rng.choice([512, 1024])
        return {"kind": "lu", "n": max(nb, n // nb * nb), "nb": nb}
    if kind == "mixed":
        prec = rng.choice(["fp32", "fp16x2", "fp16", "bf16"])
        n = _between(rng, 2000, 30000)
        nb = rng.choice([256, 512]) if n < 8000 else rng.choice([1024, 2048])
        dominant = prec in ("fp16", "bf16")
        return {"kind": "mixed", "n": n // nb * nb, "nb": nb, "prec": prec, "dominant": dominant,
                "target": 1.0 if dominant else 0.01}
    if kind == "batch":
        nmin = _between(rng, 4, 200)
        return {"kind": "batch", "systems": _between(rng, 1, 4096), "nmin": nmin, "nmax": rng.randint(nmin, 512),
                "rhs": rng.randint(1, 8), "prec": rng.choice(["fp64", "fp32"])}
    if kind == "dgemm":
        m, n, k = _between(rng, 30, 12000), _between(rng, 30, 12000), _between(rng, 16, 2048)
        return {"kind": "dgemm", "m": m, "n": n, "k": k, "ld": n + k + rng.randint(0, 31)}
    return {"kind": "residual", "n": _between(rng, 200, 40000)}


# ---------------------------------------------------------------------------
def _uniform(t, seed):
    """t (1-D, in place) i.i.d. uniform in [-0.5, 0.5), piece by piece."""
    g = _generator(seed)
    step = 1 << 28
    for at in range(0, t.numel(), step):
        t[at:at + step].uniform_(-0.5, 0.5, generator=g)


def _fill_augmented(t, case, seed):
    """lu2's kind of matrix: n x (n+1) uniform entries, zero padding; made
    diagonally dominant (a_ii += sum_j |a_ij|) for the 16-bit solves."""
    n = case["n"]
    _uniform(t, seed)
    a = t.view(n, n + 16)
    a[:, n + 1:] = 0.0
    if case.get("dominant"):
        for r in range(0, n, 4096):
            rows = torch.arange(r, min(n, r + 4096), device=t.device)
            a[rows, rows] += a[r:r + 4096, :n].abs().sum(dim=1)


def _batch_shapes(case):
    rng = np.random.default_rng([case["systems"], case["nmin"], case["nmax"], case["rhs"]])
    n = rng.integers(case["nmin"], case["nmax"] + 1, case["systems"])
    return n, rng.integers(1, case["rhs"] + 1, case["systems"])


def _fill_batch(t, n, nrhs, seed):
    """Uniform entries, plus sqrt(n)/2 on a random permutation of the diagonal:
    rows still change places, and every system is conditioned well enough for
    its solution to be compared to many digits."""
    _uniform(t, seed)
    rng = np.random.default_rng([int(seed), 1])
    base = np.concatenate([[0], np.cumsum(n * (n + nrhs))[:-1]])
    at = [b + np.arange(k) * (k + r) + rng.permutation(k) for b, k, r in zip(base, n, nrhs)]
    add = np.repeat(0.5 * np.sqrt(n), n)
    t[torch.from_numpy(np.concatenate(at)).cuda()] += torch.from_numpy(add).cuda()


def _dgemm_blocks(case):
    """(rows, element offsets of A, B and C) of C -= A B inside one matrix:
    B and C share their columns, A and C their rows."""
    return case["m"] + case["k"], case["k"] * case["ld"], case["k"], case["k"] * case["ld"] + case["k"]


def prepare(case, seed):
    ctx, kind = _context(), case["kind"]
    s = {"case": case, "ctx": ctx}
    if kind in ("lu", "mixed"):
        n = case["n"]
        s["a0"] = _Buffer(n * (n + 16), np.float64)
        _fill_augmented(s["a0"].tensor(), case, seed)
        s["x"] = _Buffer(n, np.float64)
        out = [s["x"]]
        if kind == "lu":
            s["a"], s["piv"] = _Buffer(n * (n + 16), np.float64), _Buffer(n, np.int32)
            out += [s["a"], s["piv"]]
        s["out"] = [b.tensor() for b in out]
        if kind == "lu":
            s["out"][1] = s["out"][1].view(n, n + 16)
    elif kind == "batch":
        n, nrhs = _batch_shapes(case)
        s["plan"] = L.Batch(ctx, n, nrhs, prec=L.PREC_FP64 if case["prec"] == "fp64" else L.PREC_FP32)
        s["a"], s["x"] = _Buffer(s["plan"].a_elems, np.float64), _Buffer(s["plan"].x_elems, np.float64)
        _fill_batch(s["a"].tensor(), n, nrhs, seed)
        s["out"] = s["x"].tensor()
    elif kind == "dgemm":
        rows, *s["at"] = _dgemm_blocks(case)
        s["a"] = _Buffer(rows * case["ld"], np.float64)
        _uniform(s["a"].tensor(), seed)
        s["out"] = s["a"].tensor().view(rows, case["ld"])[case["k"]:, case["k"]:case["k"] + case["n"]]
    else:
        n = case["n"]
        s["a"], s["x"] = _Buffer(n * (n + 16), np.float64), _Buffer(n, np.float64)
        _fill_augmented(s["a"].tensor(), case, seed)
        _uniform(s["x"].tensor(), seed + 1)
    torch.cuda.synchronize()   # the library's streams do not wait for torch's
    return s


_PREC = {"fp32": L.PREC_FP32, "fp16": L.PREC_FP16, "bf16": L.PREC_BF16, "fp16x2": L.PREC_FP16X2}


def run(s):
    case, ctx = s["case"], s["ctx"]
    kind = case["kind"]
    if kind == "lu":
        n = case["n"]
        s["a"].copy_from(s["a0"])
        ctx.lumcolumn_dev(n, s["a"], n + 16, case["nb"], s["piv"], s["x"])
        return s["out"]
    if kind == "mixed":
        n = case["n"]
        ctx.solve_mixed(n, s["a0"], n + 16, case["nb"], s["x"], _PREC[case["prec"]], maxiter=30,
                        target=case["target"])
        return s["out"]
    if kind == "batch":
        s["plan"].solve(s["a"], s["x"])
        return s["out"]
    if kind == "dgemm":
        a, ld = s["a"], case["ld"]
        ctx.dgemm_dev(case["m"], case["n"], case["k"], -1.0, a, ld, a, ld, 1.0, a, ld,
                      offs=tuple(8 * o for o in s["at"]))
        return s["out"]
    return ctx.residual_dev(case["n"], s["a"], case["n"] + 16, s["x"])


def work(case):
    kind = case["kind"]
    if kind == "lu":      # the matrix read and its factors written, x and the pivots written
        n = case["n"]
        return {"bytes": 16.0 * n * (n + 1) + 12.0 * n, "flops": 2.0 * n ** 3 / 3 + 2.0 * n ** 2}
    if kind == "mixed":   # the matrix read once, x written
        n = case["n"]
        return {"bytes": 8.0 * n * (n + 1) + 8.0 * n, "flops": 2.0 * n ** 3 / 3 + 2.0 * n ** 2}
    if kind == "batch":
        n, nrhs = (v.astype(np.float64) for v in _batch_shapes(case))
        return {"bytes": float(np.sum(8 * n * (n + 2 * nrhs))),
                "flops": float(np.sum(2 * n ** 3 / 3 + 2 * n ** 2 * nrhs))}
    if kind == "dgemm":
        m, n, k = case["m"], case["n"], case["k"]
        return {"bytes": 8.0 * (m * k + k * n + 2 * m * n), "flops": 2.0 * m * n * k}
    n = case["n"]
    return {"bytes": 8.0 * n * (n + 1) + 8.0 * n, "flops": 6.0 * n * n}


# ---------------------------------------------------------------------------
def _augmented(case, seed):
    n = case["n"]
    t = torch.empty(n * (n + 16), dtype=torch.float64, device="cuda")
    _fill_augmented(t, case, seed)
    return t.view(n, n + 16)


def exact(case, seed):
    kind = case["kind"]
    if kind in ("lu", "mixed"):
        n = case["n"]
        if n > 20000:   # the library solve of these takes too long
            return None
        a = _augmented(case, seed)
        x = torch.linalg.solve(a[:, :n], a[:, n])
        return [x, None, None] if kind == "lu" else [x]
    if kind == "batch":
        n, nrhs = _batch_shapes(case)
        if float(np.sum(n.astype(np.float64) ** 3)) > 2e11:
            return None
        t = torch.empty(int(np.sum(n * (n + nrhs))), dtype=torch.float64, device="cuda")
        _fill_batch(t, n, nrhs, seed)
        pool, at, out = t.cpu().numpy(), 0, []
        for k, r in zip(n, nrhs):
            a = pool[at:at + k * (k + r)].reshape(k, k + r)
            out.append(np.linalg.solve(a[:, :k], a[:, k:]).reshape(-1))
            at += k * (k + r)
        return np.concatenate(out)
    if kind == "dgemm":
        rows, a_at, b_at, c_at = _dgemm_blocks(case)
        m, n, k, ld = case["m"], case["n"], case["k"], case["ld"]
        t = torch.empty(rows * ld, dtype=torch.float64, device="cuda")
        _uniform(t, seed)
        full = t.view(rows, ld)
        return full[k:, k:k + n] - full[k:, :k].contiguous() @ full[:k, k:k + n].contiguous()
    a = _augmented(case, seed)
    n = case["n"]
    x = torch.empty(n, dtype=torch.float64, device="cuda")
    _uniform(x, seed + 1)
    r = float((a[:, :n] @ x - a[:, n]).abs().max())
    ainf, a1 = float(a[:, :n].abs().sum(dim=1).max()), float(a[:, :n].abs().sum(dim=0).max())
    xinf, x1, binf = float(x.abs().max()), float(x.abs().sum()), float(a[:, n].abs().max())
    eps, eps_lu2 = 2.0 ** -53, 2e-16
    return np.array([r, ainf, a1, xinf, x1, binf, r / (eps * (ainf * xinf + binf) * n), r / (eps_lu2 * a1 * n),
                     r / (eps_lu2 * a1 * x1), r / (eps_lu2 * ainf * xinf * n)])
