"""The work that users of mspai_amd have it do, as timed cases.

Every case is one of the workloads that mspai_amd.gen generates, at the sizes
the benchmark and the tests use or odd ones between them:

  build    a preconditioner setup in a program that solves with one sparsity
           pattern and changing values (time steps, Newton steps): new values
           of A from device memory, then a complete build of M, which stays on
           the device.  Static builds leave M's values (the pattern is the one
           given); adaptive builds leave M as CSC arrays of the caller
           ("csc", Builder.build_noalloc) or M's values ("values").
  grad     a training step through the adjoint: build M from the values of C
           (and of the target), then dL/dC (and dL/dB) for a given dL/dM.
  block    a block SPAI build of a coupled system.
  apply    the preconditioned operator of a Krylov iteration, z = A (M x), and
           M^T x for a transposed one.
  gmres    a preconditioned GMRES cycle of 30 iterations on device vectors.

Values differ from seed to seed; the pattern of a grid does not.
"""
from __future__ import annotations

import math

import numpy as np
import torch

import mspai_amd
from mspai_amd import gen
from mspai_amd.autograd import spai_values
from mspai_amd.krylov import DeviceOperators, gmres

# options of the adaptive workloads: epsilon, new indices per step, steps
_GRID = {"eps": 0.4, "mn": 5, "ns": 5}
_BAND = {"eps": 0.3, "mn": 4, "ns": 8}


def _case(name, kind, matrix, size, precision=0, tuned=False, **kw):
    c = {"kind": kind, "matrix": matrix, "size": size, "precision": precision, "tuned": tuned, "out": "values"}
    c.update(kw)
    if name:
        c["name"] = name
    return c


def listed():
    return [
        # the smallest setup in use: a 64x64 Laplacian with a 5-point pattern; launches and host latency count
        _case("static_laplace2d_64_fp64", "build", "laplace2d", 64),
        # adaptive SPAI with the reference's default options on a 2D transport operator, its headline grid
        _case("adaptive_convdiff2d_256_fp64", "build", "convdiff2d", 256, out="csc", **_GRID),
        # the same in mixed precision on an odd grid
        _case("adaptive_convdiff2d_371_mixed", "build", "convdiff2d", 371, precision=1, out="csc", **_GRID),
        # unstructured, wide index sets, default size bins: what a program gets that never tunes
        _case("adaptive_band_262144_fp64_default", "build", "random", 262144, **_BAND),
        # the benchmark's headline: the same matrix, mixed precision, size bins tuned once
        _case("adaptive_band_262144_mixed_tuned", "build", "random", 262144, precision=1, tuned=True, out="csc",
              **_BAND),
        # a ragged, smaller unstructured system in FP64, tuned once
        _case("adaptive_band_50021_fp64_tuned", "build", "random", 50021, tuned=True, out="csc", **_BAND),
        # MSPAI probing (rho = 100) on the 3D Laplacian, one training step
        _case("probing3d_64_mixed_grad", "grad", "probing3d", 64, precision=1),
        # the large static workload: P(A^2) on a 3D variable-coefficient operator, both precisions
        _case("static_varcoef3d_128_fp64", "build", "varcoef3d", 128),
        _case("static_varcoef3d_101_mixed", "build", "varcoef3d", 101, precision=1),
        # a training step with respect to the coefficients of that operator
        _case("varcoef3d_48_fp64_grad", "grad", "varcoef3d", 48),
        # three coupled fields, 3x3 blocks, adaptive
        _case("block_convdiff2d_256x3_fp64", "block", "block", 256, bs=3, **_GRID),
        # the Krylov iteration's products with A and M on the unstructured system
        _case("apply_band_262144", "apply", "random", 262144),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    prec = rng.choice([0, 1])
    k = rng.randrange(10)
    if k == 0:
        return _case(None, "build", "laplace2d", _log_int(rng, 16, 512), prec)
    if k in (1, 2):
        return _case(None, "build", "convdiff2d", _log_int(rng, 24, 600), prec, out=rng.choice(["csc", "values"]),
                     **_GRID)
    if k in (3, 4):
        return _case(None, "build", "random", _log_int(rng, 6000, 262144), prec, rng.choice([False, True]),
                     **_BAND)
    if k == 5:
        return _case(None, "grad", "probing3d", _log_int(rng, 10, 64), prec)
    if k == 6:
        return _case(None, "build", "varcoef3d", _log_int(rng, 12, 110), prec)
    if k == 7:
        return _case(None, "grad", "varcoef3d", _log_int(rng, 10, 64), prec)
    if k == 8:
        return _case(None, "block", "block", _log_int(rng, 20, 256), bs=rng.choice([2, 3, 4]), **_GRID)
    if rng.random() < 0.5:
        return _case(None, "apply", "random", _log_int(rng, 6000, 262144))
    return _case(None, "gmres", "convdiff2d", _log_int(rng, 48, 320), rng.choice([0, 1]), **_GRID)


# ---------------------------------------------------------------- inputs

def _matrix(case, seed):
    """(C, start pattern or None for the diagonal, target or None)."""
    rng = np.random.Generator(np.random.PCG64([seed, 11]))
    name, size = case["matrix"], case["size"]
    if name == "random":
        A = gen.random_band(size, seed=1000 + seed)
        return A, (gen.pattern_of(A) if case["kind"] == "apply" else None), None
    if name == "convdiff2d":
        return gen.convdiff2d(size, theta=rng.uniform(0.1, 1.4), speed=rng.uniform(20.0, 80.0)), None, None
    if name == "block":
        return gen.block_convdiff2d(size, case["bs"], seed=seed), None, None
    if name == "varcoef3d":
        A = gen.varcoef3d(size, seed)
        return A, gen.pattern_power2(A), None
    # Laplacians with a material coefficient that varies by a few per cent
    A = gen.laplace2d(size) if name == "laplace2d" else gen.laplace3d(size)
    A.data *= 1.0 + 0.03 * rng.standard_normal(A.nnz)
    P = gen.pattern_of(A)
    if name == "probing3d":
        C, B = gen.probing_system(A, 100.0)
        return C, P, B
    return A, P, None


def _opts(case):
    o = dict(precision=case["precision"], binning=2 if case["tuned"] else 1)
    if "eps" in case:
        o.update(epsilon=case["eps"], maxnew=case["mn"], max_impr_steps=case["ns"])
    else:
        o.update(max_impr_steps=0)
    return o


def _capacity(case, n):
    """Room for an adaptive M: ncols (max |J0| + mn ns), in block columns of bs columns."""
    return n * (1 + case["mn"] * case["ns"]) * case.get("bs", 1)


def prepare(case, seed):
    A, P, B = _matrix(case, seed)
    n = A.shape[1]
    rng = np.random.Generator(np.random.PCG64([seed, 12]))
    b = mspai_amd.Builder(0)
    b.upload(A)
    st = {"case": case, "b": b, "opts": _opts(case), "n": n}
    if case["kind"] == "block":
        b.set_block_size(case["bs"])
    else:
        b.set_pattern(P)
    if B is not None:
        b.set_target(B)
        st["target"] = torch.tensor(B.data, device="cuda").requires_grad_()
    st["vals"] = torch.tensor(A.data, device="cuda")
    if case["tuned"]:
        o = dict(st["opts"])
        o.pop("binning")
        b.autotune(repeats=1, **o)
    if case["kind"] == "grad":
        st["vals"].requires_grad_()
        st["gM"] = torch.tensor(rng.standard_normal(P.nnz), device="cuda")
    if "eps" in case:
        # the caller's arrays, with room for the worst case; an adaptive M fills them in part
        cap = _capacity(case, n)
        st["m"] = torch.zeros(cap, dtype=torch.float64, device="cuda")
        if case["out"] == "csc":
            st["ptr"] = torch.zeros(n + 1, dtype=torch.int32, device="cuda")
            st["ind"] = torch.zeros(cap, dtype=torch.int32, device="cuda")
    if case["kind"] in ("apply", "gmres"):
        b.build(**st["opts"])
        st["ops"] = DeviceOperators(b)
        st["x"] = torch.tensor(rng.standard_normal(n), device="cuda")
    return st


def run(st):
    case, b = st["case"], st["b"]
    kind = case["kind"]
    if kind == "apply":
        ops = st["ops"]
        y = ops.M(st["x"])
        z = ops.A(y)
        t = torch.empty_like(y)
        b.apply_device(1, True, st["x"].data_ptr(), t.data_ptr())
        return y, z, t
    if kind == "gmres":
        x, its, _ = gmres(st["ops"].A, st["x"], st["ops"].M, restart=30, rtol=1e-12, maxiter=30)
        return x, its
    if kind == "grad":
        leaves = [st["vals"]] + ([st["target"]] if "target" in st else [])
        opts = dict(st["opts"])
        m = spai_values(b, st["vals"], st.get("target"), **opts)
        return (m.detach(), *torch.autograd.grad(m, leaves, st["gM"]))
    b.update_values_device(st["vals"].data_ptr())
    if case["out"] == "csc":
        ptr, ind, val = st["ptr"], st["ind"], st["m"]
        b.build_noalloc(ptr.data_ptr(), ind.data_ptr(), val.data_ptr(), val.numel(), **st["opts"])
        return ptr, ind, val
    info = b.build(**st["opts"])
    m = st["m"] if "m" in st else torch.empty(info["nnz"], dtype=torch.float64, device="cuda")
    b.result_values_device(m.data_ptr())
    return m


# ---------------------------------------------------------------- necessary work

# per column of the workload: entries of A, entries of M, and the flop of its
# least-squares solves (2 m n^2 - 2/3 n^3 and what follows it), from the sizes
# the index sets have on that workload
_COLUMN = {
    ("laplace2d", "build"): (5, 5, 700), ("convdiff2d", "build"): (5, 3.9, 500),
    ("random", "build"): (12, 3.05, 8000), ("varcoef3d", "build"): (7, 24, 70000),
    ("probing3d", "grad"): (8, 7, 5000), ("varcoef3d", "grad"): (7, 24, 140000),
    ("random", "apply"): (12, 12, 72), ("convdiff2d", "gmres"): (5, 3.9, 4000),
}


def _columns(case):
    s = case["size"]
    return {"random": s, "laplace2d": s * s, "convdiff2d": s * s, "block": s * s * case.get("bs", 1)}.get(
        case["matrix"], s ** 3)


def work(case):
    n = _columns(case)
    if case["kind"] == "block":
        a, m, flop = 5.0 * case["bs"] * 0.9, 13.7 * case["bs"] / 3, 3000.0 * case["bs"]
    else:
        a, m, flop = _COLUMN[case["matrix"], case["kind"]]
    if case["kind"] == "gmres":
        # 30 iterations: A and M read once in each, and the basis vectors so far twice
        return {"bytes": n * (30 * (12 * a + 12 * m + 16) + 16 * 30 * 31 / 2), "flops": n * flop}
    if case["kind"] == "apply":
        return {"bytes": n * (12 * a + 2 * 12 * m + 6 * 8), "flops": n * flop}
    by = n * (12 * a + 4 + 12 * m + 4)  # A in, M out
    if case["kind"] == "grad":
        by += n * (8 * m + 8 * a)  # dL/dM in, dL/dC out
    return {"bytes": by, "flops": n * flop}


# ---------------------------------------------------------------- 64-bit results by plain torch

def _expand(ptr, idx):
    """For every list ptr[i]..ptr[i+1) of i in idx: (position in idx, entry)."""
    cnt = ptr[idx + 1] - ptr[idx]
    pos = torch.repeat_interleave(torch.arange(idx.numel(), device=idx.device), cnt)
    start = torch.cumsum(cnt, 0) - cnt
    ent = torch.arange(pos.numel(), device=idx.device) - start[pos] + ptr[idx][pos]
    return pos, ent


def _slots(col, ncol):
    """Sorted owners `col`: (slot of each element in its column, counts)."""
    cnt = torch.bincount(col, minlength=ncol)
    first = torch.cumsum(cnt, 0) - cnt
    return torch.arange(col.numel(), device=col.device) - first[col], cnt


def _cholesky(G):
    n = G.shape[1]
    R = torch.zeros_like(G)
    S = G.clone()
    for j in range(n):
        d = S[:, j, j].sqrt()
        R[:, j, j:] = S[:, j, j:] / d[:, None]
        S[:, j + 1:, j + 1:] -= R[:, j, j + 1:, None] * R[:, j, None, j + 1:]
    return R


def _chol_solve(R, B):
    n = R.shape[1]
    Y = B.clone()
    for i in range(n):
        Y[:, i] /= R[:, i, i, None]
        if i + 1 < n:
            Y[:, i + 1:] -= R[:, i, i + 1:, None] * Y[:, i, None, :]
    for i in range(n - 1, -1, -1):
        Y[:, i] /= R[:, i, i, None]
        if i > 0:
            Y[:, :i] -= R[:, :i, i, None] * Y[:, i, None, :]
    return Y


class _System:
    """C (and the target) as bs x bs blocks in CSC and CSR order."""

    def __init__(self, C, B=None, bs=1):
        t = lambda x: torch.as_tensor(x, device="cuda")  # noqa: E731
        coo = C.tocoo()
        nb = C.shape[1] // bs
        self.bs, self.nb, self.nr = bs, nb, (C.shape[0] + bs - 1) // bs
        r, c, v = t(coo.row.astype(np.int64)), t(coo.col.astype(np.int64)), t(coo.data)
        key, inv = torch.unique((c // bs) * self.nr + r // bs, return_inverse=True)
        self.val = torch.zeros(key.numel(), bs, bs, dtype=torch.float64, device="cuda")
        self.val.index_put_((inv, r % bs, c % bs), v)
        self.row, self.col = key % self.nr, key // self.nr
        zero = torch.zeros(1, dtype=torch.int64, device="cuda")
        self.ptr = torch.cat([zero, torch.cumsum(torch.bincount(self.col, minlength=nb), 0)])
        self.by_row = torch.argsort(self.row, stable=True)
        self.rptr = torch.cat([zero, torch.cumsum(torch.bincount(self.row, minlength=self.nr), 0)])
        self.entry = (inv, r % bs, c % bs, c)  # where a stored scalar entry sits, in COO order
        self.B = None
        if B is not None:
            self.B = (t(B.indptr.astype(np.int64)), t(B.indices.astype(np.int64)), t(B.data))

    def factor(self, cols, own, J):
        """Dense A(I,J) of the columns `cols`, J given as sorted (own, J)
        pairs: the rows, the right-hand sides and the Cholesky factor."""
        nk, bs, dev = cols.numel(), self.bs, cols.device
        slot, nj = _slots(own, nk)
        pos, ent = _expand(self.ptr, J)
        rows, inv = torch.unique(own[pos] * self.nr + self.row[ent], return_inverse=True)
        rown = rows // self.nr
        rslot, mi = _slots(rown, nk)
        m, n = int(mi.max()) * bs, int(nj.max()) * bs
        D = torch.zeros(nk, m // bs, bs, n // bs, bs, dtype=torch.float64, device=dev)
        D.permute(0, 1, 3, 2, 4)[own[pos], rslot[inv], slot[pos]] = self.val[ent]
        D = D.view(nk, m, n)
        rhs = torch.zeros(nk, m, bs, dtype=torch.float64, device=dev)
        if self.B is None:
            k, want, bval = torch.arange(nk, device=dev), cols, None
        else:
            k, e = _expand(self.B[0], cols)
            want, bval = self.B[1][e], self.B[2][e]
        at = torch.searchsorted(rows, k * self.nr + want).clamp(max=rows.numel() - 1)
        hit = rows[at] == k * self.nr + want
        for q in range(bs):
            rhs[k[hit], rslot[at[hit]] * bs + q, q] = 1.0 if bval is None else bval[hit]
        G = torch.bmm(D.transpose(1, 2).contiguous(), D)
        pad = torch.arange(n, device=dev)[None, :] >= nj[:, None] * bs
        G.diagonal(dim1=1, dim2=2).add_(pad.to(torch.float64))
        f = dict(D=D, R=_cholesky(G), rhs=rhs, rows=rows, rown=rown, rslot=rslot, slot=slot, pos=pos, ent=ent,
                 inv=inv, own=own, bhit=(k, at, hit), nk=nk)
        X = torch.zeros(nk, n, bs, dtype=torch.float64, device=dev)
        for _ in range(4):
            X += _chol_solve(f["R"], torch.bmm(D.transpose(1, 2).contiguous(), rhs - torch.bmm(D, X)))
        f["X"], f["res"] = X, rhs - torch.bmm(D, X)
        return f

    def augment(self, cols, own, J, f, rn, todo, maxnew):
        """The pairs (own, j) that one augmentation step adds."""
        bs, nk, dev = self.bs, cols.numel(), cols.device
        keep = todo[f["rown"]]
        ro, rr = f["rown"][keep], f["rows"][keep] % self.nr
        kk = torch.nonzero(todo).flatten()
        L = torch.unique(torch.cat([f["rows"][keep], kk * self.nr + cols[kk]]))
        pos, ent = _expand(self.rptr, L % self.nr)
        cand = torch.unique((L // self.nr)[pos] * self.nb + self.col[self.by_row[ent]])
        have = own * self.nb + J
        cand = cand[~torch.isin(cand, have)]
        co, cj = cand // self.nb, cand % self.nb
        if cand.numel() == 0:
            return co, cj
        pos, ent = _expand(self.rptr, rr)
        ent = self.by_row[ent]
        key = ro[pos] * self.nb + self.col[ent]
        at = torch.searchsorted(cand, key).clamp(max=cand.numel() - 1)
        hit = cand[at] == key
        pos, ent, at = pos[hit], ent[hit], at[hit]
        r = f["res"].view(nk, -1, bs, bs)[ro[pos], f["rslot"][keep][pos]]
        N = torch.zeros(cand.numel(), bs, bs, dtype=torch.float64, device=dev)
        N.index_add_(0, at, (self.val[ent][:, :, :, None] * r[:, :, None, :]).sum(1))
        if not hasattr(self, "S"):
            S = torch.zeros(self.nb, bs, bs, dtype=torch.float64, device=dev)
            S.index_add_(0, self.col, (self.val[:, :, :, None] * self.val[:, :, None, :]).sum(1))
            self.S = _cholesky(S)
        Y = _chol_solve(self.S[cj], N)
        rho = torch.sqrt(rn[co] ** 2 - (N * Y).sum((1, 2)))
        cnt = torch.bincount(co, minlength=nk)
        mean = torch.zeros(nk, dtype=torch.float64, device=dev).index_add(0, co, rho) / cnt.clamp(min=1)
        ok = rho <= mean[co]
        co, cj, rho = co[ok], cj[ok], rho[ok]
        order = torch.argsort(rho, stable=True)
        order = order[torch.argsort(co[order], stable=True)]
        co, cj = co[order], cj[order]
        take = _slots(co, nk)[0] < maxnew
        return co[take], cj[take]

    def solve(self, cols, own, J, eps=0.0, maxnew=0, steps=0):
        """M's columns `cols`: (own, J) pairs and their values."""
        nk, bs = cols.numel(), self.bs
        out_o, out_j, out_x = [], [], []
        left = torch.arange(nk, device=cols.device)  # positions in `cols` of the columns still open
        for step in range(steps + 1):
            f = self.factor(cols[left], own, J)
            rn = f["res"].pow(2).sum((1, 2)).sqrt()
            n_o = n_j = None
            if step < steps:
                todo = rn > eps * math.sqrt(bs)
                n_o, n_j = self.augment(cols[left], own, J, f, rn, todo, maxnew)
            grow = torch.zeros(left.numel(), dtype=torch.bool, device=cols.device)
            if n_o is not None:
                grow[n_o] = True
            fin = ~grow[own]
            out_o.append(left[own[fin]])
            out_j.append(J[fin])
            out_x.append(f["X"].view(left.numel(), -1, bs, bs)[own[fin], f["slot"][fin]])
            if not bool(grow.any()):
                break
            new = torch.cumsum(grow, 0) - 1
            key = torch.cat([new[own[~fin]] * self.nb + J[~fin], new[n_o] * self.nb + n_j])
            key = torch.sort(key)[0]
            own, J = key // self.nb, key % self.nb
            left = left[grow]
        o, j, x = torch.cat(out_o), torch.cat(out_j), torch.cat(out_x)
        order = torch.argsort(o * self.nb + j)
        return o[order], j[order], x[order]


def _chunks(nb, per):
    return [(a, min(nb, a + per)) for a in range(0, nb, per)]


def _exact_m(case, sys_, P):
    """(own, J, values) of M over all columns."""
    big = {"varcoef3d": 32768, "random": 8192, "block": 8192}.get(case["matrix"], 65536)
    parts = []
    dev = "cuda"
    if P is not None:
        pp = torch.as_tensor(P.indptr.astype(np.int64), device=dev)
        pi = torch.as_tensor(P.indices.astype(np.int64), device=dev)
    for a, b in _chunks(sys_.nb, big):
        cols = torch.arange(a, b, device=dev)
        if P is None:
            own, J = torch.arange(b - a, device=dev), cols
        else:
            own, ent = _expand(pp, cols)
            J = pi[ent]
        o, j, x = sys_.solve(cols, own, J, case.get("eps", 0.0), case.get("mn", 0), case.get("ns", 0))
        parts.append((o + a, j, x))
    return tuple(torch.cat([p[i] for p in parts]) for i in range(3))


def _spmv(rows, cols, vals, x, n):
    return torch.zeros(n, dtype=torch.float64, device=x.device).index_add(0, rows, vals * x[cols])


def _padded(x, n):
    return torch.nn.functional.pad(x, (0, n - x.numel()))


def exact(case, seed):
    if case["kind"] == "gmres":
        return None  # an iterate of a Krylov process: no value apart from its own arithmetic
    C, P, B = _matrix(case, seed)
    n = C.shape[1]
    bs = case["bs"] if case["kind"] == "block" else 1
    sys_ = _System(C, B, bs)
    if case["kind"] == "grad":
        return _exact_grad(case, seed, C, P, B, sys_)
    own, J, x = _exact_m(case, sys_, P)
    if case["kind"] == "block":
        # scalar CSC order: per scalar column, blocks by row, rows within a block; exact zeros dropped
        q = torch.arange(bs, device="cuda")
        col = (own[:, None, None] * bs + q[None, None, :]).expand_as(x)
        row = (J[:, None, None] * bs + q[None, :, None]).expand_as(x)
        v = x.reshape(-1)[torch.argsort((col * n + row).reshape(-1))]
        return _padded(v[v != 0], _capacity(case, n))
    x = x.view(-1)
    if case["kind"] == "apply":
        rng = np.random.Generator(np.random.PCG64([seed, 12]))
        v = torch.tensor(rng.standard_normal(n), device="cuda")
        y = _spmv(J, own, x, v, n)
        return y, _spmv(sys_.row, sys_.col, sys_.val.view(-1), y, n), _spmv(own, J, x, v, n)
    if case["out"] == "csc":
        ptr = torch.cat([torch.zeros(1, dtype=torch.int64, device="cuda"),
                         torch.cumsum(torch.bincount(own, minlength=n), 0)])
        cap = _capacity(case, n)
        return ptr.to(torch.int32), _padded(J.to(torch.int32), cap), _padded(x, cap)
    return x if P is not None else _padded(x, _capacity(case, n))


def _exact_grad(case, seed, C, P, B, sys_):
    """M's values, and dL/dC and dL/dB at M's fixed pattern: with r = b - C m
    and C^T C lambda = dL/dm per column, dL/dC_ij = r_i lambda_j -
    (C lambda)_i m_j summed over the columns, dL/db = C lambda."""
    rng = np.random.Generator(np.random.PCG64([seed, 12]))
    g = torch.tensor(rng.standard_normal(P.nnz), device="cuda")
    pp = torch.as_tensor(P.indptr.astype(np.int64), device="cuda")
    pi = torch.as_tensor(P.indices.astype(np.int64), device="cuda")
    gC = torch.zeros(sys_.val.shape[0], dtype=torch.float64, device="cuda")
    gB = torch.zeros(B.nnz, dtype=torch.float64, device="cuda") if B is not None else None
    m = torch.zeros(P.nnz, dtype=torch.float64, device="cuda")
    for a, b in _chunks(sys_.nb, 32768):
        cols = torch.arange(a, b, device="cuda")
        own, ent = _expand(pp, cols)
        f = sys_.factor(cols, own, pi[ent])
        D, X, r = f["D"], f["X"][:, :, 0], f["res"][:, :, 0]
        m[ent] = X[own, f["slot"]]
        gm = torch.zeros_like(X)
        gm[own, f["slot"]] = g[ent]
        Dt = D.transpose(1, 2).contiguous()
        lam = torch.zeros_like(gm)
        for _ in range(4):
            lam += _chol_solve(f["R"], (gm - torch.bmm(Dt, torch.bmm(D, lam[:, :, None]))[:, :, 0])[:, :, None])[:, :, 0]
        s = torch.bmm(D, lam[:, :, None])[:, :, 0]
        k, sl, rs = own[f["pos"]], f["slot"][f["pos"]], f["rslot"][f["inv"]]
        gC.index_add_(0, f["ent"], r[k, rs] * lam[k, sl] - s[k, rs] * X[k, sl])
        if gB is not None:
            kb, at, hit = f["bhit"]
            eb = _expand(sys_.B[0], cols)[1]
            gB[eb[hit]] = s[kb[hit], f["rslot"][at[hit]]]
    # sys_ holds the entries in CSC order, as C does
    return (m, gC) if gB is None else (m, gC, gB)
