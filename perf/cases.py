"""The work whose time this library is judged by: calls that programs make of
it, each through its public entry points, over the sizes, patterns, formats
and value types in use.

Every case names a `kind`:

  block      BlockSparseMatrix / BlockBandedMatrix products of a DC optimal
             power flow operator (one period, or T periods with ramp coupling)
  spmv       y = A*x, plain or from a handle, A as CSR, COO or CSC
  spmm       C = A*B with k columns, plain or from a handle, CSR, COO or CSC
  sddmm      C.val = mask .* (A*B at C's entries), plain or from a handle
  graph      one message-passing layer: the product, and both of its gradients
  bsr_spmm   block CSR times k columns
  bsr_spmv   the residual r = b - A*x of a block CSR matrix
  convert    a change of format

and a `pattern` of the matrix (of its blocks for the bsr kinds):

  uniform    `mean` distinct random columns in every row
  powerlaw   row lengths Pareto(1.8) with that mean, random columns
  mesh       the 27-point neighbourhood on a gx x gy x gz grid
  band       `mean` distinct columns within `band` of the diagonal

Sizes are those of this repository's own benchmark configurations and block
operators, or generic ones of the same kinds.
"""
import numpy as np
import torch

import jlust_amd as J
from jlust_amd import workloads as W

DEV = "cuda"


# ------------------------------------------------------------------- the cases

def listed():
    return [
        # One product of an optimal power flow operator inside a solver's
        # iteration: a few microseconds of work, so launches and the host count.
        dict(name="block_dcopf", kind="block", bus=30000, line=35393, gen=3526, periods=1, dtype="f64"),
        # The same operator over a day of hourly periods with ramp coupling.
        dict(name="block_dcopf_day", kind="block", bus=30000, line=35393, gen=3526, periods=24, dtype="f64"),
        # A Krylov iteration on a small matrix that the caches hold.
        dict(name="spmv_100k", kind="spmv", pattern="uniform", m=100000, n=100000, mean=16,
             dtype="f64", format="csr", call="handle"),
        # A ranking iteration on a large scale-free graph.
        dict(name="spmv_powerlaw_4m", kind="spmv", pattern="powerlaw", m=4000000, n=4000000, mean=16,
             dtype="f64", format="csr", call="handle"),
        # Feature aggregation over a large random graph, one plain call.
        dict(name="spmm_1m_k128", kind="spmm", pattern="uniform", m=1000000, n=1000000, mean=32, k=128,
             dtype="f32", format="csr", call="plain"),
        # A block eigensolver's product on a 3D mesh: local columns, few of
        # them at once, an odd grid, double precision.
        dict(name="spmm_mesh_k20", kind="spmm", pattern="mesh", gx=67, gy=61, gz=64, k=20,
             dtype="f64", format="csr", call="handle"),
        # Sampled scores over a large random mask.
        dict(name="sddmm_500k_k128", kind="sddmm", pattern="uniform", m=500000, n=500000, mean=32, K=128,
             dtype="f32", format="csr", masked=True, call="plain"),
        # Training on a scale-free graph with learned edge weights: forward,
        # the gradient of the features (the transposed product, over the same
        # buffers as CSC) and that of the weights; a feature count that is no
        # power of two.
        dict(name="graph_200k_k100", kind="graph", pattern="powerlaw", m=200003, n=200003, mean=14, K=100,
             dtype="f32"),
        # Block-banded matrix of 16 x 16 blocks times a tall dense one.
        dict(name="bsr16_band_k256", kind="bsr_spmm", pattern="band", m=65536, mean=8, band=32, b=16, k=256,
             dtype="f32", row_major=True, call="plain"),
        # Four unknowns a node, several right-hand sides: block Krylov on a
        # finite element matrix.
        dict(name="bsr4_mesh_k24", kind="bsr_spmm", pattern="mesh", gx=40, gy=37, gz=41, b=4, k=24,
             dtype="f64", row_major=True, call="handle"),
        # Three displacements a node: the residual of an elasticity solve.
        dict(name="bsr3_mesh_residual", kind="bsr_spmv", pattern="mesh", gx=48, gy=45, gz=47, b=3,
             dtype="f64", row_major=True, call="plain"),
        # The transpose of a scale-free matrix as a matrix of its own (its
        # CSC arrays), taken once for every new pattern.
        dict(name="convert_csc_1m", kind="convert", pattern="powerlaw", m=1000003, n=1000003, mean=16,
             dtype="f64", src="csr", dst="csc"),
    ]


def _log(rng, lo, hi):
    return int(round(lo * (hi / lo) ** rng.random()))


def _mesh(rng, lo, hi):
    """Three sides whose product lies near a logarithmic draw of [lo, hi]."""
    side = _log(rng, lo, hi) ** (1.0 / 3.0)
    gx = max(3, int(side * rng.uniform(0.7, 1.4)))
    gy = max(3, int(side * rng.uniform(0.7, 1.4)))
    return dict(gx=gx, gy=gy, gz=max(3, int(side ** 3 / (gx * gy))))


def _pattern(rng, lo, hi, means, kinds=("uniform", "powerlaw", "mesh", "band")):
    p = rng.choice(kinds)
    if p == "mesh":
        return dict(pattern=p, **_mesh(rng, lo, hi // 2))
    m = _log(rng, lo, hi)
    out = dict(pattern=p, m=m, mean=rng.randint(*means))
    if p == "band":
        out["band"] = rng.choice((16, 32, 100))
    else:
        out["n"] = m if rng.random() < 0.6 else _log(rng, max(lo, m // 3), min(hi, m * 3))
    return out


def draw(rng):
    kind = rng.choice(("block", "spmv", "spmv", "spmm", "spmm", "sddmm", "graph", "bsr_spmm", "bsr_spmm",
                       "bsr_spmv", "convert"))
    dtype = rng.choice(("f32", "f64"))
    fmt = rng.choice(("csr", "csr", "coo", "csc"))
    call = rng.choice(("plain", "handle"))
    if kind == "block":
        bus = _log(rng, 1000, 30000)
        return dict(kind=kind, bus=bus, line=int(bus * rng.uniform(1.1, 1.5)), gen=max(8, bus // rng.randint(6, 12)),
                    periods=rng.choice((1, 1, 6, 12, 24)), dtype="f64")
    if kind == "spmv":
        return dict(kind=kind, **_pattern(rng, 10000, 2000000, (3, 24)), dtype=dtype, format=fmt, call=call)
    if kind == "spmm":
        return dict(kind=kind, **_pattern(rng, 10000, 300000, (4, 32)), k=_log(rng, 2, 128),
                    dtype=dtype, format=fmt, call=call)
    if kind == "sddmm":
        return dict(kind=kind, **_pattern(rng, 10000, 250000, (4, 32)), K=_log(rng, 4, 128),
                    dtype=dtype, format=fmt, masked=rng.random() < 0.5, call=call)
    if kind == "graph":
        m = _log(rng, 10000, 200000)
        return dict(kind=kind, pattern=rng.choice(("uniform", "powerlaw")), m=m, n=m, mean=rng.randint(4, 24),
                    K=_log(rng, 8, 128), dtype="f32")
    if kind == "bsr_spmm":
        b = rng.choice((2, 3, 4, 4, 5, 6, 8, 16, 16))
        return dict(kind=kind, **_pattern(rng, 2000, 24000 if b > 8 else 60000, (4, 16), ("mesh", "band")), b=b,
                    k=_log(rng, 4, 128 if b > 8 else 48), dtype=dtype, row_major=rng.random() < 0.7, call=call)
    if kind == "bsr_spmv":
        return dict(kind=kind, **_pattern(rng, 2000, 60000, (4, 32), ("mesh", "band", "powerlaw")),
                    b=rng.choice((2, 3, 4, 6, 8, 16)), dtype=dtype, row_major=rng.random() < 0.7, call=call)
    src, dst = rng.choice((("csr", "csc"), ("csc", "csr"), ("csr", "coo"), ("coo", "csr"), ("coo", "csc"),
                           ("csr", "bsr")))
    out = dict(kind="convert", **_pattern(rng, 10000, 1000000, (3, 16)), dtype=dtype, src=src, dst=dst)
    if dst == "bsr":          # a format for matrices whose entries come in blocks
        out = dict(kind="convert", pattern="mesh", **_mesh(rng, 2000, 60000), b=rng.choice((2, 3, 4)), dtype=dtype,
                   src="csr", dst="bsr")
    return out


# ------------------------------------------------------------------- the inputs

def _dt(case):
    return torch.float64 if case["dtype"] == "f64" else torch.float32


def _shape(case):
    """Rows and columns of the pattern (block rows and columns for bsr)."""
    if case["pattern"] == "mesh":
        m = case["gx"] * case["gy"] * case["gz"]
        return m, m
    return case["m"], case.get("n", case["m"])


def _mesh_nnz(case):
    return (3 * case["gx"] - 2) * (3 * case["gy"] - 2) * (3 * case["gz"] - 2)


def _entries(case):
    """Stored entries (blocks) of the pattern."""
    return _mesh_nnz(case) if case["pattern"] == "mesh" else _shape(case)[0] * case["mean"]


def _csr(case, gen):
    """(rows, rowptr, cols) of the pattern: 0-based int64 rows and columns,
    rows in order, columns increasing in each."""
    m, n = _shape(case)
    if case["pattern"] == "mesh":
        gx, gy, gz = case["gx"], case["gy"], case["gz"]
        r = torch.arange(m, device=DEV)
        x, y, z = r % gx, r // gx % gy, r // (gx * gy)
        cols = []
        for dz in (-1, 0, 1):
            for dy in (-1, 0, 1):
                for dx in (-1, 0, 1):
                    ok = ((x + dx >= 0) & (x + dx < gx) & (y + dy >= 0) & (y + dy < gy) &
                          (z + dz >= 0) & (z + dz < gz))
                    cols.append(torch.where(ok, r + dx + gx * (dy + gy * dz), -1))
        cols = torch.stack(cols, 1)
        keep = cols >= 0
        lens = keep.sum(1)
        cols = cols[keep]
    elif case["pattern"] == "band":
        width = min(2 * case["band"] + 1, n)
        mean = min(case["mean"], width)
        start = (torch.arange(m, device=DEV) - case["band"]).clamp(0, n - width)
        pick = torch.rand(m, width, generator=gen, device=DEV).topk(mean, dim=1).indices.sort(1).values
        cols = (start[:, None] + pick).reshape(-1)
        lens = torch.full((m,), mean, device=DEV)
    else:
        if case["pattern"] == "uniform":
            lens = torch.full((m,), min(case["mean"], n), device=DEV)
        else:
            top = min(100000, n)
            w = torch.rand(m, generator=gen, device=DEV, dtype=torch.float64).clamp_min(1e-12) ** (-1.0 / 1.8)
            scale = 1.0
            for _ in range(4):
                lens = (w * scale).round().clamp(1, top)
                scale *= case["mean"] / float(lens.mean())
            lens = lens.long()
            # One entry more or less in some rows, so that every seed has m*mean of them.
            off = int(lens.sum()) - m * case["mean"]
            change = torch.randperm(m, generator=gen, device=DEV)
            change = change[(lens[change] > 1) if off > 0 else (lens[change] < n)][:abs(off)]
            lens[change] -= 1 if off > 0 else -1
        rows = torch.repeat_interleave(torch.arange(m, device=DEV), lens)
        first = torch.cumsum(lens, 0) - lens
        # Sorted draws of [0, n - length] with their place in the row added:
        # increasing, so distinct.
        span = (n - lens + 1)[rows]
        low = (torch.rand(rows.numel(), generator=gen, device=DEV, dtype=torch.float64) * span).long()
        key, _ = torch.sort(rows * (1 << 31) + torch.minimum(low, span - 1))
        cols = (key & ((1 << 31) - 1)) + torch.arange(rows.numel(), device=DEV) - first[rows]
        return rows, torch.cat((lens.new_zeros(1), lens.cumsum(0))), cols
    rows = torch.repeat_interleave(torch.arange(m, device=DEV), lens)
    return rows, torch.cat((lens.new_zeros(1), lens.cumsum(0))), cols


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(count, dtype, gen):
    return torch.randn(count, generator=gen, device=DEV, dtype=dtype)


def _matrix(rows, cols, dtype, gen):
    """A rows x cols column-major normal matrix."""
    return _normal(rows * cols, dtype, gen).view(cols, rows).t()


def _i32(t):
    return t.int() + 1


def _tensor(fmt, rows, ptr, cols, val, shape):
    """The entries (CSR order) as a 1-based CSR, COO or CSC tensor."""
    if fmt == "csr":
        return J.csr_tensor(_i32(ptr), _i32(cols), val, shape)
    if fmt == "coo":
        return J.coo_tensor(_i32(rows), _i32(cols), val, shape)
    order = torch.sort(cols, stable=True).indices
    colptr = torch.zeros(shape[1] + 1, dtype=torch.int64, device=DEV)
    colptr[1:] = torch.cumsum(torch.bincount(cols, minlength=shape[1]), 0)
    return J.csc_tensor(_i32(colptr), _i32(rows[order]), val[order].contiguous(), shape)


def _dcopf(case, seed):
    """The operator's blocks as host CSR triplets: [Cg 0 -Bbus; 0 -I Bf] and
    the ramp selectors (-R, R)."""
    d = W.dcopf(case["bus"], case["line"], case["gen"], seed=int(seed))
    nb, nl, ng, nv = d["n_bus"], d["n_line"], d["n_gen"], d["n_var"]

    def eye(k, v):
        p = np.arange(1, k + 2, dtype=np.int32)
        return p, p[:-1].copy(), np.full(k, v)
    neg = lambda t: (t[0], t[1], -t[2])  # noqa: E731
    blocks = [[(d["Cg"], nb, ng), None, (neg(d["Bbus"]), nb, nb)],
              [None, (eye(nl, -1.0), nl, nl), (d["Bf"], nl, nb)]]
    return blocks, (eye(ng, -1.0), ng, nv), (eye(ng, 1.0), ng, nv), d


def _size_of_block(case):
    """Rows, columns and entries of the block operator, near enough for its work."""
    nb, nl, ng, T = case["bus"], case["line"], case["gen"], case["periods"]
    one = ng + nl + 2 * nl + nb + 2 * nl         # Cg, -I, Bf, Bbus
    return T * (nb + nl) + (T - 1) * ng, T * (ng + nl + nb), one + 2 * ng * (T > 1)


def prepare(case, seed):
    gen, dt, kind = _gen(seed), _dt(case), case["kind"]
    if kind == "block":
        blocks, neg, pos, d = _dcopf(case, seed)
        dev = lambda t: torch.from_numpy(t).to(DEV)  # noqa: E731
        ten = lambda b: None if b is None else J.csr_tensor(*map(dev, b[0]), (b[1], b[2]))  # noqa: E731
        A = J.BlockSparseMatrix([[ten(b) for b in row] for row in blocks])
        if case["periods"] > 1:
            A = J.BlockBandedMatrix(A, ten(neg), ten(pos), case["periods"], d["n_con"], d["n_gen"], d["n_var"])
        m, n = A.size()
        x, y = _normal(n, dt, gen), torch.empty(m, dtype=dt, device=DEV)
        J.mul_(y, A, x)                          # a solver's first product assembles the operator
        return dict(kind=kind, A=A, x=x, y=y)
    if kind in ("bsr_spmm", "bsr_spmv"):
        mb, nb = _shape(case)
        b = case["b"]
        _, ptr, cols = _csr(case, gen)
        A = J.bsr_tensor(_i32(ptr), _i32(cols), _normal(cols.numel() * b * b, dt, gen), (mb * b, nb * b), (b, b),
                         row_major_blocks=case["row_major"])
        st = dict(kind=kind, A=A)
        if kind == "bsr_spmm":
            st.update(B=_matrix(nb * b, case["k"], dt, gen), C=J.dense_matrix(mb * b, case["k"], dtype=dt, device=DEV))
            if case["call"] == "handle":
                st["h"] = J.prepare(J.HIPBackend(), J.SpMMOp, A, n_cols=case["k"])
        else:
            st.update(x=_normal(nb * b, dt, gen), b=_normal(mb * b, dt, gen),
                      r=torch.empty(mb * b, dtype=dt, device=DEV))
            if case["call"] == "handle":
                st["h"] = J.prepare(J.HIPBackend(), J.SpMVOp, A)
        return st
    m, n = _shape(case)
    rows, ptr, cols = _csr(case, gen)
    val = _normal(cols.numel(), dt, gen)
    if kind == "convert":
        if case["dst"] == "bsr":
            # Every entry of the pattern a dense b x b block, as CSR.
            b = case["b"]
            lens = (ptr[1:] - ptr[:-1])
            r = torch.repeat_interleave(torch.arange(m * b, device=DEV), lens.repeat_interleave(b) * b)
            ptr = torch.cat((ptr.new_zeros(1), (lens.repeat_interleave(b) * b).cumsum(0)))
            at = torch.arange(r.numel(), device=DEV) - ptr[r]
            first = torch.cumsum(lens, 0) - lens
            cols = cols[first[r // b] + at // b] * b + at % b
            rows, m, n = r, m * b, n * b
            val = _normal(cols.numel(), dt, gen)
            dst = J.Formats.BSRRight((b, b))
        else:
            dst = {"csr": J.Formats.CSR, "csc": J.Formats.CSC, "coo": J.Formats.COO}[case["dst"]]
        return dict(kind=kind, A=_tensor(case["src"], rows, ptr, cols, val, (m, n)), dst=dst)
    if kind == "spmv":
        A = _tensor(case["format"], rows, ptr, cols, val, (m, n))
        st = dict(kind=kind, A=A, x=_normal(n, dt, gen), y=torch.empty(m, dtype=dt, device=DEV))
        if case["call"] == "handle":
            st["h"] = J.prepare(J.HIPBackend(), J.SpMVOp, A)
        return st
    if kind == "spmm":
        A = _tensor(case["format"], rows, ptr, cols, val, (m, n))
        st = dict(kind=kind, A=A, B=_matrix(n, case["k"], dt, gen), C=J.dense_matrix(m, case["k"], dtype=dt, device=DEV))
        if case["call"] == "handle":
            st["h"] = J.prepare(J.HIPBackend(), J.SpMMOp, A, n_cols=case["k"])
        return st
    if kind == "sddmm":
        K = case["K"]
        # Values of the mask in [0.5, 1.5], in its storage order.
        mask = _tensor(case["format"], rows, ptr, cols,
                       torch.rand(cols.numel(), generator=gen, device=DEV, dtype=dt) + 0.5, (m, n))
        C = J.USTensor(mask.extents, mask.format, mask.pos_buffers, mask.crd_buffers, torch.empty_like(mask.val),
                       None, mask.origin)
        st = dict(kind=kind, C=C, mask=mask.val if case["masked"] else None,
                  A=_matrix(m, K, dt, gen), B=_matrix(K, n, dt, gen))
        if case["call"] == "handle":
            st["h"] = J.prepare(J.HIPBackend(), J.SDDMMOp, C, n_inner=K)
        return st
    # graph: A as CSR; its own buffers read as CSC are its transpose.
    K = case["K"]
    A = _tensor("csr", rows, ptr, cols, val, (m, n))
    At = J.csc_tensor(A.pos_buffers[1], A.crd_buffers[1], A.val, (n, m))
    G = J.csr_tensor(A.pos_buffers[1], A.crd_buffers[1], torch.empty_like(A.val), (m, n))
    X, dY = _matrix(n, K, dt, gen), _matrix(m, K, dt, gen)
    be = J.HIPBackend()
    return dict(kind=kind, h=J.prepare(be, J.SpMMOp, A, n_cols=K), ht=J.prepare(be, J.SpMMOp, At, n_cols=K),
                hg=J.prepare(be, J.SDDMMOp, G, n_inner=K), G=G, X=X, Xt=X.contiguous().t(), dY=dY,
                Y=J.dense_matrix(m, K, dtype=dt, device=DEV), dX=J.dense_matrix(n, K, dtype=dt, device=DEV))


# ------------------------------------------------------------------- one pass

def run(st):
    kind = st["kind"]
    if kind == "block":
        return J.mul_(st["y"], st["A"], st["x"])
    if kind == "spmv":
        if "h" in st:
            J.execute(st["h"], st["x"], st["y"])
        else:
            J.execute(J.SpMVOp, st["A"], st["x"], st["y"])
        return st["y"]
    if kind in ("spmm", "bsr_spmm"):
        if "h" in st:
            J.execute(st["h"], st["B"], st["C"])
        else:
            J.mul_(st["C"], st["A"], st["B"])
        return st["C"]
    if kind == "bsr_spmv":
        st["r"].copy_(st["b"])
        J.execute(st["h"] if "h" in st else J.SpMVOp, *(() if "h" in st else (st["A"],)), st["x"], st["r"],
                  alpha=-1.0, beta=1.0)
        return st["r"]
    if kind == "sddmm":
        if "h" in st:
            J.execute(st["h"], st["A"], st["B"], mask=st["mask"])
        else:
            J.execute(J.SDDMMOp, st["A"], st["B"], st["C"], mask=st["mask"])
        return st["C"].val
    if kind == "graph":
        J.execute(st["h"], st["X"], st["Y"])
        J.execute(st["ht"], st["dY"], st["dX"])
        J.execute(st["hg"], st["dY"], st["Xt"])
        return dict(out=st["Y"], grad_features=st["dX"], grad_weights=st["G"].val)
    out = J.convert_format(st["A"], st["dst"])
    return [t for t in (*out.pos_buffers, *out.crd_buffers, out.val) if t is not None]


# ------------------------------------------------------------------- its cost

def work(case):
    """Every input read once, every output written once."""
    s, kind = (8 if case["dtype"] == "f64" else 4), case["kind"]
    if kind == "block":
        m, n, nnz = _size_of_block(case)
        return dict(bytes=s * (m + n) + (s + 4) * nnz + 4 * (case["bus"] + case["line"]),
                    flops=2.0 * nnz * case["periods"])
    m, n = _shape(case)
    nnz = _entries(case)
    if kind == "spmv":
        ptr = {"csr": 4 * m, "csc": 4 * n, "coo": 4 * nnz}[case["format"]]
        return dict(bytes=(s + 4) * nnz + ptr + s * (m + n), flops=2.0 * nnz)
    if kind == "spmm":
        ptr = {"csr": 4 * m, "csc": 4 * n, "coo": 4 * nnz}[case["format"]]
        return dict(bytes=(s + 4) * nnz + ptr + s * (m + n) * case["k"], flops=2.0 * nnz * case["k"])
    if kind == "sddmm":
        ptr = {"csr": 4 * m, "csc": 4 * n, "coo": 4 * nnz}[case["format"]]
        return dict(bytes=(4 + s + s * case["masked"]) * nnz + ptr + s * (m + n) * case["K"],
                    flops=2.0 * nnz * case["K"])
    if kind == "graph":
        # A, X, dY read once; Y, dX and the edge gradients written once.
        return dict(bytes=(4 + 2 * s) * nnz + 4 * m + 4 * s * m * case["K"], flops=6.0 * nnz * case["K"])
    if kind == "bsr_spmm":
        b = case["b"]
        return dict(bytes=(s * b * b + 4) * nnz + 4 * m + s * (m + n) * b * case["k"],
                    flops=2.0 * nnz * b * b * case["k"])
    if kind == "bsr_spmv":
        b = case["b"]
        return dict(bytes=(s * b * b + 4) * nnz + 4 * m + s * (2 * m + n) * b, flops=2.0 * nnz * b * b)
    entries = nnz * case.get("b", 1) ** 2
    side = {"csr": 4 * m * case.get("b", 1) + 4 * entries, "csc": 4 * n + 4 * entries, "coo": 8 * entries,
            "bsr": 4 * m + 4 * nnz}
    return dict(bytes=2 * s * entries + side[case["src"]] + side[case["dst"]], flops=0.0)


def tolerance(case):
    """Formats move values and indices as they are.  Sums are of a few to some
    hundreds of products of normal values, in any order, with or without
    fused multiply-adds.  Against 64 bits the results were up to 2.0e-7 (f32)
    and 7.1e-16 (f64) off, and single values up to 2.1e-6 and 5.2e-15, or
    1.5e-5 and 2.8e-14 in the rows of up to 100,000 entries that powerlaw
    holds; four times that is stated."""
    if case["kind"] == "convert":
        return "exact"
    long_rows = case.get("pattern") == "powerlaw"
    if case["dtype"] == "f32":
        return dict(rel=8e-7, max=6e-5 if long_rows else 8e-6)
    return dict(rel=3e-15, max=1.2e-13 if long_rows else 2.1e-14)


# ------------------------------------------------------------------- in 64 bits

def _f64(t):
    return t.double()


def _coo(u):
    """0-based rows and columns of a CSR, COO or CSC tensor, in storage order."""
    pos, crd = u.pos_buffers, u.crd_buffers
    if crd[0] is not None:
        return crd[0].long() - 1, crd[1].long() - 1
    ptr = pos[1].long()
    outer = torch.repeat_interleave(torch.arange(ptr.numel() - 1, device=DEV), ptr[1:] - ptr[:-1])
    inner = crd[1].long() - 1
    return (outer, inner) if u.format == J.Formats.CSR else (inner, outer)


def _product(rows, cols, val, B, m):
    """sum_k val[k] * B[cols[k], :] into row rows[k]; B is n x k in 64 bits."""
    Bt = B.contiguous()
    out = torch.zeros(m, Bt.shape[1], dtype=torch.float64, device=DEV)
    step = max(1, (1 << 25) // Bt.shape[1])
    for s in range(0, rows.numel(), step):
        e = slice(s, s + step)
        out.index_add_(0, rows[e], _f64(val[e])[:, None] * Bt[cols[e]])
    return out


def _sampled(rows, cols, A, B):
    """A[rows[k], :] . B[:, cols[k]] in 64 bits."""
    Ar, Bc = _f64(A).contiguous(), _f64(B).t().contiguous()
    step = max(1, (1 << 25) // Ar.shape[1])
    return torch.cat([(Ar[rows[s:s + step]] * Bc[cols[s:s + step]]).sum(1) for s in range(0, rows.numel(), step)])


def _blocks_times(st, case, B):
    """A*B for a BSR matrix, block by block."""
    mb, nb = _shape(case)
    b, A = case["b"], st["A"]
    ptr, cols = A.pos_buffers[1].long() - 1, A.crd_buffers[1].long() - 1
    rows = torch.repeat_interleave(torch.arange(mb, device=DEV), ptr[1:] - ptr[:-1])
    V = A.val.view(-1, b, b)
    V = V if case["row_major"] else V.transpose(1, 2)
    k = B.shape[1]
    Bb = B.contiguous().view(nb, b, k)
    out = torch.zeros(mb, b, k, dtype=torch.float64, device=DEV)
    step = max(1, (1 << 25) // (b * k))
    for s in range(0, rows.numel(), step):
        e = slice(s, s + step)
        X, P = Bb[cols[e]], _f64(V[e])
        out.index_add_(0, rows[e], sum(P[:, :, j, None] * X[:, j, None, :] for j in range(b)))
    return out.view(mb * b, k)


def exact(case, seed):
    kind = case["kind"]
    if kind == "convert":
        return None                              # nothing is computed: entries are moved
    st = prepare(case, seed)
    if kind == "block":
        blocks, neg, pos, d = _dcopf(case, seed)
        T, nv, nc = case["periods"], d["n_var"], d["n_con"]
        off_r, off_c = [0, d["n_bus"]], [0, d["n_gen"], d["n_gen"] + d["n_line"]]
        put = []
        for t in range(T):
            r0, c0 = t * (nc + d["n_gen"]), t * nv
            put += [(b, r0 + off_r[i], c0 + off_c[j]) for i, row in enumerate(blocks) for j, b in enumerate(row) if b]
            if t + 1 < T:
                put += [(neg, r0 + nc, c0), (pos, r0 + nc, c0 + nv)]
        rows, cols, vals = [], [], []
        for ((ptr, ci, v), mm, _), r0, c0 in put:
            rows.append(np.repeat(np.arange(mm), np.diff(ptr)) + r0)
            cols.append(ci.astype(np.int64) - 1 + c0)
            vals.append(v)
        up = lambda a: torch.from_numpy(np.concatenate(a)).to(DEV)  # noqa: E731
        return _product(up(rows), up(cols), up(vals), _f64(st["x"])[:, None], st["y"].numel())[:, 0]
    if kind == "spmv":
        return _product(*_coo(st["A"]), st["A"].val, _f64(st["x"])[:, None], st["y"].numel())[:, 0]
    if kind == "spmm":
        return _product(*_coo(st["A"]), st["A"].val, _f64(st["B"]), st["C"].shape[0])
    if kind == "sddmm":
        out = _sampled(*_coo(st["C"]), st["A"], st["B"])
        return out if st["mask"] is None else out * _f64(st["mask"])
    if kind == "graph":
        A = st["h"].u_A
        rows, cols = _coo(A)
        return dict(out=_product(rows, cols, A.val, _f64(st["X"]), st["Y"].shape[0]),
                    grad_features=_product(cols, rows, A.val, _f64(st["dY"]), st["dX"].shape[0]),
                    grad_weights=_sampled(rows, cols, st["dY"], st["Xt"]))
    if kind == "bsr_spmm":
        return _blocks_times(st, case, _f64(st["B"]))
    return _f64(st["b"]) - _blocks_times(st, case, _f64(st["x"])[:, None])[:, 0]
