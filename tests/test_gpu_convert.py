"""GPU format conversions (jlust_hip_convert_*, sparse_to_dense, shift_index)
against the numpy restatement of src/convert.jl (oracle/convert_oracle.py):
bit-exact index arrays and values, for every (source, target) pair of CSR,
CSC, COO, DCSR and BSR, both origins, f32/f64, with explicit zeros,
duplicates and empty rows; plus the reference's own expected arrays and
full-size round trips."""
import json
import os

import numpy as np
import pytest

from tests._util import dev, host

pytestmark = pytest.mark.gpu

GOLDEN = json.load(open(os.path.join(os.path.dirname(__file__), "golden",
                                     "reference_fixtures.json")))


@pytest.fixture(scope="module")
def J():
    import torch
    assert torch.cuda.is_available(), "GPU tests need a GPU"
    import jlust_amd
    return jlust_amd


@pytest.fixture(scope="module")
def CO():
    from oracle import convert_oracle
    return convert_oracle


def to_ust(J, d):
    """oracle dict -> device USTensor."""
    o = J.OneBased() if d["origin"] == 1 else J.ZeroBased()
    f, m, n = d["format"], d["m"], d["n"]
    if f == "CSR":
        return J.csr_tensor(dev(d["pos2"]), dev(d["crd2"]), dev(d["val"]), (m, n), origin=o)
    if f == "CSC":
        return J.csc_tensor(dev(d["pos2"]), dev(d["crd2"]), dev(d["val"]), (m, n), origin=o)
    if f == "COO":
        return J.coo_tensor(dev(d["crd1"]), dev(d["crd2"]), dev(d["val"]), (m, n), origin=o)
    if f == "DCSR":
        return J.dcsr_tensor(dev(d["crd1"]), dev(d["pos2"]), dev(d["crd2"]), dev(d["val"]), (m, n),
                             origin=o)
    return J.bsr_tensor(dev(d["pos2"]), dev(d["crd2"]), dev(d["val"]), (m, n), (d["b1"], d["b2"]),
                        row_major_blocks=d["row_major"], origin=o)


def fmt_of(J, name, b1=None, b2=None, rm=True):
    if name == "BSR":
        return J.Formats.BSRRight((b1, b2)) if rm else J.Formats.BSRLeft((b1, b2))
    return getattr(J.Formats, name)


def assert_same(J, u, d, what):
    """Device tensor u equals oracle dict d bit for bit."""
    f = d["format"]
    pos, crd = u.pos_buffers, u.crd_buffers
    lv2 = 1
    if f in ("CSR", "CSC", "DCSR", "BSR"):
        assert np.array_equal(host(pos[lv2]), d["pos2"]), what + " pos2"
        assert np.array_equal(host(crd[lv2]), d["crd2"]), what + " crd2"
    if f in ("COO", "DCSR"):
        assert np.array_equal(host(pos[0]), d["pos1"]), what + " pos1"
        assert np.array_equal(host(crd[0]), d["crd1"]), what + " crd1"
    if f == "COO":
        assert np.array_equal(host(crd[1]), d["crd2"]), what + " crd2"
    got, want = host(u.val), np.asarray(d["val"])
    assert got.dtype == want.dtype and got.shape == want.shape, what + " val shape"
    ui = np.uint64 if got.dtype == np.float64 else np.uint32
    assert np.array_equal(got.view(ui), want.view(ui)), what + " val bits"
    assert u.origin.offset == d["origin"]


def random_source(CO, seed, origin, dtype, m=24, n=20, b1=4, b2=2):
    """A CSR with explicit zeros, -0.0, an empty row band and a dense row; its
    COO with duplicates appended in row order."""
    rng = np.random.default_rng(seed)
    D = np.zeros((m, n))
    mask = rng.random((m, n)) < 0.25
    D[mask] = rng.standard_normal(mask.sum())
    D[5:9] = 0
    D[13] = rng.standard_normal(n)
    rows, cols = np.nonzero(D)
    vals = D[rows, cols].astype(dtype)
    z = rng.random(vals.size) < 0.15
    vals[z] = 0.0
    vals[np.flatnonzero(z)[::2]] = -0.0
    rowptr = np.searchsorted(rows, np.arange(m + 1)).astype(np.int32)
    csr = dict(format="CSR", origin=origin, m=m, n=n, pos2=rowptr + origin,
               crd2=(cols + origin).astype(np.int32), val=vals)
    # COO with duplicates: repeat some entries right after themselves.
    dup = rng.random(vals.size) < 0.2
    idx = np.sort(np.r_[np.arange(vals.size), np.flatnonzero(dup)], kind="stable")
    dv = vals[idx].copy()
    dv[np.r_[False, idx[1:] == idx[:-1]]] *= 3          # duplicates carry other values
    coo = dict(format="COO", origin=origin, m=m, n=n, crd1=(rows[idx] + origin).astype(np.int32),
               crd2=(cols[idx] + origin).astype(np.int32), val=dv.astype(dtype))
    return csr, coo


SOURCES = [("CSR", None), ("COO", None), ("CSC", None), ("DCSR", None), ("BSR", (4, 2, True)),
           ("BSR", (4, 2, False))]
TARGETS = [("CSR", ()), ("CSC", ()), ("COO", ()), ("DCSR", ()), ("BSR", (4, 2, True)),
           ("BSR", (2, 4, False)), ("BSR", (1, 1, True))]


@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("origin", [0, 1])
@pytest.mark.parametrize("src", SOURCES, ids=lambda s: s[0] + ("" if s[1] is None else str(s[1])))
def test_all_pairs_vs_oracle(J, CO, src, origin, dtype):
    csr, coo = random_source(CO, 7, origin, dtype)
    name, extra = src
    if name == "CSR":
        s = csr
    elif name == "COO":
        s = coo
    else:      # the source itself from the oracle (CSC, DCSR, BSR), explicit zeros dropped
        s = CO.convert_format(coo, name, *(extra or ()))
    u = to_ust(J, s)
    for tname, textra in TARGETS:
        want = CO.convert_format(s, tname, *textra)
        got = J.convert_format(u, fmt_of(J, tname, *textra))
        assert_same(J, got, want, f"{name}->{tname}{textra}")


def test_reference_arrays(J):
    """test/test_convert.jl:44-116 through the GPU path."""
    c = GOLDEN["convert"]
    u = J.csr_tensor(dev(np.int32(c["rowptr"])), dev(np.int32(c["colind"])),
                     dev(np.float32(c["val"])), (3, 4), origin=J.ZeroBased())
    w = J.convert_format(u, J.Formats.CSC)
    assert host(w.pos_buffers[1]).tolist() == c["csc_colptr"]
    assert host(w.crd_buffers[1]).tolist() == c["csc_rowind"]
    assert host(w.val).tolist() == c["csc_val"]
    q = J.convert_format(u, J.Formats.COO)
    assert host(q.pos_buffers[0]).tolist() == c["coo_pos"]
    assert host(q.crd_buffers[0]).tolist() == c["coo_rows"]
    for fmt in (J.Formats.CSC, J.Formats.COO, J.Formats.DCSR):
        back = J.convert_format(J.convert_format(u, fmt), J.Formats.CSR)
        assert host(back.pos_buffers[1]).tolist() == c["rowptr"]
        assert host(back.crd_buffers[1]).tolist() == c["colind"]
    g = GOLDEN["bsr_layout"]
    D = np.array(g["dense"])
    r, cc = np.nonzero(D)
    A = J.csr_tensor(dev(np.searchsorted(r, np.arange(5)).astype(np.int32) + 1),
                     dev((cc + 1).astype(np.int32)), dev(D[r, cc]), (4, 4))
    b = J.convert_format(A, J.Formats.BSRRight((2, 2)))
    assert host(b.pos_buffers[1]).tolist() == g["browptr"]
    assert host(b.crd_buffers[1]).tolist() == g["bcolind"]
    assert host(b.val).tolist() == g["val_row_major"]


def test_unsorted_rows_raise_for_csr_target(J):
    u = J.coo_tensor(dev(np.int32([3, 1, 2])), dev(np.int32([1, 2, 3])), dev(np.ones(3)), (3, 3))
    with pytest.raises(J.NonCanonicalStorage):
        J.convert_format(u, J.Formats.CSR)
    d = J.convert_format(u, J.Formats.DCSR)
    assert host(d.crd_buffers[0]).tolist() == [3, 1, 2]


def test_empty_and_all_zero(J, CO):
    for vals in (np.zeros(0), np.zeros(3)):
        k = vals.size
        u = J.csr_tensor(dev(np.int32([0, k, k])), dev(np.int32([0, 1, 2][:k])), dev(vals), (2, 3),
                         origin=J.ZeroBased())
        for fmt in (J.Formats.CSC, J.Formats.COO, J.Formats.DCSR, J.Formats.BSRRight((2, 3))):
            w = J.convert_format(u, fmt)
            assert w.val.numel() == 0


def test_errors(J):
    import torch
    u = J.csr_tensor(torch.tensor([1, 2], dtype=torch.int32), torch.tensor([1], dtype=torch.int32),
                     torch.ones(1, dtype=torch.float64), (1, 1))
    with pytest.raises(J.UnsupportedFormat, match="HIP device"):
        J.convert_format(u, J.Formats.CSC)
    g = J.csr_tensor(dev(np.int32([1, 2])), dev(np.int32([5])), dev(np.ones(1)), (1, 3))
    with pytest.raises(J.IncompatibleExtents, match="outside"):
        J.convert_format(g, J.Formats.CSC)
    b = J.csr_tensor(dev(np.int32([1, 2])), dev(np.int32([1])), dev(np.ones(1)), (3, 3))
    with pytest.raises(J.IncompatibleExtents, match="tile"):
        J.convert_format(b, J.Formats.BSRRight((2, 2)))


@pytest.mark.parametrize("name", ["CSR", "COO", "BSR"])
def test_sparse_to_dense(J, CO, name):
    csr, coo = random_source(CO, 3, 1, np.float64)
    # Without duplicates: the reference leaves their dense value undefined.
    s = {"CSR": csr, "COO": CO.convert_format(csr, "COO"),
         "BSR": CO.convert_format(csr, "BSR", 4, 2, False)}[name]
    D = J.sparse_to_dense(to_ust(J, s))
    assert np.array_equal(host(D), CO.to_dense(s))
    g = GOLDEN["to_dense"][0]
    u = J.csr_tensor(dev(np.int32(g["rowptr"])), dev(np.int32(g["colind"])), dev(np.float64(g["val"])),
                     (g["m"], g["n"]))
    assert host(J.sparse_to_dense(u)).tolist() == g["dense"]


def test_materialize_origin_shift_on_device(J):
    import torch
    c = GOLDEN["convert"]
    u = J.csr_tensor(dev(np.int32(c["onebased_rowptr"])), dev(np.int32(c["onebased_colind"])),
                     dev(np.float32(c["val"])), (3, 4))
    z = J.materialize(u, J.HIPDevice(0), origin=J.ZeroBased())
    assert host(z.pos_buffers[1]).tolist() == c["rowptr"]
    assert host(z.crd_buffers[1]).tolist() == c["colind"]
    h = J.materialize(z, J.CPUDevice(), origin=J.OneBased())         # shifted on the GPU first
    assert h.val.device.type == "cpu"
    assert h.pos_buffers[1].tolist() == c["onebased_rowptr"]
    cpu = J.csr_tensor(torch.tensor(c["rowptr"], dtype=torch.int32),
                       torch.tensor(c["colind"], dtype=torch.int32),
                       torch.tensor(c["val"], dtype=torch.float32), (3, 4), origin=J.ZeroBased())
    g = J.materialize(cpu, J.HIPDevice(0), origin=J.OneBased())       # moved, then shifted
    assert host(g.crd_buffers[1]).tolist() == c["onebased_colind"]


def test_config3_round_trip_full_size(J):
    """CSR -> CSC -> CSR at BASELINE config 3 (1M x 1M, 32M nonzeros) is the
    identity, bit for bit; CSC sampled against column extraction."""
    from jlust_amd import workloads as W
    cfg = W.make(3)
    u = J.csr_tensor(dev(cfg["rowptr"]), dev(cfg["colind"]), dev(cfg["val"]), (cfg["m"], cfg["n"]))
    c = J.convert_format(u, J.Formats.CSC)
    back = J.convert_format(c, J.Formats.CSR)
    assert np.array_equal(host(back.pos_buffers[1]), cfg["rowptr"])
    assert np.array_equal(host(back.crd_buffers[1]), cfg["colind"])
    assert np.array_equal(host(back.val).view(np.uint32), cfg["val"].view(np.uint32))
    colptr = host(c.pos_buffers[1])
    assert colptr[0] == 1 and colptr[-1] == cfg["colind"].size + 1
    rowind, cval = host(c.crd_buffers[1]), host(c.val)
    rng = np.random.default_rng(0)
    rows = np.repeat(np.arange(cfg["m"]), np.diff(cfg["rowptr"]))
    for j in rng.choice(cfg["n"], 8, replace=False):
        sel = cfg["colind"] == j + 1
        a, b = colptr[j] - 1, colptr[j + 1] - 1
        assert np.array_equal(rowind[a:b], rows[sel] + 1)
        assert np.array_equal(cval[a:b], cfg["val"][sel])


def test_config5_bsr_round_trip_full_size(J):
    """BSR (config 5, 134M values) -> CSR -> BSR is the identity when no stored
    value is zero (N(0,1) values)."""
    from jlust_amd import workloads as W
    cfg = W.make(5)
    assert not (cfg["val"] == 0).any()
    u = J.bsr_tensor(dev(cfg["browptr"]), dev(cfg["bcolind"]), dev(cfg["val"]), (cfg["m"], cfg["n"]))
    c = J.convert_format(u, J.Formats.CSR)
    assert c.val.numel() == cfg["val"].size
    b = J.convert_format(c, J.Formats.BSRRight((16, 16)))
    assert np.array_equal(host(b.pos_buffers[1]), cfg["browptr"])
    assert np.array_equal(host(b.crd_buffers[1]), cfg["bcolind"])
    assert np.array_equal(host(b.val).view(np.uint32), cfg["val"].view(np.uint32))


@pytest.mark.parametrize("dst", ["CSC", "COO", "DCSR", "BSR"])
def test_workspace_of_the_caller(J, CO, dst):
    """convert_analyze (the handle's own workspace) and convert_analyze_ws
    (the caller's) analyse alike; a workspace that is too small or not
    aligned is refused."""
    import ctypes
    import torch
    from jlust_amd import _lib
    from jlust_amd import convert as CV
    csr, _ = random_source(CO, 3, 1, np.float64)
    u = to_ust(J, csr)
    fid, b1, b2, rm = CV._format_id(fmt_of(J, dst, 4, 2))
    L, src = _lib.lib(), CV._descriptor(u)
    args = (ctypes.byref(src), fid, b1, b2, int(rm), 0)
    stream = CV._stream(u.val.device)

    def run(ws, size):
        h, nz, no = ctypes.c_void_p(), ctypes.c_int64(-1), ctypes.c_int64(-1)
        tail = (stream, ctypes.byref(h), ctypes.byref(nz), ctypes.byref(no))
        st = (L.jlust_hip_convert_analyze(*args, *tail) if size is None else
              L.jlust_hip_convert_analyze_ws(*args, ws, size, *tail))
        if h.value:
            L.jlust_hip_convert_destroy(h)
        return st, nz.value, no.value

    need = ctypes.c_int64()
    assert L.jlust_hip_convert_workspace(*args, ctypes.byref(need)) == 0 and need.value > 0
    buf = torch.empty(need.value + 256, dtype=torch.uint8, device="cuda")
    own = run(None, None)
    assert own[0] == 0 and run(buf.data_ptr(), need.value) == own
    assert run(buf.data_ptr(), need.value - 1)[0] != 0
    assert run(buf.data_ptr() + 8, need.value)[0] != 0
    assert run(None, need.value)[0] != 0
    got = J.convert_format(u, fmt_of(J, dst, 4, 2))
    assert got.val.numel() == own[1]


@pytest.mark.parametrize("src,dst", [("CSR", "CSC"), ("CSC", "CSR"), ("CSC", "COO")])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("origin", [0, 1])
def test_direct_equals_two_steps(J, src, dst, dtype, origin, monkeypatch):
    """convert_direct against the two-step conversion, bit for bit: one to
    three passes (coordinates below 2^11, 2^22, above), entries at the edges
    of 8,192-entry tiles, segments over several tiles, empty ones at either
    end, unordered and repeated coordinates, explicit zeros (-0.0), NaN, all
    zeros, and pointers that do not cover the entries (two steps)."""
    import torch
    from jlust_amd import convert as CV
    rng = np.random.default_rng(17)
    direct, taken = CV._convert_direct, []

    def recorded(*a):
        r = direct(*a)
        taken.append(r is not None)
        return r

    def run(nseg, ncoord, lens, repeat=False, zeros=0.0, ptr=None):
        ends = np.r_[0, np.cumsum(lens)]
        n = int(ends[-1])
        p = (ends if ptr is None else ptr) + origin
        c = rng.integers(0, ncoord, n)
        if not repeat:                                      # distinct in each segment where they fit
            for s in np.flatnonzero(np.asarray(lens) <= ncoord):
                a, b = int(ends[s]), int(ends[s + 1])
                if b - a > 1 and ncoord < 100000:
                    c[a:b] = rng.permutation(ncoord)[:b - a]
        v = rng.standard_normal(n).astype(dtype)
        v[rng.random(n) < zeros] = -0.0
        if n > 3 and zeros < 1:
            v[2] = np.nan
        dims = (nseg, ncoord) if src == "CSR" else (ncoord, nseg)
        og = J.OneBased() if origin else J.ZeroBased()
        make = J.csr_tensor if src == "CSR" else CV.csc_tensor
        u = make(*(torch.from_numpy(t).cuda() for t in (p.astype(np.int32), (c + origin).astype(np.int32), v)),
                 dims, og)
        out = []
        for general in (False, True):
            with monkeypatch.context() as mp:
                mp.setattr(CV, "_convert_direct", (lambda *a: None) if general else recorded)
                out.append(J.convert_format(u, fmt_of(J, dst)))
        assert taken.pop() == (ptr is None)
        a, b = out
        assert a.val.numel() == b.val.numel()
        it = torch.int64 if dtype == np.float64 else torch.int32
        assert torch.equal(a.val.view(it), b.val.view(it))
        for x, y in zip((*a.pos_buffers, *a.crd_buffers), (*b.pos_buffers, *b.crd_buffers)):
            assert (x is None) == (y is None)
            if x is not None:
                assert torch.equal(x, y)

    spread = lambda n, k: np.bincount(rng.integers(0, k, n), minlength=k)      # noqa: E731
    for n, k, dim in ((1, 1, 1), (5, 3, 2), (8191, 700, 2048), (8192, 700, 2049), (8193, 9000, 100),
                      (3 * 8192 + 5, 5000, 70000), (70001, 300, 5000000)):
        run(k, dim, spread(n, k))
        run(k, dim, spread(n, k), repeat=True, zeros=0.1)
    run(40, 30000, np.r_[np.zeros(10, int), 20000, 0, 0, 9000, np.ones(16, int), np.zeros(10, int)])
    run(5, 9000, np.r_[3, 8192 - 3, 8192, 1, 0])
    run(3, 50, np.r_[20, 0, 30], zeros=1.0)
    run(4, 60, np.r_[20, 0, 30, 5], ptr=np.array([3, 20, 20, 40, 52]))
    run(4, 60, np.r_[20, 0, 30, 5], ptr=np.array([0, 30, 20, 50, 55]))


@pytest.mark.parametrize("b1,b2,rm", [(1, 1, True), (2, 2, False), (3, 3, True), (4, 4, True), (5, 2, False), (8, 8, True),
                                      (1, 8, True), (7, 1, False)])
@pytest.mark.parametrize("dtype", [np.float64, np.float32])
@pytest.mark.parametrize("origin", [0, 1])
def test_blocks_equal_two_steps(J, b1, b2, rm, dtype, origin, monkeypatch):
    """convert_blocks against the two-step conversion, bit for bit: dense and
    ragged blocks, explicit zeros (-0.0, whole blocks of them, the first entry
    of a block), NaN, empty block-rows, block-rows of 0, 1, 63 to 65 entries and
    more, the last block-row of a workgroup's four, and what it leaves to the
    two steps: unordered and repeated columns, pointers that do not cover the
    entries, block-rows past 2048 entries or 1024 blocks."""
    import torch
    from jlust_amd import convert as CV
    rng = np.random.default_rng(23)
    og = J.OneBased() if origin else J.ZeroBased()
    taken = []
    blocks = CV._convert_blocks

    def counted(*a):
        r = blocks(*a)
        taken.append(r is not None)
        return r

    def check(mb, nb, rows, path=True, zeros=0.0, ptr=None):
        """rows: the columns of each row, in storage order."""
        assert len(rows) == mb * b1
        ends = np.r_[0, np.cumsum([len(r) for r in rows])]
        c = np.concatenate([np.asarray(r, np.int64) for r in rows]) if ends[-1] else np.zeros(0, np.int64)
        v = rng.standard_normal(c.size).astype(dtype)
        z = rng.random(c.size) < zeros
        v[z] = 0.0
        v[np.flatnonzero(z)[::2]] = -0.0
        if c.size > 3 and zeros < 1:
            v[2] = np.nan
        p = (ends if ptr is None else ptr) + origin
        u = J.csr_tensor(*(torch.from_numpy(t).cuda() for t in (p.astype(np.int32), (c + origin).astype(np.int32), v)),
                         (mb * b1, nb * b2), og)
        out = []
        for f in (counted, lambda *a: None):
            with monkeypatch.context() as mp:
                mp.setattr(CV, "_convert_blocks", f)
                out.append(J.convert_format(u, fmt_of(J, "BSR", b1, b2, rm)))
        assert taken.pop() == path
        x, y = out
        it = torch.int64 if dtype == np.float64 else torch.int32
        assert torch.equal(x.pos_buffers[1], y.pos_buffers[1]) and torch.equal(x.crd_buffers[1], y.crd_buffers[1])
        assert torch.equal(x.val.view(it), y.val.view(it))

    def pick(n, k):
        return np.sort(rng.choice(n, min(k, n), replace=False))

    def dense(mb, nb, k):
        out = []
        for _ in range(mb):
            at = pick(nb, k)
            out += [(at[:, None] * b2 + np.arange(b2)).reshape(-1)] * b1
        return out

    for mb, nb, k in ((1, 1, 1), (3, 9, 4), (4, 40, 27), (5, 300, 70), (41, 60, 16)):
        full = min(k, 2048 // (b1 * b2))
        check(mb, nb, dense(mb, nb, full))
        check(mb, nb, dense(mb, nb, full), zeros=0.3)
        check(mb, nb, [pick(nb * b2, int(rng.integers(0, 2 * k))) for _ in range(mb * b1 - 1)] + [[nb * b2 - 1]],
              zeros=0.2)
    for n in (63, 64, 65, 129):                             # entries of a block-row, all in its last row
        check(3, 200, [[]] * (2 * b1 - 1) + [pick(200 * b2, n)] + [[]] * b1)
    check(4, 20, dense(4, 20, 7), zeros=1.0)
    wide = 1024
    check(2, 1030, dense(1, 1030, min(wide, 2048 // (b1 * b2))) + [[1]] * b1)
    check(2, 1030, dense(1, 1030, 1025) + [[1]] * b1, path=False)
    check(1, 9000, [pick(9000 * b2, 2049)] + [[]] * (b1 - 1), path=False)
    r = dense(2, 20, 9)
    r[0] = np.r_[3, 1] if b2 * 20 > 3 else r[0]
    check(2, 20, r, path=False)
    r = dense(2, 20, 9)
    r[-1] = np.r_[4, 4]
    check(2, 20, r, path=False)
    r = [np.array([0, 5])] * (4 * b1)
    check(4, 20, r, path=False, ptr=np.r_[1, np.arange(1, 4 * b1 + 1) * 2])


@pytest.mark.parametrize("src,dst", [("CSR", "CSC"), ("CSC", "CSR"), ("CSC", "COO")])
@pytest.mark.parametrize("gap", [4 * 8192 - 20, 4 * 8192 + 20, 20_000_000])
def test_direct_over_empty_segments(J, src, dst, gap, monkeypatch):
    """A long run of empty segments inside one tile of entries: bit for bit the
    two-step conversion, in a time of its order (a workgroup that walked 20M
    segments would take over 30 times as long)."""
    import time

    import torch
    from jlust_amd import convert as CV
    rng = np.random.default_rng(31)
    side = 700_000                                          # entries on either side, 1 or 2 a segment
    lens = np.concatenate([np.full(side // 2, 2), np.zeros(gap, np.int64), np.ones(side, np.int64), [0, 0]])
    ncoord = 90_000
    n = int(lens.sum())
    p, c = np.r_[0, np.cumsum(lens)] + 1, rng.integers(0, ncoord, n) + 1
    c[:side:2], c[1:side:2] = np.minimum(c[:side:2], ncoord - 1), np.minimum(c[:side:2], ncoord - 1) + 1
    dims = (lens.size, ncoord) if src == "CSR" else (ncoord, lens.size)
    make = J.csr_tensor if src == "CSR" else CV.csc_tensor
    u = make(*(torch.from_numpy(t).cuda() for t in (p.astype(np.int32), c.astype(np.int32), rng.standard_normal(n))),
             dims)
    direct, out, took = CV._convert_direct, [], []
    for general in (False, True):
        monkeypatch.setattr(CV, "_convert_direct", (lambda *a: None) if general else direct)
        best = 1e9
        for _ in range(3):
            torch.cuda.synchronize()
            t = time.perf_counter()
            r = J.convert_format(u, fmt_of(J, dst))
            torch.cuda.synchronize()
            best = min(best, time.perf_counter() - t)
        out.append(r)
        took.append(best)
    monkeypatch.setattr(CV, "_convert_direct", direct)
    assert CV._convert_direct(u, fmt_of(J, dst), CV._descriptor(u), CV._format_id(fmt_of(J, dst))[0], u.val.device)
    a, b = out
    for x, y in zip((*a.pos_buffers, *a.crd_buffers, a.val), (*b.pos_buffers, *b.crd_buffers, b.val)):
        assert (x is None) == (y is None) and (x is None or torch.equal(x, y))
    assert took[0] < 4 * took[1] + 1e-3
