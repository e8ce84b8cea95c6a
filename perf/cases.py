"""The work by which this framework's speed is followed: calls of its public
entry points (include/kkmx_paths.h) at the sizes its programs use.

Kinds of case, and what each stands for in use:

  step         the eight dispatches of the bandwidth benchmark (STREAM copy,
               scale, add, triad; int64 reduce max, min, sum; inclusive int32
               scan), from a few thousand indices, where a call is launch
               latency, to 2^28
  scan_reduce  the small plain method: FP64 sum, exclusive int32 -> int64
               scan with total, a std-algorithm scan with a user operator and
               a std-algorithm dot product that returns to the host
  layout       deep_copy between a LayoutLeft and a LayoutRight View
  stencil      a time loop of 7-point sweeps over MDRangePolicy<Rank<3>>
  spmv         CSR matrix-vector product over TeamPolicy with team scratch
  histogram    counts of Zipf-distributed keys
  scatter      bins[idx[i]] += vals[i], by atomic_add or through ScatterView
  sort         Kokkos::sort of keys that arrive in a buffer of their own
  sort_by_key  Kokkos::Experimental::sort_by_key of such keys and values
  binsort      BinSort over BinOp1D with the sort inside bins, and the
               permutation of one array of values
  batch        one replayed step of many reductions and scans of uneven size
"""
import ctypes
import math

import torch

import kokkos_amd as K
from kokkos_amd import workloads

SORT_TYPES = (torch.int32, torch.int64, torch.float32, torch.float64, torch.uint32, torch.uint64)


def listed():
    return [
        # a solver's inner vector operations on a small local domain: latency
        {"name": "step_small", "kind": "step", "n": 4099},
        # the headline workload: 2 GiB arrays, bandwidth
        {"name": "step_large", "kind": "step", "n": 1 << 28},
        # the plain method at its own size
        {"name": "scan_reduce", "kind": "scan_reduce", "n": 1 << 24},
        # handing a field to a library that wants the other layout
        {"name": "layout", "kind": "layout", "n0": 512, "n1": 512, "n2": 512, "to_right": True},
        # ten time steps of an explicit scheme
        {"name": "stencil", "kind": "stencil", "n": 512, "sweeps": 10},
        # one Krylov iteration's product, rows of uneven length
        {"name": "spmv", "kind": "spmv", "rows": 1 << 20, "lo": 4, "hi": 64},
        # counting skewed keys
        {"name": "histogram", "kind": "histogram", "n": 1 << 28, "bins": 65536},
        # particle-to-grid deposition: random FP64 accumulation
        {"name": "scatter", "kind": "scatter", "n": 1 << 26, "bins": 1 << 20, "view": False},
        # a large key sort
        {"name": "sort", "kind": "sort", "type": 0, "n": 1 << 28, "bits": 31},
        # reordering particles by a 64-bit cell code, a ragged number of them
        {"name": "sort_by_key", "kind": "sort_by_key", "type": 1, "value_bytes": 8, "n": 3000017, "bits": 62},
        # neighbour-list binning of particles by coordinate
        {"name": "binsort", "kind": "binsort", "n": 1 << 24, "bins": 1 << 20},
        # a step of 4096 uneven dispatches, captured and replayed
        {"name": "batch", "kind": "batch", "ops": 4096, "lo": 8.0, "hi": 20.0},
    ]


def _size(rng, lo, hi):
    """A whole number of [lo, hi], its logarithm uniform; a power of two in one draw of six."""
    n = int(math.exp(rng.uniform(math.log(lo), math.log(hi + 1))))
    if rng.random() < 1 / 6:
        n = 1 << (n.bit_length() - 1)
    return max(lo, min(hi, n))


def draw(rng):
    kind = rng.choice(["step", "scan_reduce", "layout", "stencil", "spmv", "histogram", "scatter", "sort",
                       "sort_by_key", "binsort", "batch"])
    c = {"kind": kind}
    if kind == "step":
        c["n"] = _size(rng, 1000, 1 << 28)
    elif kind == "scan_reduce":
        c["n"] = _size(rng, 1000, 1 << 26)
    elif kind == "layout":
        c["n0"], c["n1"], c["n2"] = (_size(rng, 16, 512) for _ in range(3))
        c["to_right"] = rng.random() < 0.5
    elif kind == "stencil":
        c["n"], c["sweeps"] = _size(rng, 24, 512), rng.randint(1, 10)
    elif kind == "spmv":
        c["rows"], c["lo"] = _size(rng, 1000, 1 << 20), rng.randint(1, 8)
        c["hi"] = _size(rng, 9, 64)
    elif kind == "histogram":
        c["n"], c["bins"] = _size(rng, 10000, 1 << 28), _size(rng, 64, 1 << 17)
    elif kind == "scatter":
        c["n"], c["bins"] = _size(rng, 10000, 1 << 26), _size(rng, 1000, 1 << 21)
        c["view"] = rng.random() < 0.5
    elif kind in ("sort", "sort_by_key"):
        c["type"] = rng.randrange(6)
        wide = c["type"] in (1, 3, 5)
        c["bits"] = rng.choice((16, 62 if wide else 31, 62 if wide else 31))
        if kind == "sort":
            c["n"] = _size(rng, 1000, 1 << (26 if wide else 28))
        else:
            c["value_bytes"] = rng.choice((4, 8))
            c["n"] = _size(rng, 1000, 1 << 25)
    elif kind == "binsort":
        c["n"], c["bins"] = _size(rng, 10000, 1 << 24), _size(rng, 100, 1 << 20)
    else:
        c["ops"] = _size(rng, 16, 4096)
        c["lo"] = rng.choice((4.0, 8.0))
        c["hi"] = rng.choice((12.0, 16.0, 20.0))
    return c


# ---------------------------------------------------------------- inputs
def _rand(g, n, lo=0.0, hi=1.0):
    return torch.rand(n, generator=g, device="cuda", dtype=torch.float64).mul_(hi - lo).add_(lo)


def _ints(g, n, lo, hi, dtype):
    return torch.randint(lo, hi, (n,), generator=g, device="cuda", dtype=dtype)


def _keys(g, n, type_, bits):
    """Sort keys: whole numbers over `bits` bits (signed types on both sides
    of zero unless the range is small), floating-point keys over [-1, 1) or
    whole values of the small range."""
    dt = SORT_TYPES[type_]
    if dt in (torch.float32, torch.float64):
        return _ints(g, n, 0, 1 << bits, torch.int64).to(dt) if bits <= 16 else _rand(g, n, -1.0, 1.0).to(dt)
    if bits <= 16 or dt in (torch.uint32, torch.uint64):
        return _ints(g, n, 0, 1 << bits, torch.int64).to(dt)
    return _ints(g, n, -(1 << (bits - 1)), 1 << (bits - 1), dt)


def _inputs(c, seed):
    """The inputs of a case, from the seed alone."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    kind = c["kind"]
    if kind == "step":
        n = c["n"]
        return {"a": _rand(g, n, -1.0, 1.0), "x": _ints(g, n, -(1 << 40), (1 << 40) + 1, torch.int64),
                "s": _ints(g, n, 0, 8, torch.int32)}
    if kind == "scan_reduce":
        n = c["n"]
        return {"x": _rand(g, n), "y": _rand(g, n), "s": _ints(g, n, 0, 16, torch.int32),
                "m": _ints(g, n, -(1 << 30), 1 << 30, torch.int32)}
    if kind == "layout":
        return {"x": _rand(g, c["n0"] * c["n1"] * c["n2"], -1.0, 1.0)}
    if kind == "stencil":
        return {"u": _rand(g, (c["n"] + 2) ** 3)}
    if kind == "spmv":
        rp = torch.zeros(c["rows"] + 1, device="cuda", dtype=torch.int64)
        torch.cumsum(_ints(g, c["rows"], c["lo"], c["hi"] + 1, torch.int64), 0, out=rp[1:])
        nnz = int(rp[-1])
        return {"rp": rp, "col": _ints(g, nnz, 0, c["rows"], torch.int32), "val": _rand(g, nnz, -1.0, 1.0),
                "x": _rand(g, c["rows"], -1.0, 1.0)}
    if kind == "histogram":
        cdf = torch.arange(1, c["bins"] + 1, device="cuda", dtype=torch.float64).pow_(-1.1).cumsum(0)
        cdf /= cdf[-1].clone()
        u = _rand(g, c["n"])
        return {"keys": torch.searchsorted(cdf, u, right=True, out_int32=True).clamp_(max=c["bins"] - 1)}
    if kind == "scatter":
        return {"vals": _rand(g, c["n"]), "idx": _ints(g, c["n"], 0, c["bins"], torch.int32)}
    if kind == "sort":
        return {"keys": _keys(g, c["n"], c["type"], c["bits"])}
    if kind == "sort_by_key":
        return {"keys": _keys(g, c["n"], c["type"], c["bits"]),
                "vals": _ints(g, c["n"], 0, 1 << 31, torch.int64 if c["value_bytes"] == 8 else torch.int32)}
    if kind == "binsort":
        return {"keys": _rand(g, c["n"]), "vals": _ints(g, c["n"], 0, 1001, torch.int64)}
    wl = workloads.batch_workload(c["ops"], 10, c["lo"], c["hi"])  # the ops stay, their values change
    tot = wl["in_tot"]
    return {"wl": wl, "i32": _ints(g, max(tot[0], 1), 0, 16, torch.int32),
            "i64": _ints(g, max(tot[1], 1), 0, 16, torch.int64), "f64": _rand(g, max(tot[2], 1))}


def _empty(n, dtype=torch.float64):
    return torch.empty(max(n, 1), device="cuda", dtype=dtype)


def _words(t):
    """A contiguous tensor's bytes copied into whole 8-byte words, and how many words."""
    w = (t.numel() * t.element_size() + 7) // 8
    b = torch.zeros(max(w, 1), device="cuda", dtype=torch.float64)
    b.view(torch.uint8)[: t.numel() * t.element_size()].copy_(t.view(torch.uint8))
    return b, w


class _Batch:
    """The planned batch of a case: the handle, and the arrays its ops use."""

    def __init__(self, P, i):
        self.P, self.i = P, i
        wl = i["wl"]
        ops = len(wl["n"])
        self.out_i = _empty(wl["out_tot"]["i64"], torch.int64).zero_()
        self.out_f = _empty(wl["out_tot"]["f64"]).zero_()
        self.res_i = torch.zeros(ops, device="cuda", dtype=torch.int64)
        self.res_f = torch.zeros(ops, device="cuda", dtype=torch.float64)
        torch.cuda.synchronize()
        h = ctypes.c_void_p()
        K.check(P.kkmx_batch_create(ctypes.byref(h)), P)
        self.h = h
        src = (i["i32"], i["i64"], i["f64"])
        for k in range(ops):
            t, n, op = int(wl["type"][k]), int(wl["n"][k]), int(wl["op"][k])
            x = src[t].data_ptr() + int(wl["in_off"][k]) * src[t].element_size()
            out, res = (self.out_f, self.res_f) if t == workloads.T_F64 else (self.out_i, self.res_i)
            y = out.data_ptr() + 8 * int(wl["out_off"][k]) if op == workloads.OP_SCAN_EXCL else None
            K.check(P.kkmx_batch_add(h, op, t, x, n, y, res.data_ptr() + 8 * k, 1.0, 0.0), P)
        K.check(P.kkmx_batch_plan(h, ctypes.byref(ctypes.c_int64())), P)

    def __del__(self):
        self.P.kkmx_batch_destroy(self.h)


def prepare(case, seed):
    P = K.init(0)
    i = _inputs(case, seed)
    kind = case["kind"]
    st = {"P": P, "case": case, "in": i}
    if kind == "step":
        n = case["n"]
        st.update(c=_empty(n), b=_empty(n), d=_empty(n), e=_empty(n), r=_empty(3, torch.int64), so=_empty(n, torch.int32))
    elif kind == "scan_reduce":
        n = case["n"]
        st.update(sum=_empty(1), ex=_empty(n, torch.int64), tot=_empty(1, torch.int64), mx=_empty(n, torch.int32))
    elif kind == "layout":
        st["out"] = _empty(i["x"].numel())
    elif kind == "stencil":
        st["v"] = i["u"].clone()  # both grids hold the boundary values
    elif kind == "spmv":
        st["y"] = _empty(case["rows"])
    elif kind == "histogram":
        st["bins"] = torch.empty((case["bins"] + 1) // 2 * 2, device="cuda", dtype=torch.int32)
    elif kind == "scatter":
        st["bins"] = _empty(case["bins"])
    elif kind in ("sort", "sort_by_key"):
        st["kw"], st["nk"] = _words(i["keys"])
        st["keys"] = torch.zeros_like(st["kw"])
        if kind == "sort_by_key":
            st["vw"], st["nv"] = _words(i["vals"])
            st["vals"] = torch.zeros_like(st["vw"])
    elif kind == "binsort":
        st.update(vals=_empty(case["n"], torch.int64), perm=_empty(case["n"], torch.int32))
    else:
        st["batch"] = _Batch(P, i)
    torch.cuda.synchronize()  # the inputs are there before another stream reads them
    return st


def run(st):
    P, c, i = st["P"], st["case"], st["in"]
    kind = c["kind"]

    def call(rc):
        if rc:
            K.check(rc, P)

    if kind == "step":
        n, a, x, r = c["n"], i["a"].data_ptr(), i["x"].data_ptr(), st["r"].data_ptr()
        cc, b, d, e = (st[k].data_ptr() for k in "cbde")
        call(P.kkmx_stream_copy(a, cc, n))
        call(P.kkmx_stream_scale(b, cc, n, 3.0))
        call(P.kkmx_stream_add(a, b, d, n))
        call(P.kkmx_stream_triad(e, b, d, n, 3.0))
        call(P.kkmx_reduce_i64(x, n, 2, r))
        call(P.kkmx_reduce_i64(x, n, 1, r + 8))
        call(P.kkmx_reduce_i64(x, n, 0, r + 16))
        call(P.kkmx_scan_incl_i32(i["s"].data_ptr(), st["so"].data_ptr(), n))
        return [st["c"], st["b"], st["d"], st["e"], st["r"], st["so"]]
    if kind == "scan_reduce":
        n, dot = c["n"], ctypes.c_double()
        call(P.kkmx_reduce_sum_f64(i["x"].data_ptr(), n, st["sum"].data_ptr()))
        call(P.kkmx_scan_excl_i32_i64(i["s"].data_ptr(), st["ex"].data_ptr(), n, st["tot"].data_ptr()))
        call(P.kkmx_std_inclusive_scan_max_i32(i["m"].data_ptr(), st["mx"].data_ptr(), n))
        call(P.kkmx_std_transform_reduce_dot_f64(i["x"].data_ptr(), i["y"].data_ptr(), n, 0.0, ctypes.byref(dot)))
        return [st["sum"], st["ex"], st["tot"], st["mx"], dot.value]
    if kind == "layout":
        to = int(c["to_right"])
        call(P.kkmx_deep_copy_f64(st["out"].data_ptr(), i["x"].data_ptr(), c["n0"], c["n1"], c["n2"], to, 1 - to))
        return st["out"]
    if kind == "stencil":
        call(P.kkmx_stencil7_sweeps(i["u"].data_ptr(), st["v"].data_ptr(), c["n"], c["sweeps"], 0.4, 0.1, 0, 0, 0))
        return [i["u"], st["v"]]
    if kind == "spmv":
        call(P.kkmx_spmv_csr(i["rp"].data_ptr(), i["col"].data_ptr(), i["val"].data_ptr(), i["x"].data_ptr(),
                             st["y"].data_ptr(), c["rows"], i["col"].numel(), 1, 0, 0))
        return st["y"]
    if kind == "histogram":
        b = st["bins"]
        call(P.kkmx_deep_fill_f64(b.data_ptr(), b.numel() // 2, 0.0))
        call(P.kkmx_histogram(i["keys"].data_ptr(), c["n"], b.data_ptr(), c["bins"], 3, 0))
        return b[: c["bins"]]
    if kind == "scatter":
        b = st["bins"]
        call(P.kkmx_deep_fill_f64(b.data_ptr(), c["bins"], 0.0))
        if c["view"]:
            call(P.kkmx_scatter_view_f64(i["vals"].data_ptr(), i["idx"].data_ptr(), c["n"], b.data_ptr(), c["bins"], 0))
        else:
            call(P.kkmx_scatter_add_f64(i["vals"].data_ptr(), i["idx"].data_ptr(), c["n"], b.data_ptr(), c["bins"]))
        return b
    if kind in ("sort", "sort_by_key"):
        keys = st["keys"]
        call(P.kkmx_deep_copy_f64(keys.data_ptr(), st["kw"].data_ptr(), st["nk"], 1, 1, 0, 0))
        if kind == "sort":
            call(P.kkmx_sort(keys.data_ptr(), c["n"], c["type"]))
            return keys.view(_plain(i["keys"].dtype))[: c["n"]]
        vals = st["vals"]
        call(P.kkmx_deep_copy_f64(vals.data_ptr(), st["vw"].data_ptr(), st["nv"], 1, 1, 0, 0))
        call(P.kkmx_sort_by_key(keys.data_ptr(), vals.data_ptr(), c["n"], c["type"], c["value_bytes"], 0))
        return [keys.view(_plain(i["keys"].dtype))[: c["n"]], vals.view(i["vals"].dtype)[: c["n"]]]
    if kind == "binsort":
        call(P.kkmx_deep_copy_f64(st["vals"].data_ptr(), i["vals"].data_ptr(), c["n"], 1, 1, 0, 0))
        call(P.kkmx_binsort_f64(i["keys"].data_ptr(), st["vals"].data_ptr(), c["n"], c["bins"], 0.0, 1.0, 1,
                                st["perm"].data_ptr()))
        return [st["vals"], st["perm"]]
    b = st["batch"]
    call(P.kkmx_batch_run(b.h, 2, 1))
    return [b.res_i, b.res_f, b.out_i, b.out_f]


def _plain(dtype):
    """Unsigned words are returned as signed ones of the same bits."""
    return {torch.uint32: torch.int32, torch.uint64: torch.int64}.get(dtype, dtype)


def work(case):
    """Bytes: every input element read once, every output element written once."""
    kind, n = case["kind"], case.get("n", 0)
    if kind == "step":
        b = n * (16 + 16 + 24 + 24 + 3 * 8 + 8)
    elif kind == "scan_reduce":
        b = n * (8 + 12 + 8 + 16)
    elif kind == "layout":
        b = 16 * case["n0"] * case["n1"] * case["n2"]
    elif kind == "stencil":
        b = 16 * n**3 * case["sweeps"]
    elif kind == "spmv":
        b = case["rows"] * (24 + 12 * (case["lo"] + case["hi"]) / 2)
    elif kind == "histogram":
        b = 4 * n + 4 * case["bins"]
    elif kind == "scatter":
        b = 12 * n + 8 * case["bins"]
    elif kind == "sort":
        b = 2 * n * (8 if case["type"] in (1, 3, 5) else 4)
    elif kind == "sort_by_key":
        b = 2 * n * ((8 if case["type"] in (1, 3, 5) else 4) + case["value_bytes"])
    elif kind == "binsort":
        b = n * (8 + 16 + 4)
    else:
        # sizes are log-uniform over [2^lo, 2^hi]; a third of the inputs are
        # 4-byte, half of the ops write 8-byte prefixes
        mean = (2 ** case["hi"] - 2 ** case["lo"]) / ((case["hi"] - case["lo"]) * math.log(2))
        b = case["ops"] * mean * (20 / 3 + 4)
    return {"bytes": float(b), "flops": 0.0}


def tolerance(case):
    """Whole numbers, copies and keys are exact.  Elementwise FP64 results are
    allowed one rounding more or less (fused or unfused multiply-add), sums
    another order of their terms."""
    kind = case["kind"]
    if kind == "step":
        return {"rel": 2.5e-16, "max": 1e-15}  # triad: one rounding of its product
    if kind == "scan_reduce":
        return {"rel": 1e-15, "max": 1e-15}  # sums of up to 2^26 positive values
    if kind == "stencil":
        return {"rel": 6e-16, "max": 1e-14}  # ten sweeps of seven-term sums
    if kind == "spmv":
        return {"rel": 1e-15, "max": 1e-14}  # sums of up to 64 products of both signs
    if kind == "scatter":
        return {"rel": 1e-15, "max": 4e-15}  # sums of positive values in any order
    if kind == "batch":
        return {"rel": 1e-15, "max": 1e-14}  # sums and prefixes of up to 2^20 positive values
    return "exact"


# ---------------------------------------------------------------- the same results by plain torch
def exact(case, seed):
    i = _inputs(case, seed)
    kind = case["kind"]
    if kind == "step":
        a = i["a"]
        x = i["x"]
        r = torch.stack([x.max(), x.min(), x.sum()])
        b = 3.0 * a
        d = a + b
        return [a, b, d, b + 3.0 * d, r, i["s"].cumsum(0, dtype=torch.int32)]
    if kind == "scan_reduce":
        s = i["s"].cumsum(0, dtype=torch.int64)
        return [i["x"].sum().reshape(1), s - i["s"], s[-1:], i["m"].cummax(0).values, float((i["x"] * i["y"]).sum())]
    if kind == "layout":
        n0, n1, n2 = case["n0"], case["n1"], case["n2"]
        if case["to_right"]:  # the first index is fastest in the source
            return i["x"].view(n2, n1, n0).permute(2, 1, 0).reshape(-1)
        return i["x"].view(n0, n1, n2).permute(2, 1, 0).reshape(-1)
    if kind == "stencil":
        m = case["n"] + 2
        u, v = i["u"].view(m, m, m), i["u"].clone().view(m, m, m)
        w = slice(1, m - 1)
        for _ in range(case["sweeps"]):
            s = u[w, w, : m - 2] + u[w, w, 2:] + u[w, : m - 2, w] + u[w, 2:, w] + u[: m - 2, w, w] + u[2:, w, w]
            v[w, w, w] = 0.4 * u[w, w, w] + 0.1 * s
            u, v = v, u
        if case["sweeps"] % 2:
            u, v = v, u
        return [u.reshape(-1), v.reshape(-1)]
    if kind == "spmv":
        rows = torch.repeat_interleave(torch.arange(case["rows"], device="cuda"), i["rp"][1:] - i["rp"][:-1])
        p = i["val"] * i["x"][i["col"].long()]
        return torch.zeros(case["rows"], device="cuda", dtype=torch.float64).index_add_(0, rows, p)
    if kind == "histogram":
        return torch.bincount(i["keys"], minlength=case["bins"]).to(torch.int32)
    if kind == "scatter":
        return torch.zeros(case["bins"], device="cuda", dtype=torch.float64).index_add_(0, i["idx"], i["vals"])
    if kind in ("sort", "sort_by_key"):
        k = i["keys"]
        if k.dtype in (torch.uint32, torch.uint64):  # all below 2^62: the order of signed words
            k = k.view(torch.int32 if k.dtype == torch.uint32 else torch.int64)
        k, at = torch.sort(k, stable=True)
        return k if kind == "sort" else [k, i["vals"][at]]
    if kind == "binsort":
        at = torch.sort(i["keys"], stable=True).indices
        return [i["vals"][at], at.to(torch.int32)]
    return None  # thousands of ops of two kinds and three types


if __name__ == "__main__":
    for c in listed():
        print(c["name"], work(c)["bytes"])
