"""Kokkos::sort (LSD radix sort on gfx950) and Kokkos::BinSort / BinOp1D
through the C ABI (algorithms/src/sorting/Kokkos_SortPublicAPI.hpp,
Kokkos_BinSortPublicAPI.hpp), checked against numpy on the same seeded
inputs: sorted keys bit-exact; BinSort's permutation equal to numpy's stable
argsort when keys are sorted within bins, and bin-monotone otherwise."""
import numpy as np
import pytest

import kokkos_amd as K

pytestmark = pytest.mark.gpu
TYPES = {0: np.int32, 1: np.int64, 2: np.float32, 3: np.float64, 4: np.uint32, 5: np.uint64}


def run(P, rc):
    K.check(rc, P)
    K.fence()


def keys_for(oracle, code, n, seed):
    dt = TYPES[code]
    if code in (2, 3):
        x = oracle.fill_uniform_f64(n, seed, -1e6, 1e6)
        x[::7] = np.round(x[::7])  # ties
        x[::11] *= -1e-30          # tiny magnitudes of both signs
        x[3::13] = 0.0             # signed zeros, interleaved: they compare
        x[5::26] = -0.0            # equal and keep their input order
        x[::97] = np.inf
        x[1::97] = -np.inf
        return x.astype(dt)
    r = oracle.fill_uniform_i64(n, seed, -(1 << 62), 1 << 62)
    if code in (0, 4):
        r = r >> 32
    if code == 0:
        r[::5] = r[::5] % 50       # many duplicates
    return r.astype(dt)


@pytest.mark.parametrize("code", sorted(TYPES))
@pytest.mark.parametrize("n", [1, 2, 1000, 4097, 1 << 20])
def test_sort_matches_numpy(paths, oracle, code, n):
    P = paths
    x = keys_for(oracle, code, n, 70 + code)
    D = K.DeviceBuffer.from_array(x)
    run(P, P.kkmx_sort(D.ptr, n, code))
    got = D.download(TYPES[code], n)
    want = np.sort(x, kind="stable")
    bits = {4: np.uint32, 8: np.uint64}[x.dtype.itemsize]
    assert np.array_equal(got.view(bits), want.view(bits))  # bitwise: -0.0 != +0.0 here


def test_sort_large_int32(paths, oracle):
    P = paths
    n = 1 << 26
    D = K.DeviceBuffer(n * 4)
    run(P, P.kkmx_fill_uniform_i32(D.ptr, n, 77, -(1 << 30), 1 << 30))
    x = D.download(np.int32, n)
    run(P, P.kkmx_sort(D.ptr, n, 0))
    assert np.array_equal(D.download(np.int32, n), np.sort(x))


@pytest.mark.parametrize("n,nbins", [(1, 4), (1000, 16), (1 << 20, 1 << 12)])
def test_binsort_within_bins_is_stable_argsort(paths, oracle, n, nbins):
    P = paths
    # keys on a 2^-16 grid: equal keys (16 per value at 2^20) must keep index
    # order; bins stay small, since the within-bin sort is an insertion sort
    # per bin (quadratic in the bin size, as in the reference)
    keys = np.floor(oracle.fill_uniform_f64(n, 81, 0.0, 1.0) * 65536.0) / 65536.0
    vals = np.arange(n, dtype=np.int64) * 3
    Kd, Vd, Pd = K.DeviceBuffer.from_array(keys), K.DeviceBuffer.from_array(vals), K.DeviceBuffer(n * 4)
    run(P, P.kkmx_binsort_f64(Kd.ptr, Vd.ptr, n, nbins, 0.0, 1.0, 1, Pd.ptr))
    perm = Pd.download(np.int32, n)
    ref = np.argsort(keys, kind="stable")
    assert np.array_equal(perm, ref)
    assert np.array_equal(Vd.download(np.int64, n), vals[ref])


@pytest.mark.parametrize("n", [1, 8193, (1 << 21) + 3])
@pytest.mark.parametrize("form", ["crowded", "pairs", "outside"])
def test_binsort_within_bins_forms(paths, oracle, n, form):
    """Keys crowded into one cell of the quantised range, keys that meet in
    pairs there, and keys that fall in no bin (NaN): the permutation is the
    stable order of the keys in every form (numpy puts NaN last, too)."""
    P = paths
    keys = oracle.fill_uniform_f64(n, 83, 0.0, 1.0)
    if form == "crowded":
        keys = 0.5 + keys * 1e-12
    elif form == "pairs":
        keys[1::2] = np.nextafter(keys[: n - n // 2][: len(keys[1::2])], -1.0)
    else:
        keys[n // 2] = np.nan
    vals = np.arange(n, dtype=np.int64) * 3
    Kd, Vd, Pd = K.DeviceBuffer.from_array(keys), K.DeviceBuffer.from_array(vals), K.DeviceBuffer(n * 4)
    run(P, P.kkmx_binsort_f64(Kd.ptr, Vd.ptr, n, 1000, 0.0, 1.0, 1, Pd.ptr))
    ref = np.argsort(keys, kind="stable")
    assert np.array_equal(Pd.download(np.int32, n), ref)
    assert np.array_equal(Vd.download(np.int64, n), vals[ref])


@pytest.mark.parametrize("nbins", [1, 3, 5000, 1 << 20])
@pytest.mark.parametrize("n", [2, 4096, 4097, 24 * 1024 + 1, 24 * 4096, 24 * 4096 + 1])
def test_binsort_sizes(paths, oracle, n, nbins):
    """Either side of the codes' sorts, each size right after a call that met a
    key in no bin."""
    P = paths
    for form in ("outside", "any"):
        keys = np.floor(oracle.fill_uniform_f64(n, 84, 0.0, 1.0) * 30000.0) / 30000.0
        if form == "outside":
            keys[0] = np.nan
        vals = np.arange(n, dtype=np.int64) * 3
        Kd, Vd, Pd = K.DeviceBuffer.from_array(keys), K.DeviceBuffer.from_array(vals), K.DeviceBuffer(n * 4)
        run(P, P.kkmx_binsort_f64(Kd.ptr, Vd.ptr, n, nbins, 0.0, 1.0, 1, Pd.ptr))
        ref = np.argsort(keys, kind="stable")
        assert np.array_equal(Pd.download(np.int32, n), ref)
        assert np.array_equal(Vd.download(np.int64, n), vals[ref])


def test_binsort_without_bin_sort_is_bin_monotone(paths, oracle):
    P = paths
    n, nbins = 1 << 18, 1000
    keys = oracle.fill_uniform_f64(n, 82, -5.0, 5.0)
    vals = np.arange(n, dtype=np.int64)
    Kd, Vd, Pd = K.DeviceBuffer.from_array(keys), K.DeviceBuffer.from_array(vals), K.DeviceBuffer(n * 4)
    run(P, P.kkmx_binsort_f64(Kd.ptr, Vd.ptr, n, nbins, -5.0, 5.0, 0, Pd.ptr))
    perm = Pd.download(np.int32, n)
    assert np.array_equal(np.sort(perm), np.arange(n))
    bins = (nbins / 10.0 * (keys[perm] + 5.0)).astype(np.int64)
    assert np.all(np.diff(bins) >= 0)
    assert np.array_equal(Vd.download(np.int64, n), vals[perm])


@pytest.mark.parametrize("code", sorted(TYPES))
@pytest.mark.parametrize("n", [1, 2, 4097, 1 << 20])
@pytest.mark.parametrize("vbytes", [4, 8])
def test_sort_by_key_is_stable(paths, oracle, code, n, vbytes):
    """Kokkos::Experimental::sort_by_key (Kokkos_SortByKeyPublicAPI.hpp:27-64):
    keys as numpy's stable sort (bitwise), values moved with their keys, and
    equal keys keeping their input order (values = input positions here)."""
    P = paths
    x = keys_for(oracle, code, n, 90 + code)
    vdt = np.uint32 if vbytes == 4 else np.uint64
    vals = (np.arange(n, dtype=np.uint64) * 2654435761 % (1 << 32)).astype(vdt)
    Dk, Dv = K.DeviceBuffer.from_array(x), K.DeviceBuffer.from_array(vals)
    run(P, P.kkmx_sort_by_key(Dk.ptr, Dv.ptr, n, code, vbytes, 0))
    order = np.argsort(x, kind="stable")
    bits = {4: np.uint32, 8: np.uint64}[x.dtype.itemsize]
    assert np.array_equal(Dk.download(TYPES[code], n).view(bits), x[order].view(bits))
    assert np.array_equal(Dv.download(vdt, n), vals[order])


# Edges of the radix sort's forms: rounds of a block's sort, runs with a ragged
# last one, the last size of the passes whose segments add up their counts
# themselves and the first that does not (48 tiles of 4096), several tiles per segment with a ragged last one, and both
# sides of the switch to larger tiles (2^21 keys).
@pytest.mark.parametrize("n", [1023, 1025, 8191, 8192, 8193, 12289, 48 * 4096, 48 * 4096 + 1, 1024 * 4096 + 5,
                               (1 << 21) - 1, 1 << 21, 3000017])
@pytest.mark.parametrize("code,vbytes", [(0, 0), (3, 0), (4, 4), (2, 8), (1, 8), (3, 4)])
def test_sort_edges(paths, oracle, n, code, vbytes):
    P = paths
    x = keys_for(oracle, code, n, 400 + code)
    bits = {4: np.uint32, 8: np.uint64}[x.dtype.itemsize]
    order = np.argsort(x, kind="stable")
    Dk = K.DeviceBuffer.from_array(x)
    if vbytes == 0:
        run(P, P.kkmx_sort(Dk.ptr, n, code))
    else:
        vdt = np.uint32 if vbytes == 4 else np.uint64
        Dv = K.DeviceBuffer.from_array(np.arange(n, dtype=vdt))
        run(P, P.kkmx_sort_by_key(Dk.ptr, Dv.ptr, n, code, vbytes, 0))
        assert np.array_equal(Dv.download(vdt, n), order.astype(vdt))
    assert np.array_equal(Dk.download(TYPES[code], n).view(bits), x[order].view(bits))


@pytest.mark.parametrize("form", ["any", "few", "equal", "ascending", "descending"])
@pytest.mark.parametrize("n", [2048, 2049, 4096, 4097, 24 * 1024, 24 * 1024 + 1, 7 * 4096 + 1, 24 * 4096, 24 * 4096 + 1])
@pytest.mark.parametrize("code,vbytes", [(0, 0), (1, 8), (2, 8), (3, 4), (4, 4), (5, 0)])
def test_sort_in_runs(paths, oracle, n, code, vbytes, form):
    """Either side of one block, of 24 runs of 1024 keys and of 24 runs of 4096;
    equal keys keep their order across runs."""
    P = paths
    x = keys_for(oracle, code, n, 500 + code)
    if form == "few":
        x = x[np.arange(n) * 7919 % 5]
    elif form == "equal":
        x[:] = x[0]
    elif form != "any":
        x = np.sort(x)[:: 1 if form == "ascending" else -1].copy()
    order = np.argsort(x, kind="stable")
    bits = {4: np.uint32, 8: np.uint64}[x.dtype.itemsize]
    Dk = K.DeviceBuffer.from_array(x)
    if vbytes == 0:
        run(P, P.kkmx_sort(Dk.ptr, n, code))
    else:
        vdt = np.uint32 if vbytes == 4 else np.uint64
        Dv = K.DeviceBuffer.from_array(np.arange(n, dtype=vdt))
        run(P, P.kkmx_sort_by_key(Dk.ptr, Dv.ptr, n, code, vbytes, 0))
        assert np.array_equal(Dv.download(vdt, n), order.astype(vdt))
    assert np.array_equal(Dk.download(TYPES[code], n).view(bits), x[order].view(bits))


def put_hidden_runs(oracle, r, m, runs, seed):
    """m of the int64 keys r become members of `runs` runs of about the same
    length that share all but their lowest 20 bits, at places that a sample of
    every (n // 4096)-th key does not touch."""
    n = len(r)
    hidden = np.flatnonzero(np.arange(n) % max(1, n // 4096) != 0)
    at = np.sort(hidden[np.argsort(oracle.fill_uniform_i64(len(hidden), seed, 0, 1 << 62), kind="stable")[:m]])
    base = oracle.fill_uniform_i64(runs, seed + 1, -(1 << 62), 1 << 62) & ~np.int64((1 << 20) - 1)
    r[at] = base[np.arange(m) % runs] | oracle.fill_uniform_i64(m, seed + 2, 0, (1 << 20) - 1)


@pytest.mark.parametrize("form", ["spread", "runs", "crowd", "one_long_run", "equal", "six_digits"])
@pytest.mark.parametrize("n", [8193, 100003, (1 << 21) + 5])
@pytest.mark.parametrize("code,vbytes", [(1, 0), (3, 0), (5, 8), (3, 4)])
def test_sort_of_8_byte_keys_by_their_highest_digits(paths, oracle, n, code, vbytes, form):
    """8-byte keys are sorted by their five highest digits that vary where
    those tell them apart: spread keys (no digits to spare), runs of up to 40
    keys that share them out of order, keys all crowded into few runs (seen in
    the sample: all digits), one run of 300 among spread keys (not seen, found
    at the end: sorted apart), many equal keys, and keys of six digits.  The
    smallest size takes the sort of few keys."""
    P = paths
    r = oracle.fill_uniform_i64(n, 500 + code, -(1 << 62), 1 << 62)
    low = oracle.fill_uniform_i64(n, 600 + code, 0, (1 << 20) - 1)
    if form == "runs":
        put_hidden_runs(oracle, r, n // 10, -(-(n // 10) // 40), 1000 + code)
    elif form == "crowd":
        r = (r[np.arange(n) % 7] & ~np.int64((1 << 20) - 1)) | low
        r[0] = -(1 << 62)
        r[1] = (1 << 62) - 1
    elif form == "one_long_run":
        put_hidden_runs(oracle, r, 300, 1, 1000 + code)
    elif form == "equal":
        r = r[np.arange(n) % 1009]
    elif form == "six_digits":
        r = r & ((1 << 48) - 1)
    x = r.view(np.float64) if code == 3 else r.astype(TYPES[code])
    if code == 3:
        x = np.where(np.isnan(x), 1.5, x)
    order = np.argsort(x, kind="stable")
    Dk = K.DeviceBuffer.from_array(x)
    if vbytes:
        vdt = np.uint32 if vbytes == 4 else np.uint64
        Dv = K.DeviceBuffer.from_array(np.arange(n, dtype=vdt))
        run(P, P.kkmx_sort_by_key(Dk.ptr, Dv.ptr, n, code, vbytes, 0))
        assert np.array_equal(Dv.download(vdt, n), order.astype(vdt))
    else:
        run(P, P.kkmx_sort(Dk.ptr, n, code))
    assert np.array_equal(Dk.download(TYPES[code], n).view(np.uint64), x[order].view(np.uint64))


# Runs of keys that share their five highest digits, out of sight of the sample
# that decides to sort by those: short ones, put in order in place, up to the
# longest of 63, and longer ones; of the latter, fewer keys than a block sorts
# (2048), just more, as many as are sorted apart (a fifth of all) and more.
@pytest.mark.parametrize("n,m", [(100003, 64), (100003, 2048), (100003, 2049), (100003, 20000), (100003, 20001),
                                 (100003, 90000), ((1 << 21) + 5, 400000), ((1 << 21) + 5, 1900000)])
@pytest.mark.parametrize("code,vbytes,run_length", [(1, 0, 64), (5, 8, 100), (3, 4, 3000), (1, 8, 63), (5, 0, 40),
                                                    (3, 8, 3), (1, 4, 2)])
def test_sort_of_8_byte_keys_with_hidden_runs(paths, oracle, n, m, code, vbytes, run_length):
    P = paths
    r = oracle.fill_uniform_i64(n, 700 + code, -(1 << 62), 1 << 62)
    # at least run_length keys each, or, of the short ones, at most
    put_hidden_runs(oracle, r, m, max(1, m // run_length) if run_length >= 64 else -(-m // run_length), 800 + code)
    x = r.view(np.float64) if code == 3 else r.astype(TYPES[code])
    if code == 3:
        x = np.where(np.isnan(x), 1.5, x)
    order = np.argsort(x, kind="stable")
    Dk = K.DeviceBuffer.from_array(x)
    for again in range(2):  # the second call finds the sort's state as the first left it
        if vbytes:
            vdt = np.uint32 if vbytes == 4 else np.uint64
            Dk.upload(x)
            Dv = K.DeviceBuffer.from_array(np.arange(n, dtype=vdt))
            run(P, P.kkmx_sort_by_key(Dk.ptr, Dv.ptr, n, code, vbytes, 0))
            assert np.array_equal(Dv.download(vdt, n), order.astype(vdt))
        else:
            Dk.upload(x)
            run(P, P.kkmx_sort(Dk.ptr, n, code))
        assert np.array_equal(Dk.download(TYPES[code], n).view(np.uint64), x[order].view(np.uint64))


@pytest.mark.parametrize("code", [0, 3])
def test_sort_by_key_with_comparator(paths, oracle, code):
    """The comparator overload (Kokkos_SortByKeyPublicAPI.hpp:67-108) with a
    greater-than comparator: descending keys, ties in input order."""
    P = paths
    n = 5000
    x = keys_for(oracle, code, n, 95)
    vals = np.arange(n, dtype=np.uint64)
    Dk, Dv = K.DeviceBuffer.from_array(x), K.DeviceBuffer.from_array(vals)
    run(P, P.kkmx_sort_by_key(Dk.ptr, Dv.ptr, n, code, 8, 1))
    # stable descending: sort by negated key; ties keep input order
    order = sorted(range(n), key=lambda i: -float(x[i]))
    assert np.array_equal(Dk.download(TYPES[code], n), x[order])
    assert np.array_equal(Dv.download(np.uint64, n), vals[order])


@pytest.mark.parametrize("code,lo,hi", [(0, 0, 1000), (0, -5, 5), (1, 0, 1 << 20), (4, 7, 8), (5, 0, 1 << 40),
                                        (1, -(1 << 40), -(1 << 39))])
@pytest.mark.parametrize("n", [4097, 1 << 20])
def test_small_range_keys_skip_constant_digits(paths, oracle, code, lo, hi, n):
    """Keys whose high (or all) digits are the same everywhere: those passes
    are skipped, with an odd or even number of passes left (the odd case takes
    in one skipped digit), or none at all; results equal numpy's stable sort and,
    for sort_by_key, its stable argsort."""
    P = paths
    dt = TYPES[code]
    x = oracle.fill_uniform_i64(n, 300 + code, lo, hi - 1).astype(dt)
    D = K.DeviceBuffer.from_array(x)
    run(P, P.kkmx_sort(D.ptr, n, code))
    assert np.array_equal(D.download(dt, n), np.sort(x, kind="stable"))
    vals = np.arange(n, dtype=np.uint32)
    Dk, Dv = K.DeviceBuffer.from_array(x), K.DeviceBuffer.from_array(vals)
    run(P, P.kkmx_sort_by_key(Dk.ptr, Dv.ptr, n, code, 4, 0))
    order = np.argsort(x, kind="stable")
    assert np.array_equal(Dk.download(dt, n), x[order])
    assert np.array_equal(Dv.download(np.uint32, n), vals[order])


def test_float_keys_with_constant_low_digits_and_signed_zeros(paths, oracle):
    """Doubles that are small integers (their low mantissa bytes are zero in
    every key) and a mix of -0.0 and +0.0 only (equal keys: nothing moves,
    the input order stays)."""
    P = paths
    n = 100000
    x = (oracle.fill_uniform_i64(n, 310, 0, 7).astype(np.float64) - 3.0)
    x[::9] = -0.0
    D = K.DeviceBuffer.from_array(x)
    run(P, P.kkmx_sort(D.ptr, n, 3))
    want = np.sort(x, kind="stable")
    assert np.array_equal(D.download(np.float64, n).view(np.uint64), want.view(np.uint64))
    z = np.where(np.arange(n) % 3 == 0, -0.0, 0.0)
    vals = np.arange(n, dtype=np.uint64)
    Dk, Dv = K.DeviceBuffer.from_array(z), K.DeviceBuffer.from_array(vals)
    run(P, P.kkmx_sort_by_key(Dk.ptr, Dv.ptr, n, 3, 8, 0))
    assert np.array_equal(Dk.download(np.float64, n).view(np.uint64), z.view(np.uint64))
    assert np.array_equal(Dv.download(np.uint64, n), vals)
