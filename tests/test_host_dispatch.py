"""The host side of dispatches, without a GPU: libkkmx_paths.so on a stand-in
for the runtime that records launches (tests/cpp/host_runtime.cpp).  Each test
runs in a process of its own, as the stand-in takes the runtime's place."""
import os
import shutil
import subprocess
import sys
import textwrap
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
PATHS = ROOT / "kokkos_amd" / "lib" / "libkkmx_paths.so"
CXX = shutil.which("g++") or shutil.which("c++")

PRELUDE = """
import ctypes as C, sys
H = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)
H.host_kernel.restype = H.host_label.restype = C.c_char_p
H.host_grid.restype = H.host_block.restype = C.c_uint64
H.host_held.restype = C.c_size_t
P = C.CDLL(sys.argv[2], mode=C.RTLD_GLOBAL)
P.kkmx_last_error.restype = P.kkmx_stream.restype = C.c_void_p
at = lambda a: C.c_void_p(a)  # addresses that no launch reads here
i64, f64, size = C.c_int64, C.c_double, C.c_size_t
def launches():
    return [(H.host_kernel(i).decode(), H.host_grid(i), H.host_block(i)) for i in range(H.host_launches())]
def labels():
    return [H.host_label(i).decode() for i in range(H.host_labels())]
def start(cus=256):
    H.host_set_cus(cus)
    P.kkmx_init(0)
    assert P.kkmx_stream()
    H.host_clear()
"""


@pytest.fixture(scope="module")
def runtime(tmp_path_factory):
    if not CXX or not PATHS.exists():
        pytest.skip("no host compiler, or the libraries are not built")
    so = tmp_path_factory.mktemp("host_runtime") / "libkkmx_rt.so"
    # the name by which libkkmx_paths.so asks for its runtime
    cmd = [CXX, "-std=c++17", "-O1", "-Wall", "-shared", "-fPIC", "-Wl,-soname,libkkmx_rt.so", "-I", str(ROOT / "include"),
           str(ROOT / "tests" / "cpp" / "host_runtime.cpp"), "-o", str(so), "-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr[-4000:]
    return so


def run(runtime, body, tools=()):
    env = dict(os.environ)
    env.pop("KOKKOS_TOOLS_LIBS", None)
    if tools:
        env["KOKKOS_TOOLS_LIBS"] = ";".join(map(str, tools))
    r = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(body), str(runtime), str(PATHS)],
                       capture_output=True, text=True, timeout=120, env=env)
    assert r.returncode == 0, r.stdout[-2000:] + r.stderr[-4000:]


@pytest.mark.parametrize("m", [(1 << 22) - 1, 1 << 22, (1 << 22) + 1, (1 << 23) + 5, 40_000_000])
@pytest.mark.parametrize("to_right", [1, 0])
def test_transpose_of_many_tiles(runtime, m, to_right):
    """16 x m x 16 doubles are m tiles.  A launch has fewer than 2^32 lanes, and
    the launches together have m workgroups."""
    run(runtime, f"""
        start()
        rc = P.kkmx_deep_copy_f64(at(1 << 46), at(1 << 45), i64(16), i64({m}), i64(16), {to_right}, {1 - to_right})
        got = launches()
        assert rc == 0 and got
        assert all('k_layout_transpose' in k for k, _, _ in got), got
        assert all(grid * block < 1 << 32 for _, grid, block in got), got
        assert sum(grid for _, grid, _ in got) == {m}, got
    """)


@pytest.mark.parametrize("across,along,middle,narrow", [
    (16, 16, 9999, 1), (512, 24, 100, 1), (48, 31, 999, 1), (512, 32, 100, 1), (16, 33, 1985, 1), (16, 33, 1986, 0),
    (512, 64, 31, 1), (512, 64, 32, 0), (100, 65, 999, 0), (16, 72, 999, 1), (512, 96, 99, 1), (512, 104, 99, 0),
    (512, 128, 99, 0), (47, 136, 999, 0), (48, 136, 999, 1), (512, 224, 99, 1), (512, 256, 99, 0), (512, 300, 99, 0),
    (63, 512, 99, 0), (64, 512, 99, 1), (512, 512, 3, 1), (512, 512, 9, 1), (512, 1000, 3, 0)])
def test_transpose_tiles(runtime, across, along, middle, narrow):
    """Which shapes of doubles take tiles of 64 x 32, in either direction."""
    run(runtime, f"""
        start()
        for right in (1, 0):
            e0, e2 = ({across}, {along}) if right else ({along}, {across})
            H.host_clear()
            assert P.kkmx_deep_copy_f64(at(1 << 46), at(1 << 45), i64(e0), i64({middle}), i64(e2), right, 1 - right) == 0
            (kernel, grid, block), = launches()
            n = 32 if {narrow} else 64
            assert f'k_layout_transposeImLb{{right}}ELi{{n}}E' in kernel, kernel
            assert grid == {middle} * -(-{across} // 64) * -(-{along} // n)
    """)


@pytest.mark.parametrize("nbins", [65536, 100000])
def test_histogram_rows_stay(runtime, nbins):
    """A call with few keys makes the table that one with many keys uses: a
    graph that captured the former keeps its address."""
    run(runtime, f"""
        start()
        for n in (1000, 1 << 18, 1 << 22, 1 << 24):
            assert P.kkmx_histogram(at(1 << 45), i64(n), at(1 << 46), {nbins}, 3, 0) == 0
            assert H.host_allocs() == (1 if n == 1000 else 0), (n, H.host_allocs())
            H.host_clear()
    """)


@pytest.mark.parametrize("n,nbins,teams", [
    (1, 65536, 1), (13107, 65536, 1), (13108, 65536, 2), (1 << 18, 65536, 21), (1 << 22, 65536, 256),
    (1024, 1000, 1), (1025, 1000, 2), (100000, 1000, 98), (1 << 18, 300, 256), (2000, 100000, 1), (2001, 100000, 2),
    (100000, 100000, 50), (1 << 20, 100000, 256)])
def test_histogram_teams(runtime, n, nbins, teams):
    """Teams by what a row of bins costs against keys that all meet in one
    counter, in LDS (up to about 70000 bins) and in the team's row."""
    run(runtime, f"""
        start()
        assert P.kkmx_histogram(at(1 << 45), i64({n}), at(1 << 46), {nbins}, 3, 0) == 0
        assert launches()[0][1] == {teams} and len(launches()) == 2, launches()
    """)


@pytest.mark.parametrize("cus", [8, 24, 25, 32, 256])
def test_scatter_moves_by_summed_counts(runtime, cus):
    """However many segments the CUs give the move, its last kernel is told that
    the counts were summed; a sort's, where the launch before it did that."""
    run(runtime, f"""
        start({cus})
        def check():
            got = [k for k, _, _ in launches()]
            for i, k in enumerate(got):
                if 'k_radix_scatter' in k:
                    assert H.host_arg(i, H.host_args(i) - 1) == ('k_radix_offsets' in got[i - 1]), got
            return sum('k_radix_scatter' in k for k in got), sum('k_radix_offsets' in k for k in got)
        assert P.kkmx_scatter_add_f64(at(1 << 45), at(1 << 46), i64(1 << 20), at(1 << 47), 1 << 20) == 0
        assert check() == (1, 1)
        H.host_clear()
        for n in (100000, 1 << 20, 1 << 24):
            assert P.kkmx_sort(at(1 << 45), i64(n), 0) == 0
        check()
    """)


def test_scatter_without_memory(runtime):
    """Without memory for its workspace the scatter-add runs by atomics, which
    need none, and takes the workspace up again once there is some."""
    run(runtime, """
        start()
        call = lambda: P.kkmx_scatter_add_f64(at(1 << 45), at(1 << 46), i64(1 << 24), at(1 << 47), 1 << 20)
        for limit, binned in ((1 << 20, False), (1 << 30, True)):
            H.host_set_limit(size(limit))
            H.host_clear()
            assert call() == 0
            got = launches()
            assert len(got) == (4 if binned else 1) and any('k_scatter_bins' in k for k, _, _ in got) == binned, got
        held = H.host_held()
        H.host_set_limit(size(0))
        assert call() == 0 and H.host_held() == held
    """)


@pytest.mark.parametrize("n,nbins", [(1000, 100), (1 << 18, 4096), (1 << 20, 4097), (1 << 25, 1 << 20)])
def test_scatter_is_one_dispatch_to_a_tool(runtime, n, nbins):
    run(runtime, f"""
        start()
        for limit in (1 << 40, 0):
            H.host_set_limit(size(limit))
            H.host_clear()
            assert P.kkmx_scatter_add_f64(at(1 << 45), at(1 << 46), i64({n}), at(1 << 47), {nbins}) == 0
            assert labels() == ['kkmx::scatter_f64'], labels()
    """, tools=[runtime])


def test_stencil_sweeps_and_tuning_tools(runtime, tmp_path):
    """Ten sweeps with the default tile: four pairs and two single sweeps, and
    ten MDRange dispatches, whose tile it chooses, where a tuning tool is loaded."""
    tuner = tmp_path / "libtuner.so"
    src = tmp_path / "tuner.c"
    src.write_text("void kokkosp_request_values(unsigned long a, unsigned long b, void* c, unsigned long d, void* e) {}")
    r = subprocess.run([CXX, "-x", "c", "-shared", "-fPIC", str(src), "-o", str(tuner)], capture_output=True, text=True)
    assert r.returncode == 0, r.stderr
    for tools, want in (([runtime], ["kkmx::stencil7_pair"] * 4 + ["kkmx::stencil7"] * 2),
                        ([runtime, tuner], ["kkmx::stencil7"] * 10)):
        run(runtime, f"""
            start()
            assert P.kkmx_stencil7_sweeps(at(1 << 45), at(1 << 46), i64(200), 10, f64(.4), f64(.1), 0, 0, 0) == 0
            assert labels() == {want}, labels()
        """, tools=tools)


@pytest.mark.parametrize("n,kept", [(1 << 25, 1 << 28), ((1 << 25) + 1024, 0)])
def test_binsort_keeps_no_large_values(runtime, n, kept):
    """Up to 256 MiB of values leave their scratch for the next call."""
    run(runtime, f"""
        start()
        before = H.host_held()
        assert P.kkmx_binsort_f64(at(1 << 45), at(1 << 46), i64({n}), 100, f64(0), f64(1), 0, None) == 0
        assert {kept} <= H.host_held() - before < {kept} + (1 << 20), H.host_held() - before
        assert sum('CopyRows' in k for k, _, _ in launches()) == 1, launches()
    """)
