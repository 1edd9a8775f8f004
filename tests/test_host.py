"""Host-side checks that need no GPU: the C-ABI library loads and exports what include/nplm_dwconv.h
declares, argument errors are reported before anything is launched, the workspace arithmetic, the
boundary cursor (run on the host over a host copy of cu_seqlens), the Python surface's validation,
and the workload generators."""
import ctypes
import os
import re

import numpy as np
import pytest
import torch

import nanoplm_amd
from nanoplm_amd import _lib
from nanoplm_amd.dwconv import exec_kernel_size
from nanoplm_amd.workloads import cu_from_lengths, make_workload, static_packed_cu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_library_exports_every_declared_symbol():
    header = open(os.path.join(ROOT, "include", "nplm_dwconv.h")).read()
    declared = set(re.findall(r"\b(nplm_dwconv_[a-z_]+)\s*\(", header))
    assert declared == set(_lib.PUBLIC_SYMBOLS)
    lib = ctypes.CDLL(_lib.LIB_PATH)
    for name in declared:
        assert hasattr(lib, name), name


def test_header_is_plain_c_and_a_c_program_links_and_calls_the_library(tmp_path):
    """include/nplm_dwconv.h compiles as strict C11 (no C++ left in it), every function it declares links from C against
    the shared object, and a C caller gets the version, the error strings, the workspace size and the argument errors
    (reported before anything is launched, so no GPU is needed)."""
    import shutil
    import subprocess
    if shutil.which("gcc") is None:
        pytest.skip("no C compiler")
    header = open(os.path.join(ROOT, "include", "nplm_dwconv.h")).read()
    names = sorted(set(re.findall(r"\b(nplm_dwconv_[a-z_]+)\s*\(", header)))
    src = tmp_path / "abi.c"
    src.write_text(
        "#include <stdio.h>\n#include <string.h>\n#include \"nplm_dwconv.h\"\n"
        "typedef void (*fn)(void);\n"
        "int main(void) {\n"
        "    fn all[] = {" + ", ".join(f"(fn){n}" for n in names) + "};\n"
        "    char fake[64];\n"
        "    void* a = (void*)(((size_t)fake + 15) & ~(size_t)15);   /* aligned, never dereferenced */\n"
        "    if (sizeof(all) / sizeof(all[0]) != " + str(len(names)) + ") return 10;\n"
        "    if (nplm_dwconv_version() < 100) return 11;\n"
        "    if (strcmp(nplm_dwconv_strerror(0), \"success\") != 0) return 12;\n"
        "    if (!strstr(nplm_dwconv_strerror(-NPLM_DWCONV_EKSIZE), \"odd\")) return 13;\n"
        "    if (nplm_dwconv_fwd(NULL, a, a, a, a, 128, 64, 3, 1, NPLM_DWCONV_BF16, NPLM_DWCONV_BF16, NULL) != -NPLM_DWCONV_ENULL) return 14;\n"
        "    if (nplm_dwconv_fwd(a, a, a, a, a, 128, 64, 4, 1, NPLM_DWCONV_BF16, NPLM_DWCONV_BF16, NULL) != -NPLM_DWCONV_EKSIZE) return 15;\n"
        "    if (nplm_dwconv_bwd(a, a, a, a, a, a, a, NULL, 0, 128, 64, 3, 1, NPLM_DWCONV_F32, NPLM_DWCONV_F32, NULL) != -NPLM_DWCONV_EWORKSPACE) return 16;\n"
        "    if (nplm_dwconv_fwd(NULL, NULL, NULL, NULL, NULL, 0, 64, 3, 0, NPLM_DWCONV_F32, NPLM_DWCONV_F32, NULL) != 0) return 17;   /* empty batch */\n"
        "    printf(\"%zu %zu\\n\", nplm_dwconv_bwd_workspace_bytes(131072, 1024, 7, NPLM_DWCONV_BF16), nplm_dwconv_bwd_workspace_bytes(131072, 1024, 11, NPLM_DWCONV_BF16));\n"
        "    return 0;\n}\n")
    exe = tmp_path / "abi"
    libdir = os.path.dirname(_lib.LIB_PATH)
    cc = subprocess.run(["gcc", "-std=c11", "-Wall", "-Wextra", "-Werror", "-pedantic", "-I", os.path.join(ROOT, "include"),
                         str(src), "-o", str(exe), "-L", libdir, "-l:" + os.path.basename(_lib.LIB_PATH), "-Wl,-rpath," + libdir,
                         "-Wl,-rpath-link,/opt/rocm/lib"], capture_output=True, text=True)
    assert cc.returncode == 0, cc.stderr
    run = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert run.returncode == 0, (run.returncode, run.stderr)
    lib = _lib.load()
    want = f"{lib.nplm_dwconv_bwd_workspace_bytes(131072, 1024, 7, 1)} {lib.nplm_dwconv_bwd_workspace_bytes(131072, 1024, 11, 1)}"
    assert run.stdout.strip() == want


def test_version_and_strerror():
    lib = _lib.load()
    assert lib.nplm_dwconv_version() >= 100
    assert _lib.strerror(0) == "success"
    for code in range(-8, 0):
        assert "nplm_dwconv" in _lib.strerror(code)


A = 0x10000   # a fake, well-aligned, never dereferenced device address


def _fwd(x=A, cu=A, w=A, b=A, y=A, T=128, C=64, K=3, S=1, act=1, wd=1):
    return _lib.load().nplm_dwconv_fwd(x, cu, w, b, y, T, C, K, S, act, wd, None)


def _bwd(x=A, dy=A, cu=A, w=A, dx=A, dw=A, db=A, ws=A, wsb=0, T=128, C=64, K=3, S=1, act=1, wd=1):
    return _lib.load().nplm_dwconv_bwd(x, dy, cu, w, dx, dw, db, ws, wsb, T, C, K, S, act, wd, None)


def test_argument_errors_are_reported_before_any_launch():
    assert _fwd(x=None) == -1 and _fwd(y=None) == -1 and _fwd(cu=None) == -1 and _fwd(w=None) == -1
    assert _fwd(T=-1) == -2 and _fwd(C=0) == -2 and _fwd(S=-1) == -2 and _fwd(T=2 ** 31) == -2
    assert _fwd(K=4) == -3 and _fwd(K=0) == -3 and _fwd(K=257) == -3
    assert _fwd(act=2) == -4 and _fwd(wd=7) == -4
    assert _fwd(x=A + 1) == -5 and _fwd(act=0, y=A + 2) == -5 and _fwd(wd=0, w=A + 2) == -5
    assert _fwd(T=0, x=None, y=None) == 0            # empty batch: nothing to do
    assert _bwd(dy=None) == -1 and _bwd(x=None) == -1 and _bwd(w=None) == -1
    assert _bwd(K=2) == -3 and _bwd(act=5) == -4 and _bwd(dx=A + 1) == -5
    assert _bwd(ws=None) == -6 and _bwd(ws=A + 64, wsb=1 << 30) == -6 and _bwd(wsb=16) == -6
    assert _bwd(dx=None, dw=None, db=None) == 0      # nothing requested


@pytest.mark.skipif(torch.cuda.is_available(), reason="the calls pass every check and would launch on made-up pointers")
def test_rows_too_wide_for_the_matrix_cores_tiles_keep_their_kernels():
    """Rows whose 64-row tiles pass the 2 GiB limit of a tile still take the kernels with shorter tiles, which refuse them at
    a limit of their own: without a GPU an accepted call ends with the runtime's (positive) error."""
    lib, p, bf16 = _lib.load(), 1 << 20, 1
    for K, C in ((11, 14_000_000), (15, 17_000_000), (15, 13_000_000)):
        assert lib.nplm_dwconv_fwd(p, p, p, None, p, 4096, C, K, 1, bf16, bf16, None) > 0
    for K, C, ok in ((31, 5_500_000, True), (31, 6_000_000, True), (31, 7_400_000, True), (31, 7_500_000, False)):
        rc = lib.nplm_dwconv_gated_bwd(p, p, p, p, p, p, p, p, 1 << 60, 4096, C, K, 1, bf16, bf16, 0, None)
        assert rc > 0 if ok else rc == -2, (C, rc)


def test_workspace_bytes_arithmetic():
    lib = _lib.load()
    for (T, C, K, act) in [(131072, 1024, 7, 1), (131072, 2048, 31, 1), (65536, 1024, 7, 1), (776, 64, 3, 0),
                           (1, 8, 1, 1), (1000, 1000, 11, 0)]:
        n = lib.nplm_dwconv_bwd_workspace_bytes(T, C, K, act)
        slabs = lib.nplm_dwconv_bwd_slabs(T, C, K, act, None)
        assert slabs >= 1
        # enough for the library's default kernel and for the sliding-window kernel that a request for dx alone or
        # dw/db alone may take instead (K = 31), and no more than the larger of the two
        most = max(slabs, lib.nplm_dwconv_bwd_slabs(T, C, K, act, _lib.Tuning(algo=1)))
        Kx = exec_kernel_size(K)        # K = 1 is planned as 3 taps and K = 11 as 15, with room for slabs of that many rows
        assert Kx == {7: 7, 31: 31, 3: 3, 1: 3, 11: 15}[K]
        assert n % 256 == 0 and n >= most * (Kx + 1) * C * 4 > n - 256
        assert n <= (16 << 20) + (Kx + 1) * C * 4       # partials are capped (one slab minimum)
    assert lib.nplm_dwconv_bwd_workspace_bytes(0, 64, 3, 1) == 0
    assert lib.nplm_dwconv_bwd_workspace_bytes(100, 64, 4, 1) == 0


def test_column_block_width_follows_the_row_width():
    """The LDS-staged backward deals one token block per CU and column block, so its slab count (256 / column
    blocks per row) shows which column-block width the planner picked: 1 KiB by default, 768 bytes for rows that
    are a multiple of that (C = 768, 1152 in bf16; 576 in fp32), 1280 bytes for rows of 1280 and 2560 bytes."""
    lib = _lib.load()
    lds = _lib.Tuning(algo=2)
    for (C, act, slabs) in [(1024, 1, 128), (2048, 1, 64), (512, 1, 256), (896, 1, 128), (768, 1, 128),
                            (1152, 1, 85), (640, 1, 256), (1280, 1, 128), (576, 0, 85), (512, 0, 128)]:
        assert lib.nplm_dwconv_bwd_slabs(131072, C, 7, act, lds) == slabs, (C, act)


# ---- boundary cursor ---------------------------------------------------------------------------
def _intervals(cu, T, start=0, step=1, relocate_every=0):
    cu = np.ascontiguousarray(np.asarray(cu, dtype=np.int32))
    n = max(0, (T - start + step - 1) // step)
    cs = np.full(n, -7, dtype=np.int32)
    ce = np.full(n, -7, dtype=np.int32)
    got = _lib.load().nplm_dwconv_debug_intervals(cu.ctypes.data, len(cu) - 1, T, start, step, relocate_every,
                                                  cs.ctypes.data, ce.ctypes.data)
    assert got == n
    return cs, ce


def _expected_intervals(cu, T):
    cs = np.empty(T, dtype=np.int32)
    ce = np.empty(T, dtype=np.int32)
    for s, e in zip(cu[:-1], cu[1:]):
        cs[s:e] = s
        ce[s:e] = e
    return cs, ce


def test_cursor_reproduces_the_reference_position_id_example():
    # src/nanoplm/pretraining/models/modern_bert/modeling.py:204: cu=[0,3,5,9] -> pos=[0,1,2,0,1,0,1,2,3]
    cs, ce = _intervals([0, 3, 5, 9], 9)
    assert (np.arange(9) - cs).tolist() == [0, 1, 2, 0, 1, 0, 1, 2, 3]
    assert ce.tolist() == [3, 3, 3, 5, 5, 9, 9, 9, 9]


@pytest.mark.parametrize("relocate_every", [0, 1, 5, 64])
@pytest.mark.parametrize("step", [1, 3, 8])
def test_cursor_on_random_cu_with_empty_sequences(step, relocate_every):
    rng = np.random.default_rng(1)
    for _ in range(20):
        lens = rng.integers(0, 12, size=rng.integers(1, 40))
        lens[rng.random(len(lens)) < 0.3] = 0
        if lens.sum() == 0:
            lens[0] = 3
        cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        T = int(cu[-1])
        want_cs, want_ce = _expected_intervals(cu, T)
        for start in (0, 1, T // 2):
            cs, ce = _intervals(cu, T, start, step, relocate_every)
            assert np.array_equal(cs, want_cs[start::step]) and np.array_equal(ce, want_ce[start::step])


def test_cursor_on_static_packed_cu():
    """Fixed-length cu_seqlens of the static-shape collator (collator.py:430-450): pad pseudo-sequences
    after the real ones and trailing zero-length entries equal to F."""
    real = cu_from_lengths(torch.tensor([30, 17, 64, 5]))
    F, W = 256, 64
    cu = static_packed_cu(real, F, W, cu_len=12).numpy()
    assert cu.tolist() == [0, 30, 47, 111, 116, 180, 244, 256, 256, 256, 256, 256]
    want_cs, want_ce = _expected_intervals(cu, F)
    for relocate_every in (0, 16):
        cs, ce = _intervals(cu, F, 0, 1, relocate_every)
        assert np.array_equal(cs, want_cs) and np.array_equal(ce, want_ce)


def test_cursor_never_leaves_the_array_on_malformed_cu():
    # rows before cu[0] and after cu[S] form pseudo-sequences; decreasing entries cannot loop forever
    cs, ce = _intervals([4, 6, 9], 12)
    assert cs.tolist() == [0] * 4 + [4, 4] + [6, 6, 6] + [9] * 3
    assert ce.tolist() == [4] * 4 + [6, 6] + [9, 9, 9] + [12] * 3
    cs, ce = _intervals([0], 5)              # S = 0: one pseudo-sequence [0, T)
    assert cs.tolist() == [0] * 5 and ce.tolist() == [5] * 5
    _intervals([0, 9, 3, 7, 2, 12], 12)      # decreasing: only termination is asserted
    _intervals([0, 50, 100], 12)             # entries beyond T


# ---- boundary walk of the matrix-core kernels -----------------------------------------------------
def _starts(cu, a, n):
    words = np.zeros(8, dtype=np.uint32)
    reads = _lib.load().nplm_dwconv_debug_starts(cu.ctypes.data, len(cu) - 1, int(cu[-1]), a, n, words.ctypes.data)
    assert reads >= 1
    bits = np.unpackbits(words.view(np.uint8), bitorder="little")[:n - 1]
    return (a + 1 + np.flatnonzero(bits)).tolist(), reads


def test_boundary_walk_marks_every_start_in_the_window():
    rng = np.random.default_rng(3)
    for _ in range(200):
        lens = rng.integers(0, rng.integers(2, 60), size=rng.integers(1, 400))
        cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
        T = int(cu[-1])
        for a in (-15, 0, 1, T // 2, max(T - 20, 0), T):
            n = int(rng.integers(2, 95))
            rows, _ = _starts(cu, a, n)
            assert rows == sorted({int(r) for r in cu if a < r < a + n})


def test_boundary_walk_of_the_largest_number_of_sequences():
    """S = 2^31 - 1, all but the last sequence empty: entry numbers of the probes need 32 bits. (The array is 8 GiB of address
    space, of which the walk touches a few hundred pages.)"""
    cu = np.zeros(2 ** 31, dtype=np.int32)
    cu[-1] = 64
    assert _starts(cu, 10, 60)[0] == [64]
    cu[-3:-1] = 30
    assert _starts(cu, 10, 60)[0] == [30, 64]
    assert _starts(cu, 30, 40)[0] == [64]


@pytest.mark.parametrize("front,inside,tail", [(0, 0, 70000), (0, 70000, 0), (70000, 0, 0), (5000, 3000, 9000)])
def test_boundary_walk_does_not_walk_runs_of_empty_sequences(front, inside, tail):
    """Empty sequences in front of the rows, between them and behind (the static collator's tail): read 64 at a time they would
    be over a thousand reads in the tiles that hold them."""
    T = 4096
    lens = [0] * front + [1000, 30] + [0] * inside + [7] + [0] * inside + [3, 2000, T - 3040] + [0] * tail
    cu = np.concatenate([[0], np.cumsum(lens)]).astype(np.int32)
    for a in [-15, 0] + list(range(49, T, 64)):
        rows, reads = _starts(cu, a, 94)
        assert rows == sorted({int(r) for r in cu if a < r < a + 94})
        # three probes find an entry among 2^18; the window has at most four starts, each with a read, a search and a read behind it
        assert reads <= 4 + 4 * 5


def test_boundary_walk_ends_on_malformed_cu():
    rng = np.random.default_rng(4)
    for _ in range(50):
        cu = rng.integers(-2 ** 31, 2 ** 31, size=rng.integers(1, 2000)).astype(np.int32)
        words = np.zeros(8, dtype=np.uint32)
        for a in (-15, 0, 1000, 2 ** 31 - 2 ** 20 - 64):
            reads = _lib.load().nplm_dwconv_debug_starts(cu.ctypes.data, len(cu) - 1, 2 ** 31 - 2 ** 20 - 1, a, 94, words.ctypes.data)
            assert 1 <= reads <= 5 * len(cu)


# ---- which kernels a call runs on ----------------------------------------------------------------
@pytest.mark.parametrize("bwd,T,C,K,S,algo", [
    (0, 4096, 256, 31, 1, 4), (0, 4095, 256, 31, 1, 3), (0, 4096, 248, 31, 1, 1), (0, 131072, 1024, 7, 500, 2), (1, 131072, 1024, 7, 500, 2),
    # rows of partial cache lines: forward of 11 and 15 taps from 200 MiB of output on, if their column blocks are filled to 3/5
    (0, 131072, 1000, 11, 500, 2), (0, 131072, 1000, 15, 500, 2), (0, 104000, 1000, 15, 400, 4), (0, 262144, 584, 15, 900, 4), (0, 131072, 1000, 21, 500, 4),
    (0, 131072, 1000, 31, 500, 4), (0, 131072, 1024, 11, 500, 4),
    # backward: rows a sequence, and rows of partial cache lines from 270 MiB on
    (1, 131072, 2048, 31, 4096, 4), (1, 131072, 2048, 31, 4097, 3), (1, 131072, 1024, 15, 2048, 4), (1, 131072, 1024, 15, 2049, 3),
    (1, 131072, 1024, 21, 256, 4), (1, 131072, 1024, 21, 257, 3), (1, 142000, 1000, 15, 500, 3), (1, 141000, 1000, 15, 500, 4), (1, 142000, 1000, 21, 100, 4),
    (1, 142000, 1000, 31, 500, 4), (1, 142000, 1000, 11, 100, 3), (1, 131072, 1000, 11, 100, 4)])
def test_which_kernels_a_bf16_call_takes(bwd, T, C, K, S, algo):
    assert _lib.load().nplm_dwconv_debug_algo(bwd, T, C, K, S, _lib.BF16, _lib.BF16) == algo
    assert _lib.load().nplm_dwconv_debug_algo(bwd, T, C, K, S, _lib.BF16, _lib.F32) in (1, 2, 3)


@pytest.mark.parametrize("bwd,T,C,K,S,algo", [
    # forward, up to 2048 rows: steps of 64 rows a block (T * C / 2^21), then rows a sequence (below 6; from 192 on)
    (0, 2048, 1024, 11, 100, 4), (0, 2048, 1152, 11, 100, 3), (0, 2048, 1152, 15, 100, 3), (0, 2048, 1152, 15, 342, 4), (0, 2048, 1152, 15, 341, 3),
    (0, 2048, 2048, 15, 10, 4), (0, 2048, 2048, 15, 11, 3), (0, 2048, 4096, 11, 128, 3), (0, 2048, 4096, 11, 1, 3), (0, 512, 8192, 11, 32, 3),
    (0, 1024, 2048, 13, 100, 4), (0, 2048, 2048, 21, 100, 4), (0, 2048, 2176, 21, 100, 3), (0, 2048, 4096, 21, 10, 4), (0, 2048, 4096, 21, 11, 3),
    (0, 1, 512, 15, 1, 4),
    # up to 16384 rows, and 31 taps
    (0, 2049, 512, 15, 10, 4), (0, 2049, 512, 15, 11, 3), (0, 16384, 4096, 21, 85, 4), (0, 16384, 512, 11, 86, 3), (0, 16385, 512, 15, 1, 3),
    (0, 16384, 8192, 31, 16384, 4), (0, 16385, 512, 31, 512, 4), (0, 16385, 512, 31, 513, 3), (0, 131072, 1000, 31, 500, 4), (0, 64, 512, 29, 64, 4),
    # backward: 31 taps; up to 4 tiles a block below 4096 rows, short calls and long sequences, whole cache lines from 30 MiB of output on
    (1, 2048, 4096, 31, 128, 4), (1, 4000, 4096, 31, 800, 3), (1, 4000, 4096, 31, 801, 4), (1, 4000, 4096, 31, 62, 4), (1, 4000, 4096, 31, 63, 3),
    (1, 4095, 2048, 31, 256, 4), (1, 4095, 2560, 31, 256, 3), (1, 4096, 2560, 31, 256, 4),
    (1, 1, 512, 31, 1, 4), (1, 16384, 512, 31, 16384, 4), (1, 16385, 512, 31, 85, 4), (1, 16385, 512, 31, 86, 3), (1, 16385, 512, 21, 1, 3),
    (1, 16384, 1000, 31, 1, 3), (1, 15700, 1000, 31, 1, 4), (1, 4096, 512, 15, 1, 3),
    # rows of less than 1 KiB, sizes with other kernels, none
    (0, 4096, 256, 31, 1, -10), (1, 4096, 256, 31, 1, 4), (0, 4096, 512, 7, 1, 2), (1, 4096, 512, 7, 1, 2), (0, 4096, 512, 33, 1, -10)])
def test_which_kernels_a_bf16_gated_call_takes(bwd, T, C, K, S, algo):
    assert _lib.load().nplm_dwconv_debug_gated_algo(bwd, T, C, K, S, _lib.BF16, _lib.BF16) == algo
    assert _lib.load().nplm_dwconv_debug_gated_algo(bwd, T, C, K, S, _lib.BF16, _lib.F32) == min(algo, 3)


@pytest.mark.parametrize("K", [11, 13])
def test_gated_forwards_of_11_to_15_taps_take_one_kernel_as_the_same_taps_padded_to_15(K):
    lib, rng = _lib.load(), np.random.default_rng(K)
    for _ in range(4000):
        T, C = int(np.exp(rng.uniform(0, np.log(200000)))), 8 * int(rng.integers(64, 1100))
        S = int(np.exp(rng.uniform(0, np.log(2 * T + 1))))
        assert lib.nplm_dwconv_debug_gated_algo(0, T, C, K, S, 1, 1) == lib.nplm_dwconv_debug_gated_algo(0, T, C, 15, S, 1, 1), (T, C, S)


# ---- Python surface -----------------------------------------------------------------------------
def test_cpu_tensors_are_refused():
    x = torch.randn(10, 8)
    cu = torch.tensor([0, 10], dtype=torch.int32)
    w = torch.randn(8, 3)
    with pytest.raises(RuntimeError, match="no CPU implementation"):
        nanoplm_amd.varlen_dwconv_fwd(x, cu, w)
    with pytest.raises(RuntimeError, match="no CPU implementation"):
        nanoplm_amd.VarlenDWConv1d(8, 3)(x, cu)
    with pytest.raises(RuntimeError, match="no CPU implementation"):
        nanoplm_amd.VarlenDWConv1dFunction.apply(x, cu, w, None)


def test_python_validation():
    cu = torch.tensor([0, 10], dtype=torch.int32)
    w = torch.randn(8, 3)
    from nanoplm_amd.dwconv import _validate
    with pytest.raises(ValueError):
        _validate(torch.randn(10), cu, w, None)
    with pytest.raises(TypeError):
        _validate(torch.randn(10, 8).half(), cu, w, None)
    with pytest.raises(ValueError):
        nanoplm_amd.VarlenDWConv1d(8, 4)
    m = nanoplm_amd.VarlenDWConv1d(16, 7)
    assert m.weight.shape == (16, 7) and m.bias.shape == (16,)
    assert nanoplm_amd.VarlenDWConv1d(16, 7, bias=False).bias is None


def test_missing_library_fails_loudly(monkeypatch):
    monkeypatch.setattr(_lib, "_lib", None)
    monkeypatch.setattr(_lib, "LIB_PATH", "/nonexistent/libnplm_dwconv.so")
    with pytest.raises(RuntimeError, match="is missing"):
        _lib.load()


@pytest.mark.parametrize("case", ["missing", "other symbols", "other version"])
def test_without_loadable_native_nodes_calls_are_left_to_the_python_route(monkeypatch, case):
    import types
    monkeypatch.setattr(_lib, "_node", None)
    if case == "missing":
        monkeypatch.setattr(_lib, "NODE_PATH", "/nonexistent/_node.so")
    else:
        def other(name):
            if case == "other symbols":
                raise ImportError("_node.so: undefined symbol: _ZN5torch3jit")
            return types.SimpleNamespace(torch_version="2.0.0")
        monkeypatch.setattr(_lib.importlib, "import_module", other)
    with pytest.warns(RuntimeWarning, match="native autograd nodes are not in use"):
        node = _lib.load_node()
    assert node.dwconv(*range(5)) is None and node.gated_dwconv(*range(5)) is None and node.ln_dwconv(*range(8)) is None
    assert _lib.load_node() is node
    with pytest.raises(RuntimeError, match="no CPU implementation"):          # (the Python route's own message)
        nanoplm_amd.VarlenDWConv1d(8, 3)(torch.randn(10, 8), torch.tensor([0, 10], dtype=torch.int32))


def test_native_nodes_are_for_the_torch_that_runs():
    node = _lib.load_node()
    assert node.__name__ == "nanoplm_amd._node" and node.torch_version == torch.__version__.split("+")[0]


@pytest.mark.parametrize("args", [["lib"], ["PYTHON=/nonexistent/python"], ["CXX=/nonexistent/g++"]])
def test_the_library_builds_without_python_torch_or_a_host_compiler(args):
    import subprocess
    out = subprocess.run(["make", "-n", "-B", "-C", os.path.join(ROOT, "nanoplm_amd", "csrc"), *args], capture_output=True, text=True)
    assert out.returncode == 0 and not out.stderr.strip(), out.stderr
    assert "-o ../libnplm_dwconv.so" in out.stdout and "node" not in out.stdout


def test_product_does_not_import_the_oracle():
    pkg = os.path.join(ROOT, "nanoplm_amd")
    for dirpath, _, files in os.walk(pkg):
        for f in files:
            if f.endswith((".py", ".h", ".hip", ".inc")):
                text = open(os.path.join(dirpath, f)).read()
                assert "oracle" not in text.lower() or f == "workloads.py", f


# ---- workloads ----------------------------------------------------------------------------------
def test_workload_generators_follow_the_config_definitions():
    w1 = make_workload(1)
    assert w1.S == 8 and w1.C == 64 and w1.K == 3 and w1.dtype == torch.float32 and w1.dy is None
    assert 20 <= int(w1.lengths.min()) and int(w1.lengths.max()) <= 128
    w2 = make_workload(2, C=16)
    assert w2.T == 32768 and w2.K == 7 and w2.dtype == torch.bfloat16 and w2.passes == "fwd"
    assert int(w2.lengths[:-1].min()) >= 20 and int(w2.lengths.max()) <= 512
    w5 = make_workload(5, C=8)
    assert w5.T == 65536 and w5.passes == "fwd+bwd" and w5.dy is not None
    ln = w5.lengths[:-1]
    short = ln <= 8
    assert bool(((ln >= 1) & (ln <= 8) | (ln >= 400) & (ln <= 512)).all())
    assert 0.5 < float(short.float().mean()) < 0.7
    w4 = make_workload(4, T=20000, C=8)
    assert w4.K == 31 and 20 <= int(w4.lengths[:-1].min()) and int(w4.lengths.max()) <= 1024
    for w in (w1, w2, w5, w4):
        cu = w.cu_seqlens
        assert cu.dtype == torch.int32 and int(cu[0]) == 0 and int(cu[-1]) == w.T and cu.numel() == w.S + 1
        assert bool((cu[1:] >= cu[:-1]).all())
    again = make_workload(2, C=16)
    assert torch.equal(again.x, w2.x) and torch.equal(again.cu_seqlens, w2.cu_seqlens)


def test_algorithmic_bytes_of_the_headline_config():
    w3 = make_workload(3, C=8)   # C shrunk for speed; the formula is checked at the real C by hand
    T, C, K, S, e = w3.T, w3.C, w3.K, w3.S, 2
    assert w3.algorithmic_bytes("fwd") == 2 * T * C * e + C * (K + 1) * e + 4 * (S + 1)
    assert w3.algorithmic_bytes("bwd") == 3 * T * C * e + C * K * e + 4 * C * (K + 1) + 4 * (S + 1)
    # at C=1024: 5*T*C*e = 1 342 177 280
    assert 5 * 131072 * 1024 * 2 == 1342177280


# ---- torch.library registration (traceability; no kernel is run) ------------------------------------
def test_custom_ops_trace_with_fake_tensors():
    """Schemas and fake (shape/dtype) implementations of the registered ops, without a GPU. The autograd
    formula needs a device context and is exercised by the GPU tests."""
    from torch._subclasses.fake_tensor import FakeTensorMode
    from torch.fx.experimental.proxy_tensor import make_fx

    assert str(torch.ops.nanoplm_amd.varlen_dwconv_fwd.default._schema) == (
        "nanoplm_amd::varlen_dwconv_fwd(Tensor x, Tensor cu_seqlens, Tensor weight, Tensor? bias, bool residual=False) -> Tensor")
    assert str(torch.ops.nanoplm_amd.varlen_dwconv_bwd.default._schema) == (
        "nanoplm_amd::varlen_dwconv_bwd(Tensor x, Tensor dy, Tensor cu_seqlens, Tensor weight, bool residual=False, bool grads_bf16=False) -> "
        "(Tensor, Tensor, Tensor)")
    with FakeTensorMode():
        x = torch.empty(100, 64, dtype=torch.bfloat16, device="cuda")
        cu = torch.empty(5, dtype=torch.int32, device="cuda")
        w = torch.empty(64, 7, dtype=torch.float32, device="cuda")
        b = torch.empty(64, dtype=torch.float32, device="cuda")
        y = nanoplm_amd.varlen_dwconv_compilable(x, cu, w, b)
        assert y.shape == x.shape and y.dtype == torch.bfloat16 and y.device.type == "cuda"
        dx, dw, db = nanoplm_amd.varlen_dwconv_bwd_op(x, y, cu, w)
        assert dx.shape == x.shape and dx.dtype == torch.bfloat16
        assert dw.shape == (64, 7) and dw.dtype == torch.float32 and db.shape == (64,) and db.dtype == torch.float32

    def f(x, cu, w):
        y = nanoplm_amd.varlen_dwconv_compilable(x, cu, w, None)
        return nanoplm_amd.varlen_dwconv_bwd_op(x, y, cu, w)

    with FakeTensorMode(allow_non_fake_inputs=True):
        args = (torch.empty(32, 16, device="cuda"), torch.empty(3, dtype=torch.int32, device="cuda"),
                torch.empty(16, 3, device="cuda"))
        gm = make_fx(f, tracing_mode="fake")(*args)
    targets = {str(n.target) for n in gm.graph.nodes if n.op == "call_function"}
    assert "nanoplm_amd.varlen_dwconv_fwd.default" in targets and "nanoplm_amd.varlen_dwconv_bwd.default" in targets
