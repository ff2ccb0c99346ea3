"""The library's host side without a GPU: a stand-in for the HIP runtime
(tests/native/host_runtime.cc) takes its calls, runs no kernel and keeps a
list of what was asked of it.

Each check runs in a process of its own, which loads the stand-in ahead of
libwgblas_hip.so."""
import json
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, json, sys
runtime = ctypes.CDLL({runtime!r}, ctypes.RTLD_GLOBAL)
runtime.standin_log.restype = ctypes.c_char_p
import wgblas_amd as wg
from wgblas_amd.native import WgblasError

P = 1 << 41  # a device address

def calls(f):
    "What f asked of the runtime, line by line, and the error that it raised, if any."
    runtime.standin_clear()
    error = None
    try:
        f()
    except WgblasError as e:
        error = str(e)
    return runtime.standin_log().decode().splitlines(), error

"""


@pytest.fixture(scope="module")
def child(tmp_path_factory):
    gxx, hipcc = shutil.which("g++"), shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    include = os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc))), "include")
    if gxx is None or not os.path.exists(os.path.join(include, "hip", "hip_runtime_api.h")):
        pytest.skip("g++ or the HIP headers are not available")
    so = str(tmp_path_factory.mktemp("runtime") / "host_runtime.so")
    subprocess.run([gxx, "-O1", "-std=c++17", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I", include,
                    os.path.join(HERE, "native", "host_runtime.cc"), "-o", so], check=True)

    def run(script):
        res = subprocess.run([sys.executable, "-c", PRELUDE.format(runtime=so) + script], cwd=ROOT,
                             capture_output=True, text=True, timeout=300)
        assert res.returncode == 0, res.stderr
        return json.loads(res.stdout)

    return run


@pytest.mark.parametrize("n", [1, 100_003, 1 << 28])  # one block, one launch, two launches
def test_a_host_result_that_never_arrives_is_an_error(child, n):
    """No kernel runs, so nothing stores the result: every host form has to say so instead of
    returning what the slot holds."""
    got = child(f"""
ctx, n, out = wg.Context(0), {n}, {{}}
for t in "sd":
    for op in ("dot", "asum", "nrm2", "amax"):
        name = "i" + t + op if op == "amax" else t + op
        args = (n, P, 1, P, 1) if op == "dot" else (n, P, 1)
        out[name] = calls(lambda: getattr(ctx, name)(*args))[1]
print(json.dumps(out))
""")
    assert len(got) == 8
    for name, error in got.items():
        assert error and "result" in error and "status -2" in error, (name, error)


def test_empty_vectors_need_no_result(child):
    got = child("""
ctx = wg.Context(0)
log, error = calls(lambda: None)
values = [float(ctx.sdot(0, None, 1, None, 1)), float(ctx.dnrm2(0, None, 1)), ctx.isamax(0, None, 1)]
print(json.dumps([values, calls(lambda: ctx.sasum(0, None, 1))]))
""")
    assert got == [[0.0, 0.0, -1], [[], None]]


def test_a_captured_reduction_keeps_no_arrival_count(child):
    """A captured graph may be replayed on another stream, beside the context's own calls, and a
    count that two launches share would stay wrong for good: under capture the blocks' partials are
    folded by a second launch. One block has nothing to count."""
    got = child("""
ctx, out = wg.Context(0), []
for capturing in (0, 1, 0):
    runtime.standin_capture(capturing)
    for n, inc in ((4096, 1), (100_003, 1), (100_003, 3), (100_003, 5), (1 << 22, 1)):
        log, error = calls(lambda: ctx.ddot_dev(n, P, inc, P, inc, P))
        assert error is None, error
        out.append([capturing, n, ["fold_kernel" in line for line in log if line.startswith("launch")]])
print(json.dumps(out))
""")
    assert len(got) == 15
    for capturing, n, launches in got:
        two = n == 1 << 22 or (capturing and n > 4096)
        assert launches == ([False, True] if two else [False]), (capturing, n, launches)


def test_a_captured_host_result_ends_the_capture(child):
    """The host forms do not ask whether the stream is capturing: their wait for it is refused there."""
    got = child("""
ctx = wg.Context(0)
runtime.standin_capture(1)
print(json.dumps(calls(lambda: ctx.sasum(100_003, P, 1))))
""")
    assert got[0][-1] == "synchronize" and "status -2" in got[1], got


def test_a_missing_result_clears_the_arrival_count(child):
    """The next call starts from 0 whatever kept this one from storing its result."""
    got = child("""
ctx = wg.Context(0)
print(json.dumps(calls(lambda: ctx.sasum(100_003, P, 1))[0]))
""")
    kinds = [line.split()[0] for line in got]
    assert kinds == ["launch", "synchronize", "launch"], got
    assert "set_value" in got[2], got


def test_the_result_slot_is_coherent_memory(child):
    """A kernel's stores to the slot are read while its stream goes on, which only coherent host
    memory allows; without the flag the runtime's environment may choose otherwise."""
    got = child("print(json.dumps(calls(lambda: wg.Context(0))[0]))")
    flags = [int(line.split()[2]) for line in got if line.startswith("host_malloc")]
    coherent, non_coherent = 0x40000000, 0x80000000
    assert len(flags) == 1 and flags[0] & coherent and not flags[0] & non_coherent, got


def test_reductions_fold_in_the_same_launch_only_where_that_is_no_slower(child):
    """Sums of one word up to 256 first-pass blocks of 4096 elements, folds of up to 16 bytes and
    strided reads up to 192, larger folds and strided reads of 8-byte elements up to 112."""
    got = child("""
ctx, out = wg.Context(0), []
for name, two, blocks, inc in (("sdot", 1, 256, 1), ("ddot", 1, 256, 1), ("dasum", 0, 256, 1), ("snrm2", 0, 192, 1),
                               ("dnrm2", 0, 112, 1), ("isamax", 0, 192, 1), ("idamax", 0, 192, 1),
                               ("ddot", 1, 112, 5), ("sasum", 0, 192, 7), ("dnrm2", 0, 112, 6)):
    for n in (blocks * 4096, blocks * 4096 + 1):
        args = (n, P, inc, P, inc, P) if two else (n, P, inc, P)
        log, error = calls(lambda: getattr(ctx, name + "_dev")(*args))
        assert error is None, error
        out.append([name, inc, n > blocks * 4096, sum(line.startswith("launch") for line in log)])
print(json.dumps(out))
""")
    assert len(got) == 20
    for name, inc, above, launches in got:
        assert launches == (2 if above else 1), (name, inc, above, launches)


def test_transposed_gemv_accesses_by_alignment(child):
    """Aligned columns: vectors past the caches (2). Others: element by element (0) below 64 rows, else vectors
    through the caches (1), or past them in fp32 where A is larger than they are. A strided x: by element."""
    got = child("""
ctx, out = wg.Context(0), []
for name in ("sgemv", "dgemv"):
    for m, n, lda, shift, incx in ((300, 300, 300, 0, 1), (300, 300, 300, 8, 1), (300, 300, 301, 0, 1), (5000, 5000, 5002, 0, 1),
                                   (300, 300, 300, 0, 2), (60, 9000, 60, 0, 1), (63, 9000, 65, 0, 1), (64, 9000, 65, 0, 1),
                                   (8191, 8191, 8191, 0, 1), (8191, 8194, 8193, 0, 1)):
        log, error = calls(lambda: getattr(ctx, name)(1, m, n, 1.0, P + shift, lda, P, incx, 0.0, P, 1))
        assert error is None, error
        out.append(next(line.split()[-1] for line in log if "gemv_t_kernel" in line))
print(json.dumps(out))
""")
    kinds = [name.split("gemv_t_kernelI")[1][:4] for name in got]
    assert kinds == ["fLi" + k for k in "2111020112"] + ["dLi" + k for k in "2111020111"], kinds


def test_gemv_blocks_by_the_busiest_cu(child):
    """gemv N's two kinds of block, 256 rows (1 x 8 waves) or 1024 (4 x 1), on both sides of each
    of the rule's lines; with one block per CU or fewer beside each other, no CU gets two."""
    shapes = {
        # narrow in both
        (4096, 4096): "nn", (2000, 30000): "nn", (7000, 7000): "nn", (50000, 768): "nn", (300, 1000): "nn",
        # few rows, whatever the columns
        (1, 200000): "nn", (250, 70000): "nn", (512, 160000): "nn", (513, 160000): "ww",
        # the wide blocks fill the CUs
        (8192, 8192): "ww", (16384, 16384): "ww", (1025, 40000): "ww", (400000, 10): "ww",
        # splits that do not divide the CUs' work evenly
        (15000, 4000): "nw", (25000, 2304): "nw", (1024, 57000): "nn", (1024, 65000): "nw",
        (964, 61000): "nw", (800, 65000): "nw",
        # more than one narrow block per CU beside each other
        (150000, 256): "nn", (205000, 200): "nw", (255000, 200): "ww", (255000, 32): "nw", (200000, 4): "nw",
    }
    got = child(f"""
ctx, out = wg.Context(0), []
for m, n in {list(shapes)}:
    for gemv in (ctx.sgemv, ctx.dgemv):
        log, error = calls(lambda: gemv(0, m, n, 1.0, P, m, P, 1, 0.0, P, 1))
        assert error is None, error
        out.append(next(line.split() for line in log if "gemv_n_kernel" in line))
print(json.dumps(out))
""")
    kinds = {}
    for k, (m, n) in enumerate(shapes):
        for line in got[2 * k:2 * k + 2]:
            across, splits, threads = int(line[1]), int(line[2]), int(line[4])
            narrow = threads == 512
            kinds[m, n] = kinds.get((m, n), "") + ("n" if narrow else "w")
            rows = 256 if narrow else 1024
            assert (across - 1) * rows < m <= across * rows
            if narrow and across <= 256:
                assert across * splits <= 256, (m, n, across, splits)
    assert kinds == shapes


def test_long_reductions_keep_the_plain_remainder_loop(child):
    """Where a thread has more than a few vectors, taking what steps of 16 leave four at a time (and the
    folding code beside it) was slower than one at a time, unless nearly a whole step is left."""
    got = child("""
ctx, out = wg.Context(0), []
for name, n in (("isamax", 24_000_000), ("isamax", 32_000_000), ("idamax", 20_000_000), ("idamax", 24_000_000),
                ("isamax", 1), ("isamax", 1_000_000), ("idamax", 1_000_000),
                # a step of 16 vectors nearly whole, whole, and well short of it
                ("idamax", 33_344_000), ("isamax", 4096 * 256 * 63), ("isamax", 4096 * 256 * 64),
                ("idamax", 4096 * 256 * 32), ("isamax", 4096 * 256 * 60)):
    log, error = calls(lambda: getattr(ctx, name + "_dev")(n, P, 1, P))
    assert error is None, error
    out.append(next(line.split()[-1] for line in log if "reduce_vec" in line))
print(json.dumps(out))
""")
    assert ["Lb1E" in name for name in got] == [True, False, True, False] + [True] * 3 + [True, True] + [False] * 3, got


def test_sgemm_k_groups_are_reached(child):
    """The shapes of the k-group tests launch the kernel that they are there for, in every layout; one k-tile or
    one tile fewer or more than the rule's lines does not."""
    from tests.test_gpu_dispatch_edges import K_GROUPS, ONE_GROUP

    assert {case[-1] for case in K_GROUPS} == {2, 4}
    got = child(f"""
out = []
ctx = wg.Context(0)
for m, n, k, pad, groups in {K_GROUPS + ONE_GROUP}:
    for ta in (0, 1):
        for tb in (0, 1):
            log, error = calls(lambda: ctx.sgemm(ta, tb, m, n, k, 1.0, P, (k if ta else m) + pad, P, (n if tb else k) + pad,
                                                 -1.0, P, m + pad))
            out.append([groups, log[-1].split()])
for n, k, groups in ((1001, 1040, 2), (700, 2113, 4)):
    log, error = calls(lambda: ctx.sgemmtr(1, 0, 0, n, n, k, 1.0, P, n, P, k, -1.0, P, n))
    out.append([groups, log[-1].split()])
for m, n, k in ((1024, 1024, 480), (1024, 1088, 1000), (2048, 1088, 2048), (2048, 1024, 2016)):
    log, error = calls(lambda: ctx.sgemm(0, 1, m, n, k, 1.0, P, m, P, n, -1.0, P, m))
    out.append([1, log[-1].split()])
print(json.dumps(out))
""")
    for groups, (_, _, _, _, threads, name) in got:
        assert int(threads) == 256 * groups, (groups, threads, name)
        assert ("gemm_kgroup_kernelILi%dE" % groups in name) == (groups > 1), (groups, name)


@pytest.mark.parametrize("prefix,size", [("s", 4), ("d", 8)])
def test_symv_plan(child, prefix, size):
    """The runs of symv / trmv: at most 512 columns (the LDS of their sums), the workspace large enough for
    every chunk's row slots and column slots, and all columns covered."""
    got = child(f"""
out = []
for n in list(range(1, 70)) + [1023, 1024, 1025, 2049, 4096, 5120, 5121, 6001, 8191, 8192, 16383, 22528, 23000, 32769, 65536]:
    for uplo in (1, 2):
        ctx = wg.Context(0)  # a workspace of its own
        log, error = calls(lambda: ctx.{prefix}symv(uplo, n, 1.0, P, n, P, 1, 0.0, P, 1))
        assert error is None, error
        ws = [int(line.split()[1]) for line in log if line.startswith("malloc")]
        blocks = next(int(line.split()[1]) for line in log if "symv_kernel" in line)
        out.append([n, uplo, blocks, ws])
        ctx.close()
print(json.dumps(out))
""")
    for n, uplo, blocks, ws in got:
        chunks = -(-n // 1024)
        n8 = -(-n // 8) * 8
        columns = [min((r + 1) * 1024, n8) if uplo == 1 else n8 - r * 1024 for r in range(chunks)]
        # the run is not in the log: some multiple of 8 that gives this many blocks
        total = sum(columns)
        runs = [run for run in range(8, 513, 8) if -(-total // run) == blocks]
        assert runs, (n, uplo, blocks)
        starts = [sum(columns[:r]) for r in range(chunks)]
        need = min(max((s + c - 1) // run - s // run + 1 for s, c in zip(starts, columns)) for run in runs)
        assert len(ws) == 1 and ws[0] >= (need + chunks) * n * size, (n, uplo, blocks, ws)
