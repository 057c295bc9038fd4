"""The library's host side on the CPU: libprism_hip.so over a HIP runtime without a device
(hip_stub.cpp), which writes down allocations, copies and launches and runs no kernel.  Covers
what no result shows: the stream an array is copied on, and what a graph may hold.
"""

import os
import subprocess
import sys
import textwrap

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
LIB = os.path.join(ROOT, "prism-inference_amd", "libprism_hip.so")

PRELUDE = """
import ctypes, sys
import numpy as np
S = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
S.stub_log.restype = ctypes.c_char_p
S.stub_largest.argtypes = [ctypes.c_size_t]
S.hipHostMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t, ctypes.c_uint]
S.hipMalloc.argtypes = [ctypes.POINTER(ctypes.c_void_p), ctypes.c_size_t]
sys.path.insert(0, sys.argv[2])
import prism_hip as ph
P, L = ctypes.c_void_p, ph.lib()
X, OUT = P(0x10000000), P(0x20000000)  # device arrays of the caller; nothing reads them
def log():
    return S.stub_log().decode().splitlines()
def weight(c, kind, cols, rows):
    return L.prism_hip_weight_wrap_tiled(c, kind, cols, rows, P(0x70000000), L.prism_hip_weight_tiled_bytes(c, kind, cols, rows))
def project(c, w, path, tokens, pinned):
    return L.prism_hip_project_device(c, w, path, X, tokens, int(pinned), OUT, None)
def captured(call):
    S.stub_capture(1)
    rc = call()
    S.stub_capture(0)
    return rc
"""


@pytest.fixture(scope="module")
def stub(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("stub") / "hip_stub.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "hip_stub.cpp"), "-o", so], check=True)

    def run(code, *args):
        src = PRELUDE + textwrap.dedent(code)
        p = subprocess.run([sys.executable, "-c", src, so, os.path.dirname(LIB), *map(str, args)], capture_output=True,
                           text=True, timeout=300)
        assert p.returncode == 0, p.stdout + p.stderr
        return p.stdout

    return run


@pytest.mark.parametrize("memory", ["pinned", "device", "pageable"])
def test_ffn_residual_is_copied_behind_the_callers_work(stub, memory):
    """Memory HIP reads when the copy's turn comes is copied on the context stream, where the caller
    orders its work; only pageable memory, read before the call returns, may take another."""
    stub("""
        c = L.prism_hip_create(0, 0, 0)
        hidden, ffn, tokens = 1024, 1536, 300
        g, u, d = weight(c, ph.KIND_PTQ1, hidden, ffn), weight(c, ph.KIND_PTQ1, hidden, ffn), weight(c, ph.KIND_PTQ1, ffn, hidden)
        n = tokens * hidden * 4
        keep = [np.zeros(tokens * hidden, np.float32) for _ in range(3)]
        x, res, out = (P(a.ctypes.data) for a in keep)
        if sys.argv[3] != "pageable":
            res = P()
            assert (S.hipHostMalloc(ctypes.byref(res), n, 0) if sys.argv[3] == "pinned" else S.hipMalloc(ctypes.byref(res), n)) == 0
        log()
        assert L.prism_hip_ffn_chain_tokens(c, g, u, d, x, res, tokens, 0, 0, out) == 0
        stream = "stream " + hex(L.prism_hip_stream(c))
        copies = [l for l in log() if l.startswith("copy ")]
        if sys.argv[3] == "pageable":
            assert any(not l.endswith(stream) for l in copies), copies
        else:
            assert all(l.endswith(stream) for l in copies) and any(f"<- {hex(res.value)} " in l for l in copies), copies
        L.prism_hip_destroy(c)
        """, memory)


@pytest.mark.parametrize("memory", ["pinned", "pageable"])
@pytest.mark.parametrize("tokens,staged", [(300, False), (511, False), (512, True), (1100, True)])
def test_large_pageable_arrays_pass_through_the_pinned_slots(stub, memory, tokens, staged):
    """From 4 MiB a pageable array moves in pieces through pinned slots, allocated for the first such
    call; a smaller one, and pinned memory of any size, in one copy of its own."""
    stub("""
        tokens, staged = int(sys.argv[4]), sys.argv[5] == "True" and sys.argv[3] == "pageable"
        c = L.prism_hip_create(0, 0, 0)
        w = weight(c, ph.KIND_Q2_K, 2048, 2048)
        n = tokens * 2048 * 4
        if sys.argv[3] == "pinned":
            x, out = P(), P()
            assert S.hipHostMalloc(ctypes.byref(x), n, 0) == 0 and S.hipHostMalloc(ctypes.byref(out), n, 0) == 0
        else:
            keep = [np.zeros(n // 4, np.float32) for _ in range(2)]
            x, out = (P(a.ctypes.data) for a in keep)
        log()
        for call in range(2):
            assert L.prism_hip_project_f32(c, w, x, tokens, 0, out) == 0
            lines = log()
            assert any(l.startswith("host_malloc") for l in lines) == (staged and call == 0), lines
            sizes = [int(l.split()[4]) for l in lines if l.startswith("copy ") and int(l.split()[4]) > 4]
            pieces = -(-n // (1536 * 1024))
            assert len(sizes) == (2 * pieces if staged else 2) and sum(sizes) == 2 * n, lines
            direct = sum(f"<- {hex(x.value)} {n} " in l or f"copy {hex(out.value)} " in l for l in lines)
            assert direct == (0 if staged else 2), lines
        L.prism_hip_destroy(c)
        """, memory, tokens, staged)


@pytest.mark.parametrize("seed", [1, 2])
def test_a_call_made_once_uncaptured_can_be_captured(stub, seed):
    """Every form of a device call, at sizes on all routes: scratch never grows under capture, and one
    uncaptured call of the same arguments is all that a capture needs.  Both take the same kernels."""
    stub("""
        import random
        rng = random.Random(int(sys.argv[3]))
        kinds = [ph.KIND_PTQ1, ph.KIND_PQ2, ph.KIND_Q2_K, ph.KIND_Q8_0, ph.KIND_TQ1_0, ph.KIND_TQ2_0]
        launches = lambda: [l.split(" stream")[0] for l in log() if l.startswith("launch ")]
        for i in range(3000):
            kind = kinds[i % 6]
            unit = ph.LAYOUT[kind][0] if kind not in (ph.KIND_Q8_0,) else 128
            rows = int(2 ** rng.uniform(0, 10 if i % 2 else 17))
            cols = max(1, int(2 ** rng.uniform(7, 14.2)) // unit) * unit
            tokens = rng.choice([1, 2, 3, rng.randint(4, 16), rng.randint(17, 600), rng.randint(17, 600)])
            pinned = rng.random() < 0.5
            q8k = kind in (ph.KIND_Q2_K, ph.KIND_TQ1_0, ph.KIND_TQ2_0) or (kind == ph.KIND_PQ2 and cols % 256 == 0)
            path = rng.choice([ph.PATH_F32, ph.PATH_Q8K if q8k else ph.PATH_Q8])
            c = L.prism_hip_create(0, 0, 0)
            w = weight(c, kind, cols, rows)
            log()
            case = (kind, rows, cols, tokens, pinned, path)
            assert project(c, w, path, tokens, pinned) == 0, case
            eager = launches()
            assert captured(lambda: project(c, w, path, tokens, pinned)) == 0, (case, L.prism_hip_last_error(c))
            assert launches() == eager, case
            L.prism_hip_destroy(c)
        """, seed)


@pytest.mark.parametrize("kind,rows,cols,first,then,pinned,path", [
    ("PTQ1", 50, 3584, 100, 86, True, "F32"), ("PTQ1", 50, 3584, 86, 100, True, "F32"),
    ("PTQ1", 1754, 2048, 65, 124, True, "Q8"), ("Q2_K", 300, 2048, 70, 128, False, "F32"),
    ("PTQ1", 745, 8192, 64, 8, False, "Q8"), ("PTQ1", 1108, 11136, 64, 3, False, "Q8")])
def test_a_call_of_another_token_count_can_be_captured(stub, kind, rows, cols, first, then, pinned, path):
    """Token counts that pad to the same GEMM size, and few tokens after many: the scratch that one leaves
    is enough for the other, whichever kernels run them."""
    stub("""
        kind, path = getattr(ph, "KIND_" + sys.argv[3]), getattr(ph, "PATH_" + sys.argv[9])
        rows, cols, first, then = (int(a) for a in sys.argv[4:8])
        c = L.prism_hip_create(0, 0, 0)
        w = weight(c, kind, cols, rows)
        assert project(c, w, path, first, sys.argv[8] == "True") == 0
        assert captured(lambda: project(c, w, path, then, sys.argv[8] == "True")) == 0, L.prism_hip_last_error(c)
        L.prism_hip_destroy(c)
        """, kind, rows, cols, first, then, pinned, path)


@pytest.mark.parametrize("cols,tokens", [(65536, 520), (1 << 20, 512), (3959808, 65), (3959808, 2750), (30000128, 600)])
def test_scratch_of_very_long_rows(stub, cols, tokens):
    """The lane-ordered copies stay bounded, and their size is not cut to 32 bits: 32 chunks of 3.7
    million inputs, or four of 30 million, pass 2 GiB."""
    stub("""
        cols, tokens = int(sys.argv[3]), int(sys.argv[4])
        for kind, unit in ((ph.KIND_Q8_0, 128), (ph.KIND_PQ2, 128), (ph.KIND_PTQ1, 128), (ph.KIND_TQ1_0, 256)):
            for rows in (97, 2100):
                c = L.prism_hip_create(0, 0, 0)
                w = weight(c, kind, cols // unit * unit, rows)
                log()
                assert project(c, w, ph.PATH_F32, tokens, False) == 0, (kind, rows, L.prism_hip_last_error(c))
                sizes = [int(l.split()[2]) for l in log() if l.startswith("malloc ")]
                copies = max(32 << 20, 4 * (cols // 128 + 1) * 64 * 68)  # four chunks, at most 64 + 4 bytes a lane
                blocks = tokens * cols // 32 * 40  # the prepared activations: Q8_0, larger than Q8_K
                gemm = (tokens + 127) // 128 * 128 * cols * 3
                # Where the GEMM covers the call, its scratch twice: of f32 input and of prepared blocks.
                assert len(sizes) <= 3 and sum(sizes) <= blocks + max(copies, 2 * gemm if cols <= 65536 else 0) + 8192, (kind, rows, sizes)
                L.prism_hip_destroy(c)
        """, cols, tokens)


CAPTURED = [  # kind, rows, cols, tokens, pinned, path, and the tokens of the call that outgrows its scratch
    ("PTQ1", 5120, 17408, 1, False, "F32", 40), ("PQ2", 5120, 17408, 1, True, "F32", 40),  # a quantizer of its own
    ("PTQ1", 8256, 4096, 1, True, "F32", 40),  # the stream form
    ("Q2_K", 500, 2048, 7, False, "F32", 90), ("Q8_0", 500, 2048, 12, True, "F32", 90),  # few rows
    ("PTQ1", 8200, 6144, 2, True, "Q8", 30), ("PTQ1", 6144, 2048, 64, False, "F32", 600),  # copies; a GEMM
    ("PTQ1", 5120, 6144, 2, False, "Q8", 40)]  # split-K


@pytest.mark.parametrize("kind,rows,cols,tokens,pinned,path,more", CAPTURED)
@pytest.mark.parametrize("ffn", [False, True])
def test_scratch_of_a_captured_call_outlives_larger_calls(stub, kind, rows, cols, tokens, pinned, path, more, ffn):
    """Every buffer there was when a call was captured is still there after calls that need more, the
    kept ones stay below the current ones, and the context gives all of them back."""
    stub("""
        kind, path = getattr(ph, "KIND_" + sys.argv[3]), getattr(ph, "PATH_" + sys.argv[8])
        rows, cols, tokens, more, pinned, ffn = (int(a) for a in sys.argv[4:7] + sys.argv[9:10] + [sys.argv[7] == "True", sys.argv[10] == "True"])
        c = L.prism_hip_create(0, 0, 0)
        empty = S.stub_allocations()
        w = weight(c, kind, cols, rows)
        g, u, d = weight(c, kind, cols, 8192), weight(c, kind, cols, 8192), weight(c, kind, 8192, cols)
        def call():
            if ffn:
                return L.prism_hip_ffn_chain_device(c, g, u, d, X, None, 64, int(pinned), OUT, None, None)
            return project(c, w, path, tokens, pinned)
        assert call() == 0
        log()
        # Uncaptured so far: an outgrown buffer is given back at once.
        assert project(c, w, path, tokens + 1, pinned) == 0 and call() == 0
        log()
        assert captured(call) == 0
        assert not any(l.startswith(("malloc", "free")) for l in log())
        sizes = {}
        def grow(t):
            for k in (ph.PATH_F32, path):
                assert project(c, w, k, t, pinned) == 0
            for l in log():
                f = l.split()
                assert f[0] != "free", l
                if f[0] == "malloc":
                    sizes[f[1]] = int(f[2])
        for t in range(more, more + 200):
            grow(t)
        assert sizes and len(sizes) <= 4 * 3, sizes  # doubling: few buffers a role
        assert captured(lambda: project(c, w, path, more, pinned)) == 0
        # Memory for the exact size only, and then none: the old buffer keeps serving.
        big = 40 * more
        need = max(sizes.values()) * 4
        S.stub_largest(need)
        while project(c, w, path, big, pinned) == 0 and big < 4000000:
            big *= 2
        assert big < 4000000
        assert not any(l.startswith("free") for l in log())
        assert call() == 0 and captured(call) == 0
        L.prism_hip_destroy(c)
        assert S.stub_allocations() == empty - 1, (S.stub_allocations(), empty)  # and the error flag
        """, kind, rows, cols, tokens, pinned, path, more, ffn)


# The kernels a call is made of, at the lines between two of them (kind, rows, cols, tokens, pinned,
# path, the launches' kernels in order); where each line lies is measured, at the rule in the source.
ROUTES = [
    # Short rows whose skinny batch would copy its activations stay on the GEMM.
    ("PQ2", 74, 1024, 94, False, "F32", "prefill prefill_kq"),
    ("PQ2", 74, 1280, 94, False, "F32", "quantize sk_prep skinny"),
    ("TQ1_0", 700, 1024, 106, False, "F32", "prefill prefill_kq"),
    ("TQ1_0", 700, 1280, 106, False, "Q8K", "sk_prep skinny"),
    ("Q8_0", 1100, 512, 120, False, "Q8", "prefill prefill_kq"),
    ("Q8_0", 1100, 768, 120, False, "F32", "quantize sk_prep skinny"),
    ("Q2_K", 1100, 256, 120, False, "F32", "quantize skinny"),
    # Two (three) tokens of long rows on few rows stay on the one-token kernels.
    ("Q8_0", 500, 6144, 2, False, "F32", "mv_split mv_split"),
    ("Q8_0", 500, 5120, 2, False, "F32", "quantize skinny"),
    ("Q8_0", 500, 6144, 2, False, "Q8", "mv_split mv_split"),
    ("Q8_0", 500, 14336, 3, False, "Q8", "mv_split mv_split mv_split"),
    ("Q8_0", 500, 14336, 3, False, "F32", "quantize mv_split mv_split mv_split"),
    ("Q8_0", 1024, 14336, 2, False, "Q8", "sk_prep skinny"),
    ("TQ1_0", 500, 16384, 2, False, "F32", "mv_split mv_split"),
    ("TQ1_0", 500, 12288, 2, False, "F32", "quantize skinny"),
    ("TQ1_0", 500, 14336, 2, False, "F32", "quantize mv_split mv_split"),
    ("TQ1_0", 500, 14336, 2, False, "Q8K", "mv_split mv_split"),
    # Five to eight tokens copy their activations where many units would be gathered.
    ("PQ2", 1204, 4096, 6, False, "F32", "quantize skinny"),
    ("PQ2", 1204, 4352, 6, False, "F32", "quantize sk_prep skinny"),
    ("TQ1_0", 4334, 4096, 6, False, "F32", "quantize skinny"),
    ("TQ1_0", 4334, 4096, 7, False, "F32", "quantize sk_prep skinny"),
    ("TQ1_0", 4000, 4096, 7, False, "F32", "quantize skinny"),
    # Few rows between the skinny kernel and the GEMMs.
    ("PTQ1", 1638, 3456, 95, False, "F32", "prefill_prep prefill_ptq1_split"),
    ("PTQ1", 1500, 3456, 95, False, "F32", "quantize sk_prep skinny"),
    ("PTQ1", 6231, 7168, 70, False, "F32", "prefill_prep prefill_ptq1"),
    ("PTQ1", 627, 2560, 422, True, "F32", "prefill_prep prefill_ptq1_pinned"),
    ("PTQ1", 627, 2560, 390, True, "F32", "quantize sk_prep skinny"),
    ("Q2_K", 1692, 16384, 250, False, "F32", "prefill prefill_kq"),
    ("Q2_K", 1692, 8192, 250, False, "F32", "quantize skinny"),
    ("TQ1_0", 1056, 2304, 320, False, "F32", "prefill prefill_kq"),
    ("TQ1_0", 1056, 4352, 320, False, "F32", "quantize sk_prep skinny"),
    ("TQ2_0", 2699, 8192, 127, False, "F32", "prefill prefill_kq"),
    # One token of long rows: its quantizer in the prologue, or a launch of its own.
    ("PQ2", 8192, 10240, 1, True, "F32", "mv_split"),
    ("PQ2", 8128, 10240, 1, True, "F32", "quantize mv_split"),
    ("TQ2_0", 8192, 12288, 1, False, "F32", "mv_split"),
    ("TQ2_0", 8000, 12288, 1, False, "F32", "quantize mv_split"),
    ("PTQ1", 8192, 16384, 1, False, "F32", "mv_split"),
    ("Q2_K", 8256, 16384, 1, False, "F32", "quantize mv_rowsn"),
    ("Q2_K", 8256, 14336, 1, False, "F32", "mv_split"),
    ("Q2_K", 4096, 16384, 1, False, "F32", "mv_split"),
    # Wavefronts of a skinny workgroup (the kernel's last template argument).
    ("PTQ1", 16384, 5120, 17, False, "F32", "quantize sk_prep skinnyILNS0_2OpE0ELb1ELi8"),
    ("PTQ1", 16448, 5120, 17, False, "F32", "quantize sk_prep skinnyILNS0_2OpE0ELb1ELi4"),
    ("PTQ1", 32768, 5120, 7, False, "F32", "quantize sk_prep skinnyILNS0_2OpE0ELb1ELi4"),
    ("PTQ1", 65536, 5120, 7, False, "F32", "quantize sk_prep skinnyILNS0_2OpE0ELb1ELi1"),
    # Long Q8_0 rows beside the GEMM.
    ("Q8_0", 17408, 16384, 17, False, "F32", "prefill prefill_kq"),
    ("Q8_0", 17408, 14336, 17, False, "F32", "quantize sk_prep skinny"),
]


@pytest.mark.parametrize("kind,rows,cols,tokens,pinned,path,kernels", ROUTES)
def test_dispatch_lines(stub, kind, rows, cols, tokens, pinned, path, kernels):
    stub("""
        kind, path = getattr(ph, "KIND_" + sys.argv[3]), getattr(ph, "PATH_" + sys.argv[8])
        rows, cols, tokens = (int(a) for a in sys.argv[4:7])
        c = L.prism_hip_create(0, 0, 0)
        w = weight(c, kind, cols, rows)
        log()
        assert project(c, w, path, tokens, sys.argv[7] == "True") == 0
        names = [l.split()[1] for l in log() if l.startswith("launch ")]
        want = sys.argv[9].split()
        assert len(names) == len(want) and all(k in n for k, n in zip(want, names)), names
        """, kind, rows, cols, tokens, pinned, path, kernels)


# 64 x 64 (64-row tiles by groups of 64), 128 x 32 throughout (128-row blocks by groups of 32), by XCD.
@pytest.mark.parametrize("rows,cols,tokens,path,grid", [
    (20000, 4096, 65, "F32", "313 2 1"), (8192, 896, 96, "F32", "64 3 1"), (8192, 1024, 96, "F32", "128 2 1"),
    (8192, 896, 128, "F32", "64 4 1"), (32768, 256, 64, "F32", "256 2 1"), (65536, 384, 256, "F32", "8 512 1"),
    (65536, 512, 256, "F32", "1024 4 1"),
    (20000, 896, 160, "F32", "313 3 1"), (6144, 2048, 512, "F32", "8 96 1"), (6144, 2048, 449, "F32", "8 96 1"), (6200, 2048, 449, "F32", "97 8 1"),
    (13817, 9728, 51, "Q8", "108 2 1"), (20000, 4096, 64, "Q8", "313 1 1"), (16384, 4096, 64, "Q8", "128 2 1"),
    (12064, 512, 360, "Q8", "95 12 1"), (12064, 1536, 360, "Q8", "95 12 1"), (12064, 1664, 360, "Q8", "189 6 1")])
def test_pinned_gemm_grid(stub, rows, cols, tokens, path, grid):
    stub("""
        c = L.prism_hip_create(0, 0, 0)
        w = weight(c, ph.KIND_PTQ1, int(sys.argv[4]), int(sys.argv[3]))
        assert project(c, w, getattr(ph, "PATH_" + sys.argv[6]), int(sys.argv[5]), True) == 0
        gemm = [l for l in log() if "k_prefill_ptq1_pinned" in l]
        assert len(gemm) == 1 and f" grid {sys.argv[7]} block 256" in gemm[0], gemm
        """, rows, cols, tokens, path, grid)
