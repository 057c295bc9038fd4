"""Matrices of few rows at two and more tokens: the skinny matrix-core kernel with eight, four
or one wavefronts per 16-row block (pinned PTQ1 folds its native lanes on all of them), its
activations gathered or in lane order, up to 32 chunks of 16 tokens a launch, and the line
between it and the prefill GEMMs.  Every token row equals the oracle's own matvec bit for bit:
each row is one serial binary32 chain on either path, so no tolerance applies.
"""

import os

import numpy as np
import pytest

import prism_hip as ph
import synth
from hiprt import DeviceBuffer

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


@pytest.fixture(scope="module")
def ctx():
    c = ph.Context(0)
    yield c
    c.close()


def _bits(a):
    return np.ascontiguousarray(a, np.float32).reshape(-1).view(np.uint32)


# (rows, cols, tokens): one row; a partial 16-row block; the last row below and the first at
# 1024; two, eight, nine, sixteen and seventeen tokens (gathered up to eight); a chunk more than
# 64 tokens; 512 tokens (32 chunks) and one more (the GEMM); unit counts below, at and past the
# wavefronts of a block; grids on both sides of one and two workgroups per CU.
SHAPES = [(1, 256, 2), (37, 512, 9), (513, 2048, 2), (513, 2304, 17), (1023, 1280, 8), (1024, 1024, 16),
          (200, 3328, 65), (250, 768, 512), (250, 768, 513), (2048 + 37, 1024, 33), (4096 + 5, 512, 16),
          (4160, 256, 40), (8200, 256, 70), (1500, 2560, 100)]


@pytest.mark.parametrize("kind", [ph.KIND_PTQ1, ph.KIND_PQ2, ph.KIND_Q2_K, ph.KIND_Q8_0, ph.KIND_TQ1_0, ph.KIND_TQ2_0])
@pytest.mark.parametrize("rows,cols,tokens", SHAPES)
def test_gpu_few_rows_match_oracle(ctx, kind, rows, cols, tokens):
    import oracle

    w = synth.weights(kind, rows, cols, seed=rows + tokens)
    X = synth.activations(cols, seed=tokens + kind, tokens=tokens).reshape(tokens, cols)
    wid = ctx.weight(kind, cols, rows, w)
    try:
        for pinned in (False, True):
            ref = oracle.prefill(kind, cols, rows, w, X, pinned, threads=THREADS)
            got = ctx.project_f32(wid, rows, X, tokens=tokens, pinned=pinned)
            assert np.array_equal(_bits(got), _bits(ref)), (kind, rows, cols, tokens, pinned)
    finally:
        ctx.release(wid)


@pytest.mark.parametrize("rows,cols,tokens", [(37, 384, 5), (500, 2176, 12), (300, 512, 130)])
def test_gpu_few_rows_prepared_pinned_ptq1_and_odd_pq2(ctx, rows, cols, tokens):
    """Prepared blocks, which ran token by token below 1024 rows: pinned PTQ1 and PQ2 rows of an
    odd number of 128-element groups (Q8_0 activations)."""
    import oracle

    X = synth.activations(cols, seed=tokens, tokens=tokens).reshape(tokens, cols)
    nb = cols // 32
    for kind, contract, pinned in ((ph.KIND_PTQ1, 2, True), (ph.KIND_PTQ1, 0, False), (ph.KIND_PQ2, 1, True)):
        w = synth.weights(kind, rows, cols, seed=rows)
        wid = ctx.weight(kind, cols, rows, w)
        act = np.concatenate([oracle.quantize_q8_0(X[t], contract) for t in range(tokens)])
        ref = np.stack([oracle.project_q8(kind, cols, rows, w, act[t * nb:(t + 1) * nb], pinned, threads=THREADS)
                        for t in range(tokens)])
        got = ctx.project_q8(wid, rows, act.view(ph.Q8_DTYPE), tokens=tokens, pinned=pinned)
        ctx.release(wid)
        assert np.array_equal(_bits(got), _bits(ref)), (kind, pinned)


def test_gpu_few_rows_keep_the_scratch_free_path():
    """Where the prepared blocks do not fit the fixed scratch (800 tokens of 17280 inputs, 17 MB
    of Q8_0 blocks against 16 MiB) a call that ran token by token without scratch still does, and
    so does the first call of a context that is being captured (scratch may not grow then)."""
    import hiprt

    kind, rows, cols, tokens = ph.KIND_PQ2, 40, 17280, 800
    with ph.Context(0) as c:
        wid = c.weight(kind, cols, rows, synth.weights(kind, rows, cols, seed=3))
        x = DeviceBuffer.from_numpy(np.ascontiguousarray(synth.activations(cols, seed=4, tokens=tokens), np.float32))
        a, b = DeviceBuffer(rows * tokens * 4), DeviceBuffer(rows * tokens * 4)
        c.project_device_noalloc(wid, ph.PATH_F32, x, tokens, False, a)
        assert c.sync() == 0
        c.project_device(wid, ph.PATH_F32, x, tokens, False, b)
        assert c.sync() == 0
        assert np.array_equal(a.to_numpy(np.uint32), b.to_numpy(np.uint32))
        with ph.Context(0) as d:
            wd = d.weight(kind, cols, rows, synth.weights(kind, rows, cols, seed=3))
            out = DeviceBuffer(rows * 3 * 4)
            g = hiprt.Graph(d.stream(), lambda: d.project_device(wd, ph.PATH_F32, x, 3, False, out))
            for _ in range(3):
                g.launch()
                assert d.sync() == 0
                assert np.array_equal(out.to_numpy(np.uint32), b.to_numpy(np.uint32)[:rows * 3])


@pytest.mark.parametrize("kind,rows,cols,tokens,pinned", [
    (ph.KIND_PTQ1, 200, 8192, 3, False),   # split-K with scratch
    (ph.KIND_PTQ1, 8200, 6144, 2, True),   # lane-ordered copy, prepared blocks only
    (ph.KIND_Q8_0, 500, 2048, 12, True),   # lane-ordered copy
    (ph.KIND_PTQ1, 8200, 5120, 1, False),  # a quantizer of its own: one token
    (ph.KIND_PTQ1, 8256, 4096, 1, True)])  # the stream form: one token
def test_gpu_first_call_under_capture(kind, rows, cols, tokens, pinned):
    """The first call of a context may be captured where its former path needed no scratch: it
    gives the same bits as an uncaptured call."""
    import hiprt

    w = synth.weights(kind, rows, cols, seed=9)
    X = np.ascontiguousarray(synth.activations(cols, seed=10, tokens=tokens).reshape(tokens, cols), np.float32)
    with ph.Context(0) as c, ph.Context(0) as d:
        wc, wd = c.weight(kind, cols, rows, w), d.weight(kind, cols, rows, w)
        x, a, b = DeviceBuffer.from_numpy(X), DeviceBuffer(rows * tokens * 4), DeviceBuffer(rows * tokens * 4)
        path, inp = ph.PATH_F32, x
        if kind == ph.KIND_PTQ1 and pinned and tokens > 1:
            path, inp = ph.PATH_Q8, DeviceBuffer(tokens * cols // 32 * 40)
            c.quantize_q8_device(x, cols, tokens, ph.Q8_PINNED_NATIVE, inp)
        c.project_device(wc, path, inp, tokens, pinned, a)
        assert c.sync() == 0
        g = hiprt.Graph(d.stream(), lambda: d.project_device(wd, path, inp, tokens, pinned, b))
        for _ in range(3):
            g.launch()
            assert d.sync() == 0
            assert np.array_equal(a.to_numpy(np.uint32), b.to_numpy(np.uint32))


@pytest.mark.parametrize("kind,rows,cols,tokens,pinned", [
    (ph.KIND_PTQ1, 8200, 5120, 1, False),  # a quantizer of its own: one token
    (ph.KIND_PTQ1, 8256, 4096, 1, True),  # the stream form: one token
    (ph.KIND_PTQ1, 2048, 2048, 7, True), (ph.KIND_Q8_0, 500, 2048, 12, True)])  # few rows, gathered and copied
def test_gpu_replay_after_a_larger_call(kind, rows, cols, tokens, pinned):
    """A captured call's scratch outlives larger calls of its context (tests/test_host_scratch.py shows
    that its buffers are kept): replays before and after one give the uncaptured call's bits."""
    import hiprt

    X = np.ascontiguousarray(synth.activations(cols, seed=11, tokens=300).reshape(300, cols), np.float32)
    with ph.Context(0) as c:
        w = c.weight(kind, cols, rows, synth.weights(kind, rows, cols, seed=12))
        x, a, b = DeviceBuffer.from_numpy(X), DeviceBuffer(rows * 300 * 4), DeviceBuffer(rows * tokens * 4)
        c.project_device(w, ph.PATH_F32, x, tokens, pinned, b)
        assert c.sync() == 0
        want = b.to_numpy(np.uint32)
        g = hiprt.Graph(c.stream(), lambda: c.project_device(w, ph.PATH_F32, x, tokens, pinned, b))
        for larger in (0, 40, 300):
            if larger:
                c.project_device(w, ph.PATH_F32, x, larger, pinned, a)
                assert c.sync() == 0
            for _ in range(2):
                b.zero()
                g.launch()
                assert c.sync() == 0
                assert np.array_equal(b.to_numpy(np.uint32), want)
        c.project_device(w, ph.PATH_F32, x, 300, pinned, a)
        assert c.sync() == 0
        assert np.array_equal(a.to_numpy(np.uint32)[:rows * tokens], want)
        del g
