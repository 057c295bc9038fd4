"""The stream form of the PTQ1 table kernel (sixteen units of a workgroup's tiles at a time, their
terms folded behind the next sixteen) and the split kernel's fold of pinned rows by native lane:
one token on long rows, against the oracle's matvec bit for bit (one serial binary32 chain per
row, or four per pinned row, so no tolerance applies).
"""

import os

import numpy as np
import pytest

import prism_hip as ph
import synth
from hiprt import cu_count

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


@pytest.fixture(scope="module")
def ctx():
    c = ph.Context(0)
    yield c
    c.close()


# Tiles as (quarters per CU, extra rows) and units per row: just over half a tile per CU at the
# first pinned unit count, one tile and its last partial one, two, three and five tiles for some
# workgroups only; unit counts that are no multiple of sixteen, leave one unit over, or exceed
# the spread form's 64; the longest row of few tiles (17408 inputs) and one past 256 units.
@pytest.mark.parametrize("per_cu4,extra,units", [(2, 1, 25), (2, 37, 57), (4, -3, 41), (5, 5, 65), (9, 64, 66), (13, 9, 26),
                                                 (17, 1, 66), (1, 17, 136), (1, 1, 257), (9, 1, 17)])
@pytest.mark.parametrize("pinned", [False, True])
def test_gpu_stream_rows_match_oracle(ctx, per_cu4, extra, units, pinned):
    import oracle

    rows, cols = cu_count() * 16 * per_cu4 + extra, units * 128
    w = synth.ptq1_weights(rows, cols, seed=rows % 1000 + units)
    x = synth.activations(cols, seed=units)
    wid = ctx.weight(ph.KIND_PTQ1, cols, rows, w)
    try:
        ref = oracle.matvec(oracle.KIND_PTQ1, cols, rows, w, x, pinned, threads=THREADS)
        got = ctx.project_f32(wid, rows, x, pinned=pinned)
        assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
        if not pinned and units % 2 == 0:  # Q8_K activations: sampled rows
            act = oracle.quantize_q8k(x, False)
            got = ctx.project_q8k(wid, rows, act.view(ph.Q8K_DTYPE), tokens=1, fused=False).reshape(-1)
            sample = list(range(0, rows, max(1, rows // 300))) + list(range(rows - 3, rows))
            nb = units * 28
            want = np.array([oracle.dot_ptq1_q8k(w[r * nb:(r + 1) * nb], act) for r in sample], np.float32)
            assert np.array_equal(got[sample].view(np.uint32), want.view(np.uint32))
    finally:
        ctx.release(wid)


@pytest.mark.parametrize("rows,cols", [(1, 128), (9, 17408), (100, 2048), (2053, 5120), (4100, 1280)])
def test_gpu_split_pinned_fold_matches_oracle(ctx, rows, cols):
    """8 to 64 rows per workgroup, folded by native lane on one or several wavefronts."""
    import oracle

    w = synth.ptq1_weights(rows, cols, seed=rows)
    x = synth.activations(cols, seed=cols)
    wid = ctx.weight(ph.KIND_PTQ1, cols, rows, w)
    ref = oracle.matvec(oracle.KIND_PTQ1, cols, rows, w, x, True, threads=THREADS)
    got = ctx.project_f32(wid, rows, x, pinned=True)
    ctx.release(wid)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("hidden,ffn", [(256, 512), (2560, 2048), (1024, 4352)])
def test_gpu_pinned_gate_up_fold_matches_oracle(ctx, hidden, ffn):
    """Gate and up share the workgroup and its fold (two matrices of rows)."""
    import oracle

    g, u = (synth.ptq1_weights(ffn, hidden, seed=s) for s in (1, 2))
    x = synth.activations(hidden, seed=3)
    wg, wu = ctx.weight(ph.KIND_PTQ1, hidden, ffn, g), ctx.weight(ph.KIND_PTQ1, hidden, ffn, u)
    got = ctx.ffn_swiglu(wg, wu, ffn, x, pinned=True)
    gv, uv = (oracle.matvec(oracle.KIND_PTQ1, hidden, ffn, m, x, True, threads=THREADS) for m in (g, u))
    want = oracle.swiglu(gv, uv, True)
    ctx.release(wg)
    ctx.release(wu)
    assert np.array_equal(np.asarray(got, np.float32).view(np.uint32), np.asarray(want, np.float32).view(np.uint32))


@pytest.mark.parametrize("kind,pinned", [(ph.KIND_PQ2, True), (ph.KIND_PQ2, False), (ph.KIND_Q2_K, False), (ph.KIND_Q8_0, True),
                                         (ph.KIND_TQ1_0, False), (ph.KIND_TQ2_0, False), (ph.KIND_PTQ1, False)])
@pytest.mark.parametrize("per_cu4,extra,cols", [(1, 5, 10240), (1, 64, 17408), (2, 70, 16640), (2, 70, 4864)])
def test_gpu_long_rows_separate_quantizer_matches_oracle(ctx, kind, pinned, per_cu4, extra, cols):
    """A quarter to one tile per CU on long rows: sixteen split wavefronts per CU, and f32 input
    quantized by a launch of its own."""
    import oracle

    rows = cu_count() * 16 * per_cu4 + extra
    w = synth.weights(kind, rows, cols, seed=cols)
    x = synth.activations(cols, seed=rows)
    wid = ctx.weight(kind, cols, rows, w)
    ref = oracle.matvec(kind, cols, rows, w, x, pinned, threads=THREADS)
    got = ctx.project_f32(wid, rows, x, pinned=pinned)
    ctx.release(wid)
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))
