"""The prefill GEMMs' scale products on the f16 matrix cores, against the oracle bit for bit: the
products of two binary16 scales are exact in binary32, so subnormal scales on either side, their
zeros and the largest ones have to come out as the VALU's.  And the pinned PTQ1 GEMM's tiles: 64
rows by 64 tokens, two halves of a block, with rows and tokens missing from each quarter.
"""

import os

import numpy as np
import pytest

import prism_hip as ph
import synth

pytestmark = pytest.mark.gpu

THREADS = min(16, os.cpu_count() or 1)


@pytest.fixture(scope="module")
def ctx():
    c = ph.Context(0)
    yield c
    c.close()


def _check(ctx, kind, rows, cols, w, X, pinned, tokens):
    import oracle

    wid = ctx.weight(kind, cols, rows, w)
    try:
        ref = oracle.prefill(kind, cols, rows, w, X, pinned, threads=THREADS)
        got = ctx.project_f32(wid, rows, X, tokens=tokens, pinned=pinned)
        g, r = (np.ascontiguousarray(a, np.float32).reshape(-1).view(np.uint32) for a in (got, ref))
        assert np.array_equal(g, r), (kind, rows, cols, tokens, pinned, int((g != r).sum()))
    finally:
        ctx.release(wid)


@pytest.mark.parametrize("kind,at,block", [(ph.KIND_PTQ1, 26, 28), (ph.KIND_Q8_0, 0, 34)])
@pytest.mark.parametrize("pinned", [False, True])
@pytest.mark.parametrize("rows,tokens", [(200, 520), (9000, 96)])
def test_gpu_prefill_subnormal_and_large_scales(ctx, kind, at, block, pinned, rows, tokens):
    """520 tokens of 200 rows and 96 of 9000 take the GEMMs.  Weight scales over every binary16
    exponent (subnormals, zero, up to 2^14) and tokens from 1e-9 (scale zero) over 1e-5 (subnormal)
    to 1e3."""
    cols = 512
    rng = np.random.default_rng(rows + tokens)
    w = np.array(synth.weights(kind, rows, cols, seed=7), np.uint8).reshape(-1, block).copy()
    bits = rng.integers(0, 0x7400, w.shape[0]).astype(np.uint16)
    bits[::5] = rng.integers(0, 0x400, bits[::5].size)
    w[:, at:at + 2] = bits.view(np.uint8).reshape(-1, 2)
    X = synth.activations(cols, seed=8, tokens=tokens).reshape(tokens, cols).astype(np.float32)
    X *= np.float32(10.0) ** rng.integers(-9, 4, tokens).astype(np.float32)[:, None]
    _check(ctx, kind, rows, cols, w.reshape(-1), X, pinned, tokens)


@pytest.mark.parametrize("rows,cols,tokens", [(64, 128, 513), (33, 256, 577), (97, 384, 545), (6144 + 31, 640, 97),
                                              (8192 + 64, 1152, 160), (4160, 128, 513)])
def test_gpu_pinned_prefill_tiles_match_oracle(ctx, rows, cols, tokens):
    """One to nine blocks (the halves staged three ahead run past the row's end), partial row
    halves and token halves, and (513 tokens) a token half without tokens."""
    _check(ctx, ph.KIND_PTQ1, rows, cols, synth.ptq1_weights(rows, cols, seed=rows),
           synth.activations(cols, seed=tokens, tokens=tokens).reshape(tokens, cols), True, tokens)


# The last group of at most 32 tokens on 128-row workgroups: alone, behind one, two and seven groups
# of 64 (eight groups, of which seven are whole), its rows a partial tile, one tile of two, or two; and
# short rows (under eight blocks) on those workgroups only, with the first of eight blocks beside them.
@pytest.mark.parametrize("rows,cols,tokens", [(8192 + 37, 1280, 32), (8192 + 100, 1152, 65), (4096 + 64, 1664, 150),
                                              (6144 + 31, 1152, 449), (8192 + 5, 896, 96), (8192 + 5, 1024, 96),
                                              (8192 + 97, 256, 32)])
@pytest.mark.parametrize("prepared", [False, True])
def test_gpu_pinned_prefill_half_group_matches_oracle(ctx, rows, cols, tokens, prepared):
    import oracle

    w = synth.ptq1_weights(rows, cols, seed=rows)
    X = synth.activations(cols, seed=tokens, tokens=tokens).reshape(tokens, cols)
    if not prepared:
        return _check(ctx, ph.KIND_PTQ1, rows, cols, w, X, True, tokens)
    act = np.concatenate([oracle.quantize_q8_0(X[t], 2) for t in range(tokens)])
    ref = oracle.prefill(ph.KIND_PTQ1, cols, rows, w, X, True, threads=THREADS)
    wid = ctx.weight(ph.KIND_PTQ1, cols, rows, w)
    try:
        got = ctx.project_q8(wid, rows, act.view(ph.Q8_DTYPE), tokens=tokens, pinned=True)
        g, r = (np.ascontiguousarray(a, np.float32).reshape(-1).view(np.uint32) for a in (got, ref))
        assert np.array_equal(g, r), int((g != r).sum())
    finally:
        ctx.release(wid)
