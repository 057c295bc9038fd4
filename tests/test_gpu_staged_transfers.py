"""Host arrays of several staging slots (from 4 MiB; 1.5 MiB a slot, four of them): projections, groups and the FFN chain with
its residual on the side stream, from pageable and from pinned memory, against the device-pointer
calls of the same inputs bit for bit, several calls in a row on one context.
"""

import ctypes

import numpy as np
import pytest

import prism_hip as ph
import synth
from hiprt import DeviceBuffer, hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens", [64, 512, 513, 1100])  # below, at and past 4 MiB of input; six slots
@pytest.mark.parametrize("kind", [ph.KIND_PTQ1, ph.KIND_Q2_K])
def test_gpu_staged_projection_equals_device_call(kind, tokens):
    cols, rows = 2048, 2100  # 1100 tokens: 9.2 MB of output
    with ph.Context(0) as ctx:
        wid = ctx.weight(kind, cols, rows, synth.weights(kind, rows, cols, seed=1))
        for seed in (2, 3):
            X = np.ascontiguousarray(synth.activations(cols, seed=seed, tokens=tokens).reshape(tokens, cols), np.float32)
            d, o = DeviceBuffer.from_numpy(X), DeviceBuffer(rows * tokens * 4)
            ctx.project_device(wid, ph.PATH_F32, d, tokens, False, o)
            assert ctx.sync() == 0
            want = o.to_numpy(np.uint32)
            got = ctx.project_f32(wid, rows, X, tokens=tokens)
            assert np.array_equal(np.asarray(got, np.float32).reshape(-1).view(np.uint32), want)
            outs = ctx.project_f32_group_tokens([wid, wid], [rows, rows], X)
            for g in outs:
                assert np.array_equal(np.asarray(g, np.float32).reshape(-1).view(np.uint32), want)


@pytest.mark.parametrize("tokens", [1, 40, 256, 257, 1100])  # the side stream from 256 tokens (1 MiB)
def test_gpu_staged_ffn_residual(tokens):
    """Each token's row of the chain equals its own one-token call; a non-finite input then fails
    the call, clears the output and leaves the context usable."""
    hidden, ffn = 1024, 1536
    with ph.Context(0) as ctx:
        g, u = (ctx.weight(ph.KIND_PTQ1, hidden, ffn, synth.ptq1_weights(ffn, hidden, seed=s)) for s in (1, 2))
        d = ctx.weight(ph.KIND_PTQ1, ffn, hidden, synth.ptq1_weights(hidden, ffn, seed=3))
        X = np.ascontiguousarray(synth.activations(hidden, seed=4, tokens=tokens).reshape(tokens, hidden), np.float32)
        R = np.ascontiguousarray(synth.activations(hidden, seed=5, tokens=tokens).reshape(tokens, hidden), np.float32)
        for _ in range(2):
            got = ctx.ffn_chain_tokens(g, u, d, hidden, X, residual=R, pinned=True)
            for t in sorted({0, tokens // 2, tokens - 1}):
                one = ctx.ffn_chain(g, u, d, hidden, X[t], residual=R[t], pinned=True)
                assert np.array_equal(got[t].view(np.uint32), np.asarray(one, np.float32).reshape(-1).view(np.uint32))
        bad = X.copy()
        bad[tokens // 2, 3] = np.inf
        rc, out = ctx.ffn_chain_tokens(g, u, d, hidden, bad, residual=R, pinned=True, check=False)
        assert rc == ph.ERR_NONFINITE and not np.any(out)
        again = ctx.ffn_chain_tokens(g, u, d, hidden, X, residual=R, pinned=True)
        assert np.array_equal(again.view(np.uint32), got.view(np.uint32))


def _pinned(shape):
    p = ctypes.c_void_p()
    assert hip().hipHostMalloc(ctypes.byref(p), ctypes.c_size_t(int(np.prod(shape)) * 4), 0) == 0
    return p, np.ctypeslib.as_array(ctypes.cast(p, ctypes.POINTER(ctypes.c_float)), shape)


@pytest.mark.parametrize("tokens", [300, 1100])  # 2.5 MB each way, below the slots' line; 9.0 and 9.2 MB
def test_gpu_pinned_host_arrays_transfer_directly(tokens):
    """Pinned input and output of a call give the pageable call's bits (that they bypass the slots is
    shown where the copies are written down, test_host_scratch.py)."""
    cols, rows = 2048, 2100
    with ph.Context(0) as ctx:
        wid = ctx.weight(ph.KIND_Q2_K, cols, rows, synth.weights(ph.KIND_Q2_K, rows, cols, seed=1))
        X = np.ascontiguousarray(synth.activations(cols, seed=2, tokens=tokens).reshape(tokens, cols), np.float32)
        want = ctx.project_f32(wid, rows, X, tokens=tokens)
        (px, x), (po, out) = _pinned(X.shape), _pinned((tokens, rows))
        x[:] = X
        for _ in range(2):
            out[:] = 7
            assert ph.lib().prism_hip_project_f32(ctx._h, wid, px, tokens, 0, po) == 0
            assert np.array_equal(out.view(np.uint32), np.asarray(want).view(np.uint32))
        for p in (px, po):
            hip().hipHostFree(p)


@pytest.mark.parametrize("memory", ["pinned", "pinned, null stream", "device"])
@pytest.mark.parametrize("tokens", [256, 1030])  # the smallest residual of the side stream (1 MiB), and staged sizes
@pytest.mark.parametrize("which", ["input", "residual"])
def test_gpu_host_call_reads_behind_queued_work(memory, tokens, which):
    """A pinned or device array filled by a copy queued on the context stream (or the null stream,
    which the context stream orders itself with) behind some ten milliseconds of kernels is read
    when its turn comes: same bits as the synchronized call."""
    hidden, ffn = 1024, 1536
    with ph.Context(0) as ctx:
        g, u = (ctx.weight(ph.KIND_PTQ1, hidden, ffn, synth.ptq1_weights(ffn, hidden, seed=s)) for s in (1, 2))
        d = ctx.weight(ph.KIND_PTQ1, ffn, hidden, synth.ptq1_weights(hidden, ffn, seed=3))
        big = ctx.weight(ph.KIND_PTQ1, 2048, 20000, synth.ptq1_weights(20000, 2048, seed=6))
        bx = DeviceBuffer.from_numpy(np.ascontiguousarray(synth.activations(2048, seed=7, tokens=512), np.float32))
        bo = DeviceBuffer(20000 * 512 * 4)
        X, R = (np.ascontiguousarray(synth.activations(hidden, seed=s, tokens=tokens).reshape(tokens, hidden), np.float32)
                for s in (4, 5))
        want = ctx.ffn_chain_tokens(g, u, d, hidden, X, residual=R)
        src = X if which == "input" else R
        dsrc = DeviceBuffer.from_numpy(src)
        own, late = None, None
        if memory == "device":
            late = DeviceBuffer.from_numpy(np.zeros_like(src))
            ptr, kind = late.ptr, 3
        else:
            own, late = _pinned(src.shape)
            late[:] = 0
            ptr, kind = own.value, 2
        out = np.full((tokens, hidden), 7.0, np.float32)
        ctx.project_device(big, ph.PATH_F32, bx, 512, False, bo)
        assert ctx.sync() == 0
        for _ in range(100):
            ctx.project_device(big, ph.PATH_F32, bx, 512, False, bo)
        stream = None if memory.endswith("null stream") else ctx.stream()
        assert hip().hipMemcpyAsync(ptr, dsrc.ptr, src.nbytes, kind, stream) == 0
        px, pr = (ptr, R.ctypes.data) if which == "input" else (X.ctypes.data, ptr)
        rc = ph.lib().prism_hip_ffn_chain_tokens(ctx._h, g, u, d, ctypes.c_void_p(px), ctypes.c_void_p(pr), tokens, 0, 0,
                                                 ctypes.c_void_p(out.ctypes.data))
        assert rc == 0
        assert np.array_equal(out.view(np.uint32), want.view(np.uint32))
        if own:
            hip().hipHostFree(own)
