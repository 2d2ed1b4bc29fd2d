"""The forms of the batched Q4_0 GEMV (af_q4_gemm): packed halves up to 8 tokens, one or two token groups,
8- or 16-wave workgroups, K in one range, in ranges the last workgroup adds and in ranges a reduce launch
adds, at the edges of row tiles, super-tiles and token groups."""
import ctypes
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from adaforge_amd import _native as N, hip, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("columns,rows,tokens", [
    (32, 1, 1), (128, 64, 8), (160, 65, 8),        # packed: one block, whole tiles, one past each
    (4128, 63, 8), (16384, 130, 2),                # packed: several ranges of K, added by the last workgroup
    (32, 16, 9), (2080, 1000, 16), (16384, 70, 9), # one group of 16 tokens
    (32, 17, 17), (1056, 999, 17), (4096, 3840, 32),  # two groups
    (3840, 15360, 16), (15360, 3856, 13),          # 16 waves, 2 row waves
    (3840, 15361, 17), (3872, 15360, 32),          # 16 waves, 4 row waves, the last workgroup adds
    (15360, 3844, 31),                             # and with a reduce launch
    (512, 16384, 16), (512, 16385, 16), (512, 16384, 17),  # 256 workgroups of 8 waves, and past one round of them
    (256, 20480, 9), (32, 16400, 32),              # 16 waves, fewer super-tiles than waves along K
    (4096, 5120, 16), (4096, 5120, 17),
])
def test_forms_match_oracle(columns, rows, tokens):
    w = synth.q4(f"forms{columns}x{rows}", columns, rows, signed=True)
    rng = np.random.default_rng(columns * 7 + rows + tokens)
    xs = rng.standard_normal((tokens, columns)).astype(np.float32)
    xs[tokens // 2] *= np.float32(2.0 ** 40)  # scales are per token
    h = N.P()
    N.check(N.lib().af_q4_upload(w.ctypes.data_as(N.u8p), w.size, columns, rows, ctypes.byref(h)))
    try:
        xb, yb = hip.Buffer.from_numpy(xs), hip.Buffer(tokens * rows)
        got = []
        for _ in range(3):  # the tickets start every call at zero
            yb.upload(np.full(tokens * rows, np.nan, np.float32))
            N.check(N.lib().af_q4_gemm(h, xb.ptr, tokens, yb.ptr, None))
            hip.synchronize()
            got.append(yb.numpy().reshape(tokens, rows))
    finally:
        N.lib().af_q4_free(h)
    assert np.array_equal(got[0], got[1]) and np.array_equal(got[0], got[2])
    for t in {0, tokens // 2, tokens - 1}:
        ref = oracle.q4_matvec(w, columns, rows, xs[t])
        # inputs to 22 bits and fp32 sums in any order: the 2-norm of the error is far below 2^-20 of
        # the 2-norm of the products it sums
        scale = np.sqrt(columns) * np.abs(xs[t]).max() * 0.02 * 8
        assert np.abs(got[0][t] - ref).max() <= 2.0 ** -20 * scale
        if t != tokens // 2:
            oracle.compare(ref, got[0][t])


def test_non_finite_inputs_stay_in_their_token():
    """An infinity or NaN makes its own token's outputs non-finite and no other's."""
    columns, rows = 256, 48
    w = synth.q4("forms-nan", columns, rows, signed=True)
    h = N.P()
    N.check(N.lib().af_q4_upload(w.ctypes.data_as(N.u8p), w.size, columns, rows, ctypes.byref(h)))
    try:
        for tokens in (5, 12, 30):
            xs = np.random.default_rng(tokens).standard_normal((tokens, columns)).astype(np.float32)
            xs[1, 7], xs[3, 200] = np.inf, np.nan
            xb, yb = hip.Buffer.from_numpy(xs), hip.Buffer(tokens * rows)
            N.check(N.lib().af_q4_gemm(h, xb.ptr, tokens, yb.ptr, None))
            hip.synchronize()
            y = yb.numpy().reshape(tokens, rows)
            for t in range(tokens):
                if t in (1, 3):
                    assert not np.isfinite(y[t]).any()
                else:
                    oracle.compare(oracle.q4_matvec(w, columns, rows, xs[t]), y[t])
    finally:
        N.lib().af_q4_free(h)


@pytest.mark.parametrize("columns,rows,tokens", [(160, 65, 8), (4128, 63, 5), (2080, 1000, 16), (1056, 999, 17),
                                                 (3840, 15361, 16), (3872, 15360, 30), (16384, 130, 32)])
def test_small_blocks_beside_an_outlier(columns, rows, tokens):
    """Some tokens hold one element 2^30 above the rest, in a block whose weights are zero: their products come from
    the small blocks alone, to the tolerance of the tokens without one."""
    w = synth.q4(f"outlier{columns}x{rows}", columns, rows, signed=True)
    w.reshape(rows, columns // 32, 18)[:, 2, :2] = 0
    rng = np.random.default_rng(columns + rows + tokens)
    xs = rng.standard_normal((tokens, columns)).astype(np.float32)
    small = xs.copy()
    small[:, 64:96] = 0.0
    xs[1::2, 70] = np.float32(2.0 ** 30)
    h = N.P()
    N.check(N.lib().af_q4_upload(w.ctypes.data_as(N.u8p), w.size, columns, rows, ctypes.byref(h)))
    try:
        xb, yb = hip.Buffer.from_numpy(xs), hip.Buffer(tokens * rows)
        N.check(N.lib().af_q4_gemm(h, xb.ptr, tokens, yb.ptr, None))
        hip.synchronize()
        y = yb.numpy().reshape(tokens, rows)
    finally:
        N.lib().af_q4_free(h)
    for t in {0, 1, 2, tokens // 2, tokens - 1}:
        ref = oracle.q4_matvec(w, columns, rows, small[t])
        # inputs to 22 bits of their block's largest and fp32 sums, as in test_forms_match_oracle
        scale = np.sqrt(columns) * np.abs(small[t]).max() * 0.02 * 8
        assert np.abs(y[t] - ref).max() <= 2.0 ** -20 * scale
        oracle.compare(ref, y[t])


@pytest.mark.parametrize("n,tokens,offset", [(1024, 5, 0), (3840, 12, 0), (3840, 32, 0), (2080, 30, 2080 * 4), (2080, 8, -64)])
def test_outputs_over_the_inputs(n, tokens, offset):
    """y in place of x, or overlapping it by any number of elements: the vectors are read before any is written."""
    w = synth.q4(f"inplace{n}", n, n, signed=True)
    xs = np.random.default_rng(n + tokens).standard_normal((tokens, n)).astype(np.float32)
    h = N.P()
    N.check(N.lib().af_q4_upload(w.ctypes.data_as(N.u8p), w.size, n, n, ctypes.byref(h)))
    try:
        b = hip.Buffer(3 * tokens * n)
        whole = np.zeros(3 * tokens * n, np.float32)
        whole[tokens * n:2 * tokens * n] = xs.ravel()
        for _ in range(3):
            b.upload(whole)
            at = b.ptr + tokens * n * 4
            N.check(N.lib().af_q4_gemm(h, at, tokens, at + 4 * offset, None))
            hip.synchronize()
            y = b.numpy()[tokens * n + offset:][:tokens * n].reshape(tokens, n)
            for t in {0, tokens // 2, tokens - 1}:
                oracle.compare(oracle.q4_matvec(w, n, n, xs[t]), y[t])
    finally:
        N.lib().af_q4_free(h)


def test_captured_calls_replay_among_direct_ones():
    """A captured call's tickets serve every replay, with direct calls (whose tickets count from higher) in between."""
    columns, rows, tokens = 15360, 3840, 5
    w = synth.q4("replay", columns, rows, signed=True)
    xs = np.random.default_rng(7).standard_normal((4, tokens, columns)).astype(np.float32)
    h = N.P()
    N.check(N.lib().af_q4_upload(w.ctypes.data_as(N.u8p), w.size, columns, rows, ctypes.byref(h)))
    try:
        xb, yb = hip.Buffer.from_numpy(xs[0]), hip.Buffer(tokens * rows)
        s = hip.Stream()

        def call():
            N.check(N.lib().af_q4_gemm(h, xb.ptr, tokens, yb.ptr, s.handle))

        call()
        s.synchronize()
        graph = hip.Graph(s, call)
        for x in xs:
            xb.upload(x)
            got = []
            for run in (call, lambda: graph.launch(s), lambda: graph.launch(s), call):
                yb.upload(np.full(tokens * rows, np.nan, np.float32))
                run()
                s.synchronize()
                got.append(yb.numpy())
            assert all(np.array_equal(got[0], g) for g in got[1:])
            oracle.compare(oracle.q4_matvec(w, columns, rows, x[0]), got[0][:rows])
    finally:
        N.lib().af_q4_free(h)


LEFT = """
import ctypes
import numpy as np
import oracle
from adaforge_amd import _native as N, hip, synth
for columns, rows, tokens in [(15360, 3840, 5), (4096, 3840, 32), (3840, 15361, 17)]:
    w = synth.q4(f"left{columns}", columns, rows, signed=True)
    xs = np.random.default_rng(rows).standard_normal((tokens, columns)).astype(np.float32)
    h = N.P()
    N.check(N.lib().af_q4_upload(w.ctypes.data_as(N.u8p), w.size, columns, rows, ctypes.byref(h)))
    xb, yb = hip.Buffer.from_numpy(xs), hip.Buffer(tokens * rows)
    for _ in range(2):
        yb.upload(np.full(tokens * rows, np.nan, np.float32))
        N.check(N.lib().af_q4_gemm(h, xb.ptr, tokens, yb.ptr, None))
        hip.synchronize()
        for t in (0, tokens - 1):
            oracle.compare(oracle.q4_matvec(w, columns, rows, xs[t]), yb.numpy().reshape(tokens, rows)[t])
print("sums complete")
"""


@pytest.mark.parametrize("left", [1, 3, 17])
def test_tickets_left_by_overlapping_calls(left):
    """Counts in the completion tickets, as two calls that overlapped on different streams may leave them (set from the
    host where the tickets are allocated): the calls that follow are complete."""
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    r = subprocess.run([sys.executable, "-c", LEFT], cwd=root, env=dict(os.environ, AF_GEMM_TICKETS_LEFT=str(left)),
                       capture_output=True, text=True, timeout=100)
    assert r.returncode == 0 and "sums complete" in r.stdout, r.stdout[-2000:] + r.stderr[-2000:]
