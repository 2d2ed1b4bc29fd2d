"""Prefill passes of more than 32 positions (wide_gemm_kernel, its input images and the batched
attention over whole passes) against the CPU oracle, teacher-forced per layer."""
import os

import numpy as np
import pytest

import oracle
from adaforge_amd import synth
from tests.test_gpu_batch import THREADS, open_with_env

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q_heads,kv_heads,window,intermediate,n,batch", [
    (16, 8, 16, 2048, 33, 33),     # one 64-token tile, nearly half padding
    (16, 8, 100, 2080, 64, 64),    # a full 64-token tile; FFN rows and columns off every tile
    (8, 8, 24, 1056, 150, 65),     # 128-token tiles, nearly half padding; passes of 65 + 65 + 20
    (16, 4, 64, 2048, 280, 128),   # full 128-token tiles; two passes and a narrow remainder
    (16, 8, 40, 2080, 330, 161),   # two 128-token tiles, the second mostly padding; the ring wraps inside the pass
    (16, 8, 1024, 2048, 530, 512), # the largest pass, then a narrow one
])
def test_wide_trace_teacher_forced(q_heads, kv_heads, window, intermediate, n, batch):
    """Layer outputs within the oracle's tolerance (|gpu - ref| <= 1e-4 + 1e-4 |ref|) and K/V within one
    fp16 ulp at tile, window and pass boundaries."""
    model = synth.model(name=f"wide{q_heads}x{kv_heads}", layers=3, hidden=1024, intermediate=intermediate,
                        q_heads=q_heads, kv_heads=kv_heads, head_width=256, vocabulary=2048, window=window,
                        global_every=3)
    ids = [int(i) for i in synth.prompt_ids(n, model.vocabulary, name=f"wide{n}.ids")]
    with open_with_env(model, n + 8, AF_TRACE_BATCH=batch) as s:
        outputs, kv, logits, hidden = s.trace(ids, kv_rows=kv_heads * 256)
    marks = {0, 1, 15, 16, 31, 32, 63, 64, 127, 128, window - 1, window, batch - 1, batch, batch + 1, n - 1}
    positions = sorted(p for p in marks if 0 <= p < n)
    ratio, ulps, differ = oracle.check_layer_stack(model, ids, outputs, kv, threads=THREADS, positions=positions)
    print(f"wide trace n={n} batch={batch}: layer ratio {ratio:.3f}, K/V ratio {ulps:.3f}, {differ} fp16 values differ",
          flush=True)
    nrm = oracle.rmsnorm(model.final_norm, model.final_eps, hidden).astype(np.float32)
    oracle.compare(oracle.q6_matvec(model.table, model.hidden, model.vocabulary, nrm, threads=THREADS), logits)


@pytest.mark.parametrize("hidden,intermediate,n", [
    (1024, 4128, 33),     # two octets per thread in the down projection's image, the second nearly empty; 64-token tile
    (1024, 8192, 64),     # both whole
    (1024, 15360, 65),    # four octets per thread, the last not whole; splits of a long K, 128-token tiles
    (3840, 15360, 128),   # the 12B shape
    (1024, 16384, 200),   # the longest K
    (3840, 15360, 512),   # the largest pass
])
def test_wide_trace_long_columns(hidden, intermediate, n):
    """Down projections of 4,128 to 16,384 columns (the image's wider forms, more splits of K) per layer against the oracle."""
    model = synth.model(name=f"long{hidden}x{intermediate}", layers=1, hidden=hidden, intermediate=intermediate, q_heads=16,
                        kv_heads=8, head_width=256, vocabulary=2048, window=1024, global_every=2)
    ids = [int(i) for i in synth.prompt_ids(n, model.vocabulary, name=f"long{n}.ids")]
    with open_with_env(model, n + 8, AF_TRACE_BATCH=512) as s:
        outputs, kv, _, _ = s.trace(ids, kv_rows=8 * 256, logits=False, hidden=False)
    positions = sorted({p for p in (0, 15, 16, 31, 32, 63, 64, 127, 128, 255, 256, n - 1) if p < n})
    ratio, ulps, differ = oracle.check_layer_stack(model, ids, outputs, kv, threads=THREADS, positions=positions)
    print(f"long columns {hidden}x{intermediate} n={n}: layer ratio {ratio:.3f}, K/V ratio {ulps:.3f}, {differ} fp16 "
          f"values differ", flush=True)


def test_wide_trace_gemma4_width_512_shared_v():
    """The 512-wide global layer (16 query heads on one KV head, V from K's weights) in wide passes."""
    model = synth.gemma4_model(name="gemma4-wide", layers=6, hidden=1024, intermediate=2048, local_q=(16, 8, 256),
                               global_q=(16, 1, 512), vocabulary=2048, window=48)
    n = 150
    ids = [int(i) for i in synth.prompt_ids(n, model.vocabulary, name="gemma4-wide.ids")]
    kv_rows = max(L.kv_heads * L.head_width for L in model.layers)
    with open_with_env(model, n + 8, AF_TRACE_BATCH=100) as s:
        outputs, kv, _, _ = s.trace(ids, kv_rows=kv_rows, logits=False, hidden=False)
    positions = [0, 1, 15, 16, 47, 48, 63, 64, 99, 100, 101, 147, 149]
    ratio, ulps, differ = oracle.check_layer_stack(model, ids, outputs, kv, threads=THREADS, positions=positions)
    print(f"gemma4 wide: layer ratio {ratio:.3f}, K/V ratio {ulps:.3f}, {differ} fp16 values differ", flush=True)


def one_channel_model(name, special, q_heads=16, **kw):
    """A one-layer model whose embeddings are zero in channel 5 for every id not in `special`, and large there."""
    model = synth.model(name=name, layers=1, hidden=1024, q_heads=q_heads, kv_heads=8, head_width=256,
                        vocabulary=2048, **kw)
    rows = model.table.reshape(model.vocabulary, model.hidden // 256, 210)  # Q6_K: ql[128], qh[64], scales, d
    keep = np.isin(np.arange(model.vocabulary), special)
    rows[~keep, 0, 5] &= 0xF0
    rows[~keep, 0, 128 + 5] = rows[~keep, 0, 128 + 5] & 0xFC | 2  # code 32: weight 0
    rows[keep, 0, 5] |= 0x0F
    rows[keep, 0, 128 + 5] |= 3  # code 63: weight 31
    rows[keep, 0, 192] = 127     # (the scale of channels 0-15)
    return model


def zero_block(matrix, columns):
    """The Q4_0 matrix with the scales of its first 32 columns' blocks zero."""
    blocks = matrix.reshape(-1, columns // 32, 18)
    blocks[:, 0, :2] = 0
    return matrix


@pytest.mark.parametrize("n", [40, 100])
def test_wide_trace_keeps_small_blocks_beside_an_outlier(n):
    """A channel 2^30 above the others in some tokens' GEMM inputs, in a block whose weights are zero: the
    products come from the small blocks alone and are as exact as without it (K/V within one fp16 ulp, layer
    outputs within the oracle's tolerance)."""
    ids = [int(i) for i in synth.prompt_ids(n, 2048, name=f"outlier{n}.ids")]
    model = one_channel_model(f"outlier{n}", ids[3::2], intermediate=2048, window=0, global_every=1)
    L = model.layers[0]
    L.input_norm[5] = L.ffn_norm[5] = np.float32(2.0 ** 30)
    for m in (L.q, L.k, L.v, L.gate, L.up):
        zero_block(m, model.hidden)
    with open_with_env(model, n + 8, AF_TRACE_BATCH=512) as s:
        outputs, kv, _, _ = s.trace(ids, kv_rows=8 * 256, logits=False, hidden=False)
    positions = [0, 1, 2, 3, 4, 15, 16, 31, 32, n - 2, n - 1]
    ratio, ulps, differ = oracle.check_layer_stack(model, ids, outputs, kv, threads=THREADS, positions=positions)
    print(f"outlier n={n}: layer ratio {ratio:.3f}, K/V ratio {ulps:.3f}, {differ} fp16 values differ", flush=True)


@pytest.mark.parametrize("n", [40, 100])
def test_wide_trace_non_finite_token(n):
    """One token's GEMM input overflows fp32 (beside other tokens and the tile's padding): no position that does not see
    it changes."""
    at, window = 19, 8
    ids = [int(i) for i in synth.prompt_ids(n, 2047, name=f"nonfinite{n}.ids")]
    ids[at] = 2047
    model = one_channel_model(f"nonfinite{n}", [2047], intermediate=2048, window=window, global_every=2)
    model.layers[0].input_norm[5] = np.float32(3e38)
    with open_with_env(model, n + 8, AF_TRACE_BATCH=512) as s:
        outputs, kv, _, _ = s.trace(ids, kv_rows=8 * 256, logits=False, hidden=False)
    assert not np.isfinite(kv[at]).any() and np.isfinite(np.delete(kv, at, 0)).all()
    kv[at] = 0.0  # (seen by none of these; the oracle takes finite histories)
    positions = [p for p in (0, 15, 16, 18, 27, 31, 32, 33, 39, 47, 48, 63, 64, 65, 99) if p < n]
    oracle.check_layer_stack(model, ids, outputs, kv, threads=THREADS, positions=positions)


@pytest.mark.parametrize("batch", [32, 512])
@pytest.mark.parametrize("q_heads,window", [(8, 0), (16, 24), (32, 24)])
def test_overflowed_value_reaches_only_the_positions_that_see_it(q_heads, window, batch):
    """One position's V overflows fp16: positions before it, and those whose window it has left, are as
    without it, also in its own tile of queries."""
    n, at = 130, 45
    ids = [int(i) for i in synth.prompt_ids(n, 2047, name="overflow.ids")]
    ids[at] = 2047
    model = one_channel_model("overflow", [2047], q_heads=q_heads, intermediate=2048, window=window,
                              global_every=2 if window else 1)
    L = model.layers[0]
    first = L.v.reshape(8 * 256, model.hidden // 32, 18)[0, 0]  # row 0, columns 0-31: only channel 5 weighs
    first[:2] = np.frombuffer(np.float16(60000.0).tobytes(), np.uint8)
    first[2:] = 0x88
    first[2 + 5] = 0x8F
    with open_with_env(model, n + 8, AF_TRACE_BATCH=batch) as s:
        outputs, kv, _, _ = s.trace(ids, kv_rows=8 * 256, logits=False, hidden=False)
    assert np.isinf(kv[at, 0, 1, 0]) and np.isfinite(np.delete(kv, at, 0)).all()
    sees = np.arange(n) >= at
    if window:
        sees &= np.arange(n) < at + window
    bad = ~np.isfinite(outputs[:, 0]).all(axis=1)
    assert np.array_equal(bad, sees), np.nonzero(bad != sees)[0]
    kv[at] = 0.0  # (seen by none of these; the oracle takes finite histories)
    positions = [p for p in (0, 15, 16, 31, 32, 40, 44, 63, 64, 69, 70, 95, 96, 129) if not sees[p]]
    oracle.check_layer_stack(model, ids, outputs, kv, threads=THREADS, positions=positions)


@pytest.mark.parametrize("batch", [32, 100])
def test_batched_trace_of_tiny_queries(batch):
    """Queries of about 2^-130 (a subnormal query norm): every key weighs the same, in narrow and wide passes."""
    model = synth.model(name="tinyq", layers=1, hidden=1024, intermediate=2048, q_heads=16, kv_heads=8, head_width=256,
                        vocabulary=2048, window=64, global_every=2)
    model.layers[0].q_norm *= np.float32(2.0 ** -130)
    n = 100
    ids = [int(i) for i in synth.prompt_ids(n, model.vocabulary, name="tinyq.ids")]
    with open_with_env(model, n + 8, AF_TRACE_BATCH=batch) as s:
        outputs, kv, _, _ = s.trace(ids, kv_rows=8 * 256, logits=False, hidden=False)
    oracle.check_layer_stack(model, ids, outputs, kv, threads=THREADS, positions=[0, 1, 31, 32, 63, 64, 99])


def test_wide_pass_is_no_less_exact_than_narrow_ones():
    """A layer's error against the oracle over 512 positions: in one pass no larger than in passes of 32 (scores
    summed in one chain made it 3 % larger)."""
    model = synth.model(name="exact", layers=1, hidden=1024, intermediate=2048, q_heads=16, kv_heads=8, head_width=256,
                        vocabulary=2048, window=1024, global_every=2)
    n = 512
    ids = np.array(synth.prompt_ids(n, model.vocabulary, name="exact.ids"), np.uint32)
    emb = np.concatenate([oracle.embedding(model.table, 1024, 2048, ids[i:i + 256]) for i in (0, 256)]).reshape(n, -1)
    table, error = oracle.layer_table(model), []
    for batch in (32, 512):
        with open_with_env(model, n + 8, AF_TRACE_BATCH=batch) as s:
            out, kv, _, _ = s.trace(ids, kv_rows=8 * 256, logits=False, hidden=False)
        num = den = 0.0
        for t in range(1, n, 3):
            k, v = (np.ascontiguousarray(kv[:t + 1, 0, i]) for i in (0, 1))
            ref = oracle.layer_forward(model, table, 0, emb[t], k, v, t, given_kv=True, threads=THREADS)[0].astype(np.float64)
            num += ((out[t, 0] - ref) ** 2).sum()
            den += (ref ** 2).sum()
        error.append((num / den) ** 0.5)
    print(f"layer error over {n} positions: {error[0]:.3e} in passes of 32, {error[1]:.3e} in one", flush=True)
    assert error[1] <= error[0]


def test_wide_prefill_ids_match_one_position_at_a_time():
    """Greedy ids after a 300-token prompt: one wide pass against one step-kernel launch per position, and
    again on a follow-up turn whose pass starts in the middle of the ring."""
    model = synth.model(name="wide-gen", layers=3, hidden=1024, intermediate=2048, q_heads=16, kv_heads=8,
                        head_width=256, vocabulary=2048, window=64, global_every=3)
    prompt = [int(i) for i in synth.prompt_ids(300, model.vocabulary, name="wide-gen.prompt")]
    more = [int(i) for i in synth.prompt_ids(90, model.vocabulary, name="wide-gen.more")]
    got = []
    for batch in (512, 0):
        with open_with_env(model, 420, AF_PREFILL_BATCH=batch) as s:
            first = s.generate(prompt, [2047], 8)
            got.append((first.ids, s.generate(prompt + first.ids + more, [2047], 8).ids))
    assert got[0] == got[1]
