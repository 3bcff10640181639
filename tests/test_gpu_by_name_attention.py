"""attn-causal-gqa by name on its matrix-core form (full float4 rows, head dims
32, 64, 80, 96, 128) against the CPU restatement, at the sizes where it can go
wrong: the edges of its 32-query tiles and 32-key blocks, one to four key
blocks per wave, every instantiated head dim, partial grids, a V of infinities
and NaNs after a query, and buffers that take the general kernel instead.
decode-attn(-b) on its split form likewise: every lanes-per-row form, one and
many workgroups per head (a call under capture takes one), positions at the
edges of its blocks and past the cache, NaN in every row not attended."""
import gc

import numpy as np
import pytest

import nlg_oracle as orc
import nlgpu

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nlgpu.init()
    yield


def inputs(seq, heads, kvh, hd, seed=0):
    rng = np.random.default_rng(seq * 131 + heads * 7 + hd + seed)
    q = (rng.standard_normal(seq * heads * hd) * 1.5).astype(f32)
    return q, rng.standard_normal(seq * kvh * hd).astype(f32), rng.standard_normal(seq * kvh * hd).astype(f32)


def both(q, k, v, push, groups, fill=0.0):
    out = np.full(push[0] * push[1] * push[3], fill, f32)
    devs = [nlgpu.to_device(b) for b in (q, k, v, out)]
    nlgpu.dispatch("attn-causal-gqa", devs, push, groups)
    got = devs[-1].download(f32, out.size)
    want = out.copy()
    orc.dispatch("attn-causal-gqa", [q.copy(), k.copy(), v.copy(), want], push, groups)
    return got, want


# f32 sums of at most 200 terms of size ~1 in another order, relative to the
# largest output: 200 x 2^-24 = 1.2e-5 in the worst case, 1e-5 is the bar the
# by-name cases state
@pytest.mark.parametrize("hd", [32, 64, 80, 96, 128])
@pytest.mark.parametrize("seq,heads,kvh", [(1, 4, 2), (31, 4, 4), (32, 8, 2), (33, 4, 1), (65, 6, 3), (200, 4, 2)])
def test_prompt_attention_f32(seq, heads, kvh, hd):
    print(f"[gpu] attn-causal-gqa seq={seq} heads={heads}/{kvh} hd={hd}", flush=True)
    q, k, v = inputs(seq, heads, kvh, hd)
    got, want = both(q, k, v, [seq, heads, kvh, hd], (heads * seq + 63) // 64)
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))


@pytest.mark.parametrize("hd", [32, 64, 80, 96, 128])
@pytest.mark.parametrize("seq", [2, 5, 6, 7, 8, 9])
def test_prompt_attention_f32_few_queries(seq, hd):
    """On both sides of the lengths up to which the walk over the keys is taken."""
    q, k, v = inputs(seq, 6, 3, hd)
    got, want = both(q, k, v, [seq, 6, 3, hd], (6 * seq + 63) // 64)
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))


# 2-norm error against 64 bits.  A score rounded after each of 128 dimensions is
# off by ~sqrt(128 / 2) half-ulps of its size, one summed in chains of 8 that meet
# in pairs by ~sqrt(4 + 4); the first shows as 2.1e-7 of the result at 40
# positions, the second as 1.06e-7, the rest (exponentials, sums) as 0.9e-7.
@pytest.mark.parametrize("seq,hd,bar", [(40, 128, 1.5e-7), (40, 96, 1.5e-7), (300, 128, 2.1e-7)])
def test_prompt_attention_f32_precision(seq, hd, bar):
    heads, kvh = 8, 2
    print(f"[gpu] attn-causal-gqa precision seq={seq} hd={hd}", flush=True)
    q, k, v = inputs(seq, heads, kvh, hd)
    q = (q / 1.5).astype(f32)
    out = np.zeros(q.size, f32)
    devs = [nlgpu.to_device(b) for b in (q, k, v, out)]
    nlgpu.dispatch("attn-causal-gqa", devs, [seq, heads, kvh, hd], (heads * seq + 63) // 64)
    got = devs[-1].download(f32, out.size).reshape(seq, heads, hd).astype(np.float64)
    q64, k64, v64 = (b.astype(np.float64).reshape(seq, -1, hd) for b in (q, k, v))
    s = np.einsum("qhd,khd->hqk", q64, np.repeat(k64, heads // kvh, axis=1)) / np.sqrt(hd)
    s = np.where(np.tril(np.ones((seq, seq), bool)), s, -np.inf)
    p = np.exp(s - s.max(axis=2, keepdims=True))
    p /= p.sum(axis=2, keepdims=True)
    want = np.einsum("hqk,khd->qhd", p, np.repeat(v64, heads // kvh, axis=1))
    assert np.linalg.norm(got - want) <= bar * np.linalg.norm(want)


@pytest.mark.parametrize("groups", [1, 3, 5])
def test_prompt_attention_f32_partial_grid(groups):
    seq, heads, kvh, hd = 75, 6, 2, 64
    print(f"[gpu] attn-causal-gqa partial grid groups={groups}", flush=True)
    q, k, v = inputs(seq, heads, kvh, hd)
    got, want = both(q, k, v, [seq, heads, kvh, hd], groups, fill=-7.0)
    untouched = want == -7.0
    assert untouched.any() and np.array_equal(got[untouched], want[untouched])
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))


@pytest.mark.parametrize("hd,at", [(64, 40), (128, 5), (80, 69)])
def test_prompt_attention_f32_values_not_attended(hd, at):
    """Position `at` of V is Inf, -Inf or NaN by column: only the queries from
    `at` on see it."""
    seq, heads, kvh = 70, 4, 2
    print(f"[gpu] attn-causal-gqa non-finite V hd={hd} at={at}", flush=True)
    q, k, v = inputs(seq, heads, kvh, hd)
    row = v.reshape(seq, kvh * hd)
    row[at, 0::3], row[at, 1::3], row[at, 2::7] = np.inf, -np.inf, np.nan
    got, want = both(q, k, v, [seq, heads, kvh, hd], (heads * seq + 63) // 64)
    fine = np.isfinite(want)
    assert np.array_equal(np.isfinite(got), fine) and np.array_equal(np.isnan(got), np.isnan(want))
    assert np.array_equal(got[~fine & ~np.isnan(want)], want[~fine & ~np.isnan(want)])
    assert np.max(np.abs(got[fine] - want[fine])) <= 1e-5 * np.max(np.abs(want[fine]))


def test_prompt_attention_f32_scores_of_minus_infinity():
    """Keys of -Inf scores: a row that attends nothing else divides 0 by 0, as
    the reference's seeded maximum does."""
    seq, heads, kvh, hd = 40, 2, 1, 64
    q, k, v = inputs(seq, heads, kvh, hd)
    q = np.abs(q)
    k.reshape(seq, hd)[:3] = -np.inf
    got, want = both(q, k, v, [seq, heads, kvh, hd], (heads * seq + 63) // 64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.isnan(want).any()
    fine = np.isfinite(want)
    assert np.max(np.abs(got[fine] - want[fine])) <= 1e-5 * np.max(np.abs(want[fine]))


@pytest.mark.parametrize("form", ["short", "unaligned", "heads"])
def test_prompt_attention_f32_general_form(form):
    """Forms the matrix-core kernel does not take: a short V (read as zeros), a
    Q that is not 16-byte aligned, heads that are no multiple of the kv heads."""
    seq, heads, kvh, hd = 37, 5 if form == "heads" else 4, 2, 64
    print(f"[gpu] attn-causal-gqa general form: {form}", flush=True)
    q, k, v = inputs(seq, heads, kvh, hd)
    out = np.zeros(seq * heads * hd, f32)
    push, groups = [seq, heads, kvh, hd], (heads * seq + 63) // 64
    devs = [nlgpu.to_device(b) for b in (q, k, v, out)]
    bufs, short = list(devs), v.copy()
    if form == "short":
        bufs[2] = (devs[2], v.size - 3 * hd)
        short = v[:v.size - 3 * hd].copy()
    if form == "unaligned":
        devs[0] = nlgpu.to_device(np.concatenate([np.zeros(1, f32), q]))

        class Off:
            def as_buffer(self, n=None):
                return nlgpu.Buffer(devs[0].ptr + 4, q.size)
        bufs[0] = Off()
    nlgpu.dispatch("attn-causal-gqa", bufs, push, groups)
    got = devs[-1].download(f32, out.size)
    want = out.copy()
    orc.dispatch("attn-causal-gqa", [q.copy(), k.copy(), short, want], push, groups)
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))


def decode_inputs(batch, heads, kvh, hd, maxseq, seed=0):
    rng = np.random.default_rng(batch * 31 + heads * 7 + hd + maxseq + seed)
    q = (rng.standard_normal(batch * heads * hd) * 1.5).astype(f32)
    n = batch * maxseq * kvh * hd
    return q, rng.standard_normal(n).astype(f32), rng.standard_normal(n).astype(f32)


def decode_both(q, k, v, pos, push, groups=None, fill=0.0, stale=np.nan, graph=False):
    """The split decode attention and the oracle; rows past `pos` of every
    sequence hold `stale` on the device (nobody attends them)."""
    batch, dim, heads, kvh, maxseq = push
    kvd = kvh * (dim // heads)
    kd, vd = k.copy(), v.copy()
    for x in (kd, vd):
        x.reshape(batch, maxseq, kvd)[:, pos + 1:] = stale
    out = np.full(batch * dim, fill, f32)
    devs = [nlgpu.to_device(b) for b in (q, kd, vd, np.array([pos], f32), out)]
    groups = (batch * dim + 63) // 64 if groups is None else groups
    if graph:
        s = nlgpu.lib().nlg_stream_create()
        nlgpu.graph_begin(s)
        nlgpu.dispatch("decode-attn-b", devs, push, groups, stream=s)
        g = nlgpu.graph_end(s)
        for _ in range(3):
            devs[-1].upload(out)
            nlgpu.graph_launch(g, s)
            nlgpu.sync(s)
        nlgpu.graph_destroy(g)
        nlgpu.lib().nlg_stream_destroy(s)
    else:
        nlgpu.dispatch("decode-attn-b", devs, push, groups)
    got = devs[-1].download(f32, out.size)
    want = out.copy()
    orc.dispatch("decode-attn-b", [q.copy(), k.copy(), v.copy(), np.array([pos], f32), want], push, groups)
    return got, want


# sums of up to 1,500 terms, the error of a random order about sqrt(1500) x
# 2^-24 = 2e-6 of the output: the 1e-5 bar the by-name cases state
@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("batch,heads,kvh,hd,maxseq,pos", [
    (1, 4, 1, 128, 40, 0), (2, 4, 2, 128, 300, 15), (1, 20, 5, 128, 1500, 1499), (3, 6, 2, 64, 700, 511),
    (2, 8, 8, 80, 260, 129), (1, 14, 2, 96, 600, 513), (2, 4, 2, 256, 200, 64), (40, 16, 16, 32, 33, 20),
    (1, 5, 5, 20, 77, 76)])
def test_decode_attention_f32(batch, heads, kvh, hd, maxseq, pos, graph):
    print(f"[gpu] decode-attn-b batch={batch} heads={heads}/{kvh} hd={hd} pos={pos}/{maxseq} graph={graph}", flush=True)
    q, k, v = decode_inputs(batch, heads, kvh, hd, maxseq)
    got, want = decode_both(q, k, v, pos, [batch, heads * hd, heads, kvh, maxseq], graph=graph)
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))


@pytest.mark.parametrize("pos", [299, 300, 1000])
def test_decode_attention_f32_past_the_cache(pos):
    """Positions past the last sequence's rows read as zeros: score 0, no V."""
    batch, heads, kvh, hd, maxseq = 1, 4, 2, 64, 300
    q, k, v = decode_inputs(batch, heads, kvh, hd, maxseq)
    got, want = decode_both(q, k, v, pos, [batch, heads * hd, heads, kvh, maxseq])
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))


def test_decode_attention_f32_partial_grid_and_single():
    batch, heads, kvh, hd, maxseq, pos = 3, 4, 2, 64, 130, 100
    q, k, v = decode_inputs(batch, heads, kvh, hd, maxseq)
    got, want = decode_both(q, k, v, pos, [batch, heads * hd, heads, kvh, maxseq], groups=5, fill=-7.0)
    assert np.array_equal(got[320:], want[320:]) and np.all(want[320:] == -7.0)
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))
    one = maxseq * kvh * hd
    out = np.zeros(heads * hd, f32)
    bufs = [q[:heads * hd], k[:one], v[:one], np.array([pos], f32), out]
    devs = [nlgpu.to_device(b) for b in bufs]
    nlgpu.dispatch("decode-attn", devs, [heads * hd, heads, kvh], 4)
    want = out.copy()
    orc.dispatch("decode-attn", [b.copy() for b in bufs[:4]] + [want], [heads * hd, heads, kvh], 4)
    assert np.max(np.abs(devs[-1].download(f32, out.size) - want)) <= 1e-5 * np.max(np.abs(want))


def test_decode_attention_f32_more_units_than_a_grid_holds():
    """2^23 (sequence, kv head) pairs: 512 threads each are more than a grid's x
    dimension holds, 256 are not."""
    batch, heads, hd = 1 << 21, 4, 4
    n = batch * heads * hd
    print(f"[gpu] decode-attn-b batch={batch}", flush=True)
    v = np.random.default_rng(3).standard_normal(n).astype(f32)
    dv = nlgpu.to_device(v)
    out = nlgpu.to_device(np.zeros(n, f32))
    nlgpu.dispatch("decode-attn-b", [dv, dv, dv, nlgpu.to_device(np.array([0], f32)), out], [batch, heads * hd, heads, heads, 1],
                   n // 64)
    assert np.array_equal(out.download(f32, n), v)  # one position: its values


def test_decode_attention_f32_infinities():
    """An attended V of infinities and an attended K whose score is NaN."""
    batch, heads, kvh, hd, maxseq, pos = 1, 4, 2, 64, 200, 150
    for bad in ("v", "k"):
        q, k, v = decode_inputs(batch, heads, kvh, hd, maxseq)
        x = (v if bad == "v" else k).reshape(maxseq, kvh, hd)
        x[40, 0, :] = np.inf if bad == "v" else np.nan
        got, want = decode_both(q, k, v, pos, [batch, heads * hd, heads, kvh, maxseq])
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        fine = np.isfinite(want)
        assert fine.any() and not fine.all()
        assert np.max(np.abs(got[fine] - want[fine])) <= 1e-5 * np.max(np.abs(want[fine]))


@pytest.mark.parametrize("graph", [False, True])
@pytest.mark.parametrize("size", [1e8, 1e10, 5e10, 1e15, 1e20])
@pytest.mark.parametrize("heads,kvh,hd,maxseq,pos", [(4, 2, 128, 600, 0), (6, 2, 64, 300, 299), (8, 2, 128, 700, 511),
                                                     (2, 2, 256, 200, 150)])
def test_decode_attention_f32_large_scores(heads, kvh, hd, maxseq, pos, size, graph):
    """q.k of any finite size.  Where every key is the same the values' mean is the
    answer; where they differ by far more than 1 the largest score's value is."""
    print(f"[gpu] decode-attn-b scores of {size:g} heads={heads}/{kvh} hd={hd} pos={pos} graph={graph}", flush=True)
    q, k, v = decode_inputs(1, heads, kvh, hd, maxseq, seed=5)
    push = [1, heads * hd, heads, kvh, maxseq]
    val = v.reshape(maxseq, kvh, hd)[:pos + 1].astype(np.float64)
    same = np.tile(k[:kvh * hd], maxseq).copy()
    dots = np.einsum("hd,hd->h", q.reshape(heads, hd).astype(np.float64),
                     np.repeat(same[:kvh * hd].reshape(kvh, hd), heads // kvh, axis=0))
    qs = (q.reshape(heads, hd) * (size / np.abs(dots))[:, None]).astype(f32).reshape(-1)
    got, _ = decode_both(qs, same, v, pos, push, graph=graph)
    mean = np.repeat(val.mean(axis=0), heads // kvh, axis=0).reshape(-1)
    assert np.max(np.abs(got - mean)) <= 1e-5 * np.max(np.abs(val))
    got, _ = decode_both(qs, k, v, pos, push, graph=graph)
    s = np.einsum("hd,jhd->jh", qs.reshape(heads, hd).astype(np.float64),
                  np.repeat(k.reshape(maxseq, kvh, hd)[:pos + 1], heads // kvh, axis=1))
    top = s.max(axis=0)
    for h in range(heads):
        near = s[:, h] >= top[h] - max(1e-4 * abs(top[h]), 1e3 * np.sqrt(hd))
        if near.sum() == 1:  # an f32 score is good to ~1e-6 of itself
            assert np.max(np.abs(got.reshape(heads, hd)[h] - val[int(s[:, h].argmax()), h // (heads // kvh)])) <= 1e-5


# 2-norm error against 64 bits at 34 positions: the per-position kernel's own is 1.26e-7
@pytest.mark.parametrize("hd", [64, 128])
def test_decode_attention_f32_precision(hd):
    batch, heads, kvh, maxseq, pos = 16, 20, 5, 60, 33
    q, k, v = decode_inputs(batch, heads, kvh, hd, maxseq, seed=9)
    q = (q / 1.5).astype(f32)
    got, _ = decode_both(q, k, v, pos, [batch, heads * hd, heads, kvh, maxseq])
    q64 = q.astype(np.float64).reshape(batch, heads, hd)
    k64, v64 = (np.repeat(x.astype(np.float64).reshape(batch, maxseq, kvh, hd)[:, :pos + 1], heads // kvh, axis=2)
                for x in (k, v))
    s = np.einsum("bhd,bjhd->bhj", q64, k64) / np.sqrt(hd)
    p = np.exp(s - s.max(axis=2, keepdims=True))
    want = np.einsum("bhj,bjhd->bhd", p / p.sum(axis=2, keepdims=True), v64).reshape(-1)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    print(f"[gpu] decode-attn-b error against 64 bits, head dim {hd}: {err:.3g}", flush=True)
    assert err <= 1.3e-7


def test_decode_attention_f32_general_form():
    """K shorter than V by part of a row: the general kernel (zeros past it)."""
    batch, heads, kvh, hd, maxseq, pos = 1, 4, 2, 64, 90, 89
    q, k, v = decode_inputs(batch, heads, kvh, hd, maxseq)
    push, out = [batch, heads * hd, heads, kvh, maxseq], np.zeros(heads * hd, f32)
    devs = [nlgpu.to_device(b) for b in (q, k, v, np.array([pos], f32), out)]
    nlgpu.dispatch("decode-attn-b", [devs[0], (devs[1], k.size - 70)] + devs[2:], push, 4)
    want = out.copy()
    orc.dispatch("decode-attn-b", [q.copy(), k[:k.size - 70].copy(), v.copy(), np.array([pos], f32), want], push, 4)
    assert np.max(np.abs(devs[-1].download(f32, out.size) - want)) <= 1e-5 * np.max(np.abs(want))


def test_a_collection_inside_a_capture_frees_nothing():
    """An array that only a dead reference cycle holds is freed before a capture
    begins, not by a collection that falls inside it."""
    x = np.arange(256, dtype=f32)
    devs = [nlgpu.to_device(b) for b in (x, x, np.zeros(256, f32))]
    s = nlgpu.lib().nlg_stream_create()
    cycle = [nlgpu.DeviceArray(4096)]
    cycle.append(cycle)
    del cycle
    nlgpu.graph_begin(s)
    gc.collect()
    nlgpu.dispatch("vadd", devs, [256], 4, stream=s)
    g = nlgpu.graph_end(s)
    for _ in range(3):
        nlgpu.graph_launch(g, s)
        nlgpu.sync(s)
        assert np.array_equal(devs[2].download(f32, 256), 2 * x)
    nlgpu.graph_destroy(g)
    nlgpu.lib().nlg_stream_destroy(s)


def test_decode_attention_f32_beside_a_capture():
    """A call whose scratch is allocated while another stream of the thread is
    being captured: it runs, and the capture stays valid."""
    batch, heads, kvh, hd, maxseq, pos = 2, 4, 2, 64, 900, 800
    q, k, v = decode_inputs(batch, heads, kvh, hd, maxseq)
    push, groups = [batch, heads * hd, heads, kvh, maxseq], (batch * heads * hd + 63) // 64
    x = np.arange(256, dtype=f32)
    adds = [nlgpu.to_device(b) for b in (x, 2 * x, np.zeros(256, f32))]
    devs = [nlgpu.to_device(b) for b in (q, k, v, np.array([pos], f32), np.zeros(batch * heads * hd, f32))]
    captured, other = nlgpu.lib().nlg_stream_create(), nlgpu.lib().nlg_stream_create()
    nlgpu.graph_begin(captured)
    nlgpu.dispatch("vadd", adds, [256], 4, stream=captured)
    rc = nlgpu.dispatch("decode-attn-b", devs, push, groups, stream=other, check=False)
    nlgpu.dispatch("vadd", [adds[2], adds[0], adds[2]], [256], 4, stream=captured)
    g = nlgpu.graph_end(captured)
    assert rc == 0, nlgpu.last_error()
    nlgpu.sync(other)
    for _ in range(3):
        nlgpu.graph_launch(g, captured)
        nlgpu.sync(captured)
        assert np.array_equal(adds[2].download(f32, 256), 4 * x)
    nlgpu.graph_destroy(g)
    want = np.zeros(batch * heads * hd, f32)
    orc.dispatch("decode-attn-b", [q.copy(), k.copy(), v.copy(), np.array([pos], f32), want], push, groups)
    assert np.max(np.abs(devs[-1].download(f32, want.size) - want)) <= 1e-5 * np.max(np.abs(want))
    nlgpu.lib().nlg_stream_destroy(captured)
    nlgpu.lib().nlg_stream_destroy(other)
