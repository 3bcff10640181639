"""attn-causal-gqa by name on its matrix-core form (full float4 rows, head dims
32, 64, 80, 96, 128) against the CPU restatement, at the sizes where it can go
wrong: the edges of its 32-query tiles and 32-key blocks, one to four key
blocks per wave, every instantiated head dim, partial grids, a V of infinities
and NaNs after a query, and buffers that take the general kernel instead."""
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
