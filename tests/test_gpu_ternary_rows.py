"""ternary-rows by name (f32 activations) on its forms, two or four rows and
up to four tokens per wave and 32-token tiles on the bf16 matrix cores, against the CPU
restatement: edges of the tiles and of the 128-column blocks, word strides and
block counts that cover more or less than the columns, partial grids,
infinities and NaNs, buffers that are not 16-byte aligned."""
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


def inputs(seq, out, cols, nblk, wng, seed=0, scale=1.0):
    rng = np.random.default_rng(seq * 1009 + out * 31 + cols + seed)
    w = rng.integers(0, 2 ** 32, out * wng, dtype=np.uint64).astype(np.uint32).view(f32)  # code 10 (-2) included
    x = (rng.standard_normal(seq * cols) * scale).astype(f32)
    return x, w, rng.standard_normal(out).astype(f32), (np.abs(rng.standard_normal(out * nblk)) * 0.05).astype(f32)


def both(x, w, bias, beta, push, groups=None, fill=0.0, shift=False):
    seq, out = push[:2]
    y = np.full(seq * out, fill, f32)
    devs = [nlgpu.to_device(b) for b in (x, w, bias, beta, y)]
    bufs = list(devs)
    if shift:  # x one float into its allocation
        devs[0] = nlgpu.to_device(np.concatenate([np.zeros(1, f32), x]))

        class Off:
            def as_buffer(self, n=None):
                return nlgpu.Buffer(devs[0].ptr + 4, x.size)
        bufs[0] = Off()
    groups = (seq * out + 63) // 64 if groups is None else groups
    nlgpu.dispatch("ternary-rows", bufs, push, groups)
    got = devs[-1].download(f32, y.size)
    want = y.copy()
    orc.dispatch("ternary-rows", [x.copy(), w.copy(), bias, beta, want], push, groups)
    return got, want


def close(got, want, terms):
    """f32 sums of `terms` products in another order: sqrt(terms) roundings of
    half an ulp of the largest output, with a factor of eight for a row that cancels."""
    fine = np.isfinite(want)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[~fine & ~np.isnan(want)],
                                                                            want[~fine & ~np.isnan(want)])
    bar = min(1e-5, 8 * np.sqrt(terms) * 2.0 ** -24)
    assert np.max(np.abs(got[fine] - want[fine])) <= bar * np.max(np.abs(want[fine]))


@pytest.mark.parametrize("seq", [1, 2, 3, 5, 11, 12, 32, 33, 70])
@pytest.mark.parametrize("out,cols,nblk,wng", [(6, 256, 2, 16), (65, 300, 3, 19), (130, 1028, 9, 68),
                                               (64, 640, 3, 44), (33, 36, 1, 3), (129, 260, 5, 20)])
def test_ternary_rows(seq, out, cols, nblk, wng):
    print(f"[gpu] ternary-rows seq={seq} out={out} cols={cols}/{nblk} wng={wng}", flush=True)
    got, want = both(*inputs(seq, out, cols, nblk, wng), [seq, out, cols, nblk, wng])
    close(got, want, cols)


@pytest.mark.parametrize("seq,out,cols", [(200, 9400, 132), (130, 2500, 1300), (33, 8200, 132)])
def test_ternary_rows_many_tiles(seq, out, cols):
    """Enough tiles for 64- and 128-row workgroups."""
    nblk, wng = (cols + 127) // 128, (cols + 15) // 16
    got, want = both(*inputs(seq, out, cols, nblk, wng), [seq, out, cols, nblk, wng])
    close(got, want, cols)


@pytest.mark.parametrize("seq,out,cols", [(1, 8300, 256), (2, 4200, 256), (3, 2800, 256), (1, 2600, 37), (2, 2600, 37),
                                          (4, 2600, 37), (5, 2700, 302), (24, 64, 512), (25, 64, 512)])
def test_ternary_rows_many_outputs(seq, out, cols):
    """Few tokens past the counts of outputs up to which a wave takes two rows."""
    nblk, wng = (cols + 127) // 128, (cols + 15) // 16
    got, want = both(*inputs(seq, out, cols, nblk, wng), [seq, out, cols, nblk, wng])
    close(got, want, cols)


@pytest.mark.parametrize("seq,cols", [(5, 301), (40, 301), (40, 300)])
def test_ternary_rows_unaligned(seq, cols):
    out, nblk, wng = 37, 3, 19
    got, want = both(*inputs(seq, out, cols, nblk, wng), [seq, out, cols, nblk, wng], shift=True)
    close(got, want, cols)


@pytest.mark.parametrize("seq,groups", [(3, 2), (50, 40), (50, 1)])
def test_ternary_rows_partial_grid(seq, groups):
    out, cols, nblk, wng = 100, 256, 2, 16
    got, want = both(*inputs(seq, out, cols, nblk, wng), [seq, out, cols, nblk, wng], groups=groups, fill=-7.0)
    assert np.array_equal(got[64 * groups:], want[64 * groups:])
    close(got[:64 * groups], want[:64 * groups], cols)


@pytest.mark.parametrize("seq", [4, 40])
def test_ternary_rows_non_finite_and_wide(seq):
    """An infinity meets weights 0 (NaN), +-1, -2; NaN with a payload the upper
    half does not show; activations over the whole exponent range."""
    out, cols, nblk, wng = 70, 256, 2, 16
    push = [seq, out, cols, nblk, wng]
    x, w, bias, beta = inputs(seq, out, cols, nblk, wng)
    x = x.reshape(seq, cols)
    x[1, 17] = np.inf
    x[2, 200] = np.uint32(0x7f800001).view(f32)
    x[3] *= 2.0 ** 100
    w = w.view(np.uint32).reshape(out, wng)
    w[::2] |= 0x55555555  # every second row: fields 01 and 11 only, no zero
    got, want = both(x.reshape(-1), w.reshape(-1).view(f32), bias, beta, push)
    got, want = got.reshape(seq, out), want.reshape(seq, out)
    assert np.isinf(want[1]).any() and np.isnan(want[1]).any() and np.isnan(want[2]).all()
    close(got[:3].reshape(-1), want[:3].reshape(-1), cols)
    close(got[3], want[3], cols)


@pytest.mark.parametrize("seq,out", [(3, 70), (40, 70), (70, 300)])
def test_ternary_rows_tiny_activations(seq, out):
    """Rows of activations near and below the smallest normal number, whose lower
    parts no bf16 holds, each compared on its own scale (beta 1, no bias)."""
    cols, nblk, wng = 260, 3, 17
    push = [seq, out, cols, nblk, wng]
    x, w, bias, beta = inputs(seq, out, cols, nblk, wng)
    x = x.reshape(seq, cols)
    exps = [0, -90, -100, -108, -112, -115, -120, -126, -132, -140, -147]
    for r in range(seq):
        x[r] = np.ldexp(x[r].astype(np.float64), exps[r % len(exps)]).astype(f32)
    x[0, ::2] = np.ldexp(1.5, -130)  # among normal ones
    got, want = both(x.reshape(-1), w, 0 * bias, np.ones_like(beta), push)
    got, want = got.reshape(seq, out), want.reshape(seq, out)
    bar = min(1e-5, 8 * np.sqrt(cols) * 2.0 ** -24)
    for r in range(seq):
        err = np.max(np.abs(got[r].astype(np.float64) - want[r]))
        assert err <= bar * np.max(np.abs(want[r])) + cols * 2.0 ** -149, (r, exps[r % len(exps)], err, np.max(np.abs(want[r])))
