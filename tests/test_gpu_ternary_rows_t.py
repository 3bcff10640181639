"""ternary-rows-t by name on its matrix-core form (one row per step, the
reference's order), bit for bit against the CPU restatement: tiles of 32 and
64 positions and their edges (a handful of positions stay on the kernel of one
chain per 64 columns), row counts around its 64-row chunks, padded word
strides, partial grids, denormal products, infinities, products that overflow
only before the sum, and buffers that take the general kernel."""
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


def inputs(out, cols, wng, seq, seed=0):
    rng = np.random.default_rng(out * 1009 + cols * 31 + seq + seed)
    nblk = (cols + 127) // 128
    w = rng.integers(0, 2 ** 32, out * wng, dtype=np.uint64).astype(np.uint32).view(f32)
    beta = (np.abs(rng.standard_normal(out * nblk)) * 0.05).astype(f32)
    return w, beta, rng.standard_normal(seq * out).astype(f32), [out, cols, nblk, wng, seq]


def both(w, beta, g, push, groups=None, fill=0.0, shift=False, short=0):
    out, cols, _, _, seq = push
    x = np.full(seq * cols, fill, f32)
    devs = [nlgpu.to_device(b) for b in (w, beta, g, x)]
    bufs, gw = list(devs), g
    if shift:  # g one float into its allocation
        devs[2] = nlgpu.to_device(np.concatenate([np.zeros(1, f32), g]))

        class Off:
            def as_buffer(self, n=None):
                return nlgpu.Buffer(devs[2].ptr + 4, g.size)
        bufs[2] = Off()
    if short:  # the last values of g are not bound: they read as zeros
        bufs[2], gw = (devs[2], g.size - short), g[:g.size - short].copy()
    groups = (seq * cols + 63) // 64 if groups is None else groups
    with np.errstate(all="ignore"):
        nlgpu.dispatch("ternary-rows-t", bufs, push, groups)
        got = devs[-1].download(f32, x.size)
        want = x.copy()
        orc.dispatch("ternary-rows-t", [w.copy(), beta, gw, want], push, groups)
    return got, want


def same(got, want):
    nan = np.isnan(want)
    return np.array_equal(np.isnan(got), nan) and np.array_equal(got[~nan].view(np.uint32), want[~nan].view(np.uint32))


@pytest.mark.parametrize("seq", [1, 5, 16, 17, 32, 33, 64, 65, 130])
@pytest.mark.parametrize("out,cols,wng", [(1, 16, 1), (63, 40, 3), (64, 128, 8), (65, 300, 20), (200, 260, 17),
                                          (322, 1000, 63), (70, 17000, 1063)])
def test_ternary_rows_t_positions(seq, out, cols, wng):
    print(f"[gpu] ternary-rows-t out={out} cols={cols} wng={wng} seq={seq}", flush=True)
    assert same(*both(*inputs(out, cols, wng, seq)))


@pytest.mark.parametrize("seq,cols", [(3, 17000), (3, 200), (20, 4000), (70, 3000), (200, 5600)])
def test_ternary_rows_t_forms(seq, cols):
    w, beta, g, push = inputs(72, cols, (cols + 15) // 16, seq)
    assert same(*both(w, beta, g, push, shift=True))
    assert same(*both(w, beta, g, push, short=7))
    got, want = both(w, beta, g, push, groups=seq * cols // 64 - 2, fill=-7.0)
    assert same(got, want) and (want == -7.0).any()


def test_ternary_rows_t_too_many_positions():
    """More than 65,535 positions are refused, whichever form would take them."""
    w, beta, g, push = inputs(3, 16, 1, 65536)
    devs = [nlgpu.to_device(b) for b in (w, beta, g, np.full(16 * 65536, -7.0, f32))]
    with pytest.raises(nlgpu.NlgError, match="65535"):
        nlgpu.dispatch("ternary-rows-t", devs, push, 65536 * 16 // 64)
    assert np.all(devs[3].download(f32, 1024) == -7.0)


@pytest.mark.parametrize("seq,cols", [(2, 17000), (2, 200), (24, 2000), (66, 1300), (260, 20000)])
def test_ternary_rows_t_extremes(seq, cols):
    """Products and sums below the normal range; infinities and NaNs of G; and
    -2 x BETA*G that overflows although the sum would not."""
    wng = (cols + 15) // 16
    w, beta, g, push = inputs(140, cols, wng, seq)
    tiny = (g.astype(np.float64) * 2.0 ** -141).astype(f32)
    got, want = both(w, beta, tiny, push)
    assert same(got, want) and (np.abs(want[want != 0]) < 2.0 ** -126).any()
    bad = g.copy().reshape(seq, -1)
    bad[0, 70], bad[1, 3], bad[-1, 139] = np.inf, np.nan, -np.inf
    got, want = both(w, beta, bad.reshape(-1), push)
    assert same(got, want) and np.isnan(want).any()
    huge = np.zeros_like(g).reshape(seq, -1)
    ones = np.ones_like(beta)
    huge[:, 65], huge[:, 66] = f32(2.5e38), f32(2.4e38)
    words = w.view(np.uint32).copy().reshape(140, wng)
    words[65], words[66] = 0x55555555, 0xAAAAAAAA  # +1, then -2
    got, want = both(words.reshape(-1).view(f32), ones, huge.reshape(-1), push)
    assert same(got, want) and np.isinf(want).all()
