"""The f32 products by name on their larger tiles (32 x 32, 64 x 32 and 64 x
64 outputs, chosen by their estimated time: tests/test_mm_tile.py), bit for bit against the CPU
restatement: ragged rows and columns, k at and around the LDS stages, aligned
and unaligned row lengths, partial grids, -0 biases."""
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


def check(name, m, k, n, groups=None, seed=0):
    print(f"[gpu] {name} {m}x{k}x{n} groups={groups}", flush=True)
    rng = np.random.default_rng(m * 7 + k * 3 + n + seed)
    a = rng.standard_normal(m * k).astype(f32)
    b = rng.standard_normal(k * n).astype(f32)
    a[::5] = 0.0
    b[::7] *= f32(-0.0)
    c = np.full(m * n, -7.0, f32)
    bufs = [a, b] + ([np.where(np.arange(n) % 3, rng.standard_normal(n), -0.0).astype(f32)] if name == "linear" else []) + [c]
    full = {"matmul-tiled": ((m + 15) // 16) * ((n + 15) // 16), "matmul-reg": (m * n // 16 + 63) // 64}
    groups = full.get(name, (m * n + 63) // 64) if groups is None else groups
    devs = [nlgpu.to_device(x) for x in bufs]
    nlgpu.dispatch(name, devs, [m, k, n], groups)
    got = devs[-1].download(f32, c.size)
    want = c.copy()
    orc.dispatch(name, [x.copy() for x in bufs[:-1]] + [want], [m, k, n], groups)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("name", ["matmul", "matmul-tiled", "linear"])
@pytest.mark.parametrize("m,k,n", [(512, 32, 512), (530, 33, 515), (520, 1, 516), (16, 70, 9000),
                                   (1024, 40, 1024), (1030, 31, 1027), (40, 64, 20000),
                                   (2048, 20, 2048), (2050, 17, 2041), (2052, 48, 2044),
                                   (2040, 17, 2035), (2036, 48, 2044), (33, 36, 8200), (1, 40, 32000)])
def test_tiles_bit_exact(name, m, k, n):
    check(name, m, k, n)


@pytest.mark.parametrize("m,k,n", [(512, 36, 516), (1028, 32, 1024), (2052, 8, 2048)])
def test_register_blocks_bit_exact(m, k, n):
    check("matmul-reg", m, k, n)
    check("matmul-reg", m, k, n, groups=m * n // 16 // 64 - 5)


@pytest.mark.parametrize("m,k,n", [(530, 33, 515), (1030, 8, 1027), (2050, 17, 2041)])
def test_partial_grids_bit_exact(m, k, n):
    check("matmul", m, k, n, groups=m * n // 64 // 2)
    check("matmul-tiled", m, k, n, groups=77)
