"""fp16 decode attention over large caches of many chunks, where the chunks past
the position start last (contiguous) or a workgroup takes several of its unit's
(paged) and the merge skips those past the position: against float64, for the matrix-core and the vector form, contiguous and paged,
at positions on and around the chunk edges; every row not attended holds NaN, and
the workspace too (a chunk nobody wrote must not reach the result)."""
import numpy as np
import pytest

import nlgpu

pytestmark = pytest.mark.gpu
f32 = np.float32


@pytest.fixture(scope="module", autouse=True)
def device():
    nlgpu.init()
    yield


def attend(q, k, v):
    """q [heads, hd], k and v [n, kvheads, hd]: float64 attention."""
    heads, hd = q.shape
    grp = heads // k.shape[1]
    out = np.empty((heads, hd))
    for h in range(heads):
        s = k[:, h // grp].astype(np.float64) @ q[h].astype(np.float64) / np.sqrt(hd)
        e = np.exp(s - s.max())
        out[h] = e @ v[:, h // grp].astype(np.float64) / e.sum()
    return out


def close(got, want):
    # f32 sums of a few thousand probabilities (and q in two fp16 halves, 22
    # bits): 3e-7 of the result measured, the bar the prompt attention has
    assert np.max(np.abs(got - want)) <= 1e-5 * np.max(np.abs(want))


@pytest.mark.parametrize("heads,kvh,hd,max_seq", [
    (32, 8, 128, 2400), (16, 8, 128, 2400), (32, 8, 128, 3400), (16, 4, 64, 8800),
    (8, 1, 128, 17000), (24, 3, 64, 3100), (24, 3, 128, 500)])  # eight heads a group: two workgroups
def test_contiguous(heads, kvh, hd, max_seq):
    batch = 17 if heads == 8 * kvh else 16  # (17: units that are no multiple of the XCDs)
    print(f"[gpu] decode attention heads={heads}/{kvh} hd={hd} max_seq={max_seq}", flush=True)
    rng = np.random.default_rng(heads + hd)
    q = rng.standard_normal((batch, heads, hd)).astype(f32)
    chunk = 256 if hd == 128 else 512
    hi = min(chunk * 6 + 3, max_seq)
    k = np.full((batch, kvh, max_seq, hd), np.nan, np.float16)
    v = np.full_like(k, np.nan)
    rows = rng.standard_normal((batch, kvh, hi, hd)).astype(np.float16)
    vals = rng.standard_normal((batch, kvh, hi, hd)).astype(np.float16)
    ws = nlgpu.DeviceArray(nlgpu.decode_attn_f16_workspace(batch, heads, kvh, hd, max_seq))
    dq, out = nlgpu.to_device(q), nlgpu.DeviceArray(q.nbytes)
    for pos in (0, chunk - 1, chunk, min(4 * chunk + 17, hi - 2), hi - 1):
        k[:, :, :pos + 1], v[:, :, :pos + 1] = rows[:, :, :pos + 1], vals[:, :, :pos + 1]
        dk, dv = nlgpu.to_device(k), nlgpu.to_device(v)
        ws.upload(np.full(ws.nbytes // 4, np.nan, f32))
        nlgpu.decode_attn_f16(dq, dk, dv, nlgpu.to_device(np.array([pos], np.int32)), out, batch, heads, kvh, hd,
                              max_seq, ws)
        got = out.download(f32, q.size).reshape(q.shape)
        for b in (0, 7, batch - 1):
            close(got[b], attend(q[b], rows[b, :, :pos + 1].transpose(1, 0, 2), vals[b, :, :pos + 1].transpose(1, 0, 2)))


@pytest.mark.parametrize("heads,kvh,hd,bs,mbps", [(20, 5, 128, 16, 150), (16, 8, 64, 32, 160), (8, 1, 128, 16, 600)])
def test_paged(heads, kvh, hd, bs, mbps):
    batch = 32
    print(f"[gpu] paged attention heads={heads}/{kvh} hd={hd} bs={bs} mbps={mbps}", flush=True)
    rng = np.random.default_rng(heads * 3 + hd)
    chunk = 256 if hd == 128 else 512
    q = rng.standard_normal((batch, heads, hd)).astype(f32)
    lens = rng.integers(0, 3 * chunk, batch).astype(np.int32)
    lens[:6] = [0, chunk - 1, chunk, bs * mbps - 1, 5 * chunk + 1, bs - 1]
    need = [(int(n) // bs) + 1 for n in lens]
    npool = sum(need) + 3
    k = np.full((npool, bs, kvh, hd), np.nan, np.float16)
    v = np.full_like(k, np.nan)
    table = np.full((batch, mbps), npool + 5, np.int32)  # entries past a sequence: no block
    order = rng.permutation(npool)
    at, seqs = 0, []
    for b in range(batch):
        n = int(lens[b]) + 1
        blocks = order[at:at + need[b]]
        at += need[b]
        table[b, :need[b]] = blocks
        kk, vv = (rng.standard_normal((n, kvh, hd)).astype(np.float16) for _ in range(2))
        for j, blk in enumerate(blocks):
            part = slice(j * bs, min(n, (j + 1) * bs))
            k[blk, :part.stop - part.start], v[blk, :part.stop - part.start] = kk[part], vv[part]
        seqs.append((kk, vv))
    ws = nlgpu.DeviceArray(nlgpu.decode_attn_paged_f16_workspace(batch, heads, kvh, hd, bs, mbps))
    ws.upload(np.full(ws.nbytes // 4, np.nan, f32))
    dq, out = nlgpu.to_device(q), nlgpu.DeviceArray(q.nbytes)
    nlgpu.decode_attn_paged_f16(dq, nlgpu.to_device(k), nlgpu.to_device(v), nlgpu.to_device(lens),
                                nlgpu.to_device(table), npool, out, batch, heads, kvh, hd, bs, mbps, ws)
    got = out.download(f32, q.size).reshape(q.shape)
    for b in range(batch):
        close(got[b], attend(q[b], *seqs[b]))


@pytest.mark.parametrize("heads,kvh,batch", [(32, 32, 256), (64, 8, 512)])
def test_paged_past_the_one_dimensional_grid(heads, kvh, batch):
    """More chunk workgroups (2^23 of 512 threads) than a grid's x dimension holds,
    one head each or two of a group's four."""
    hd, bs, mbps = 64, 4096, 129  # 1,032 chunks of 512 positions; a pool that all sequences share
    print(f"[gpu] paged attention heads={heads}/{kvh} batch={batch} reach={bs * mbps}", flush=True)
    rng = np.random.default_rng(heads)
    npool = 3
    k, v = (rng.standard_normal((npool, bs, kvh, hd)).astype(np.float16) for _ in range(2))
    q = rng.standard_normal((batch, heads, hd)).astype(f32)
    lens = rng.integers(0, 1200, batch).astype(np.int32)
    lens[[0, 100, batch - 1]] = [9000, 511, 4097]
    table = rng.integers(0, npool, (batch, mbps)).astype(np.int32)
    ws = nlgpu.DeviceArray(nlgpu.decode_attn_paged_f16_workspace(batch, heads, kvh, hd, bs, mbps))
    dq, out = nlgpu.to_device(q), nlgpu.to_device(np.full(q.size, 7.0, f32))
    nlgpu.decode_attn_paged_f16(dq, nlgpu.to_device(k), nlgpu.to_device(v), nlgpu.to_device(lens),
                                nlgpu.to_device(table), npool, out, batch, heads, kvh, hd, bs, mbps, ws)
    got = out.download(f32, q.size).reshape(q.shape)
    for b in (0, 1, 100, batch // 2, batch - 1):
        n = int(lens[b]) + 1
        kk, vv = (x[table[b, :n // bs + 1]].reshape(-1, kvh, hd)[:n] for x in (k, v))
        close(got[b], attend(q[b], kk, vv))
