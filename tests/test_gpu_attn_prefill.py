"""GPU tests of the prompt attention kernels (q8_attn_prefill, q8_attn_prefill_k8)
at the edges of their tiles: 32 queries a workgroup, 32 keys a tile dealt to
four or eight waves, eight where the workgroups would not fill the chip.

Bar: a score is a sum of 64 products of an f16 key and a query split into two
f16 parts (2^-22 each) in f32, so its error, and with it a weight's relative
error, is at most delta = 2^-21 max_t sum_d |q_d k_d| scale; the output moves
by at most 2 delta max|v|, plus the f32 bar of the weighted sum.
"""
import numpy as np
import pytest

import oracle
from llm_amd import q8
from test_gpu_decoder import cache_pair, int_buffer

pytestmark = pytest.mark.gpu
SEED = 0xA77


@pytest.fixture(scope="module")
def gpu():
    g = q8.Gpu(0)
    yield g
    g.close()


# (n, start, heads, kv heads, scale, query std, capacity beyond start + n)
CASES = [
    (2, 0, 3, 1, 0.125, 1, 5), (31, 0, 5, 5, 0.125, 1, 0), (33, 31, 4, 2, 0.125, 1, 1),
    (64, 64, 4, 4, 0.125, 1, 0), (65, 191, 2, 1, 0.125, 1, 7),     # last tiles full, one key, one query
    (40, 500, 2, 2, 0.125, 1, 3), (96, 1, 9, 3, 0.125, 1, 9),      # every wave of eight holds several tiles
    (290, 0, 29, 29, 0.125, 1, 2), (300, 77, 26, 13, 0.125, 1, 0),  # more than 256 workgroups: four waves
    (33, 70, 2, 2, 0.3, 1, 0), (48, 30, 2, 1, 1.0, 1, 0), (40, 20, 2, 2, -0.125, 1, 0),  # other scales
    (70, 200, 3, 3, 0.125, 12, 0), (280, 40, 29, 29, 0.125, 12, 0),  # peaked rows: the running max moves often
]


@pytest.mark.parametrize("n,start,heads,kv,scale,std,room", CASES)
def test_tile_edges(gpu, n, start, heads, kv, scale, std, room):
    r = np.random.default_rng(SEED + n + start + heads)
    capacity = start + n + room
    kf, vf, kc, vc = cache_pair(gpu, r, start + n, capacity, kv)
    q = (r.standard_normal((n, heads, 64)) * std).astype(np.float32)
    qb, out, pos = gpu.alloc(q.nbytes), gpu.alloc(q.nbytes), int_buffer(gpu, start)
    qb.upload(q)
    print(f"\nprompt attention n={n} start={start} heads={heads}/{kv} scale={scale} std={std}", flush=True)
    gpu.attention(qb, kc, vc, out, n, heads, kv, 64, capacity, scale, pos)
    got = out.download(np.float32, q.size).reshape(q.shape)
    ref = oracle.attention(q, kf, vf, start, scale)
    size = max((np.abs(q[:, h]).astype(np.float64) @ np.abs(kf[:start + n, h // (heads // kv)]).T.astype(np.float64)).max()
               for h in range(heads))
    delta = 2.0 ** -21 * size * abs(scale)
    bar = 2 * delta * np.abs(vf).max() + 2e-6 + 1e-5 * np.abs(ref)
    worst = (np.abs(got - ref) / bar).max()
    assert worst <= 1, f"{worst:.2f} of the bar"
    for b in (qb, out, kc, vc, pos):
        b.free()


def test_rows_past_the_context_are_not_read(gpu):
    """Cache rows past the last visible key hold NaN: they reach no output,
    also in the tile that holds the last key and in the tokens before it."""
    n, start, heads = 37, 50, 2
    r = np.random.default_rng(SEED)
    capacity = 160
    kf, vf, kc, vc = cache_pair(gpu, r, start + n, capacity, heads)
    nan = np.full((capacity - start - n) * heads * 64, np.nan, np.float16)
    for b in (kc, vc):
        b.upload(nan, (start + n) * heads * 64 * 2)
    q = r.standard_normal((n, heads, 64)).astype(np.float32)
    qb, out, pos = gpu.alloc(q.nbytes), gpu.alloc(q.nbytes), int_buffer(gpu, start)
    qb.upload(q)
    gpu.attention(qb, kc, vc, out, n, heads, heads, 64, capacity, 0.125, pos)
    got = out.download(np.float32, q.size).reshape(q.shape)
    ref = oracle.attention(q, kf, vf, start, 0.125)
    assert np.abs(got - ref).max() <= 5e-6
    for b in (qb, out, kc, vc, pos):
        b.free()
