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


@pytest.mark.parametrize("scale", [0.125, 0.09, -0.125, 0.36])
@pytest.mark.parametrize("n,start,heads", [(40, 30, 3), (290, 10, 29)])
def test_small_queries_against_large_keys(gpu, n, start, heads, scale):
    """A query's two f16 parts carry 22 bits of each element at any size: the bar
    above, with elements of 2^-16 and keys of 2^15.  Split at its own size such an element's
    second part is an f16 subnormal, rounded at 2^-25, which is 2^-10 of a key."""
    r = np.random.default_rng(SEED + n)
    capacity = start + n
    kf = (r.uniform(-1, 1, (capacity, heads, 64)) * 32000).astype(np.float16).astype(np.float32)
    vf = r.standard_normal((capacity, heads, 64)).astype(np.float16).astype(np.float32)
    q = (r.integers(-255, 256, (n, heads, 64)) * 2.0 ** -24).astype(np.float32)
    kc, vc, qb, out = gpu.alloc(2 * kf.size), gpu.alloc(2 * vf.size), gpu.alloc(q.nbytes), gpu.alloc(q.nbytes)
    kc.upload(kf.astype(np.float16))
    vc.upload(vf.astype(np.float16))
    qb.upload(q)
    pos = int_buffer(gpu, start)
    print(f"\nsmall queries n={n} heads={heads} scale={scale}", flush=True)
    gpu.attention(qb, kc, vc, out, n, heads, heads, 64, capacity, scale, pos)
    got = out.download(np.float32, q.size).reshape(q.shape)
    ref = oracle.attention(q, kf, vf, start, scale)
    size = max((np.abs(q[:, h]).astype(np.float64) @ np.abs(kf[:, h]).T.astype(np.float64)).max() for h in range(heads))
    delta = 2.0 ** -21 * size * abs(scale)
    bar = 2 * delta * np.abs(vf).max() + 2e-6 + 1e-5 * np.abs(ref)
    worst = (np.abs(got - ref) / bar).max()
    assert worst <= 1, f"{worst:.2f} of the bar"
    for b in (qb, out, kc, vc, pos):
        b.free()


# (scale, query std): scores near 8 std^2 scale
@pytest.mark.parametrize("scale,std", [(1e20, 1), (-1e20, 1), (1e30, 1), (-1e30, 1), (1e36, 1), (3e38, 1e-3),
                                       (-3.4e38, 1e-3)])
@pytest.mark.parametrize("n,heads", [(40, 2), (290, 29)])
def test_scores_far_apart_pick_one_key(gpu, n, heads, scale, std):
    """At such scales every query's weights are one 1 and zeros: the output is its best key's
    value, exactly, also where all the scores that a query sees are far below zero."""
    r = np.random.default_rng(SEED + n)
    kf, vf, kc, vc = cache_pair(gpu, r, n, n, heads)
    q = (r.standard_normal((n, heads, 64)) * std).astype(np.float32)
    qb, out, pos = gpu.alloc(q.nbytes), gpu.alloc(q.nbytes), int_buffer(gpu, 0)
    qb.upload(q)
    print(f"\nscale {scale} n={n} heads={heads}", flush=True)
    gpu.attention(qb, kc, vc, out, n, heads, heads, 64, n, scale, pos)
    got = out.download(np.float32, q.size).reshape(q.shape)
    checked = 0
    for h in range(heads):
        s = (q[:, h].astype(np.float64) @ kf[:, h].T.astype(np.float64)) * np.sign(scale)
        s[np.triu_indices(n, 1)] = -np.inf
        top = np.sort(s, axis=1)
        # two f16 parts of q and a f32 sum: the order of scores further apart than this is certain
        apart = np.full(n, True)
        apart[1:] = top[1:, -1] - top[1:, -2] > 2.0 ** -18 * np.abs(q[1:, h]).max() * 64 * np.abs(kf[:, h]).max()
        want = vf[s.argmax(1), h]
        assert np.array_equal(got[apart, h], want[apart]), f"head {h}"
        checked += int(apart.sum())
    assert checked >= 0.95 * n * heads
    for b in (qb, out, kc, vc, pos):
        b.free()


def test_scores_near_the_end_of_the_range(gpu):
    """All of a row's scores at -2.2e38, -3.2e38 in units of log2: equal, so its keys weigh alike."""
    n, heads = 40, 2
    r = np.random.default_rng(SEED)
    kf, vf, kc, vc = cache_pair(gpu, r, n, n, heads)
    kc.upload(np.full(n * heads * 64, 1.25, np.float16))
    q = np.full((n, heads, 64), 1.25, np.float32)
    qb, out, pos = gpu.alloc(q.nbytes), gpu.alloc(q.nbytes), int_buffer(gpu, 0)
    qb.upload(q)
    gpu.attention(qb, kc, vc, out, n, heads, heads, 64, n, -2.22e36, pos)
    got = out.download(np.float32, q.size).reshape(q.shape)
    want = np.cumsum(vf.astype(np.float64), axis=0) / np.arange(1, n + 1)[:, None, None]
    assert np.abs(got - want).max() <= 5e-6
    for b in (qb, out, kc, vc, pos):
        b.free()


def test_zero_scale_averages(gpu):
    """Scale 0 and the least subnormal weigh every visible key alike."""
    n, heads = 45, 2
    r = np.random.default_rng(SEED)
    kf, vf, kc, vc = cache_pair(gpu, r, n, n, heads)
    q = r.standard_normal((n, heads, 64)).astype(np.float32)
    qb, out, pos = gpu.alloc(q.nbytes), gpu.alloc(q.nbytes), int_buffer(gpu, 0)
    qb.upload(q)
    for scale in (0.0, -0.0, 1e-45, -1e-45):
        gpu.attention(qb, kc, vc, out, n, heads, heads, 64, n, scale, pos)
        got = out.download(np.float32, q.size).reshape(q.shape)
        ref = oracle.attention(q, kf, vf, 0, scale)
        assert np.abs(got - ref).max() <= 5e-6, scale
    for b in (qb, out, kc, vc, pos):
        b.free()


def test_a_nan_key_reaches_the_queries_that_see_it(gpu):
    """A score that is no number makes its query's output no number (the reference's softmax
    sums it) and leaves the queries before it, in the same tile, as they were."""
    n, heads, at = 70, 2, 41
    r = np.random.default_rng(SEED)
    kf, vf, kc, vc = cache_pair(gpu, r, n, n, heads)
    q = r.standard_normal((n, heads, 64)).astype(np.float32)
    ref = oracle.attention(q, kf, vf, 0, 0.125)
    kc.upload(np.full(heads * 64, np.nan, np.float16), at * heads * 64 * 2)
    qb, out, pos = gpu.alloc(q.nbytes), gpu.alloc(q.nbytes), int_buffer(gpu, 0)
    qb.upload(q)
    gpu.attention(qb, kc, vc, out, n, heads, heads, 64, n, 0.125, pos)
    got = out.download(np.float32, q.size).reshape(q.shape)
    assert np.abs(got[:at] - ref[:at]).max() <= 5e-6
    assert np.isnan(got[at:]).all()
    for b in (qb, out, kc, vc, pos):
        b.free()
