"""GPU test of the decode attention's grouped-query order: a kv head's heads run
as one contiguous run per XCD, so launches that don't divide by eight, groups
that straddle two runs, and every launch smaller than eight workgroups have to
reach each (head, split) once.

Bar: test_gpu_decoder's, 2e-6 + 1e-5 |ref| of the exact attention formula.
"""
import numpy as np
import pytest

import oracle
from llm_amd import q8
from test_gpu_decoder import cache_pair, int_buffer
from test_gpu_q8 import assert_close

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def gpu():
    g = q8.Gpu(0)
    yield g
    g.close()


# (visible, splits, heads, kv heads): 45, 28, 3, 6, 14, 36, 99 and 288 workgroups
@pytest.mark.parametrize("visible,splits,heads,kv", [
    (700, 3, 15, 5), (520, 2, 14, 2), (90, 1, 3, 1), (70, 1, 6, 3), (1, 7, 2, 1), (300, 4, 9, 3), (2100, 3, 33, 11),
    (4000, 8, 36, 4)])
def test_every_head_and_split_once(gpu, visible, splits, heads, kv):
    r = np.random.default_rng(0xDEC0 + visible + heads)
    kf, vf, kc, vc = cache_pair(gpu, r, visible, visible + 60, kv)
    q = (r.standard_normal((1, heads, 64)) * 2).astype(np.float32)
    qb, out, pos = gpu.alloc(q.nbytes), gpu.alloc(q.nbytes), int_buffer(gpu, visible - 1)
    qb.upload(q)
    print(f"\ndecode attention visible={visible} splits={splits} heads={heads}/{kv}", flush=True)
    gpu.attention(qb, kc, vc, out, 1, heads, kv, 64, visible + 60, 0.125, pos, splits)
    got = out.download(np.float32, q.size).reshape(q.shape)
    assert_close(got, oracle.attention(q, kf, vf, visible - 1, 0.125), f"visible={visible} splits={splits}")
    for b in (qb, out, kc, vc, pos):
        b.free()
