"""GPU tests of the rotations in the q/k/v epilogues at head widths that divide
neither a slice of 8 or 16 rows nor a tile of 32: a slice and a tile then hold rows of
several heads, heads straddle their edges, and members end inside a tile.

Bar: the fused launches give the bits of the plain group followed by
q8_rope_append (the decode group in the exact order).
"""
import numpy as np
import pytest

import oracle
from llm_amd import q8
from test_gpu_decoder import f16_buffer, int_buffer, q8w, read_f16
from test_gpu_q8 import assert_bits

pytestmark = pytest.mark.gpu
SEED = 0x207A
BASE = 10000.0


@pytest.fixture(scope="module")
def gpu():
    g = q8.Gpu(0)
    yield g
    g.close()


# (heads, kv heads, head width, rotated dims)
HEADS = [(10, 5, 6, 4), (7, 7, 20, 20), (9, 3, 48, 24), (5, 5, 2, 2), (12, 4, 10, 0), (3, 1, 128, 128), (11, 11, 36, 34)]


def check(gpu, got, want, heads, hd, n, capacity, kvw):
    assert_bits(got[0].download(np.float32, n * heads * hd), want[0].download(np.float32, n * heads * hd), "q")
    for name, a, b in (("key", got[1], want[1]), ("value", got[2], want[2])):
        a, b = (read_f16(c, capacity, kvw).view(np.uint16) for c in (a, b))
        assert np.array_equal(a, b), f"{name} cache: {int((a != b).sum())} halves differ"


@pytest.mark.parametrize("heads,kv,hd,n_rot", HEADS)
@pytest.mark.parametrize("n,options", [(5, {}), (70, {}), (70, {"gemm.tpw": 2}), (70, {"gemm.tpw": 4}),
                                       (70, {"gemm.twaves": 2}), (40, {"gemm.kwaves": 1}), (40, {"gemm.slices": 2}),
                                       (40, {"gemm.smode": 0}), (40, {"gemm.pipe": 1}), (40, {"gemm.lds": 1})])
def test_prompt_rotation(gpu, n, options, heads, kv, hd, n_rot):
    r = np.random.default_rng(SEED + n + heads + hd)
    e, position, kvw = 544, 3, kv * hd
    capacity = position + n
    weights = [q8w(r, heads * hd, e), q8w(r, kvw, e), q8w(r, kvw, e)]
    x, pos = gpu.alloc(4 * n * e), int_buffer(gpu, position)
    x.upload(oracle.make_activations(r, n, e))
    plain, fused = ([gpu.alloc(4 * n * heads * hd), f16_buffer(gpu, capacity, kvw), f16_buffer(gpu, capacity, kvw)]
                    for _ in range(2))
    k, v = gpu.alloc(4 * n * kvw), gpu.alloc(4 * n * kvw)
    try:
        print(f"\nprompt rotation n={n} heads={heads}/{kv} of {hd} rot={n_rot} {options}", flush=True)
        for name, value in options.items():
            gpu.set_option(name, value)
        p = gpu.prepare(x, 0, n, e)
        gpu.matmul_prompt_group(list(zip(weights, (plain[0], k, v), (0, 0, 0))), p, n, e)
        gpu.rope_append(plain[0], k, v, *plain[1:], n, heads, kv, hd, n_rot, BASE, capacity, pos)
        gpu.prompt_qkv_rope(*weights, p, n, fused[0], *fused[1:], heads, kv, hd, n_rot, BASE, capacity, pos)
        gpu.sync()
        check(gpu, fused, plain, heads, hd, n, capacity, kvw)
    finally:
        for name in options:
            gpu.set_option(name, -1)
        for b in (x, pos, k, v, *plain, *fused):
            b.free()
        for w in weights:
            gpu.release(w)


@pytest.mark.parametrize("heads,kv,hd,n_rot", HEADS)
@pytest.mark.parametrize("group,options", [(False, {}), (False, {"gemv.group_rows": 8}), (False, {"gemv.group_rows": 16}),
                                           (True, {}), (True, {"gemv.group_rows": 8}), (True, {"gemv.slice_copy": 0})])
def test_decode_rotation(gpu, group, options, heads, kv, hd, n_rot):
    r = np.random.default_rng(SEED + heads + hd)
    e, position, capacity, kvw, eps = 544, 11, 16, kv * hd, 1e-6
    datas = [oracle.make_q8_weight(r, o, e) for o in (heads * hd, kvw, kvw)]
    single, fused_w = ([q8.Weight(d.copy(), e, o) for d, o in zip(datas, (heads * hd, kvw, kvw))] for _ in range(2))
    xv = (r.standard_normal(e) * 2).astype(np.float32)
    nw = (1 + 0.1 * r.standard_normal(e)).astype(np.float32)
    x, xn, pos = gpu.alloc(4 * e), gpu.alloc(4 * e), int_buffer(gpu, position)
    x.upload(xv)
    plain, fused = ([gpu.alloc(4 * heads * hd), f16_buffer(gpu, capacity, kvw), f16_buffer(gpu, capacity, kvw)]
                    for _ in range(2))
    k, v = gpu.alloc(4 * kvw), gpu.alloc(4 * kvw)
    try:
        print(f"\ndecode rotation heads={heads}/{kv} of {hd} rot={n_rot} group={group} {options}", flush=True)
        gpu.set_option("gemv.exact", 1)
        gpu.rmsnorm(x, 0, nw, eps, 1, xn)
        gpu.matmul_decode_group(list(zip(single, (plain[0], k, v), (0, 0, 0))), xn, 0, e)
        gpu.rope_append(plain[0], k, v, *plain[1:], 1, heads, kv, hd, n_rot, BASE, capacity, pos)
        for name, value in options.items():
            gpu.set_option(name, value)
        if group:
            gpu.resident_group(fused_w)
        gpu.norm_qkv_rope(nw, eps, *fused_w, x, 0, fused[0], 0, *fused[1:], heads, kv, hd, n_rot, BASE, capacity, pos)
        gpu.sync()
        check(gpu, fused, plain, heads, hd, 1, capacity, kvw)
    finally:
        for name in ("gemv.exact", *options):
            gpu.set_option(name, -1)
        for b in (x, xn, pos, k, v, *plain, *fused):
            b.free()
        for w in single + fused_w:
            gpu.release(w)
