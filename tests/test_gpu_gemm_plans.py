"""GPU tests of the prompt GEMM's launch shapes (q8_gemm_shape, q8_gemm_rope_shape,
q8_gemm_silu_kwaves) on both sides of their lines: where a wave takes a second
token tile, where the K range splits over 1, 2, 4 or 8 waves, and where two
token-tile waves of a q/k/v group share a workgroup.

Bars: the plain GEMM within 2e-6 + 1e-5 |ref| of the oracle (assert_parity);
the rotated group the same bits as the plain group followed by q8_rope_append
(its K split is the plain group's); the fused gate/up launch the same bytes as
the unfused one at the same K split.
"""
import numpy as np
import pytest

import oracle
from llm_amd import q8
from test_gpu_decoder import f16_buffer, int_buffer, q8w, read_f16
from test_gpu_q8 import assert_bits, assert_parity, exact_at, unpack_prepared

pytestmark = pytest.mark.gpu
SEED = 0x61A5


@pytest.fixture(scope="module")
def gpu():
    g = q8.Gpu(0)
    yield g
    g.close()


# (n, rows, k, token tiles a wave, K waves)
PLANS = [
    (64, 100, 448, 1, 1), (33, 100, 480, 1, 4),                 # seven pairs: unsplit; eight: two each
    (5, 2304, 1024, 1, 8), (32, 1300, 544, 1, 3),               # two each over eight waves; nine pairs in three
    (97, 2048, 2304, 1, 8), (97, 2720, 2304, 1, 4),             # 256 tiles: a CU each, eight waves; 340: token tiles paired
    (64, 4128, 2304, 1, 4), (129, 2304, 5760, 1, 4),            # 258 tiles, paired; 360 in five: unpaired
    (480, 2624, 3328, 1, 4), (480, 2624, 4096, 2, 4),           # 63 960 and 78 720 tile-pairs
    (512, 2624, 4096, 2, 4), (512, 2624, 3872, 2, 4),
    (512, 2624, 3840, 2, 4), (256, 4000, 4736, 2, 4),           # paired: two token tiles in each of two waves
    (489, 5000, 2080, 2, 2), (1000, 6912, 1088, 2, 1),          # a half-empty last token tile; no K split
]


@pytest.mark.parametrize("n,rows,k,tpw,kwaves", PLANS)
def test_gemm_on_both_sides_of_the_lines(gpu, n, rows, k, tpw, kwaves):
    t = gpu.plan(n, rows, k)
    assert (t["tpw"], t["kwaves"]) == (tpw, kwaves)
    r = np.random.default_rng(SEED + n + rows + k)
    w = q8.Weight(oracle.make_q8_weight(r, rows, k), k, rows)
    x = oracle.make_activations(r, n, k, outlier_rate=0.01)
    xb, yb = gpu.alloc(4 * n * k), gpu.alloc(4 * n * rows)
    xb.upload(x)
    try:
        print(f"\ngemm n={n} rows={rows} k={k} tpw={tpw} kwaves={kwaves}", flush=True)
        gpu.matmul(w, xb, 0, n, yb, 0)
        got = yb.download(np.float32, n * rows).reshape(n, rows)
        assert_parity(got, oracle.matmul(w.data, k, rows, x, n), exact_at(w.data, k, rows, x, n),
                      f"gemm n={n} rows={rows} k={k}")
    finally:
        xb.free()
        yb.free()
        gpu.release(w)


# workgroup counts on both sides of a multiple of the eight XCDs, and below it
@pytest.mark.parametrize("tiles", [1, 7, 8, 9, 15, 41])
@pytest.mark.parametrize("option", [None, "gemm.pipe", "gemm.lds", "gemm.f16"])
def test_every_tile_has_its_workgroup(gpu, option, tiles):
    n, rows, k = 20, 32 * tiles, 544
    r = np.random.default_rng(SEED + tiles)
    w = q8.Weight(oracle.make_q8_weight(r, rows, k), k, rows)
    x = oracle.make_activations(r, n, k, outlier_rate=0.01)
    xb, yb = gpu.alloc(4 * n * k), gpu.alloc(4 * n * rows)
    xb.upload(x)
    yb.upload(np.full(n * rows, np.nan, np.float32))
    try:
        print(f"\n{option} {tiles} row tiles", flush=True)
        if option:
            gpu.set_option(option, 1)
        gpu.matmul(w, xb, 0, n, yb, 0)
        got = yb.download(np.float32, n * rows).reshape(n, rows)
        assert_parity(got, oracle.matmul(w.data, k, rows, x, n), exact_at(w.data, k, rows, x, n),
                      f"{option} n={n} rows={rows} k={k}")
    finally:
        if option:
            gpu.set_option(option, -1)
        xb.free()
        yb.free()
        gpu.release(w)


@pytest.mark.parametrize("n,heads,kv,n_rot,e,position,kwaves", [(*c, -1) for c in [
    (2, 4, 2, 64, 256, 0), (32, 22, 11, 64, 1536, 5),       # one token tile
    (33, 24, 24, 64, 1536, 9), (64, 32, 16, 64, 1536, 0),   # 144 and 128 row tiles, paired: 1024 threads
    (64, 30, 15, 64, 1536, 3), (65, 24, 24, 64, 1536, 3),   # 120 row tiles; three token tiles: unpaired
    (250, 36, 36, 16, 1152, 1), (290, 36, 36, 64, 1152, 0), (256, 9, 3, 0, 576, 40),
    (96, 24, 24, 64, 224, 2), (64, 24, 24, 64, 32, 7),       # short rows: no K split
    (416, 64, 64, 64, 2560, 3), (420, 64, 64, 48, 2560, 0)]] +  # 4992 and 5376 tiles: one and two token tiles a wave
    [(64, 24, 24, 64, 1536, 0, 16)])                       # K over all of a workgroup's waves: unpaired
def test_rotated_group_equals_the_plain_one(gpu, n, heads, kv, n_rot, e, position, kwaves):
    r = np.random.default_rng(SEED + n + heads + kv + e)
    capacity, kvw, base = position + n, kv * 64, 10000.0
    weights = [q8w(r, heads * 64, e), q8w(r, kvw, e), q8w(r, kvw, e)]
    xb = gpu.alloc(4 * n * e)
    xb.upload(oracle.make_activations(r, n, e))
    q1, q2 = gpu.alloc(4 * n * heads * 64), gpu.alloc(4 * n * heads * 64)
    k1, v1 = gpu.alloc(4 * n * kvw), gpu.alloc(4 * n * kvw)
    plain, fused = ([f16_buffer(gpu, capacity, kvw) for _ in range(2)] for _ in range(2))
    pos = int_buffer(gpu, position)
    try:
        print(f"\nrotated group n={n} heads={heads}/{kv} rot={n_rot} e={e}", flush=True)
        p = gpu.prepare(xb, 0, n, e)
        gpu.set_option("gemm.kwaves", kwaves)
        gpu.matmul_prompt_group(list(zip(weights, (q1, k1, v1), (0, 0, 0))), p, n, e)
        gpu.rope_append(q1, k1, v1, *plain, n, heads, kv, 64, n_rot, base, capacity, pos)
        gpu.prompt_qkv_rope(*weights, p, n, q2, *fused, heads, kv, 64, n_rot, base, capacity, pos)
        gpu.sync()
        assert_bits(q2.download(np.float32, n * heads * 64), q1.download(np.float32, n * heads * 64), "q")
        for name, a, b in zip(("key", "value"), fused, plain):
            got, want = (read_f16(c, capacity, kvw).view(np.uint16) for c in (a, b))
            assert np.array_equal(got, want), f"{name} cache: {int((got != want).sum())} halves differ"
    finally:
        gpu.set_option("gemm.kwaves", -1)
        for b in (xb, q1, q2, k1, v1, pos, *plain, *fused):
            b.free()
        for w in weights:
            gpu.release(w)


# (n, ffn, k, K waves)
@pytest.mark.parametrize("n,ffn,k,kwaves", [(64, 96, 224, 1), (33, 96, 512, 4), (128, 4992, 2304, 4),
                                            (129, 4032, 2304, 2), (250, 4992, 1056, 2), (257, 4480, 1056, 2),
                                            (250, 6144, 1056, 2), (250, 6176, 1056, 1),  # six tiles a CU
                                            # 80 pairs: half a tile and five tiles a CU
                                            (64, 2048, 5120, 8), (64, 2080, 5120, 4), (64, 2048, 5056, 4),
                                            (250, 5120, 5120, 4), (250, 5152, 5120, 2)])
def test_gate_up_on_both_sides_of_the_lines(gpu, n, ffn, k, kwaves):
    r = np.random.default_rng(SEED + n + ffn + k)
    g, u = q8w(r, ffn, k), q8w(r, ffn, k)
    xb = gpu.alloc(4 * n * k)
    xb.upload(oracle.make_activations(r, n, k, outlier_rate=0.01))
    try:
        print(f"\ngate/up n={n} ffn={ffn} k={k} kwaves={kwaves}", flush=True)
        p = gpu.prepare(xb, 0, n, k)
        got = unpack_prepared(gpu, gpu.gate_up_silu_prepared(g, u, p), n, ffn)
        for name, value in (("gemm.silu", 0), ("gemm.tpw", 1), ("gemm.twaves", 1), ("gemm.kwaves", kwaves)):
            gpu.set_option(name, value)
        want = unpack_prepared(gpu, gpu.gate_up_silu_prepared(g, u, p), n, ffn)
        for a, b in zip(got, want):
            assert np.array_equal(a, b), f"{int((a != b).sum())} of {a.size} differ"
    finally:
        for name in ("gemm.silu", "gemm.tpw", "gemm.twaves", "gemm.kwaves"):
            gpu.set_option(name, -1)
        xb.free()
        gpu.release(g)
        gpu.release(u)
