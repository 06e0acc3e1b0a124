"""CPU tests of the prompt GEMM's launch rule (q8_gemm_shape through q8_plan,
256 CUs): the shape it takes on both sides of each of its lines.  The rule's
reasons, with times of both sides, are written beside it.
"""
import pytest

from llm_amd import q8

# (n, rows, k, token tiles a wave, token-tile waves, K waves)
LINES = [
    # eight K waves while every workgroup has a CU: 256 and 260 tiles
    (97, 2048, 2304, 1, 1, 8), (97, 2080, 2304, 1, 2, 4),
    # one to two workgroups a CU: two or four token tiles pair, three and six do not
    (64, 4096, 2304, 1, 1, 8), (64, 4128, 2304, 1, 2, 4), (64, 5760, 2304, 1, 2, 4), (64, 8192, 2304, 1, 2, 4),
    (64, 8224, 2304, 1, 1, 4), (65, 3072, 2304, 1, 1, 4), (97, 2720, 2304, 1, 2, 4), (192, 2304, 5760, 1, 1, 4),
    (256, 4000, 4736, 2, 2, 4),
    # waves resident at once: 700 tiles of four K waves
    (129, 4480, 2304, 1, 1, 4), (129, 4512, 2304, 1, 1, 2),
    # four to five workgroups a CU, from 32 pairs up
    (512, 2048, 2048, 1, 1, 2), (512, 2080, 2048, 1, 1, 4), (512, 2080, 1984, 1, 1, 2), (512, 2560, 2048, 1, 1, 4),
    (512, 2592, 2048, 1, 1, 2),
    # two token tiles a wave: 870 tiles (868 and 882), 64 000 tile-pairs (63 960 and 65 190)
    (448, 1984, 4736, 1, 1, 2), (448, 2016, 4736, 2, 1, 4), (480, 2624, 3328, 1, 1, 4), (480, 2624, 3392, 2, 1, 4),
    # the benchmark's projections of 512 tokens
    (512, 2304, 2304, 1, 1, 4), (512, 2304, 5760, 2, 1, 4), (512, 6912, 2304, 2, 1, 1),
    # short rows stay unsplit
    (64, 100, 448, 1, 1, 1), (64, 5760, 448, 1, 1, 1),
]


@pytest.mark.parametrize("n,rows,k,tpw,twaves,kwaves", LINES)
def test_both_sides_of_the_lines(n, rows, k, tpw, twaves, kwaves):
    t = q8.plan(n, rows, k)
    assert (t["tpw"], t["twaves"], t["kwaves"]) == (tpw, twaves, kwaves)
    assert t["kwaves"] * t["pairs_per_wave"] >= -(-k // 64) > (t["kwaves"] - 1) * t["pairs_per_wave"]


def test_every_plan_fits_its_workgroup():
    """At most 1024 threads at one token tile a wave, 512 at two (the kernels' bounds)."""
    for n in (2, 33, 64, 97, 128, 300, 511, 1024):
        for rows in (32, 900, 2080, 4128, 8000, 12288):
            for k in (32, 480, 1056, 2304, 4736, 8192):
                t = q8.plan(max(n, 3), rows, k)
                assert 64 * t["twaves"] * t["kwaves"] <= (1024 if t["tpw"] == 1 else 512), (n, rows, k, t)
