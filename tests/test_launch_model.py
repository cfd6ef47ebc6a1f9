"""Which kernel family a quantized_matmul call runs, from the library's own
launch model (launch_model.cpp), without a GPU."""

import itertools

import pytest

import host_program
from test_gpu_stream_tile import TALL

SHAPES = [(17408, 5120), (5120, 17408), (12288, 4096), (10240, 5120), (2048, 1024), (300, 2048),
          (36000, 1024), (1000, 4160), (248320, 5120)]


def routes(cases):
    """(route, tile rows, splits, unit) of cases (M, N, K, bits, gs, ws, row identity)."""
    out = host_program.run("launch_model.cpp", [" ".join(map(str, map(int, c))) for c in cases])
    assert len(out) == len(cases)
    return [tuple(map(int, line.split())) for line in out]


@pytest.mark.parametrize("bits, gs", list(itertools.product([4, 8], [32, 64, 128])))
def test_row_identity_keeps_one_family(bits, gs):
    cases = [(M, N, K, bits, gs, ws, 1) for (N, K) in SHAPES if K % gs == 0
             for M in (1, 2, 16, 17, 20, 24, 31, 32) for ws in (0, 1)]
    assert {r[0] for r in routes(cases)} == {0}
    # without the switch, and past 32 rows, the cheaper family
    assert any(r[0] for r in routes([c[:6] + (0,) for c in cases]))
    assert all(r[0] for r in routes([(512, N, K, bits, gs, 1, 1) for N, K in SHAPES
                                     if K % gs == 0 and K % 64 == 0]))


def test_wide_heights_are_planned():
    """The shapes of test_gpu_stream_tile.TALL run the tiles they are there for,
    with the workspace; without it (and the scales at an odd address) every one
    still runs the wide kernel."""
    cases = [c[:5] for c in TALL]
    for c, r in zip(TALL, routes([(*c, 1, 0) for c in cases])):
        assert r == (1, c[6], r[2], c[7]) and (r[2] > 1) == c[8], (c, r)
    assert {(r[0]) for r in routes([(*c, 0, 0) for c in cases])} == {1}
    assert {c[6:8] for c in TALL} == set(itertools.product([128, 192, 256], [1, 2, 4]))


@pytest.mark.parametrize("M, N, K, bits, gs, wide", [
    (48, 36000, 512, 8, 64, 1),      # 12.5 us against 43.3
    (64, 8192, 512, 4, 64, 1),       # 8.3 against 18.4
    (64, 36000, 1024, 4, 64, 1),     # 13.6 against 36.7
    (64, 12288, 1536, 8, 64, 1),     # 20.6 against 38.7
    (80, 17408, 2880, 8, 64, 1),     # 34.7 against 94
    (32, 2050, 640, 8, 64, 0),       # 12.1 against 7.5
    (24, 2050, 576, 4, 64, 0),       # 9.1 against 6.2
    (64, 17408, 5120, 4, 64, 0),     # bits of 16-row calls: less than a third to gain
    (64, 5120, 17408, 4, 64, 0),
])
def test_route_of_few_rows(M, N, K, bits, gs, wide):
    """Calls where one family is far slower (wide tile against skinny launches,
    measured)."""
    assert routes([(M, N, K, bits, gs, 1, 0)])[0][0] == wide
