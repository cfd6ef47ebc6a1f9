"""Where the kernels' loads of weights and scales end: never past the arrays.

Arrays of whole 2 MiB pages may end where mapped memory does, so a load that
reaches past them can fault the GPU, while its value (of a code past K) is
multiplied by nothing: comparing results cannot show it.  Here the buffer
ranges that the kernels compute are walked on the CPU (read_ranges.cpp).

The skinny tile's steps cover 2 to 8 groups of every row; at K of partial steps
the last one ends inside the row.  Taken as a whole step there, its range
reaches past the last row: the second column of the walk, which must say so
for exactly those K, or the walk would not see the fault it is for."""

import random

import pytest

import host_program


def _step_codes(bits, gs):
    return 4 * gs * (2 if (bits, gs) == (4, 32) else 1)


def _shapes(bits, gs):
    """Sizes of linear layers and banks, whole steps of K and partial ones,
    ragged N, and banks of whole 2 MiB pages."""
    rng = random.Random(1000 * bits + gs)
    out = [(gs, 1, 1), (_step_codes(bits, gs) + gs, 17, 1), (448 * gs // 32, 1024, 64),
           (1152, 32768, 1), (640, 512, 128)]
    for _ in range(40):
        out.append((gs * rng.randint(1, 8192 // gs), rng.randint(1, 4096), rng.choice([1, 8, 64])))
    for _ in range(40):                         # as MoE layers come
        out.append((128 * rng.randint(2, 24), 128 * rng.randint(2, 24), rng.choice([64, 256, 512])))
    return out


@pytest.mark.parametrize("gs", [32, 64, 128])
@pytest.mark.parametrize("bits", [4, 8])
def test_loads_end_with_the_arrays(bits, gs):
    shapes = _shapes(bits, gs)
    lines = host_program.run("read_ranges.cpp", [f"{bits} {gs} {K} {N} {E}" for K, N, E in shapes])
    assert len(lines) == len(shapes)
    partial = 0
    for (K, N, E), line in zip(shapes, lines):
        skinny, whole_steps, quad, stream, all_read = map(int, line.split())
        assert (skinny, quad, stream) == (0, 0, 0), (K, N, E, line)
        assert all_read == 1, (K, N, E, line)
        ragged = K % _step_codes(bits, gs) != 0
        partial += ragged
        assert (whole_steps > 0) == ragged, (K, N, E, line)
    assert partial >= 10
