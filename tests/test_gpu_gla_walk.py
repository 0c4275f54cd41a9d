"""The GLA state walk and the kernels around it (``csrc/ccq_gla.hip``) at the sizes where they can go
wrong: one token, the edges of a chunk, fewer and more chunks than the ring of loads holds (six), unit
counts off the groups of eight, empty, one-token and ragged packed sequences, value widths that leave
waves of the output kernel idle (64) or need a second pass (320).  Output, final state and every gradient
against the float64 oracle, with the bounds of the other GLA cases: rel-L2 2e-3, 5e-4 for the kernels' own
error (against the oracle rounded to bf16)."""

import pytest

from test_gpu_gla import test_gla_backbone as _case

pytestmark = pytest.mark.gpu

CASES = [
    # B, T, H, K, V, gate normaliser, initial state, varlen
    (1, 1, 1, 64, 64, 16.0, True, None),
    (1, 63, 3, 128, 64, 16.0, True, None),
    (2, 65, 1, 64, 320, 16.0, True, None),
    # five, six, seven and twelve chunks, the last one full or partial
    (1, 320, 1, 64, 64, 16.0, True, None),
    (1, 383, 1, 128, 128, 16.0, True, None),
    (1, 400, 2, 64, 192, 2.0, False, None),
    (1, 705, 1, 256, 64, 16.0, True, None),
    # nine units, an empty and a one-token sequence among them
    (1, 300, 3, 64, 64, 16.0, True, [0, 130, 130, 300]),
    (1, 600, 1, 128, 320, 16.0, True, [0, 1, 65, 129, 600]),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_gla_walk(case):
    _case(case)
