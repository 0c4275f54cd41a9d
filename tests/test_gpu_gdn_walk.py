"""The K = 256 state walks (``csrc/ccq_gwalk.hip``) at the sizes where they can go wrong: one token, the
edges of a chunk, few chunks (the loads run two chunks ahead, the prefetch four), unit counts off the
groups of eight, empty and ragged packed sequences, both workgroup shapes (32 columns per workgroup once
those fill the chip).  Outputs, the final state and every gradient against the float64 oracle, with the
bounds the other head sizes are held to: rel-L2 2e-3, and per element a quarter of a bf16 ulp's share."""

import pytest
import torch

from test_gpu_workload import _gdn_case, _report

pytestmark = pytest.mark.gpu

CASES = [
    # B, T, H, V, varlen, initial states, cleaning, l2norm
    (1, 1, 1, 64, None, True, True, True),
    (1, 63, 2, 128, None, True, False, False),
    (2, 64, 1, 64, None, False, True, False),
    (1, 65, 3, 64, None, True, True, False),
    (1, 129, 1, 192, None, False, False, True),
    # six and seven chunks: the prefetch runs, the last chunk full or partial
    (1, 384, 1, 64, None, True, False, False),
    (1, 401, 2, 64, None, True, True, False),
    # nine units (one past a group of eight), an empty and a one-token sequence among them
    (1, 300, 3, 64, [0, 130, 130, 300], True, False, False),
    (1, 200, 1, 64, [0, 1, 65, 129, 200], True, True, True),
    # 16 units x 512 columns: 256 workgroups of 32 columns
    (1, 560, 2, 512, [0, 64, 129, 200, 263, 330, 400, 470, 560], True, False, False),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_gdn_walk(case):
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    print("test_gdn_walk", case, flush=True)
    B, T, H, V, cu, st, ccq, l2 = case
    errs, kerrs = _gdn_case(B, T, H, 256, V, cu, st, ccq, l2, seed=31)
    # (the bar of the K = 256 head-size case with the largest spread over seeds, for the same reason:
    # single elements of dq, dk are small differences of terms that carry 16 significant bits)
    _report(case, errs, kerrs, 1e-3)
