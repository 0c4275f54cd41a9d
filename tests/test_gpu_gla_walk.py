"""The GLA state walk and the kernels around it (``csrc/ccq_gla.hip``) at the sizes where they can go
wrong: one token, the edges of a chunk, fewer and more chunks than the ring of loads holds (six), unit
counts off the groups of eight, empty, one-token and ragged packed sequences, value widths that leave
waves of the output kernel idle (64) or need a second pass (320).  Output, final state and every gradient
against the float64 oracle, with the bounds of the other GLA cases: rel-L2 2e-3, 5e-4 for the kernels' own
error (against the oracle rounded to bf16)."""

import pytest
import torch

from ccq_amd import _lib
from ccq_amd._lib import ptr, stream_of
from test_gpu_gla import gla_inputs
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
    # two, three, four, eight and nine chunks: every wait of the last steps, with the ring not yet full and full
    (1, 100, 2, 64, 64, 16.0, True, None),
    (1, 192, 1, 256, 64, 16.0, True, None),
    (2, 250, 1, 128, 64, 16.0, True, None),
    (1, 512, 1, 128, 64, 16.0, True, None),
    (1, 570, 3, 64, 128, 16.0, True, None),
]


@pytest.mark.parametrize("case", CASES, ids=[str(i) for i in range(len(CASES))])
def test_gla_walk(case):
    _case(case)


@pytest.mark.parametrize("T,K,shift", [(64, 64, 1), (128, 256, 3), (128, 128, 2), (70, 128, 1), (33, 64, 3), (20, 64, 2)])
def test_gradients_off_16_bytes(T, K, shift):
    """The C entry takes dq_f32 and dk_f32 at any element, whatever else the call keeps there (whole, nearly whole, just
    over half full and emptier chunks): the same values as on 16 bytes, and nothing beside them."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda")
    lib = _lib.load()
    B, H, V = 1, 2, 64
    nt = (T + 63) // 64
    print("test_gradients_off_16_bytes", T, K, shift, flush=True)
    x, gen = gla_inputs(B, T, H, K, V, seed=6)
    x = {n: t.to(dev) for n, t in x.items() if t is not None}
    do = torch.randn(B, T, H, V, generator=gen).to(dev, torch.bfloat16)
    saved = torch.empty(lib.ccq_gla_saved_bytes(B * T, nt, H, K, V), device=dev, dtype=torch.uint8)
    o = torch.empty_like(do)
    head = [ptr(x["q"]), None, ptr(x["k"]), ptr(x["v"]), ptr(x["gk"])]
    tail = [B, T, H, K, V, B, K ** -0.5, stream_of(do)]
    _lib.check(lib.ccq_gla_fwd(*head, None, None, None, None, nt, ptr(o), None, ptr(saved), *tail), "ccq_gla_fwd")
    ws = torch.empty(lib.ccq_gla_bwd_workspace_bytes(B * T, nt, H, K, V), device=dev, dtype=torch.uint8)
    dv, dgk = torch.empty_like(do), torch.empty_like(x["gk"])

    def call(dq, dk):
        _lib.check(lib.ccq_gla_bwd(*head, None, None, None, nt, ptr(saved), ptr(do), None, None, ptr(ws), ptr(dq), ptr(dk),
                                   ptr(dv), None, ptr(dgk), None, *tail), "ccq_gla_bwd")
        torch.cuda.synchronize()
        return dv.clone(), dgk.clone()

    n = B * T * H * K
    want = [torch.empty(n, device=dev) for _ in range(2)]
    rest = call(*want)
    for sq, sk in ((shift, 0), (0, shift), (shift, 4 - shift)):
        buf = [torch.full((n + 8,), 7.0, device=dev) for _ in range(2)]
        got = call(buf[0][sq:], buf[1][sk:])
        for b, s, w in zip(buf, (sq, sk), want):
            assert torch.equal(b[s:s + n], w)
            assert bool((b[:s] == 7).all()) and bool((b[s + n:] == 7).all())
        assert all(torch.equal(a, b) for a, b in zip(got, rest))


@pytest.mark.parametrize("K", [64, 128, 256])
def test_no_decay_is_zero_decay(K):
    """The C entry takes no gk at all: the same as zeros, whole and partial chunks."""
    if not torch.cuda.is_available():
        pytest.skip("no GPU")
    dev = torch.device("cuda")
    lib = _lib.load()
    B, T, H, V = 1, 150, 2, 64
    print("test_no_decay_is_zero_decay", K, flush=True)
    x, _ = gla_inputs(B, T, H, K, V, seed=8)
    q, k, v = (x[n].to(dev) for n in ("q", "k", "v"))
    saved = torch.empty(lib.ccq_gla_saved_bytes(B * T, 3, H, K, V), device=dev, dtype=torch.uint8)
    out = []
    for gk in (None, torch.zeros(B, T, H, K, device=dev)):
        o, s = torch.empty_like(v), torch.empty(B, H, K, V, device=dev)
        _lib.check(lib.ccq_gla_fwd(ptr(q), None, ptr(k), ptr(v), ptr(gk), None, None, None, None, 3, ptr(o), ptr(s),
                                   ptr(saved), B, T, H, K, V, B, K ** -0.5, stream_of(q)), "ccq_gla_fwd")
        torch.cuda.synchronize()
        out.append((o, s))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
