"""Routing and dispatch on the GPU, bit for bit against the C oracle (oracle/route_ref.c).

Logits, top-k ids, gates, per-expert counts, offsets, per-source counts and the
permutation must be identical bit patterns, on the benchmark shapes (router on
full token counts for the Mixtral and DeepSeek-like layers) and on edge cases:
exact ties, NaN logits, empty experts, one token, invalid ids.
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from _helpers import DEV, host_x, say, seeded, x_kind, zipf_prior
from oracle import route_c as R
from resihp_megatron_amd import kernels as K

pytestmark = pytest.mark.gpu

# (name, T, h, E, k, x dtype, score, bias, router std)
ROUTE_CASES = [
    ("tiny-f64", 512, 64, 8, 2, torch.float64, "softmax", None, 0.125),
    ("tiny-f32", 512, 64, 8, 2, torch.float32, "softmax", None, 0.125),
    ("mixtral", 8192, 4096, 8, 2, torch.bfloat16, "softmax", None, 0.02),
    ("dsv2lite-sigmoid-bias", 16384, 2048, 64, 6, torch.bfloat16, "sigmoid", "normal", 0.02),
    ("ep128-zipf", 8192, 2048, 128, 8, torch.bfloat16, "softmax", "zipf", 0.02),
    ("reference-default", 48, 8, 6, 2, torch.float64, "softmax", None, 0.35),
    ("odd-e", 333, 256, 5, 3, torch.bfloat16, "sigmoid", None, 0.05),
    # a hidden size below one 256-element segment (ragged last 16-element batch), expert counts that are not a
    # multiple of 16, 32 segments, more expert tiles than waves, and more experts than the three-batch staging
    # of 16-token blocks leaves room for
    ("bf16-h200-e20", 130, 200, 20, 4, torch.bfloat16, "softmax", "normal", 0.05),
    ("bf16-h8192-e72", 100, 8192, 72, 6, torch.bfloat16, "sigmoid", "normal", 0.02),
    ("bf16-e200", 150, 1024, 200, 8, torch.bfloat16, "softmax", "zipf", 0.02),
    ("bf16-e300", 70, 256, 300, 4, torch.bfloat16, "softmax", None, 0.05),
]


def _bias(kind, E, dtype):
    if kind is None:
        return None
    if kind == "zipf":
        return zipf_prior(E).to(dtype)
    return seeded((E,), 99, 0.1, dtype)


@pytest.mark.parametrize("case", ROUTE_CASES, ids=[c[0] for c in ROUTE_CASES])
def test_route_bit_exact(case):
    name, T, h, E, k, xdt, score, bias_kind, wstd = case
    rdt = torch.float64 if xdt == torch.float64 else torch.float32
    x = seeded((T, h), 1, 1.0, xdt)
    w = seeded((E, h), 2, wstd, rdt)
    bias = _bias(bias_kind, E, rdt)
    say(f"route {name}: T={T} h={h} E={E} k={k} {xdt} {score}")
    logits, topi, gates = K.route(x.to(DEV), w.to(DEV), None if bias is None else bias.to(DEV), k, score,
                                  True, 1.0)
    torch.cuda.synchronize()
    ref_logits = R.router_logits(host_x(x), w.numpy(), x_kind(xdt))
    ref_topi, ref_gates = R.topk(ref_logits, k, None if bias is None else bias.numpy(), score)
    got_l = logits.cpu().numpy()
    assert got_l.dtype == ref_logits.dtype
    assert np.array_equal(got_l.view(np.uint8), ref_logits.view(np.uint8)), "logit bits differ"
    assert np.array_equal(topi.cpu().numpy(), ref_topi), "selection differs"
    assert np.array_equal(gates.cpu().numpy().view(np.uint8), ref_gates.view(np.uint8)), "gate bits differ"


# Edges of the matrix-core kernel: one token, a ragged last 16-token tile at both block sizes (16 and, from
# 8192 bf16 tokens, 32), segment counts that are not a multiple of four, more segment quads than waves (the
# sums continue over rounds), one expert, expert tiles over several rounds, and the LDS limits of its buffers:
# the last size of each (E odd or one less, plus 2 k: 255 for 32-token blocks, 1023 in bfloat16, 511 in float32)
# and the first past it, which takes 16-token blocks and, "per-thread", the kernel of a thread per chain.
EDGE_CASES = [
    ("one-token", 1, 4096, 8, 2, torch.bfloat16, "softmax", None, 0.02),
    ("t8191", 8191, 256, 16, 2, torch.bfloat16, "softmax", None, 0.05),
    ("t8197-wide", 8197, 512, 33, 4, torch.bfloat16, "sigmoid", "normal", 0.05),
    ("t8192-wide-e239", 8192, 256, 239, 8, torch.bfloat16, "softmax", "zipf", 0.05),
    ("t8192-e240", 8192, 256, 240, 8, torch.bfloat16, "softmax", "zipf", 0.05),
    ("t8192-e250", 8192, 256, 250, 8, torch.bfloat16, "softmax", "zipf", 0.05),
    ("e1007", 70, 256, 1007, 8, torch.bfloat16, "sigmoid", "normal", 0.05),
    ("e1008-per-thread", 70, 256, 1008, 8, torch.bfloat16, "sigmoid", "normal", 0.05),
    ("e1024-per-thread", 71, 256, 1024, 8, torch.bfloat16, "softmax", "zipf", 0.05),
    ("f32-e495", 37, 256, 495, 8, torch.float32, "softmax", "normal", 0.05),
    ("f32-e496-per-thread", 37, 256, 496, 8, torch.float32, "softmax", "normal", 0.05),
    ("f32-e600-h512-per-thread", 21, 512, 600, 4, torch.float32, "sigmoid", "normal", 0.05),
    ("five-segments", 77, 1280, 17, 3, torch.bfloat16, "softmax", None, 0.03),
    ("sixteen-quads", 40, 16384, 24, 4, torch.bfloat16, "softmax", None, 0.01),
    ("h8-e1", 50, 8, 1, 1, torch.bfloat16, "softmax", None, 0.3),
    ("f32-h16384", 33, 16384, 12, 3, torch.float32, "sigmoid", "normal", 0.01),
    ("f32-e400", 21, 256, 400, 16, torch.float32, "softmax", None, 0.05),
    ("f64-e70", 35, 512, 70, 6, torch.float64, "sigmoid", "normal", 0.05),
]


@pytest.mark.parametrize("case", EDGE_CASES, ids=[c[0] for c in EDGE_CASES])
def test_route_kernel_edges(case):
    test_route_bit_exact(case)


@pytest.mark.parametrize("T,h,E,k,xdt", [(16321, 4096, 320, 8, torch.bfloat16), (16320, 4096, 320, 8, torch.bfloat16),
                                         (37, 4096, 256, 8, torch.float32), (70, 16384, 500, 4, torch.bfloat16)])
def test_route_takes_any_token_count(T, h, E, k, xdt):
    """Sizes the matrix-core kernel's LDS holds are taken whatever the token count, float32 tokens too."""
    n = min(T, 37)
    base, w = seeded((n, h), 7, 1.0, xdt), seeded((E, h), 8, 0.02, torch.float32)
    x = base.repeat(T // n + 1, 1)[:T]
    say(f"route any T={T} h={h} E={E} k={k} {xdt}")
    logits, topi, gates = K.route(x.to(DEV), w.to(DEV), None, k, "softmax", True, 1.0)
    torch.cuda.synchronize()
    ref_logits = R.router_logits(host_x(base), w.numpy(), x_kind(xdt))
    ref_topi, ref_gates = R.topk(ref_logits, k)
    rows = np.arange(T) % n
    assert np.array_equal(logits.cpu().numpy().view(np.int32), ref_logits.view(np.int32)[rows])
    assert np.array_equal(topi.cpu().numpy(), ref_topi[rows])
    assert np.array_equal(gates.cpu().numpy().view(np.int32), ref_gates.view(np.int32)[rows])


@pytest.mark.parametrize("E,xdt", [(130, torch.bfloat16), (1024, torch.bfloat16), (600, torch.float32)])
def test_route_ties_over_candidates(E, xdt):
    # Experts in equal pairs two lanes' candidates apart, in both kernels: the lower id of each pair comes first.
    T, h, k = 37, 256, 8
    x = seeded((T, h), 5, 1.0, xdt)
    w = seeded((E, h), 6, 0.05, torch.float32)
    w[64:128] = w[0:64]
    w[3] = w[2]
    say(f"route ties over {E} experts {xdt}")
    logits, topi, gates = K.route(x.to(DEV), w.to(DEV), None, k, "softmax", True, 1.0)
    ref_logits = R.router_logits(host_x(x), w.numpy(), x_kind(xdt))
    ref_topi, ref_gates = R.topk(ref_logits, k)
    assert np.array_equal(topi.cpu().numpy(), ref_topi)
    assert np.array_equal(gates.cpu().numpy().view(np.uint8), ref_gates.view(np.uint8))


def test_route_ties_and_nan():
    T, h, E, k = 64, 64, 16, 4
    x = seeded((T, h), 3, 1.0, torch.float32)
    x[0] = 0.0                              # every logit of token 0 is +0: ids 0..3 win
    w = seeded((E, h), 4, 0.1, torch.float32)
    w[9] = w[2]                             # experts 2 and 9 always tie: 2 must win
    w[13] = w[5]
    x[1, 0] = float("nan")                  # NaN logits rank last
    say("route ties/nan")
    logits, topi, gates = K.route(x.to(DEV), w.to(DEV), None, k, "softmax", True, 1.0)
    torch.cuda.synchronize()
    ref_logits = R.router_logits(x.numpy(), w.numpy(), "f32")
    ref_topi, _ = R.topk(ref_logits, k)
    assert np.array_equal(topi.cpu().numpy(), ref_topi)
    assert topi[0].tolist() == [0, 1, 2, 3]
    t = topi.cpu().numpy()
    assert not ((t == 9) & ~(t == 2).any(1, keepdims=True)).any(), "expert 9 chosen without its tie twin 2"


DISPATCH_CASES = [
    # (name, T, k, E, e0, e1, n_src, skew)
    ("tiny", 512, 2, 8, 0, 8, 1, 0.0),
    ("mixtral", 8192, 2, 8, 0, 8, 1, 0.0),
    ("dsv2lite", 16384, 6, 64, 0, 64, 1, 0.0),
    ("ep128-hot-share", 32768, 8, 128, 0, 16, 8, 1.1),
    ("ep128-tail-share", 32768, 8, 128, 112, 128, 8, 1.1),
    ("one-token", 1, 2, 4, 0, 4, 1, 0.0),
    ("ragged-sources", 1001, 3, 10, 2, 9, 7, 0.5),
]

# Experts that never receive a token in the tail-share case (empty groups in the window).
EMPTY = (113, 120, 121, 127)


def _topi(T, k, E, skew, seed, never=()):
    g = torch.Generator().manual_seed(seed)
    keys = torch.randn(T, E, generator=g, dtype=torch.float64) + (zipf_prior(E, skew) if skew else 0.0)
    keys[:, list(never)] = -torch.inf
    return torch.sort(keys, dim=1, descending=True, stable=True).indices[:, :k].to(torch.int32)


@pytest.mark.parametrize("case", DISPATCH_CASES, ids=[c[0] for c in DISPATCH_CASES])
def test_dispatch_bit_exact(case):
    name, T, k, E, e0, e1, n_src, skew = case
    topi = _topi(T, k, E, skew, 7, EMPTY if e0 == 112 else ())
    say(f"dispatch {name}: T={T} k={k} E={E} window=[{e0},{e1}) n_src={n_src}")
    plan = K.dispatch(topi.to(DEV), E, e0, e1, n_src)
    torch.cuda.synchronize()
    ref = R.dispatch(topi.numpy(), E, e0, e1, n_src)
    P = int(ref["offsets"][-1])
    assert np.array_equal(plan.counts.cpu().numpy(), ref["counts"])
    assert np.array_equal(plan.offsets.cpu().numpy(), ref["offsets"])
    assert np.array_equal(plan.src_counts.cpu().numpy(), ref["src_counts"])
    assert np.array_equal(plan.perm[:P].cpu().numpy(), ref["perm"])
    assert np.array_equal(plan.pair_row.cpu().numpy(), ref["pair_row"])
    if e0 == 112:
        assert (ref["counts"][list(EMPTY)] == 0).all() and P > 0


@pytest.mark.parametrize("T,k,E,e0,e1", [
    (2048, 2, 8, 0, 8), (1365, 3, 64, 5, 63), (1366, 3, 64, 5, 63), (64, 1, 1, 0, 1), (65, 1, 1024, 0, 1024),
    (511, 8, 130, 0, 130), (43, 6, 64, 0, 64), (257, 1, 7, 6, 7),
])
def test_dispatch_few_pairs(T, k, E, e0, e1):
    """The one-block plan at the ends of its range (up to 4096 pairs), of a wave's and of a round's pairs, with
    ids outside [0, E) and a window of the experts, and the first size past it."""
    g = torch.Generator().manual_seed(T)
    topi = _topi(T, min(k, E), E, 1.0, 11)
    topi[torch.rand(topi.shape, generator=g) < 0.05] = E + 3
    topi[torch.rand(topi.shape, generator=g) < 0.05] = -1
    say(f"dispatch few pairs T={T} k={k} E={E} window=[{e0},{e1})")
    plan = K.dispatch(topi.to(DEV), E, e0, e1)
    torch.cuda.synchronize()
    ref = R.dispatch(topi.numpy(), E, e0, e1)
    assert np.array_equal(plan.counts.cpu().numpy(), ref["counts"])
    assert np.array_equal(plan.offsets.cpu().numpy(), ref["offsets"])
    assert np.array_equal(plan.src_counts.cpu().numpy(), ref["src_counts"])
    assert np.array_equal(plan.perm[:int(ref["offsets"][-1])].cpu().numpy(), ref["perm"])
    assert np.array_equal(plan.pair_row.cpu().numpy(), ref["pair_row"])


def test_dispatch_invalid_ids_dropped():
    topi = torch.tensor([[0, 9], [-1, 1], [3, 2]], dtype=torch.int32)
    say("dispatch invalid ids")
    plan = K.dispatch(topi.to(DEV), 4)
    torch.cuda.synchronize()
    ref = R.dispatch(topi.numpy(), 4)
    assert plan.counts.cpu().tolist() == ref["counts"].tolist() == [1, 1, 1, 1, 2]
    assert np.array_equal(plan.pair_row.cpu().numpy(), ref["pair_row"])


def test_expert_bias_update_matches_reference_rule():
    counts = torch.tensor([5, 1, 3, 3, 0, 6], dtype=torch.int32)   # mean 3
    bias = torch.zeros(6, dtype=torch.float64)
    say("bias update")
    b = bias.to(DEV)
    K.update_expert_bias(b, counts.to(DEV), 0.01)
    torch.cuda.synchronize()
    ref = bias + 0.01 * torch.sign(counts.double().mean() - counts.double())
    assert torch.equal(b.cpu(), ref)
