"""The E = 16 prefill's down projection over every expert at once, taken on the device when a pass
that is offered it has enough pairs: both sides of the choice and calls that are not offered it,
each told from the call's plan and its own mask; one pass and two, a ragged last row tile, tiles
cut in K and whole ones, and experts with infinite and NaN down weights, which must reach the
tokens that select them and no others (an unselected expert's act is 0, and 0 times an infinite
weight is NaN)."""
import numpy as np
import pytest
import torch

from helpers import (abi_prefill, assert_close, dev, gi, make_module, oracle, prefill_passes, sparse_expected_gpu,
                     to_gpu)

pytestmark = pytest.mark.gpu
E, G, H = 16, 64, 256


def forms(pkg, N, H, tau, mask):
    """What each pass of the call ran: "grouped" (not offered the product), "combine" (too few
    pairs for it) or "product"."""
    t0, out = 0, []
    for t, min_pairs, _ in prefill_passes(pkg._lib.lib(), N, H, E, G, tau):
        pairs = int(mask[t0:t0 + t].sum())
        out.append("grouped" if min_pairs < 0 else "product" if pairs >= min_pairs else "combine")
        t0 += t
    assert t0 == N
    return out


@pytest.mark.parametrize("H,N,tau,want_forms", [
    # the partial sums of cut tiles need more than the workspace of these holds
    (H, 2048, 0.97, ["grouped"]), (H, 4096, 0.95, ["grouped"]), (H, 4097, 0.3, ["grouped"]),
    (H, 5003, 0.99, ["grouped"]),
    (1536, 2048, 0.97, ["product"]),         # the fewest tokens and tiles
    (1536, 5003, 0.99, ["product"]),
    (1536, 8000, 0.97, ["product"]),         # one round of whole tiles, in one pass; grouped it would be two
    (1536, 8000, 0.2, ["combine"]),
    (4096, 5000, 0.97, ["product"] * 2), (4096, 5000, 0.2, ["combine"] * 2),  # two passes
    (3072, 8191, 0.95, ["product"] * 2),     # passes of 4096 and 4095 tokens, where the share changes
    (H, 9000, 0.97, ["grouped"]),            # more tokens than the form's count table
])
def test_prefill_all_experts(pkg, H, N, tau, want_forms):
    w = gi.layer_weights(N, H=H, I=E * G, E=E)
    m = make_module(pkg, w, tau)
    xg = to_gpu(gi.tokens(N + 1, N, H=H), torch.bfloat16 if N % 2 else torch.float32)
    y, lg, mk = abi_prefill(pkg, m, xg, E, G, tau=tau)
    sel = oracle.select(lg.cpu().numpy(), tau)
    np.testing.assert_array_equal(mk.cpu().numpy(), sel.mask)
    assert forms(pkg, N, H, tau, mk) == want_forms
    want = sparse_expected_gpu(xg.float().cpu().numpy(), w, sel.gates, act_bf16=True)
    assert_close(y.float().cpu().numpy(), want, what=f"N={N} tau={tau}")
    y2, _, _ = abi_prefill(pkg, m, xg, E, G, tau=tau, routed=False)
    assert torch.equal(y, y2)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
@pytest.mark.parametrize("H,N", [
    (512, 5399),   # 22 x 3 tiles, all of them cut in K
    (1664, 8192),  # 32 x 9 tiles: one round of whole tiles, the rest cut in K
])
def test_prefill_all_experts_nonfinite_weights(pkg, H, N, bad):
    """The elements that a bad weight reaches, and the bits of all others, whatever the output held
    before the call: a workgroup must not take what another has not stored yet for a result."""
    tau = 0.95
    w = gi.layer_weights(3, H=H, I=E * G, E=E)
    xg = to_gpu(gi.tokens(4, N, H=H))
    m = make_module(pkg, w, tau)
    y, _, mk = abi_prefill(pkg, m, xg, E, G, tau=tau)
    assert forms(pkg, N, H, tau, mk) == ["product"]
    perm = oracle.pack_permutation(w["expert_ids"])
    w2 = dict(w, w_down=w["w_down"].copy())
    hit = torch.zeros(N, H, dtype=torch.bool, device=dev())
    for e, g, h in [(5, 3, 7), (5, 40, H - 1), (15, 63, 200), (0, 0, 300)]:  # expert, neuron, output column
        w2["w_down"][h, perm[e * G + g]] = bad
        hit[:, h] = mk[:, e].bool()
    m2 = make_module(pkg, w2, tau)
    y2, _, mk2 = abi_prefill(pkg, m2, xg, E, G, tau=tau, fill=0.0)
    assert torch.equal(mk, mk2)
    assert bool((~torch.isfinite(y2.float()))[hit].all())
    assert torch.equal(torch.isfinite(y2.float()), ~hit)
    cols = hit.any(0)
    assert torch.equal(y2[:, ~cols], y[:, ~cols])
    # the same columns, summed over the selected experts alone
    rest = cols[None] & ~hit
    d = (y2[rest].float() - y[rest].float()).abs()
    assert bool((d <= 2e-3 + 2e-2 * y[rest].float().abs()).all())
    for fill in (float("nan"), float("inf")):
        y3, _, _ = abi_prefill(pkg, m2, xg, E, G, tau=tau, fill=fill)
        assert torch.equal(y3.view(torch.int16), y2.view(torch.int16))
