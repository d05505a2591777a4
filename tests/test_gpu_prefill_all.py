"""The E = 16 prefill's down projection over every expert at once, taken on the device when a pass
has enough pairs: both sides of the choice, one pass and two, a ragged last row tile, and experts
with infinite and NaN down weights, which must reach the tokens that select them and no others
(an unselected expert's act is 0, and 0 times an infinite weight is NaN)."""
import numpy as np
import pytest
import torch

from helpers import abi_prefill, assert_close, dev, gi, make_module, oracle, sparse_expected_gpu, to_gpu

pytestmark = pytest.mark.gpu
E, G, H = 16, 64, 256


@pytest.mark.parametrize("H,N,tau", [
    (H, 2048, 0.97), (H, 4096, 0.95), (H, 4097, 0.3), (H, 5003, 0.99),
    (4096, 5000, 0.97), (4096, 5000, 0.2),  # longer than a grouped pass of 2048 tokens: two passes
    (3072, 8191, 0.95),                     # passes of 4096 and 4095 tokens, where the share changes
    (H, 9000, 0.97),                        # more tokens than the form's count table: grouped
])
def test_prefill_all_experts(pkg, H, N, tau):
    w = gi.layer_weights(N, H=H, I=E * G, E=E)
    m = make_module(pkg, w, tau)
    xg = to_gpu(gi.tokens(N + 1, N, H=H), torch.bfloat16 if N % 2 else torch.float32)
    y, lg, mk = abi_prefill(pkg, m, xg, E, G, tau=tau)
    sel = oracle.select(lg.cpu().numpy(), tau)
    np.testing.assert_array_equal(mk.cpu().numpy(), sel.mask)
    want = sparse_expected_gpu(xg.float().cpu().numpy(), w, sel.gates, act_bf16=True)
    assert_close(y.float().cpu().numpy(), want, what=f"N={N} tau={tau}")
    y2, _, _ = abi_prefill(pkg, m, xg, E, G, tau=tau, routed=False)
    assert torch.equal(y, y2)


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_prefill_all_experts_nonfinite_weights(pkg, bad):
    N, tau = 4100, 0.9
    w = gi.layer_weights(3, H=H, I=E * G, E=E)
    xg = to_gpu(gi.tokens(4, N, H=H))
    m = make_module(pkg, w, tau)
    y, _, mk = abi_prefill(pkg, m, xg, E, G, tau=tau)
    assert mk.float().mean() > 0.5  # the side under test
    perm = oracle.pack_permutation(w["expert_ids"])
    w2 = dict(w, w_down=w["w_down"].copy())
    w2["w_down"][7, perm[5 * G + 3]] = bad  # expert 5, output column 7
    y2, _, mk2 = abi_prefill(pkg, make_module(pkg, w2, tau), xg, E, G, tau=tau)
    assert torch.equal(mk, mk2)
    hit = torch.zeros(N, H, dtype=torch.bool, device=dev())
    hit[:, 7] = mk[:, 5].bool()
    assert bool((~torch.isfinite(y2.float()))[hit].all())
    assert torch.equal(torch.isfinite(y2.float()), ~hit)
    clean = ~hit
    clean[:, 7] = False
    assert torch.equal(y2[clean], y[clean])
    rest = ~mk[:, 5].bool()  # column 7 again, summed over the selected experts alone
    d = (y2[rest, 7].float() - y[rest, 7].float()).abs()
    assert bool((d <= 2e-3 + 2e-2 * y[rest, 7].float().abs()).all())
