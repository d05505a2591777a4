"""The grouped gate/up's 32-neuron tiles, taken where the 64-neuron items would not give every CU
one: the fewest and an odd number of K blocks against their three stages, one column tile per
expert and many, experts of one ragged row tile and of two, and a batch on the other side of the
choice (more than one 64-neuron item per CU). Against the float64 restatement, acts rounded to
bf16; the selection bit-exact on the call's own logits."""
import numpy as np
import pytest
import torch

from helpers import abi_prefill, assert_close, gi, make_module, oracle, sparse_expected_gpu, to_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,E,G,N,xdt", [
    (128, 5, 64, 65, torch.float32),      # two K blocks: fewer than the stages; two narrow columns
    (192 * 2, 3, 192, 129, torch.bfloat16),
    (640, 8, 128, 300, torch.float32),    # experts of two and three row tiles
    (1536, 16, 384, 65, torch.bfloat16),
    (1536, 16, 384, 333, torch.float32),
    (1536, 16, 384, 1000, torch.bfloat16),  # 64-neuron items
])
def test_prefill_narrow_tiles(pkg, H, E, G, N, xdt):
    w = gi.layer_weights(H + E + N, H=H, I=E * G, E=E)
    m = make_module(pkg, w, 0.7)
    xg = to_gpu(gi.tokens(N, N, H=H), xdt)
    y, lg, mk = abi_prefill(pkg, m, xg, E, G)
    sel = oracle.select(lg.cpu().numpy(), 0.7)
    np.testing.assert_array_equal(mk.cpu().numpy(), sel.mask)
    want = sparse_expected_gpu(xg.float().cpu().numpy(), w, sel.gates, act_bf16=True)
    assert_close(y.float().cpu().numpy(), want, what=f"narrow tiles H={H} E={E} G={G} N={N}")
    y2, _, _ = abi_prefill(pkg, m, xg, E, G, routed=False)
    assert torch.equal(y, y2)
