"""The dense form's small-batch kernels (csrc/dense_few.h) at the sizes where their tiles end:
one token, 16-token blocks and the last of them ragged, the largest batch of the form, K steps
that do not divide over the waves, several K chunks and groups of token blocks, experts of one
and of several K steps, K parts whose last waves hold no step, and the selection inside and
outside the gate/up launch. Against the float64 restatement, the selection bit-exact on the
call's own logits, a router bias on E > 1, repeated calls bit-identical."""
import numpy as np
import pytest
import torch

from helpers import abi_prefill, assert_close, gi, make_module, oracle, sparse_expected, to_gpu

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("H,E,G,N,xdt", [
    (1536, 192, 32, 1, torch.float32),
    (1536, 192, 32, 15, torch.bfloat16),
    (1536, 192, 32, 16, torch.float32),
    (1536, 192, 32, 17, torch.bfloat16),
    (1536, 192, 32, 224, torch.float32),   # the largest batch of the form
    (1536, 192, 32, 225, torch.bfloat16),  # the first on GEMM tiles: 128-row down tiles in eight K parts
    (1536, 24, 32, 50, torch.bfloat16),    # selection in a launch of its own; 96 units in threes
    (1536, 5, 160, 33, torch.float32),     # 100 units: a last workgroup of one; five K steps an expert
    (1408, 65, 32, 70, torch.bfloat16),    # 44 K steps over eight waves; E just above the in-launch selection
    (128, 3, 32, 100, torch.float32),      # four K steps, four waves without any
    (256, 66, 32, 40, torch.float32),      # one whole K step a wave
    (512, 200, 32, 129, torch.bfloat16),   # two
    (768, 24, 32, 16, torch.float32),      # three
    (1024, 5, 160, 100, torch.bfloat16),   # four
    (1280, 100, 32, 17, torch.float32),    # five
    (128, 70, 32, 192, torch.float32),     # the largest batch below H = 512
    (384, 64, 32, 161, torch.bfloat16),    # above it with the selection apart: GEMM tiles
    (640, 200, 32, 129, torch.bfloat16),   # two groups of token blocks on weights loaded once
    (1664, 20, 96, 64, torch.float32),     # two K chunks, the second of one step
    (4096, 70, 32, 49, torch.bfloat16),    # three K chunks
    (640, 5, 160, 300, torch.float32),     # down: a 128-row tile of 44 tokens, H in a short last column tile
    (256, 70, 96, 1100, torch.bfloat16),   # nine 128-row tiles
])
def test_dense_few_shapes(pkg, H, E, G, N, xdt):
    seed = H + E * 7 + G + N
    w = gi.layer_weights(seed, H=H, I=E * G, E=E)
    m = make_module(pkg, w, 0.7, bias=gi.zipf_bias(E) if E > 1 else None)
    xg = to_gpu(gi.tokens(seed + 1, N, H=H), xdt)
    y, lg, mk = abi_prefill(pkg, m, xg, E, G)
    sel = oracle.select(lg.cpu().numpy(), 0.7)
    np.testing.assert_array_equal(mk.cpu().numpy(), sel.mask)
    assert_close(y.float().cpu().numpy(), sparse_expected(xg.float().cpu().numpy(), w, sel.gates, act_bf16=True),
                 what=f"small dense batch H={H} E={E} G={G} N={N}")
    y2, _, _ = abi_prefill(pkg, m, xg, E, G, routed=False)
    assert torch.equal(y, y2)


@pytest.mark.parametrize("xdt", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N", [1, 200, 512])
def test_few_token_logits_equal_the_staged_kernels(pkg, N, xdt):
    """Up to 512 tokens the logits come from route_logits_few_kernel, above from
    route_logits_kernel: one summation order, so the same bits for the same rows."""
    E, H = 192, 1536
    w = gi.layer_weights(5, H=H, I=E * 32, E=E)
    m = make_module(pkg, w, 0.7)
    x = to_gpu(gi.tokens(6, 600, H=H), xdt)
    full = pkg.ops.route(x, m.router_packed, E, 0.7)
    few = pkg.ops.route(x[:N].contiguous(), m.router_packed, E, 0.7)
    assert torch.equal(few["logits"], full["logits"][:N])
    assert torch.equal(few["mask"], full["mask"][:N])
