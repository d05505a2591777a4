"""How a grouped prefill call is cut into passes: every pass's buffers lie inside the workspace
that the call asks for, over widths, expert widths and token counts around the multiples of 4096
(where the share of the pairs from which the product over every expert is taken changes) and of a
grouped pass; and what the product's pass needs of its launches. Host arithmetic, no GPU."""
import pytest

from conftest import import_pkg
from helpers import prefill_passes


TOKENS = ([1, 64, 65, 2047, 2048, 2049, 5000, 8192, 8193, 9000, 11264, 20001]
          + [4096 * k + d for k in range(1, 7) for d in (-7, -4, -3, -2, -1, 0, 1, 3, 5)])


@pytest.mark.parametrize("G", [64, 128, 384, 512, 768, 960, 1024, 1408, 1664, 2944, 8192])
def test_every_pass_fits_the_workspace(G):
    lib = import_pkg()._lib.lib()
    offered = 0
    for H in range(128, 4097, 128):
        for N in TOKENS:
            have = lib.pp_prefill_workspace_bytes(N, H, 16, G)
            for tau in (0.5, 0.95):
                passes = prefill_passes(lib, N, H, 16, G, tau)
                assert sum(t for t, _, _ in passes) == N
                for i, (t, m, b) in enumerate(passes):
                    assert b <= have, (N, H, G, tau, i, t, b, have)
                    assert i + 1 == len(passes) or t % 4 == 0  # the next pass's mask rows
                    if m >= 0:  # the product is offered
                        offered += 1
                        # no short tiles and the router's count table in one kernel: the product's
                        # bucketing clears its counters and the unselected acts
                        assert 64 < t and (t + 15) // 16 * 16 <= 8192, (N, H, G, tau, i, t)
                        assert 0 < m < t * 16
                shares = {m >= 0 for _, m, _ in passes}
                assert len(shares) == 1  # one form for the call
    assert offered or G >= 2944


def test_long_calls_and_other_expert_counts():
    lib = import_pkg()._lib.lib()
    for H, E, G in [(1536, 16, 384), (4096, 16, 384), (2048, 16, 64), (1536, 96, 64), (4096, 256, 64), (256, 5, 128)]:
        for N in (1, 63, 129, 1000, 65537, 1 << 20, (1 << 20) + 4097, 0x7fffffff // 256):
            have = lib.pp_prefill_workspace_bytes(N, H, E, G)
            for t, m, b in prefill_passes(lib, N, H, E, G, 0.95, pick=(0, 1, -2, -1)):
                assert b <= have, (N, H, E, G, t, b, have)
                assert m < 0 or t > 64


def test_no_plan_for_other_shapes():
    lib = import_pkg()._lib.lib()
    for N, H, E, G in [(0, 1536, 16, 384), (-1, 1536, 16, 384), (16, 100, 16, 384), (16, 1536, 192, 32),
                       (0x7fffffff // 256 + 1, 1536, 16, 384)]:
        assert lib.pp_prefill_pass(N, H, E, G, 0.7, 0, None, None, None) == 0


@pytest.mark.parametrize("H,G,N,tau,passes,offered", [
    (1536, 384, 2047, 0.95, 1, False), (1536, 384, 2048, 0.95, 1, True), (1536, 384, 2048, 0.89, 1, False),
    (1536, 384, 8191, 0.5, 1, True),                                     # one pass less
    (1024, 384, 2600, 0.95, 1, False), (1024, 384, 3500, 0.95, 1, True),   # 66 and 84 tiles
    (640, 384, 6000, 0.95, 1, False), (640, 384, 7000, 0.95, 1, True),   # 96 and 112 tiles
    (1024, 64, 2600, 0.95, 1, True),
    (2560, 384, 6500, 0.7, 2, False), (2560, 384, 6500, 0.95, 2, True),  # as many passes as grouped
    (2560, 384, 8191, 0.7, 2, True),                                     # one less; 4096 tokens a pass
])
def test_where_the_product_is_offered(H, G, N, tau, passes, offered):
    p = prefill_passes(import_pkg()._lib.lib(), N, H, 16, G, tau)
    assert len(p) == passes
    assert all((m >= 0) == offered for _, m, _ in p)
