"""The masked-gate backward where its persistent row loop and its register-held places can go
wrong: row lengths around the steps of 2048 elements, the longest row, more rows than workgroups
(each takes several, the next one's loads in flight), experts of uneven sizes and without
neurons, one lane per expert, no d_inter. d_inter bit for bit against the products, d_gates
against float64 sums: a sum of m fp32 products carries at most about m 2^-24 of the sum of their
magnitudes (each product's rounding and m - 1 additions), and repeated calls give the same bits."""
import pytest
import torch

from helpers import dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("N,I,E", [
    (1, 8, 1), (3000, 2040, 3), (2600, 2048, 256), (1100, 2056, 100), (1500, 6152, 192), (700, 8184, 7),
    (300, 12296, 33), (530, 16384, 64),
])
def test_masked_gate_bwd_rows(pkg, N, I, E, dtype):
    g = torch.Generator(device=dev()).manual_seed(N + I + E)
    x = torch.randn(N, I, device=dev(), generator=g).to(dtype)
    d = torch.randn(N, I, device=dev(), generator=g).to(dtype)
    gates = torch.rand(N, E, device=dev(), generator=g)
    ids = (torch.rand(I, device=dev(), generator=g) ** 2 * E).long().clamp(max=E - 1)  # uneven
    if E > 2:
        ids[ids == 1] = 0  # an expert without neurons
    layout = pkg.ops.masked_gate_layout(ids, E)
    d_inter, d_gates = pkg.ops.masked_gate_bwd(d, x, gates, *layout)
    held = gates.to(dtype).float()
    assert torch.equal(d_inter, (d.float() * held[:, ids]).to(dtype))
    onehot = torch.zeros(I, E, dtype=torch.float64, device=dev())
    onehot[torch.arange(I, device=dev()), ids] = 1.0
    prod = d.double() * x.double()
    err = (d_gates.double() - prod @ onehot).abs()
    m = torch.bincount(ids, minlength=E).double()
    assert bool((err <= (prod.abs() @ onehot) * m.clamp(min=1) * 2.0 ** -24).all())
    none, again = pkg.ops.masked_gate_bwd(d, x, gates, *layout, need_d_inter=False)
    assert none is None and torch.equal(again, d_gates)


@pytest.mark.parametrize("dtype,N", [(torch.float32, 2048), (torch.float32, 2049), (torch.bfloat16, 4096),
                                     (torch.bfloat16, 4097)])
def test_masked_gate_fwd_rows(pkg, dtype, N):
    """The forward up to 128 MiB of rows and above, where its results are stored non-temporally:
    bit for bit against the products."""
    I, E = 16384, 37
    g = torch.Generator(device=dev()).manual_seed(N)
    x = torch.randn(N, I, device=dev(), generator=g).to(dtype)
    gates = torch.rand(N, E, device=dev(), generator=g)
    ids = torch.randint(E, (I,), device=dev(), generator=g)
    want = (x.float() * gates.to(dtype).float()[:, ids]).to(dtype)
    eid = pkg.ops.masked_gate_layout(ids, E)[0]
    assert torch.equal(pkg.ops.masked_gate_fwd(x, gates, eid), want)
