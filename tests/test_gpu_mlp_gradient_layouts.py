"""MLP.backward takes output gradients of every layout: rows that overlap (expanded), columns or
rows apart, other types, with the bits of the contiguous FP32 gradient of the same values."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SIZES = [8, 128, 128, 6]


def _layouts(M, n):
    row = torch.randn(1, n, device="cuda", generator=torch.Generator("cuda").manual_seed(M)) / M
    full = torch.randn(M, n, device="cuda", generator=torch.Generator("cuda").manual_seed(M + 1)) / M
    wide = torch.randn(M, n + 3, device="cuda")
    strip = torch.randn(M + n, device="cuda")
    yield "expanded row", row.expand(M, n)
    yield "expanded value", row[:, :1].expand(M, n)
    yield "expanded column", full[:, :1].expand(M, n)
    yield "overlapping rows", strip.as_strided((M, n), (1, 1))
    yield "columns of a wider tensor", wide[:, 1:n + 1]
    yield "transposed", full.t().contiguous().t()
    yield "FP64", full.double()
    yield "bf16", full.to(torch.bfloat16)


@pytest.mark.parametrize("M", [1, 33, 2049])
@pytest.mark.parametrize("tensor_sums", [False, True])
def test_layouts(M, tensor_sums):
    from opengate_amd.learn.mlp import MLP

    net = MLP(SIZES, seed=5)
    net.forward(torch.randn(M, 8, device="cuda").to(torch.bfloat16))
    assert net._zs is None  # the fused path
    for name, g in _layouts(M, SIZES[-1]):
        print(f"[gpu case] gradient layout {name} M={M} tensor_sums={tensor_sums}", flush=True)
        want = net.backward(g.float().contiguous(), tensor_sums=tensor_sums)
        got = net.backward(g, tensor_sums=tensor_sums)
        for a, b in zip(sum(got, []), sum(want, [])):
            assert torch.equal(a, b), name
