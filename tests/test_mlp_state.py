"""Networks from stored states: every floating type, with or without the padding, gives the
weights and biases of the same state in padded FP32, and results within the network's sizes."""
import pytest
import torch

from opengate_amd.learn.mlp import MLP, fragment_order, pad

GEN = [8, 256, 256, 6]
RESPONSE = [3, 128, 128, 128, 4]
DTYPES = (torch.float32, torch.bfloat16, torch.float16, torch.float64)


def _state(sizes, dtype, padded, device="cpu"):
    g = torch.Generator().manual_seed(11)
    W, b = [], []
    for k, n in zip(sizes[:-1], sizes[1:]):
        w, v = torch.randn(k, n, generator=g) * (2.0 / k) ** 0.5, 0.3 * torch.randn(n, generator=g)
        if padded:
            w = torch.nn.functional.pad(w, (0, pad(n, 8) - n, 0, pad(k, 8) - k))
            v = torch.nn.functional.pad(v, (0, pad(n, 8) - n))
        W.append(w.to(dtype).to(device))
        b.append(v.to(dtype).to(device))
    return {"W": W, "b": b}


def _loaded(sizes, state, device):
    net = MLP(sizes, device=device, seed=3)
    net.load_state_dict(state)
    return net


@pytest.mark.parametrize("sizes", [GEN, RESPONSE, [5, 24, 40, 3]])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("padded", [True, False])
def test_state_is_kept_as_padded_fp32(sizes, dtype, padded):
    st = _state(sizes, dtype, padded)
    full = _state(sizes, dtype, True)
    net = _loaded(sizes, st, "cpu")
    for l in range(len(sizes) - 1):
        assert net.W[l].dtype == net.b[l].dtype == torch.float32
        assert torch.equal(net.W[l], full["W"][l].float()) and torch.equal(net.b[l], full["b"][l].float())
        assert torch.equal(net.W16[l], full["W"][l].to(torch.bfloat16))
        if net.Wf is not None:
            assert torch.equal(net.Wf[l], fragment_order(net.W16[l].t(), torch.empty_like(net.Wf[l])))


def test_bias_of_one_row_or_one_value():
    st = _state(GEN, torch.float32, True)
    st["b"] = [st["b"][0][None], torch.tensor(0.5), st["b"][2][:6]]
    net = _loaded(GEN, st, "cpu")
    assert [tuple(b.shape) for b in net.b] == [(256,), (256,), (8,)]
    assert bool((net.b[1] == 0.5).all()) and bool((net.b[2][6:] == 0).all())


def test_a_missing_bias_is_refused():
    st = _state(GEN, torch.float32, True)
    st["b"].pop()
    with pytest.raises(IndexError):
        _loaded(GEN, st, "cpu")._fused_args()


@pytest.mark.gpu
@pytest.mark.parametrize("sizes", [GEN, RESPONSE, [5, 24, 40, 3]])
@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("padded", [True, False])
def test_results_of_any_stored_type(sizes, dtype, padded):
    print(f"[gpu case] network state {sizes} {dtype} padded={padded}", flush=True)
    want = _loaded(sizes, {k: [t.float() for t in v] for k, v in _state(sizes, dtype, True).items()}, "cuda")
    st = _state(sizes, dtype, padded, "cuda")
    net = _loaded(sizes, st, "cuda")
    X = torch.zeros(300, net.psizes[0], device="cuda", dtype=torch.bfloat16)
    X[:, : sizes[0]] = torch.randn(300, sizes[0], generator=torch.Generator().manual_seed(1)).cuda()
    for keep in (True, False):
        assert torch.equal(net.forward(X, keep=keep), want.forward(X, keep=keep))
    grad = torch.randn(300, sizes[-1], generator=torch.Generator().manual_seed(2)).cuda() / 300
    for x, y in zip(sum(net.backward(grad), []), sum(want.backward(grad), [])):
        assert torch.equal(x, y)
    # tensors set directly, then refreshed: the copies and the biases of the passes
    if net.Wf is not None and padded:
        net.W, net.b = st["W"], st["b"]
        net._refresh()
        Z = [torch.empty(300, 8, device="cuda") for _ in range(2)]
        net.infer_fused(X, Z[0])
        want.infer_fused(X, Z[1])
        assert torch.equal(Z[0][:, : sizes[-1]], Z[1][:, : sizes[-1]])


@pytest.mark.gpu
@pytest.mark.parametrize("layers", [32, 33])
def test_networks_of_many_layers(layers):
    # beyond the tensors of one packing launch the copies are made one by one
    print(f"[gpu case] network of {layers} layers", flush=True)
    sizes = [8] * (layers + 1)
    net = _loaded(sizes, _state(sizes, torch.float32, True), "cuda")
    for w, w16 in zip(net.W, net.W16):
        assert torch.equal(w.to(torch.bfloat16), w16)
    out = net.forward(torch.randn(20, 8, device="cuda").to(torch.bfloat16))
    assert out.shape == (20, 8) and bool(out.isfinite().all())
