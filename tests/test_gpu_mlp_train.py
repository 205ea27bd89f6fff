"""The fused training passes (gh_mlp_train_*) on the GPU: the forward values equal the
layer-by-layer GEMMs bit for bit, the gradients agree with FP64 products of the same bf16
operands, at the edges of the row tiles (16, 32, 64 rows), of the 128-row slices and of the
network shapes; the packed Adam step keeps both weight layouts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GEN = [8, 256, 256, 256, 256, 256, 6]


def _net(sizes, seed=7):
    from opengate_amd.learn.mlp import MLP

    net = MLP(sizes, seed=seed)
    for b, n in zip(net.b, sizes[1:]):
        b[:n].normal_(0.0, 0.3)
    net._refresh()
    return net


def _layered(net, X):
    """Hidden activations and output through gh_gemm_bf16."""
    import torch
    from opengate_amd.learn.mlp import EPI_BIAS, EPI_BIAS_RELU

    x, ys, M = X, [], X.shape[0]
    for l in range(len(net.W)):
        K, N = net.psizes[l], net.psizes[l + 1]
        last = l == len(net.W) - 1
        Z = torch.empty(M, N, device="cuda")
        Y = None if last else torch.empty(M, N, device="cuda", dtype=torch.bfloat16)
        net._gemm(x, K, 1, net.W16[l], N, 1, M, N, K, bias=net.b[l], c32=Z, c16=Y, ldc=N,
                  mode=EPI_BIAS if last else EPI_BIAS_RELU)
        if last:
            return ys, Z
        ys.append(Y)
        x = Y


@pytest.mark.parametrize("sizes,M", [(GEN, 1), (GEN, 15), (GEN, 129), (GEN, 4097), (GEN, 8193 + 31), (GEN, 16384),
                                     ([3, 128, 128, 128, 4], 5003), ([3, 128, 128, 128, 4], 8192 + 17),
                                     ([8, 256, 6], 300), ([20, 128, 128, 16], 777), ([32, 256, 256, 9], 4096)])
def test_train_passes(sizes, M):
    import torch

    print(f"[gpu case] train passes {sizes} M={M}", flush=True)
    net = _net(sizes)
    g = torch.Generator().manual_seed(M)
    X = torch.zeros(M, net.psizes[0], dtype=torch.bfloat16)
    X[:, : sizes[0]] = torch.randn(M, sizes[0], generator=g).to(torch.bfloat16)
    X, G = X.cuda(), ((0.5 + torch.randn(M, sizes[-1], generator=g)) / M).cuda()
    out = net.forward(X)
    assert net._zs is None  # the fused path
    dW, db = net.backward(G)
    ys, Z = _layered(net, X)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(out.cpu().numpy(), Z[:, : sizes[-1]].cpu().numpy())
    for a, b in zip(net._xs[1:], ys):
        assert torch.equal(a, b)
    # FP64 gradients from the same kept activations and bf16 operands; a gradient element is
    # rounded to bf16 (2^-9) on its way to the layer below and may flip there by one rounding
    # of its FP32 sum: 2^-8 of the absolute products per layer bounds both
    gr = G.double()
    mag = gr.abs()
    for l in range(len(sizes) - 2, -1, -1):
        x = net._xs[l].double()
        k, n = net.psizes[l], net.psizes[l + 1]
        pad = lambda t: torch.nn.functional.pad(t, (0, n - t.shape[1]))  # noqa: E731
        want, lim = x.T @ pad(gr), x.abs().T @ pad(mag)
        tol = (len(sizes) - 1 - l) * 2.0 ** -8
        assert torch.all((dW[l].double() - want).abs() <= tol * lim + 1e-12), l
        assert torch.all((db[l].double() - pad(gr).sum(0)).abs() <= tol * pad(mag).sum(0) + 1e-12), l
        if l:
            w = net.W16[l].double()
            m = (net._xs[l] > 0).double()
            gr, mag = (pad(gr) @ w.T) * m, (pad(mag) @ w.abs().T) * m


def test_packed_adam_layouts():
    import torch

    print("[gpu case] packed adam", flush=True)
    net = _net([8, 256, 256, 6])
    X = torch.randn(700, 8, device="cuda").to(torch.bfloat16)
    for _ in range(2):
        net.forward(X)
        net.step(*net.backward(torch.randn(700, 6, device="cuda") / 700))
    torch.cuda.synchronize()
    for w, w16, wt in zip(net.W, net.W16, net.Wt):
        assert torch.equal(w.to(torch.bfloat16), w16)
        k, n = w.shape
        assert torch.equal(wt[:n, :k], w16.t())
        assert torch.count_nonzero(wt[n:]) == 0 and torch.count_nonzero(wt[:, k:]) == 0
