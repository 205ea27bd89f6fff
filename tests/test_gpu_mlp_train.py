"""The fused training passes (gh_mlp_train_*) on the GPU: the forward values equal the
layer-by-layer GEMMs bit for bit, the gradients agree with FP64 products of the same bf16
operands, at the edges of the row tiles (16, 32, 64 rows), of the 128-row slices and of the
network shapes; the packed Adam step keeps every weight layout."""
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


def _rows(t):
    """A kept matrix (tiles of 16 rows in fragment order) as rows."""
    m, c = t.shape
    return t.reshape(m // 16, c // 32, 4, 16, 8).permute(0, 3, 1, 2, 4).reshape(m, c)


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
    _, Xt, Y = net._xs
    kept = [_rows(Xt), *(_rows(y) for y in Y)]
    assert torch.equal(kept[0][:M, : net.psizes[0]], X) and torch.count_nonzero(kept[0][M:]) == 0
    for a, b in zip(kept[1:], ys):
        assert torch.equal(a[:M], b) and torch.count_nonzero(a[M:]) == 0
    xs = [X, *ys]
    # FP64 gradients from the same kept activations and bf16 operands; a gradient element is
    # rounded to bf16 (2^-9) on its way to the layer below and may flip there by one rounding
    # of its FP32 sum: 2^-8 of the absolute products per layer bounds both
    gr = G.double()
    mag = gr.abs()
    for l in range(len(sizes) - 2, -1, -1):
        x = xs[l].double()
        k, n = net.psizes[l], net.psizes[l + 1]
        pad = lambda t: torch.nn.functional.pad(t, (0, n - t.shape[1]))  # noqa: E731
        want, lim = x.T @ pad(gr), x.abs().T @ pad(mag)
        tol = (len(sizes) - 1 - l) * 2.0 ** -8
        assert torch.all((dW[l].double() - want).abs() <= tol * lim + 1e-12), l
        assert torch.all((db[l].double() - pad(gr).sum(0)).abs() <= tol * pad(mag).sum(0) + 1e-12), l
        if l:
            w = net.W16[l].double()
            m = (xs[l] > 0).double()
            gr, mag = (pad(gr) @ w.T) * m, (pad(mag) @ w.abs().T) * m


@pytest.mark.parametrize("M", [1, 16, 4097, 8193, 32768, 32769, 65536, 65537, 65536 + 32769])
def test_packed_forward_forms(M):
    """Every form that gh_mlp_forward_packed_bf16 takes (row tiles, 8-wave, both) against the
    layer-by-layer GEMMs, bit for bit; 128 at its own edges of the same sizes."""
    import torch
    from opengate_amd.learn.mlp import _pointers

    for sizes in (GEN, [3, 128, 128, 128, 4]):
        print(f"[gpu case] packed forward {sizes} M={M}", flush=True)
        net = _net(sizes)
        X = torch.zeros(M, 8, device="cuda", dtype=torch.bfloat16)
        X[:, : sizes[0]] = torch.randn(M, sizes[0], device="cuda", generator=torch.Generator("cuda").manual_seed(M))
        Z = torch.full((M, 8), float("nan"), device="cuda")
        net.infer_fused(X, Z)
        want = _layered(net, X)[1]
        torch.cuda.synchronize()
        n = sizes[-1]
        assert torch.equal(Z[:, :n], want[:, :n]) and bool(Z[:, n:].isnan().all())
        # gh_mlp_forward_bf16: the same from rows of K values
        L = len(net.W)
        wt = [torch.zeros(16 if l == L - 1 else w.shape[1], 32 if l == 0 else w.shape[0], device="cuda",
                          dtype=torch.bfloat16) for l, w in enumerate(net.W16)]
        for a, w in zip(wt, net.W16):
            a[: w.shape[1], : w.shape[0]] = w.t()
        R = torch.empty(M, 8, device="cuda")
        assert net.lib.gh_mlp_forward_bf16(X.data_ptr(), 8, M, L, 8, net.psizes[1], n, _pointers(wt), _pointers(net.b),
                                           R.data_ptr(), 8, None) == 0
        torch.cuda.synchronize()
        assert torch.equal(R[:, :n], want[:, :n])


@pytest.mark.parametrize("n", [1, 17, 4097, 32768, 32769, 65536 + 5, 65536 + 40000])
def test_generate_in_one_call(n):
    """gh_exitplane_generate gives the bits of noise, network and decoder called one by one, for
    every split of n into launches."""
    import torch
    from opengate_amd.learn.exitplane import ExitPlaneGenerator, QuantileMap

    print(f"[gpu case] generate in one call n={n}", flush=True)
    gen = ExitPlaneGenerator((32.0, 32.0, 142.5), 0.0, seed=2)
    g = torch.Generator("cuda").manual_seed(1)
    gen.qmap = QuantileMap(torch.sort(torch.randn(6, 257, device="cuda", generator=g), 1).values, 4.0)
    assert gen._one_call()
    got = gen.generate(n, 99, first=2**33 + 7, chunk=65536, weight=0.5)
    want = gen.generate(n, 99, first=2**33 + 7, weight=0.5, events=[])
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_packed_adam_layouts():
    import torch

    from opengate_amd.learn.mlp import fragment_order

    print("[gpu case] packed adam", flush=True)
    net = _net([8, 256, 256, 6])
    X = torch.randn(700, 8, device="cuda").to(torch.bfloat16)
    for _ in range(2):
        net.forward(X)
        net.step(*net.backward(torch.randn(700, 6, device="cuda") / 700))
    torch.cuda.synchronize()
    for l, (w, w16) in enumerate(zip(net.W, net.W16)):
        assert torch.equal(w.to(torch.bfloat16), w16)
        want = torch.empty_like(net.Wf[l])
        assert torch.equal(fragment_order(w16.t(), want), net.Wf[l])
        if l:
            want = torch.empty_like(net.Wb[l])
            assert torch.equal(fragment_order(w16, want), net.Wb[l])
