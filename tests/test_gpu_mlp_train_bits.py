"""The fused backward pass against the layer-by-layer one, bit for bit: weight gradients (the split
of gh_gemm_bf16's reductions) and, with tensor_sums, bias gradients (PyTorch's sums of the FP32
gradients), at the ends of row tiles and of reduction slices, where a lost row of thousands is
below any bound on rounding. The kernels' own bias sums against FP64 sums of the same gradients."""
import pytest
import torch

pytestmark = pytest.mark.gpu

GEN = [8, 256, 256, 256, 256, 256, 6]
RESPONSE = [3, 128, 128, 128, 4]


def _net(sizes, seed=7):
    from opengate_amd.learn.mlp import MLP

    net = MLP(sizes, seed=seed)
    for b, n in zip(net.b, sizes[1:]):
        b[:n].normal_(0.0, 0.3)
    net._refresh()
    return net


def _layered(net, X, G):
    """Weight gradients and the FP32 gradients of every layer's outputs, a GEMM launch each."""
    from opengate_amd.learn.mlp import EPI_BIAS, EPI_BIAS_RELU, EPI_DRELU, EPI_STORE

    L, M, P = len(net.W), X.shape[0], net.psizes
    f32 = lambda *s: torch.empty(*s, device="cuda")  # noqa: E731
    b16 = lambda *s: torch.empty(*s, device="cuda", dtype=torch.bfloat16)  # noqa: E731
    xs, zs = [X], []
    for l in range(L):
        K, N = P[l], P[l + 1]
        zs.append(f32(M, N))
        if l < L - 1:
            xs.append(b16(M, N))
            net._gemm(xs[l], K, 1, net.W16[l], N, 1, M, N, K, bias=net.b[l], c32=zs[l], c16=xs[-1], ldc=N,
                      mode=EPI_BIAS_RELU)
        else:
            net._gemm(xs[l], K, 1, net.W16[l], N, 1, M, N, K, bias=net.b[l], c32=zs[l], ldc=N, mode=EPI_BIAS)
    g32 = torch.nn.functional.pad(G, (0, P[-1] - G.shape[1]))
    g16 = g32.to(torch.bfloat16)
    dW, grads = [None] * L, [None] * L
    for l in range(L - 1, -1, -1):
        K, N = P[l], P[l + 1]
        grads[l] = g32
        dW[l] = f32(K, N)
        net._gemm(xs[l], 1, K, g16, N, 1, K, N, M, c32=dW[l], ldc=N, mode=EPI_STORE)
        if l:
            n32, n16 = f32(M, K), b16(M, K)
            net._gemm(g16, N, 1, net.W16[l], 1, N, M, K, N, zprev=zs[l - 1], ldz=K, c32=n32, c16=n16, ldc=K,
                      mode=EPI_DRELU)
            g32, g16 = n32, n16
    return dW, grads


# row tiles of 16, 32 (from 4097 rows on) and 64 rows (from 8193); slices of about 512 rows from 2048
# rows on; beyond the column sums' 65536 rows
@pytest.mark.parametrize("sizes,M", [(GEN, 1), (GEN, 15), (GEN, 129), (GEN, 2047), (GEN, 2048), (GEN, 2561), (GEN, 4097),
                                     (GEN, 8193 + 31), (GEN, 16384), (RESPONSE, 5003), (RESPONSE, 8192 + 17),
                                     (RESPONSE, 65537), ([8, 256, 6], 300), ([20, 128, 128, 16], 2777),
                                     ([32, 256, 256, 9], 4096)])
def test_backward_bits(sizes, M):
    print(f"[gpu case] backward bits {sizes} M={M}", flush=True)
    net = _net(sizes)
    g = torch.Generator().manual_seed(M)
    X = torch.zeros(M, net.psizes[0], dtype=torch.bfloat16)
    X[:, : sizes[0]] = torch.randn(M, sizes[0], generator=g).to(torch.bfloat16)
    X, G = X.cuda(), ((0.5 + torch.randn(M, sizes[-1], generator=g)) / M).cuda()
    net.forward(X)
    assert net._zs is None  # the fused path
    want, grads = _layered(net, X, G)
    for tensor_sums in (False, True):
        dW, db = net.backward(G, tensor_sums=tensor_sums)
        for l in range(len(want)):
            assert torch.equal(dW[l], want[l]), (tensor_sums, l)
            if tensor_sums:
                assert torch.equal(db[l], grads[l].sum(0)), l
                continue
            # FP32 additions of a value's longest way: rows of a tile (4 per lane, 4 exchanges), tiles
            # (16 chains, then one), each rounding at most 2^-24 of the absolute sum
            tile = 16 if M <= 4096 else (32 if M <= 8192 else 64)
            chain = 8 + (M // tile + 16) // 16 + 16
            lim = chain * 2.0**-24 * grads[l].double().abs().sum(0)
            assert torch.all((db[l].double() - grads[l].double().sum(0)).abs() <= lim), l
