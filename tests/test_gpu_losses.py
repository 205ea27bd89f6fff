"""The training losses' kernels on the GPU: the sliced 2-Wasserstein gradient equals the
tensor form bit for bit (sorts are exact, the gradient is one product), softmax
cross-entropy agrees with FP64."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M,P,quantum", [(1, 3, None), (63, 9, None), (1000, 134, None), (4096, 17, None),
                                         (4097, 8, None), (8193, 5, 0.25), (12345, 134, None), (16384, 134, None),
                                         (16384, 7, 0.5)])
def test_sliced_w2_against_tensor_form(M, P, quantum):
    import torch
    from opengate_amd import _abi as A

    print(f"[gpu case] sliced w2 M={M} P={P} quantum={quantum}", flush=True)
    lib = A.load_library()
    g = torch.Generator("cuda").manual_seed(M)
    a = torch.randn(M, 8, device="cuda", generator=g)[:, :6]
    b = 0.7 * torch.randn(M, 6, device="cuda", generator=g) + 0.1
    th = torch.randn(6, P, device="cuda", generator=g)
    if quantum:  # many equal values, zeros among them
        a, b = torch.round(a / quantum) * quantum + 0.0, torch.round(b / quantum) * quantum + 0.0
        th = torch.round(th)
    grad, loss = torch.full((M, P), float("nan"), device="cuda"), torch.empty(P, device="cuda")
    work = torch.empty(2 * M * P, device="cuda")
    assert lib.gh_sliced_w2(a.data_ptr(), a.stride(0), b.data_ptr(), 6, th.data_ptr(), M, 6, P, work.data_ptr(),
                            grad.data_ptr(),
                            loss.data_ptr(), None) == 0
    torch.cuda.synchronize()
    # the projections: one FP32 rounding per multiply-add (a double holds the product exactly)
    x, y = torch.zeros(M, P, device="cuda"), torch.zeros(M, P, device="cuda")
    for k in range(6):
        x = (a[:, k:k + 1].double() * th[k].double() + x.double()).float()
        y = (b[:, k:k + 1].double() * th[k].double() + y.double()).float()
    x.requires_grad_(True)
    val = ((torch.sort(x, dim=0, stable=True).values - torch.sort(y, dim=0, stable=True).values) ** 2).mean()
    val.backward()
    assert torch.equal(grad, x.grad)
    d = torch.sort(x.detach().double(), 0).values - torch.sort(y.double(), 0).values
    # FP32 sums of M squares per column in 1024-lane partial sums: a relative error far below 1e-5
    assert torch.all((loss.double() - (d ** 2).sum(0)).abs() <= 1e-5 * (d ** 2).sum(0) + 1e-12)


def test_sliced_w2_rejects():
    import torch
    from opengate_amd import _abi as A

    lib = A.load_library()
    t = torch.zeros(8, device="cuda")
    p = t.data_ptr()
    assert lib.gh_sliced_w2(p, 6, p, 6, p, 16385, 6, 1, p, p, p, None) != 0
    assert lib.gh_sliced_w2(p, 6, p, 6, p, 0, 6, 1, p, p, p, None) != 0
    assert lib.gh_sliced_w2(p, 9, p, 9, p, 1, 9, 1, p, p, p, None) != 0
    assert lib.gh_softmax_ce(p, 1, 1, 17, p, None, p, p, None) != 0


@pytest.mark.parametrize("M,C,pitch", [(1, 2, 2), (255, 4, 8), (257, 4, 4), (5003, 16, 16)])
def test_softmax_ce_against_fp64(M, C, pitch):
    import torch
    from opengate_amd import _abi as A

    print(f"[gpu case] softmax ce M={M} C={C}", flush=True)
    lib = A.load_library()
    g = torch.Generator("cuda").manual_seed(M)
    Z = 3 * torch.randn(M, pitch, device="cuda", generator=g)
    cls = torch.randint(0, C, (2 * M,), device="cuda", generator=g)
    rows = torch.randint(0, 2 * M, (M,), device="cuda", generator=g)
    grad, loss = torch.empty(M, C, device="cuda"), torch.empty((M + 255) // 256, device="cuda")
    assert lib.gh_softmax_ce(Z.data_ptr(), pitch, M, C, cls.data_ptr(), rows.data_ptr(), grad.data_ptr(),
                             loss.data_ptr(), None) == 0
    torch.cuda.synchronize()
    z = Z[:, :C].double().requires_grad_(True)
    val = torch.nn.functional.cross_entropy(z, cls[rows])
    val.backward()
    val = val.detach()
    # a probability carries a few FP32 roundings of exp and log
    assert torch.all((grad.double() - z.grad).abs() <= 4e-6 / M)
    assert abs(float(loss.double().sum()) / M - float(val)) <= 1e-5 * max(1.0, float(val))
