"""The transport's short division against the correctly rounded quotient, bit for bit (an FP64
division rounded to FP32 is that: 53 bits are more than twice 24 and two): every divisor mantissa
with dividends of all kinds, and the operands of the places that use it."""
import pytest
import torch

pytestmark = pytest.mark.gpu

MEC2 = 0.51099895  # MeV


def _check(a, b, what):
    from opengate_amd import _abi as A

    a, b = a.float().contiguous(), b.float().contiguous()
    out = torch.empty_like(a)
    assert A.load_library().gh_quotient(a.data_ptr(), b.data_ptr(), a.numel(), out.data_ptr(), None) == 0
    torch.cuda.synchronize()
    want = (a.double() / b.double()).float()
    bad = torch.nonzero(out.view(torch.int32) != want.view(torch.int32))
    if bad.numel():
        i = int(bad[0])
        raise AssertionError(f"{what}: {bad.numel()} differ, {float(a[i])!r} / {float(b[i])!r} = {float(out[i])!r}")


def _divisors():
    return (torch.arange(2**23, device="cuda", dtype=torch.int32) + 0x3F800000).view(torch.float32)  # [1, 2)


@pytest.mark.parametrize("scale", [2.0**-40, 2.0**-10, 1.0, 2.0**30])
def test_every_divisor(scale):
    print(f"[gpu case] quotients by every divisor x {scale}", flush=True)
    b = _divisors()
    g = torch.Generator("cuda").manual_seed(5)
    one = torch.ones_like(b)
    up = (b.view(torch.int32) + 1).view(torch.float32)
    down = (b.view(torch.int32) - 1).view(torch.float32)
    dividends = [one, one + 2.0**-23, one * (2 - 2.0**-23), b, up, down, 0 * b, b.flip(0)]
    dividends += [(torch.randint(0, 2**23, b.shape, device="cuda", generator=g, dtype=torch.int32) + 0x3F800000)
                  .view(torch.float32) for _ in range(56)]
    for k, a in enumerate(dividends):
        _check(a, b * scale, f"dividend {k}")


@pytest.mark.parametrize("seed", range(4))
def test_operands_of_the_samplers(seed):
    print(f"[gpu case] quotients of the samplers, seed {seed}", flush=True)
    g, n = torch.Generator("cuda").manual_seed(seed), 1 << 23
    r = lambda: torch.rand(n, device="cuda", generator=g)  # noqa: E731
    E = 2.0**-10 * (10.0 / 2.0**-10) ** r()  # 1 keV to 10 MeV
    _check(E, torch.full_like(E, MEC2), "energy in electron masses")
    alpha = E / MEC2
    onep, a2 = 1 + 2 * alpha, 2 * alpha
    _check(onep, 9 + a2, "branch threshold")
    t = torch.addcmul(torch.ones_like(a2), a2, r())
    _check(onep, t, "energy ratio")
    _check(torch.ones_like(t), t, "its inverse")
    _check(t - 1, alpha, "one less the cosine")
    _check(2.0**-23 * torch.randint(0, 64, (n,), device="cuda", generator=g), alpha, "forward scatter")
    _check(E, t, "scattered energy")
    w = 0.99999 * (2 * r() - 1)
    tmp = torch.sqrt(1 - w * w)
    c = 2 * r() - 1
    _check(torch.sqrt(1 - c * c), tmp, "rotation")
    _check(2.0 ** (-24 * r()), tmp, "rotation by small angles")
    _check(torch.zeros_like(tmp), tmp, "no rotation")
    _check(torch.ones_like(tmp), 1 + 2.0**-20 * (2 * r() - 1), "normalisation")
