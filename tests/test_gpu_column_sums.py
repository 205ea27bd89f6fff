"""Column sums of several matrices in two launches: the bits of PyTorch's sum over the rows (the
order that fits' first steps depend on), at the edges of its splits."""
import ctypes as C
import random
import struct

import pytest
import torch

pytestmark = pytest.mark.gpu


def _sums(mats, pads):
    from opengate_amd import _abi as A

    lib, M, k = A.load_library(), mats[0].shape[0], len(mats)
    out = [torch.full((p,), float("nan"), device="cuda") for p in pads]
    work = torch.empty(256 * sum(pads), device="cuda")
    q = lambda ts: struct.pack(f"={k}Q", *[t.data_ptr() for t in ts])  # noqa: E731
    rc = lib.gh_column_sums(q(mats), struct.pack(f"={k}q", *[m.stride(0) for m in mats]),
                            struct.pack(f"={k}i", *[m.shape[1] for m in mats]), struct.pack(f"={k}i", *pads), k, M, q(out),
                            C.c_void_p(work.data_ptr()), work.numel(), None)
    assert rc == 0
    torch.cuda.synchronize()
    return out


# rows: thread rows used or not (15/16 by, 256), one workgroup or several (256 rows a thread row),
# 128 or 256 workgroups, the largest; and some between
@pytest.mark.parametrize("M", [1, 31, 32, 63, 64, 127, 128, 255, 256, 257, 510, 511, 512, 1020, 1021, 2041, 4096, 4097,
                               8192, 8193, 16320, 16321, 16384, 32768, 32769, 65536,
                               *random.Random(3).sample(range(2, 65536), 24)])
def test_bits(M):
    print(f"[gpu case] column sums of {M} rows", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M)
    mats = [torch.randn(M, n, device="cuda", generator=g) for n in (256, 128, 8, 64)]
    for out, m in zip(_sums(mats, [256, 128, 8, 64]), mats):
        assert torch.equal(out, m.sum(0)), m.shape


@pytest.mark.parametrize("M,n,pad", [(300, 4, 8), (5003, 6, 8), (20000, 3, 16), (20000, 32, 32)])
def test_unpadded(M, n, pad):
    print(f"[gpu case] column sums of {M} x {n} in {pad}", flush=True)
    wide = torch.randn(M, n + 3, device="cuda")
    full = torch.zeros(M, pad, device="cuda")
    full[:, :n] = wide[:, :n]
    out = _sums([wide[:, :n]], [pad])[0]
    assert torch.equal(out, full.sum(0))
