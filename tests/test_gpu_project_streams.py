"""Window probabilities added to one image from several streams at once: nothing is lost, whichever
of the accumulating kernels a call takes. The sums are FP64 of the same terms in another order."""
import math

import pytest
import torch

pytestmark = pytest.mark.gpu


def _pairs(m, n_pix, seed):
    from opengate_amd.learn.arf import PairBuffer

    g = torch.Generator("cuda").manual_seed(seed)
    buf = PairBuffer(m, "cuda")
    buf.x16.zero_()
    buf.x16[:, :3] = torch.randn(m, 3, device="cuda", generator=g).to(torch.bfloat16)
    buf.pix.copy_(torch.randint(0, n_pix, (m,), device="cuda", generator=g))
    buf.wgt.copy_(0.5 + torch.rand(m, device="cuda", generator=g))
    return buf


# pairs of a call: few (direct kernel), many (binned)
@pytest.mark.parametrize("m", [3000, 1000000])
@pytest.mark.parametrize("squared", [True, False])
def test_one_image_from_several_streams(m, squared):
    from opengate_amd.learn.arf import ArfModel

    print(f"[gpu case] one image from 3 streams, {m} pairs a call, squared={squared}", flush=True)
    heads, ny, nx, calls = 16, 64, 64, 4
    arf = ArfModel(theta_max=math.radians(10.0), seed=4)
    bufs = [_pairs(m, heads * ny * nx, k) for k in range(3)]

    def images():
        return [torch.zeros(heads * arf.n_win, ny, nx, device="cuda", dtype=torch.float64) for _ in range(2)]

    want = images()
    for buf in bufs:
        for _ in range(calls):
            arf.project(buf, m, want[0], want[1] if squared else None)
    got = images()
    streams = [torch.cuda.Stream() for _ in bufs]
    torch.cuda.synchronize()
    for _ in range(calls):
        for st, buf in zip(streams, bufs):
            with torch.cuda.stream(st):
                arf.project(buf, m, got[0], got[1] if squared else None)
    torch.cuda.synchronize()
    for a, b in zip(got, want):
        torch.testing.assert_close(a, b, rtol=1e-11, atol=0)


@pytest.mark.parametrize("squared", [True, False])
def test_own_images(squared):
    from opengate_amd.learn.arf import ArfModel

    print(f"[gpu case] own image, squared={squared}", flush=True)
    m, heads, ny, nx = 1200003, 7, 60, 70
    arf = ArfModel(theta_max=math.radians(10.0), seed=4)
    buf = _pairs(m, heads * ny * nx, 9)
    out = []
    for own in (True, False):
        img = [torch.full((heads * arf.n_win, ny, nx), 0.25, device="cuda", dtype=torch.float64) for _ in range(2)]
        arf.project(buf, m, img[0], img[1] if squared else None, own=own)
        out.append(img)
    for a, b in zip(*out):
        torch.testing.assert_close(a, b, rtol=1e-11, atol=0)
