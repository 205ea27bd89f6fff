"""Projection kernels at the edges of their workgroups: the set of (photon, head) pairs equals
the oracle's, bit for bit but for the angles."""
import math

import numpy as np
import pytest

from oracle import arf_ref as R
from oracle import mlp_ref as MR

pytestmark = pytest.mark.gpu


def _heads(n_proj, theta_deg):
    from opengate_amd.learn.arf import Heads

    return Heads(center=(100.0, 100.0, 80.0), radius=200.0, n_proj=n_proj, nx=32, ny=24, spacing=(6.0, 5.0),
                 angle0=-7.3, theta_max=math.radians(theta_deg))


def _photons(n, seed):
    g = np.random.default_rng(seed)
    p = g.uniform(60, 140, size=(n, 3))
    d = g.normal(size=(n, 3))
    d[:, 2] *= 0.1
    d /= np.linalg.norm(d, axis=1)[:, None]
    return [a.astype(np.float32) for a in (p[:, 0], p[:, 1], p[:, 2], d[:, 0], d[:, 1], d[:, 2],
                                           g.uniform(0.02, 0.15, n), g.uniform(0.5, 1.5, n))]


# one photon; a workgroup's 256 and one more; every head tested (wide acceptance, few heads) so that
# the waiting pairs overflow many times; several photons per thread
@pytest.mark.parametrize("n,n_proj,theta,det", [(1, 16, 12.0, False), (256, 16, 12.0, True), (257, 60, 10.0, False),
                                                (5000, 128, 60.0, False), (5000, 3, 80.0, True),
                                                (40000, 128, 10.0, True), (1000003, 16, 1.0, False)])
def test_pairs(n, n_proj, theta, det):
    import torch

    from opengate_amd import _abi as A
    from opengate_amd.learn.arf import PairBuffer, spect_pairs

    print(f"[gpu case] pairs n={n} heads={n_proj} theta={theta} det={det}", flush=True)
    h, rec = _heads(n_proj, theta), _photons(n, n_proj)
    ref, cnt = R.spect_pairs(rec, h.desc(), h.angle_table(), 1 << 20)
    assert cnt < 1 << 20
    buf = PairBuffer(1 << 20, "cuda", det=det)
    cs = torch.from_numpy(h.angle_table()).cuda()
    m = spect_pairs(A.load_library(), [torch.from_numpy(a).cuda() for a in rec], n, h, cs, buf)
    assert m == cnt
    pix, wgt = buf.pix[:m].cpu().numpy(), buf.wgt[:m].cpu().numpy()
    x = buf.x16[:m].float().cpu().numpy()
    xr = MR.to_bf16(ref["x3"])
    o, r = np.lexsort((wgt, x[:, 0], pix)), np.lexsort((ref["wgt"], xr[:, 0], ref["pix"]))
    np.testing.assert_array_equal(pix[o], ref["pix"][r])
    np.testing.assert_array_equal(wgt[o], ref["wgt"][r])
    np.testing.assert_array_equal(x[o][:, 0], xr[r][:, 0])
    np.testing.assert_allclose(x[o][:, 1:3], xr[r][:, 1:3], rtol=2.0**-7, atol=1e-3)
    assert np.all(x[:, 3:] == 0)
    if det:
        for k in range(8):
            np.testing.assert_array_equal(buf.det[k][:m].cpu().numpy()[o], ref["det"][k][r])


def test_pairs_beyond_capacity_are_counted():
    import ctypes as C

    import torch

    from opengate_amd import _abi as A
    from opengate_amd.learn.arf import PairBuffer

    print("[gpu case] pairs beyond the buffer", flush=True)
    h, rec = _heads(64, 20.0), _photons(20000, 4)
    ref, cnt = R.spect_pairs(rec, h.desc(), h.angle_table(), 1 << 20)
    cap = cnt // 3
    buf = PairBuffer(cnt, "cuda")
    buf.pix.fill_(-1)
    cs = torch.from_numpy(h.angle_table()).cuda()
    p = lambda t: C.c_void_p(t.data_ptr())  # noqa: E731
    dev = [torch.from_numpy(a).cuda() for a in rec]
    photons = (A.FP * 8)(*[C.cast(p(a), A.FP) for a in dev])
    rc = A.load_library().gh_spect_pairs(photons, 20000, C.byref(h.desc()), p(cs), cap, p(buf.x16), p(buf.pix),
                                         p(buf.wgt), None, C.c_void_p(), p(buf.count), None)
    assert rc == 0
    torch.cuda.synchronize()
    assert int(buf.count) == cnt
    pix = buf.pix.cpu().numpy()
    assert np.all(pix[:cap] >= 0) and np.all(pix[cap:] == -1)


# one pair; sorting workgroups of 4096 pairs; bins of 4096 pixels; every record size; one hot pixel
@pytest.mark.parametrize("m,heads,plane,n_win,squared,hot", [(1, 1, 1, 1, True, False), (4096, 1, 4096, 3, True, False),
                                                             (4097, 3, 4097, 4, False, False),
                                                             (70001, 16, 768, 3, True, True),
                                                             (100003, 128, 16384, 3, True, False),
                                                             (100000, 7, 65536, 8, True, False),
                                                             (90000, 5, 999, 7, False, True)])
def test_binned_accumulation(m, heads, plane, n_win, squared, hot):
    import ctypes as C

    import torch

    from opengate_amd import _abi as A

    print(f"[gpu case] binned accumulation m={m} heads={heads} plane={plane} windows={n_win}", flush=True)
    lib, g = A.load_library(), np.random.default_rng(m)
    n_pix = heads * plane
    logits = g.normal(size=(m, n_win + 2)).astype(np.float32)
    pix = g.integers(0, n_pix, m).astype(np.int32)
    if hot:
        pix[: m // 2] = n_pix - 1
    wgt = g.uniform(0.5, 1.5, m).astype(np.float32)
    L, P, W = (torch.from_numpy(a).cuda() for a in (logits, pix, wgt))
    p = lambda t: C.c_void_p(t.data_ptr()) if t is not None else C.c_void_p()  # noqa: E731
    bins = (n_pix + 4095) // 4096
    work = torch.full((4 * ((3 * bins + 4) // 4 * 4) + 16 * ((n_win + 4) // 4) * m,), 255, dtype=torch.uint8,
                      device="cuda")
    need = C.c_int64(-1)
    assert lib.gh_arf_accumulate_workspace(m, n_win, n_pix, int(squared), C.byref(need)) == 0
    assert need.value in (0, work.numel())
    got, want = [], []
    for out in (got, want):
        out += [torch.full((heads * n_win * plane,), 0.25, dtype=torch.float64, device="cuda") for _ in range(2)]
    i2 = lambda out: out[1] if squared else None  # noqa: E731
    args = (p(L), n_win + 2, m, p(P), p(W), n_win, plane)
    assert lib.gh_arf_accumulate_binned(*args, n_pix, p(got[0]), p(i2(got)), p(work), work.numel() - 1, None) != 0
    for _ in range(2):  # the workspace needs no clearing
        assert lib.gh_arf_accumulate_binned(*args, n_pix, p(got[0]), p(i2(got)), p(work), work.numel(), None) == 0
        assert lib.gh_arf_accumulate(*args, p(want[0]), p(i2(want)), None) == 0
    for a, b in zip(got, want):  # the same terms, FP64 sums in another order
        np.testing.assert_allclose(a.cpu().numpy(), b.cpu().numpy(), rtol=1e-11, atol=0)
    ref = 0.25 + 2 * R.accumulate_arf(logits, pix, wgt, n_win, plane, heads)
    np.testing.assert_allclose(got[0].cpu().numpy(), ref.reshape(-1), rtol=1e-5)
