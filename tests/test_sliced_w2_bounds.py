"""The fit's rule for its loss kernel stays within what gh_sliced_w2 accepts; everything else takes
the tensor form of the loss."""
import pytest


@pytest.mark.parametrize("batch,directions,taken", [(16384, 134, True), (16384, 2**17 - 1, True), (16384, 2**17, False),
                                                    (16385, 134, False), (0, 134, False), (2047, 2**20, True),
                                                    (2048, 2**20, False), (1, 2**20 + 1, False)])
def test_rule(batch, directions, taken):
    from opengate_amd.learn.exitplane import ExitPlaneGenerator

    assert ExitPlaneGenerator._w2_kernel(batch, directions) == taken


@pytest.mark.parametrize("M,P", [(16384, 2**17), (2048, 2**20), (16385, 134), (0, 134)])
def test_the_entry_refuses_the_rest(M, P):
    # (refused on the host: nothing is launched, no pointer is followed)
    from opengate_amd import _abi as A

    assert A.load_library().gh_sliced_w2(16, 8, 16, 8, 16, M, 6, P, 16, 16, 16, None) == 1


@pytest.mark.gpu
def test_a_fit_on_more_directions_than_the_kernel_takes():
    import numpy as np
    import torch

    from opengate_amd.learn.exitplane import ExitPlaneGenerator

    print("[gpu case] fit on 2^20 + 6 directions", flush=True)
    g = torch.Generator("cuda").manual_seed(3)
    u = torch.rand(4, 500, device="cuda", generator=g)
    d = torch.nn.functional.normalize(torch.stack([u[0] - 0.5, u[1] - 0.5, -4 - u[2]]), dim=0)
    rec = [22 + 20 * u[0], 22 + 20 * u[1], torch.zeros(500, device="cuda"), *d, 0.02 + 0.1 * u[3],
           torch.ones(500, device="cuda")]
    gen = ExitPlaneGenerator((32.0, 32.0, 142.5), 0.0, seed=2)
    assert not gen._w2_kernel(16, 2**20 + 6)
    loss = gen.fit(rec, steps=2, batch=16, projections=2**20)
    assert loss.shape == (2,) and np.all(np.isfinite(loss)) and np.all(loss > 0)
