"""ArfModel.fit hands the classes to a kernel by address: classes that are not one per row on the
rows' device are refused before anything is launched."""
import pytest
import torch


def _fit(X, cls, device):
    from opengate_amd.learn.arf import ArfModel

    return ArfModel(device=device, sizes=[3, 128, 128, 128, 4]).fit(X, cls, steps=1, batch=64)


def _rows(device):
    X = torch.zeros(500, 8, device=device, dtype=torch.bfloat16)
    X[:, :3] = torch.rand(500, 3, device=device).to(torch.bfloat16)
    return X


@pytest.mark.parametrize("cls", [torch.zeros(499, dtype=torch.long), torch.zeros(500, 1, dtype=torch.long),
                                 torch.zeros(0, dtype=torch.long), torch.zeros(500, dtype=torch.long, device="meta")])
def test_refused(cls):
    with pytest.raises(ValueError, match="one per row"):
        _fit(_rows("cpu"), cls, "cpu")


@pytest.mark.gpu
def test_classes_on_the_host_are_refused():
    print("[gpu case] classes on the host", flush=True)
    with pytest.raises(ValueError, match="one per row"):
        _fit(_rows("cuda"), torch.zeros(500, dtype=torch.long), "cuda")


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.uint8])
def test_more_classes_than_rows_and_other_integers(dtype):
    print(f"[gpu case] classes of {dtype}", flush=True)
    X, cls = _rows("cuda"), (torch.arange(600, device="cuda") % 4)
    assert _fit(X, cls.to(dtype), "cuda") == _fit(X, cls[:500], "cuda")
