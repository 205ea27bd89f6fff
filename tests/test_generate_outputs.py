"""ExitPlaneGenerator.generate with outputs or a chunk that it cannot use: refused on the host, by
the path that checks them (the one-call path takes 8 arrays by address)."""
import pytest
import torch


def _generator(device):
    from opengate_amd.learn.exitplane import ExitPlaneGenerator, QuantileMap

    gen = ExitPlaneGenerator((32.0, 32.0, 142.5), 0.0, device=device, seed=2)
    gen.qmap = QuantileMap(torch.linspace(-1, 1, 64, device=device).expand(6, 64).contiguous(), 4.0)
    return gen


@pytest.mark.parametrize("n_out,chunk", [(7, 4096), (9, 4096), (0, 4096), (8, 0), (8, -5)])
def test_the_one_call_path_is_not_taken(n_out, chunk, monkeypatch):
    gen = _generator("cpu")
    assert gen._one_call()

    def one_call(*a):
        raise AssertionError("taken")

    def checked(*a, **k):
        raise KeyError("the checked path")

    monkeypatch.setattr(gen, "_generate", one_call)
    monkeypatch.setattr(gen, "noise", checked)
    with pytest.raises((KeyError, ValueError, RuntimeError)):
        gen.generate(100, 1, out=[torch.empty(100) for _ in range(n_out)], chunk=chunk)


@pytest.mark.gpu
@pytest.mark.parametrize("n_out,chunk", [(7, 4096), (9, 4096), (8, 0), (8, -5)])
def test_refused(n_out, chunk):
    print(f"[gpu case] generate into {n_out} arrays, chunk {chunk}", flush=True)
    gen = _generator("cuda")
    with pytest.raises((RuntimeError, ValueError, IndexError, TypeError)):
        gen.generate(100, 1, out=[torch.empty(100, device="cuda") for _ in range(n_out)], chunk=chunk)
