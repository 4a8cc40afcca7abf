"""The sampler's host side: the parameter arrays and what it keeps of them (CPU only)."""
import pytest
import torch

from llm_infer_rust_amd import sampling
from llm_infer_rust_amd.sampling import Sampler, SamplingParams

CPU = torch.device("cpu")


@pytest.fixture
def pageable(monkeypatch):
    """torch.empty without the pinning, which needs a GPU."""
    real = torch.empty

    def empty(*args, pin_memory=False, **kw):
        return real(*args, **kw)

    monkeypatch.setattr(sampling.torch, "empty", empty)


def test_failed_build_is_not_kept(pageable, monkeypatch):
    """A list whose arrays could not be built raises again; it does not get the last one's."""
    s = Sampler()
    s._device_params([SamplingParams(0.5)], CPU)
    longer = [SamplingParams(0.7), SamplingParams(0.9)]
    with monkeypatch.context() as m:
        def fail(*args, **kw):
            raise MemoryError
        m.setattr(sampling.torch, "empty", fail)
        for _ in range(2):
            with pytest.raises(MemoryError):
                s._device_params(longer, CPU)
    temperature, _, _ = s._device_params(longer, CPU)
    assert temperature.tolist() == pytest.approx([0.7, 0.9])
