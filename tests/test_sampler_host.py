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


@pytest.mark.parametrize("params", [
    [SamplingParams(0.8, 50, 0.9)],
    [SamplingParams(0.0), SamplingParams(0.7, 200, 0.5, max_tokens=0), SamplingParams(1, 130, 1)],
    [SamplingParams(0.5, -1, 0.9), SamplingParams(0.5, 0, 1.0)],
    [SamplingParams(0.5, 129, float("nan")), SamplingParams(-1.0, 500, 0.3)],
    [SamplingParams(0.5, 128, 1.5), SamplingParams(0.5, 50, float("inf"))],
    [SamplingParams(0.9, 300, 0.0), SamplingParams(0.9, 20, -0.5)],
    [SamplingParams(0.1 + r / 256, r, r / 200) for r in range(256)]])
def test_batch_words_without_copies_of_the_parameters(pageable, monkeypatch, params):
    """The arrays and what is told from them are those of the normalized parameters, without a
    normalized copy of each row."""
    normal = [p.normalized() for p in params]
    drawn = [p for p in normal if p.temperature > 0 and p.top_p > 0]

    def copied(self):
        raise AssertionError("a copy of the parameters")

    monkeypatch.setattr(SamplingParams, "normalized", copied)
    s = Sampler()
    temperature, top_k, top_p = s._device_params(params, CPU)
    assert torch.equal(temperature, torch.tensor([float(p.temperature) for p in normal]))
    assert torch.equal(top_k, torch.tensor([p.top_k for p in normal], dtype=torch.int32))
    assert torch.equal(top_p, torch.tensor([float(p.top_p) for p in normal]))
    listed = sampling.LISTED_TOP_K
    assert s._top_p_rows == any(p.top_p < 1 and not 0 < p.top_k <= listed for p in drawn)
    assert s._all_greedy == (not drawn)
    assert s._large_k == min((p.top_k for p in drawn if p.top_k > listed), default=None)
