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
    greedy, race, few, widest, top_p_rows = s._kinds
    assert greedy == len(normal) - len(drawn) and greedy + race + few + top_p_rows == len(normal)
    assert few == sum(0 < p.top_k <= listed for p in drawn)
    assert widest == max((p.top_k for p in drawn if 0 < p.top_k <= listed), default=0)
    assert top_p_rows == sum(p.top_p < 1 and not 0 < p.top_k <= listed for p in drawn)
    assert s._large_k == min((p.top_k for p in drawn if p.top_k > listed), default=None)


GREEDY, RACE, TOP_K, TOP_P = (1, 0, 0, 0, 0), (0, 1, 0, 0, 0), (0, 0, 1, 50, 0), (0, 0, 0, 0, 1)


@pytest.mark.parametrize("kind,rows,vocab,splits", [
    (GREEDY, 1, 32000, False), (GREEDY, 1, 151936, True), (GREEDY, 64, 50257, False),
    (GREEDY, 1, 50257, True), (GREEDY, 64, 151936, True), (GREEDY, 128, 151936, False), (RACE, 5, 32000, True),
    (RACE, 256, 32000, False), (RACE, 256, 151936, True), (RACE, 320, 32000, True), (RACE, 256, 50257, True),
    (TOP_K, 5, 16385, True), (TOP_K, 256, 20000, True), (TOP_K, 256, 50257, True),
    (TOP_K, 1024, 151936, True), (TOP_P, 64, 20000, True), (TOP_P, 256, 32000, False),
    (TOP_P, 256, 151936, True)])
def test_batches_are_split_where_it_was_measured_quicker(kind, rows, vocab, splits):
    greedy, race, listed, widest, top_p = kind
    assert sampling._split_pays(rows, vocab, greedy * rows, race * rows, listed * rows, widest,
                                top_p * rows, False, vocab % 8 == 0) == splits


def test_a_large_listed_k_needs_many_segments():
    assert not sampling._split_pays(5, 16385, 0, 0, 5, 128, 0, False, True)
    assert sampling._split_pays(5, 16385, 0, 0, 5, 96, 0, False, True)
    assert sampling._split_pays(5, 151936, 0, 0, 5, 128, 0, False, True)
