"""Joint top-k/top-p sampling kernel against the reference's sampling tests and the oracle.

Follows src/engine/sampling.rs:454-546 (greedy / top-k=1 / top-p=0 fixtures), 554-659
(support, frequency within 0.02 over 20000 rows, same seed -> same ids, wide vocabulary, ties)
and 736-757 (the joint 3/7 case). Beyond those, every row of a wide random batch must equal the
oracle's draw for the same (seed, offset) exactly, unless the oracle reports a float-level near
tie for that row.
"""
import zlib

import numpy as np
import pytest
import torch

from llm_infer_rust_amd import sampling
from llm_infer_rust_amd._native import lib
from llm_infer_rust_amd.sampling import Sampler, SamplingError, SamplingParams
from oracle import bf16 as obf
from oracle import sampling as osamp

pytestmark = pytest.mark.gpu

FIVE = [4.0, 3.0, 2.0, 1.0, 0.0]


def sp(t=0.0, k=-1, p=1.0):
    return SamplingParams(temperature=t, top_k=k, top_p=p)


def test_greedy_fixtures(gpu):
    logits = torch.tensor([[0.1, 2.0, 0.2], [3.0, 1.0, 0.5]], device=gpu)
    s = Sampler(0)
    assert s.sample_batch(logits, [sp()] * 2) == [1, 0]
    assert s.sample_batch(logits, [sp(1.0, 1)] * 2) == [1, 0]
    assert s.sample_batch(logits, [sp(1.0, -1, 0.0)] * 2) == [1, 0]
    rows3 = torch.tensor([FIVE], device=gpu).repeat(3, 1)
    assert s.sample_batch(rows3, [sp(), sp(1.0, 1), sp(1.0, -1, 0.0)]) == [0, 0, 0]


@pytest.mark.parametrize("k,p", [(-1, 1.0), (-1, 0.8), (3, 0.9), (1, 1.0), (-1, 0.0)])
def test_support_frequencies_and_repeatability(gpu, k, p):
    rows = 20000
    logits = torch.tensor([FIVE], device=gpu).repeat(rows, 1)
    params = [sp(1.0, k, p)] * rows
    s = Sampler(12345)
    first = s.sample_batch(logits, params)
    s.manual_seed(12345)
    assert s.sample_batch(logits, params) == first
    if p == 0.0:
        want = np.array([1.0, 0, 0, 0, 0])
    else:
        _, kk, pp = osamp.normalized(1.0, k, p, 5)
        want = osamp.filtered_distribution(np.array(FIVE, np.float32), kk, pp)
    freq = np.bincount(first, minlength=5) / rows
    assert np.all(freq[want == 0] == 0), (freq, want)
    assert np.abs(freq - want).max() < 0.02, (freq, want)


def test_joint_uses_original_mass(gpu):
    rows = 20000
    logits = torch.log(torch.tensor([[0.4, 0.3, 0.2, 0.1]])).to(gpu).repeat(rows, 1)
    ids = Sampler(7).sample_batch(logits, [sp(1.0, 2, 0.5)] * rows)
    assert set(ids) <= {0, 1}
    assert abs(ids.count(1) / rows - 3 / 7) < 0.02


def test_ties_at_the_top_k_boundary_are_kept(gpu):
    logits = torch.tensor([[1.0, 1.0, 0.0]], device=gpu).repeat(1024, 1)
    ids = Sampler(3).sample_batch(logits, [sp(1.0, 1)] * 1024)
    assert 0 in ids and 1 in ids and 2 not in ids


def test_offset_advances_the_stream(gpu):
    logits = torch.zeros(4096, 64, device=gpu)
    s = Sampler(99)
    a = s.sample_batch(logits, [sp(1.0)] * 4096)
    b = s.sample_batch(logits, [sp(1.0)] * 4096)
    assert a != b


def test_invalid_distribution_sentinel(gpu):
    logits = torch.tensor([[0.0, float("nan"), 1.0], [float("-inf")] * 3, [0.0, 1.0, 2.0]],
                          device=gpu)
    s = Sampler(0)
    ids = s.sample_batch_device(logits, [sp(1.0, -1, 0.9), sp(1.0), sp(1.0, 2, 0.5)])
    got = ids.cpu().tolist()
    assert got[0] == -1 and got[1] == -1 and got[2] in (1, 2)
    with pytest.raises(SamplingError, match="invalid probability distribution"):
        s.sample_batch(logits, [sp(1.0)] * 3)
    pending = s.defer_batch(logits, [sp(1.0)] * 3)
    assert pending.relay().min().item() >= 0


def test_positive_infinity_makes_the_row_invalid(gpu):
    """A scaled logit of +inf makes the reference's softmax NaN throughout (sampling.rs:261):
    -1 on every filter path (unfiltered race, top-k candidate path, top-p radix path), the raw
    argmax for greedy rows; fp16 logits overflow to +inf when scaled by a small temperature."""
    row = [0.0, float("inf"), 1.0, 2.0] + [0.5] * 60
    logits = torch.tensor([row] * 4, device=gpu)
    params = [sp(1.0), sp(1.0, 2), sp(1.0, -1, 0.9), sp()]
    assert Sampler(1).sample_batch_device(logits, params).cpu().tolist() == [-1, -1, -1, 1]
    half = torch.tensor([[1.0, 30.0, 2.0] + [0.0] * 61] * 3, dtype=torch.float16, device=gpu)
    params = [sp(1e-4), sp(1e-4, 5), sp(1e-4, -1, 0.5)]
    assert Sampler(1).sample_batch_device(half, params).cpu().tolist() == [-1, -1, -1]
    assert Sampler(1).sample_batch_device(half, [sp(0.5, 5)] * 3).min().item() >= 0


def test_parameter_count_mismatch(gpu):
    with pytest.raises(SamplingError):
        Sampler(0).sample_batch(torch.zeros(2, 3, device=gpu), [sp()])
    assert Sampler(0).sample_batch(torch.zeros(0, 3, device=gpu), []) == []


@pytest.mark.parametrize("dtype,name", [(torch.bfloat16, "bf16"), (torch.float16, "f16"),
                                        (torch.float32, None)])
@pytest.mark.parametrize("k,p", [(-1, 1.0), (-1, 0.9), (50, 0.9), (50, 1.0)])
def test_wide_vocabulary_matches_oracle_draws(gpu, dtype, name, k, p):
    rows, vocab = 16, 151936
    g = torch.Generator().manual_seed(vocab + k)
    logits = (torch.randn(rows, vocab, generator=g) * 3).to(dtype)
    s = Sampler(2024)
    s.offset = 5
    t = [0.7] * rows
    ids = s.sample_batch_device(logits.to(gpu), [sp(0.7, k, p)] * rows).cpu().numpy()
    assert ((ids >= 0) & (ids < vocab)).all()
    round_to = (lambda x: obf.round_to(x, name)) if name else None
    want, margins = osamp.sample_rows(logits.float().numpy(), t, [k] * rows, [p] * rows,
                                      2024, 5, round_to)
    for r in range(rows):
        if ids[r] != want[r]:
            assert margins[r] < 1e-4, (r, ids[r], want[r], margins[r])


def test_heterogeneous_rows_one_launch(gpu):
    vocab = 1000
    g = torch.Generator().manual_seed(1)
    logits = torch.randn(6, vocab, generator=g).to(torch.bfloat16)
    params = [sp(), sp(0.7, 50, 0.9), sp(1.0, 1), sp(1.3, -1, 0.5), sp(0.5, 5), sp(0.9, -1, 2.0)]
    s = Sampler(5)
    ids = s.sample_batch(logits.to(gpu), params)
    want, margins = osamp.sample_rows(
        logits.float().numpy(), [q.temperature for q in params], [q.top_k for q in params],
        [q.top_p for q in params], 5, 0, lambda x: obf.round_to(x, "bf16"))
    for r in range(6):
        assert ids[r] == want[r] or margins[r] < 1e-4


def test_unaligned_rows_use_the_scalar_path(gpu):
    g = torch.Generator().manual_seed(9)
    base = torch.randn(8, 1003, generator=g)
    logits = base.to(gpu)[:, 1:1002]  # row stride 1003, first element misaligned
    ids = Sampler(11).sample_batch_device(logits, [sp(0.8, 20, 0.95)] * 8).cpu().numpy()
    want, margins = osamp.sample_rows(base[:, 1:1002].numpy(), [0.8] * 8, [20] * 8, [0.95] * 8,
                                      11, 0)
    for r in range(8):
        assert ids[r] == want[r] or margins[r] < 1e-4


def _edge_rows(case, vocab, g):
    """Rows that steer top-k sampling onto each branch of the candidate path and its fallbacks."""
    x = torch.randn(8, vocab, generator=g)
    if case == "ties":  # 5 distinct logits: the k-th value's bin holds thousands of tokens
        return torch.round(x).clamp(-2, 2)
    if case == "ties_fit":  # ~20 distinct logits: ties at the k-th value that still fit the list
        return torch.round(x * 2) / 2
    if case == "few_finite":  # 30 or 60 finite logits against k = 50
        keep = torch.zeros(8, vocab, dtype=torch.bool)
        for r in range(8):
            keep[r, torch.randperm(vocab, generator=g)[: 30 if r % 2 == 0 else 60]] = True
        return torch.where(keep, x, torch.full_like(x, float("-inf")))
    if case == "sharp":  # the k-th largest p underflows to zero (mass and value)
        return x * 200
    if case == "negative":
        return x - 50
    if case == "coarse":  # large offset: bf16 spacing 4-8 makes many exact ties near the top
        return x * 30 + 1000
    return x * 3


@pytest.mark.parametrize("dtype,name", [(torch.bfloat16, "bf16"), (torch.float16, "f16"),
                                        (torch.float32, None)])
@pytest.mark.parametrize("case,k,p", [
    ("ties", 50, 0.9), ("ties", 1, 1.0), ("ties_fit", 50, 0.9), ("ties_fit", 3000, 0.95),
    ("plain", 2000, 0.95), ("plain", 2048, 1.0), ("plain", 2049, 0.99), ("plain", 4000, 0.9),
    ("plain", 50, 1e-9), ("few_finite", 50, 0.9), ("few_finite", 50, 1.0),
    ("sharp", 50, 0.9), ("sharp", 50, 1.0), ("negative", 50, 0.9), ("coarse", 20, 0.8)])
def test_top_k_candidate_path_edges_match_oracle(gpu, dtype, name, case, k, p):
    """Top-k rows first try a candidate list gathered from an order-key histogram and fall back
    to the radix selection when the list overflows (heavy ties), a row has fewer than k finite
    logits or the k-th p has no fixed-point mass; every branch must give the oracle's draw."""
    vocab = 151936
    g = torch.Generator().manual_seed(zlib.crc32(f"{case}/{k}".encode()))
    logits = _edge_rows(case, vocab, g).to(dtype)
    rows = logits.shape[0]
    s = Sampler(77)
    s.offset = 3
    ids = s.sample_batch_device(logits.to(gpu), [sp(0.7, k, p)] * rows).cpu().numpy()
    round_to = (lambda v: obf.round_to(v, name)) if name else None
    want, margins = osamp.sample_rows(logits.float().numpy(), [0.7] * rows, [k] * rows,
                                      [p] * rows, 77, 3, round_to)
    for r in range(rows):
        if ids[r] != want[r]:
            assert margins[r] < 1e-4, (case, k, p, r, ids[r], want[r], margins[r])


ROW_KINDS = [sp(), sp(0.7, 50, 0.9), sp(1.0), sp(1.3, -1, 0.6), sp(0.8, 128), sp(0.5, 5, 0.3)]


@pytest.fixture
def split(monkeypatch):
    """Every batch that can be split is, also where one workgroup per row is the quicker one."""
    monkeypatch.setattr(sampling, "_split_pays", lambda *args: True)


def one_workgroup_per_row(logits, params, seed, offset):
    """mi355x_sample on the parameter arrays the sampler itself would pass."""
    s = Sampler(seed)
    t, k, p = s._device_params(params, logits.device)
    out = torch.empty(logits.size(0), dtype=torch.int64, device=logits.device)
    err = lib().mi355x_sample(logits.data_ptr(), logits.size(0), logits.size(1), logits.stride(0),
                              {torch.bfloat16: 0, torch.float16: 1, torch.float32: 2}[logits.dtype],
                              t.data_ptr(), k.data_ptr(), p.data_ptr(), seed, offset,
                              out.data_ptr(), torch.cuda.current_stream().cuda_stream)
    assert err is None
    return out


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("rows,vocab", [(6, 16384), (7, 16385), (8, 18432), (21, 30001),
                                        (40, 65539), (140, 70000), (300, 20000), (60, 151936)])
def test_split_rows_equal_one_workgroup_per_row(gpu, split, dtype, rows, vocab):
    """Nine and more segments per row, 1, 2 and 4 chunks per segment, rows that end inside a
    chunk, every kind of row in one call. Equal ids: the two differ by the fp32 rounding of the
    exponentials' sum only."""
    g = torch.Generator().manual_seed(rows + vocab)
    logits = (torch.randn(rows, vocab, generator=g) * 3).to(dtype).to(gpu)
    params = [ROW_KINDS[i % len(ROW_KINDS)] for i in range(rows)]
    s = Sampler(77)
    s.offset = 3
    got = s.sample_batch_device(logits, params)
    assert torch.equal(got, one_workgroup_per_row(logits, params, 77, 3))
    assert (lib().mi355x_sample_workspace_bytes(rows, vocab, True) == 0) == (vocab <= 16384)


def test_large_top_k_takes_one_workgroup_per_row(gpu, split):
    """A top_k past the lists: routed whole by the sampler, and correct inside a split call."""
    logits = (torch.randn(6, 30000, generator=torch.Generator().manual_seed(4)) * 3).to(gpu)
    params = [sp(0.9, 129, 0.8), sp(0.7, 50, 0.9), sp(), sp(1.0, 5000), sp(0.9, -1, 0.5), sp(1.0)]
    want = one_workgroup_per_row(logits, params, 6, 0)
    s = Sampler(6)
    assert torch.equal(s.sample_batch_device(logits, params), want)
    s.manual_seed(6)
    s._large_k = None
    assert torch.equal(s.sample_batch_device(logits, params), want)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("case", ["equal", "coarse", "few", "empty_segment", "sorted", "nan", "inf",
                                  "all_hidden"])
def test_split_rows_on_awkward_distributions(gpu, split, dtype, case):
    """Lists that overflow (ties), fewer finite logits than k, segments without a finite logit,
    every large logit in one segment, and invalid values in one segment only."""
    rows, vocab = 2 * len(ROW_KINDS), 50000
    g = torch.Generator().manual_seed(5)
    logits = torch.randn(rows, vocab, generator=g)
    if case == "equal":
        logits.zero_()
    elif case == "coarse":
        logits = logits.round()
    elif case == "few":
        logits[:, 30:].fill_(float("-inf"))
    elif case == "empty_segment":
        logits[:, 2048:12000].fill_(float("-inf"))
    elif case == "sorted":
        logits = logits.sort(1).values * 4
    elif case == "nan":
        logits[::2, 33333] = float("nan")
    elif case == "inf":
        logits[::2, 33333] = float("inf")
    else:
        logits[:] = float("-inf")
    logits = logits.to(dtype).to(gpu)
    params = [ROW_KINDS[i % len(ROW_KINDS)] for i in range(rows)]
    got = Sampler(9).sample_batch_device(logits, params)
    assert torch.equal(got, one_workgroup_per_row(logits, params, 9, 0))


def test_split_workspace_is_checked(gpu):
    logits = torch.zeros(2, 20000, device=gpu)
    need = lib().mi355x_sample_workspace_bytes(2, 20000, False)
    assert 0 < need < lib().mi355x_sample_workspace_bytes(2, 20000, True)
    t, k, p = Sampler(0)._device_params([sp(1.0)] * 2, gpu)
    out = torch.empty(2, dtype=torch.int64, device=gpu)
    ws = torch.empty(need, dtype=torch.uint8, device=gpu)
    args = (logits.data_ptr(), 2, 20000, 20000, 2, t.data_ptr(), k.data_ptr(), p.data_ptr(), 0, 0,
            out.data_ptr(), False)
    stream = torch.cuda.current_stream().cuda_stream
    assert b"workspace" in lib().mi355x_sample_split(*args, ws.data_ptr(), need - 1, stream)
    assert b"workspace" in lib().mi355x_sample_split(*args, None, need, stream)
    assert lib().mi355x_sample_split(*args, ws.data_ptr(), need, stream) is None


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("allowed", [1, 4, 30, 49, 50, 51, 127, 128, 300])
@pytest.mark.parametrize("spread", [1.0, 10.0, 40.0])
def test_split_rows_with_few_or_negligible_tokens(gpu, split, dtype, allowed, spread):
    """Fewer finite logits than k, as many and a few more, spread over the row or side by side,
    with a k-th probability that does or does not reach the fixed-point mass; masks of -inf and of
    the type's lowest value. Equal ids with one workgroup per row."""
    rows, vocab = 2 * len(ROW_KINDS), 40000
    g = torch.Generator().manual_seed(allowed + int(spread))
    values = torch.randn(rows, vocab, generator=g) * spread
    mask = torch.ones(rows, vocab, dtype=torch.bool)
    for r in range(rows):
        if r % 2:
            mask[r, 777 * r:777 * r + allowed] = False
        else:
            mask[r, torch.randperm(vocab, generator=g)[:allowed]] = False
    params = [ROW_KINDS[i % len(ROW_KINDS)] for i in range(rows)]
    for hidden in (float("-inf"), torch.finfo(dtype).min):
        logits = values.to(dtype).masked_fill(mask, hidden).to(gpu)
        got = Sampler(allowed).sample_batch_device(logits, params)
        assert torch.equal(got, one_workgroup_per_row(logits, params, allowed, 0))
    logits = values.to(dtype).to(gpu)
    got = Sampler(allowed).sample_batch_device(logits, params)
    assert torch.equal(got, one_workgroup_per_row(logits, params, allowed, 0))


def test_sampling_without_room_for_the_split_workspace(gpu, split, monkeypatch):
    """A batch that was sampled before rows were split is still sampled when there is no memory
    left for the split call's workspace."""
    g = torch.Generator().manual_seed(40)
    logits = torch.randn(len(ROW_KINDS), 40000, generator=g).to(torch.bfloat16).to(gpu)
    real = torch.empty

    def full(*args, **kw):
        if kw.get("dtype") == torch.uint8:
            raise torch.OutOfMemoryError("no room")
        return real(*args, **kw)

    s = Sampler(3)
    with monkeypatch.context() as m:
        m.setattr(torch, "empty", full)
        got = s.sample_batch_device(logits, ROW_KINDS)
    assert s.offset == 1
    assert torch.equal(got, one_workgroup_per_row(logits, ROW_KINDS, 3, 0))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("vocab", [16385, 34817, 151936, 256000])
@pytest.mark.parametrize("spread", [3.0, 40.0])
def test_split_rows_with_long_lists_and_wide_cutoffs(gpu, split, dtype, vocab, spread):
    """A k up to the lists' largest: more listed tokens in a row than are loaded before its bound is
    known (k 64 of 256,000 and 100 of 151,936 and up), 64 candidates and either side, and k-th
    probabilities without fixed-point mass. Equal ids with one workgroup per row."""
    params = [sp(0.8, k, p) for k in (40, 56, 60, 64, 65, 80, 100, 127, 128)
              for p in (1.0, 0.9, 0.3)]
    g = torch.Generator(device=gpu).manual_seed(vocab)
    logits = (torch.empty(len(params), vocab, device=gpu).normal_(generator=g) * spread).to(dtype)
    got = Sampler(7).sample_batch_device(logits, params)
    assert torch.equal(got, one_workgroup_per_row(logits, params, 7, 0))


@pytest.mark.parametrize("rows,vocab,params", [
    (16, 32000, sp()), (16, 65536, sp()), (256, 32000, sp(1.0)), (32, 32000, sp(1.0)),
    (256, 20000, sp(1.0, -1, 0.9)), (16, 20000, sp(1.0, -1, 0.9)), (5, 20000, sp(1.0, 100))])
def test_either_route_gives_the_same_ids(gpu, rows, vocab, params):
    g = torch.Generator(device=gpu).manual_seed(rows)
    logits = torch.empty(rows, vocab, device=gpu).normal_(generator=g).to(torch.bfloat16)
    got = Sampler(8).sample_batch_device(logits, [params] * rows)
    assert torch.equal(got, one_workgroup_per_row(logits, [params] * rows, 8, 0))
