"""Generation parameters: the reference's defaults, checks and choice of sampling mode."""
import pytest

from atoma_infer_amd.sampling import DEFAULT_RANDOM_SEED, GenerateParameters, ValidationError, uniform, validate


def plan(**kw):
    return validate(GenerateParameters(**kw), 10, 4096, 8192)


def test_defaults_follow_the_reference():
    """backends/vllm/src/validation.rs:226-315, types.rs:84-85."""
    p = plan()
    assert p.temperature == 1.0 and p.top_k == 0 and p.top_p == 1.0 and p.repetition_penalty == 1.0
    assert p.random_seed == DEFAULT_RANDOM_SEED == 1_283_768_955 and p.max_new_tokens == 100
    assert p.greedy and p.mode == "ArgMax"          # temperature 1.0 means argmax (llm_service.rs:346-348)
    assert plan(max_new_tokens=None).max_new_tokens == 8192 - 10   # validation.rs:133-137


def test_mode_selection():
    """backends/vllm/src/llm_service.rs:346-372."""
    assert plan(temperature=0.7).mode == "All"
    assert plan(temperature=0.7, do_sample=False).mode == "ArgMax"
    assert plan(temperature=0.7, top_p=0.9).mode == "TopP"
    assert plan(temperature=0.7, top_k=5).mode == "TopK"
    assert plan(temperature=0.7, top_k=5, top_p=0.9).mode == "TopKThenTopP"
    assert plan(temperature=1.0, top_k=5).mode == "ArgMax"


@pytest.mark.parametrize("kw", [
    {"temperature": 0.0}, {"temperature": -1.0}, {"repetition_penalty": 0.0}, {"frequency_penalty": 2.5},
    {"top_p": 1.0}, {"top_p": 0.0}, {"typical_p": 1.5}, {"top_k": 0}, {"max_new_tokens": 0},
    {"stop": ["a", "b"]}, {"top_n_tokens": 5}, {"truncate": 0}, {"truncate": 5000}, {"best_of": 2},
    {"max_new_tokens": 9000}, {"repetition_penalty": 1.2},
])
def test_invalid_parameters_are_refused(kw):
    with pytest.raises(ValidationError):
        plan(**kw)


def test_input_length_checks():
    with pytest.raises(ValidationError):
        validate(GenerateParameters(), 0, 4096, 8192)
    with pytest.raises(ValidationError):
        validate(GenerateParameters(), 5000, 4096, 8192)
    assert plan(repetition_penalty=1.2, repeat_last_n=16).repeat_last_n == 16


def test_uniform_is_a_pure_function_in_the_unit_interval():
    xs = [uniform(42, i) for i in range(2000)]
    assert all(0.0 <= x < 1.0 for x in xs)
    assert xs == [uniform(42, i) for i in range(2000)]
    assert abs(sum(xs) / len(xs) - 0.5) < 0.03 and len(set(xs)) > 1990
    assert uniform(42, 0) != uniform(43, 0)


def test_a_steps_uniform_numbers_written_natively_are_the_functions():
    import ctypes

    from atoma_infer_amd.sampling import sampler
    seeds = [0, 1, 42, -1, 2 ** 63, 2 ** 64 - 1, 2 ** 64 + 5] * 40
    steps = [i * i for i in range(len(seeds))]
    rows = len(seeds)
    for counters in (steps, [s + 2 ** 63 for s in steps]):
        got, c = (ctypes.c_float * (5 * rows))(), sampler._counters(counters)
        sampler._native().sampling_pack(b"".join([plan(do_sample=True, temperature=0.7, random_seed=s).packed for s in seeds]), c.buffer_info()[0],
                                        rows, 128, ctypes.addressof(got))
        assert list(got)[2 * rows: 3 * rows] == [uniform(s, n) for s, n in zip(seeds, counters)]


def test_a_steps_parameters_packed_natively_are_the_plans():
    """What the native packing writes and finds against the plans' own attributes, over greedy rows, cuts on both sides of the lists'
    largest, penalties and seeds beyond 64 bits."""
    import random

    import numpy as np
    import torch

    from atoma_infer_amd.kernels import ops
    from atoma_infer_amd.sampling import sampler
    pick = random.Random(5)
    for rows in (1, 5, 64, 65):
        for _ in range(40):
            plans = [validate(GenerateParameters(do_sample=pick.random() < 0.7, temperature=pick.choice([None, 0.7, 1.0, 2.0]),
                                                 top_k=pick.choice([None, 1, 128, 129]), top_p=pick.choice([None, 0.3]),
                                                 random_seed=pick.choice([None, -5, 2 ** 64 + 7, pick.randrange(2 ** 64)]),
                                                 repetition_penalty=pick.choice([None, None, 1.3]), repeat_last_n=4,
                                                 max_new_tokens=4), 3, 100, 200) for _ in range(rows)]
            steps = [pick.randrange(1000) for _ in plans]
            meta, counters = torch.zeros(5, rows), sampler._counters(steps)
            found = sampler._native().sampling_pack(b"".join([p.packed for p in plans]), counters.buffer_info()[0], rows,
                                                    ops.FEW_MAX_K, meta.data_ptr())
            assert found == sampler._found(plans)
            want = np.array([[0.0 if p.greedy else p.temperature for p in plans], [p.top_p for p in plans],
                             [uniform(p.random_seed, c) for p, c in zip(plans, steps)],
                             [p.repetition_penalty for p in plans]], np.float32)
            assert (meta.numpy()[:4] == want).all() and meta.numpy()[4].view(np.int32).tolist() == [p.top_k for p in plans]


@pytest.mark.parametrize("rows", [1, 4, 5, 64])
@pytest.mark.parametrize("top_k", [2 ** 31 - 1, 2 ** 31, 2 ** 32 + 1, 2 ** 32 + 40, 2 ** 64])
def test_a_top_k_beyond_32_bits_is_no_cut_beside_any_number_of_rows(monkeypatch, rows, top_k):
    """No vocabulary is as large as the largest number that a step's parameters hold, so that is what such a cut becomes: in the rows that
    are written one by one and in those that are packed natively, which also count it as a cut beyond the lists."""
    import torch

    from atoma_infer_amd.kernels import ops
    from atoma_infer_amd.sampling import Sampler, sampler
    empty, seen = torch.empty, {}
    monkeypatch.setattr(torch, "empty", lambda *a, pin_memory=False, **kw: empty(*a, **kw))
    monkeypatch.setattr(torch.cuda, "Event", lambda: type("E", (), {"record": lambda self: None, "synchronize": lambda self: None})())

    def draw(logits, temperature, top_k, top_p, uniform, **how):
        seen.update(top_k=top_k.tolist(), how=how)
        return torch.zeros(2, logits.shape[0])
    monkeypatch.setattr(ops, "sample_packed", draw)
    plans = [plan(do_sample=True, temperature=0.7, top_k=40) for _ in range(rows - 1)] + [plan(do_sample=True, temperature=0.7, top_k=top_k)]
    Sampler(torch.device("cpu")).launch(torch.zeros(rows, sampler.SPLIT_MIN_VOCAB), plans, [0] * rows, [()] * rows)
    assert seen["top_k"] == [40] * (rows - 1) + [2 ** 31 - 1]
    assert seen["how"] == dict(split=True, cuts=True, few=False, top_p_cuts=False)
