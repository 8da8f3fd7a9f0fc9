"""The sampler's one call on the GPU: rows' options through pinned memory, kernels, tokens back."""
import random

import numpy as np
import pytest
import torch

from ninfer_amd.sampling import SampleRow, SamplingParams
from ninfer_amd.sampling.sampler import History, Sampler, uniform

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ops():
    from ninfer_amd.kernels import load_ops
    return load_ops()


# (rows whose numbers are no multiple of four; top_k 300: by a block a row, 40: by the whole GPU, 0: cut by top-p alone)
@pytest.mark.parametrize("rows", [1, 2, 3, 65])
@pytest.mark.parametrize("penalty", [1.0, 1.2])
@pytest.mark.parametrize("top_k,temperature", [(40, 0.8), (300, 0.8), (0, 0.8), (40, 0.0)])
def test_tokens_are_those_of_the_kernels(ops, rows, penalty, top_k, temperature):
    rng, vocab = random.Random(rows), 13001
    gen = torch.Generator("cuda").manual_seed(rows)
    sampler = Sampler(ops, torch.device("cuda:0"))
    for turn in range(3):   # (buffers are used again, for rows that need more)
        logits = 3 * torch.randn(rows, vocab, generator=gen, device="cuda")
        made = [SampleRow(SamplingParams(temperature=temperature, top_k=top_k, top_p=0.9, repetition_penalty=penalty),
                          History(rng.choices(range(vocab), k=(turn + 1) * rng.randint(1, 700))), key=i, draw=turn, seed=7)
                for i in range(rows)]
        got = sampler.sample(logits, made)
        f32 = lambda v: torch.tensor(v, dtype=torch.float32, device="cuda")
        i32 = lambda v: torch.tensor(np.asarray(v, np.int32), device="cuda")
        both = [r.history.arrays() for r in made]
        out = torch.empty(rows, dtype=torch.int32, device="cuda")
        pen = dict(pen_offsets=i32(np.cumsum([0] + [len(t) for t, _ in both])), pen_tokens=i32(np.concatenate([t for t, _ in both])),
                   pen_counts=i32(np.concatenate([c for _, c in both]))) if penalty != 1.0 else {}
        ops.sample(logits, f32([temperature] * rows), f32([uniform(r.seed, r.key, r.draw) for r in made]), out,
                   top_k=i32([top_k] * rows), top_p=f32([0.9] * rows), rep_penalty=f32([penalty] * rows), **pen)
        assert got == out.tolist()
        assert len(sampler._free) == 1


def test_more_rows_than_a_grid_is_high(ops):
    rows, vocab = 65537, 12800
    logits = torch.randn(rows, vocab, device="cuda")
    params, nothing = SamplingParams(temperature=0.8, top_k=0, top_p=0.9, repetition_penalty=1.0), History([])
    got = Sampler(ops, torch.device("cuda:0")).sample(logits, [SampleRow(params, nothing, key=i, draw=0, seed=7) for i in range(rows)])
    every = list(range(0, rows, 997)) + [rows - 1]
    f32 = lambda v: torch.tensor(v, dtype=torch.float32, device="cuda")
    out = torch.empty(len(every), dtype=torch.int32, device="cuda")
    ops.sample(logits[every].contiguous(), f32([0.8] * len(every)), f32([uniform(7, i, 0) for i in every]), out, top_p=f32([0.9] * len(every)))
    assert [got[i] for i in every] == out.tolist()


def test_what_it_refuses(ops):
    from ninfer_amd.kernels.ops import KernelError
    logits, numbers = torch.zeros(2, 50, device="cuda"), torch.zeros(64, dtype=torch.int32)
    for buffer, rows, ints, n_pen in ((numbers, 2, 10, 0), (numbers.pin_memory(), 3, 15, 0), (numbers.pin_memory(), 2, 11, 0),
                                      (numbers.pin_memory(), 2, 63, 25), (torch.zeros(12, dtype=torch.int32).pin_memory(), 2, 10, 0)):
        with pytest.raises(KernelError):
            ops.sample_rows(logits, rows, buffer, ints, n_pen)
    with pytest.raises(KernelError):
        Sampler(ops, torch.device("cuda:0")).sample(logits[:0], [])


def test_rows_that_keep_few_tokens_say_how_many(ops):
    from ninfer_amd.kernels.ops import KernelError
    logits, f32 = torch.zeros(2, 50, device="cuda"), torch.ones(2, device="cuda")
    out = torch.full((2,), -7, dtype=torch.int32, device="cuda")
    with pytest.raises(KernelError, match="top_k"):
        ops.sample(logits, f32, f32 * 0.5, out, few=True)
    assert out.tolist() == [-7, -7]
