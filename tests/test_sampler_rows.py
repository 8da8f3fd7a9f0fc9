"""What the sampler hands to the kernel: the random numbers of many rows at once are those of the
rows one by one."""
import ctypes
import random

import numpy as np
import pytest
import torch

from ninfer_amd.sampling import SampleRow, SamplingParams
from ninfer_amd.sampling.sampler import History, Sampler, _streams, uniform, uniforms


@pytest.mark.parametrize("rows", [1, 8, 9, 300])
def test_uniforms_are_the_rows_own(rows):
    rng = random.Random(rows)
    made = [SampleRow(SamplingParams(), History([1]), rng.choice([0, -3, rng.getrandbits(64), rng.getrandbits(70)]),
                      rng.randrange(10 ** 6), rng.getrandbits(64)) for _ in range(rows)]
    assert uniforms(made).tolist() == [uniform(r.seed, r.key, r.draw) for r in made]


@pytest.mark.parametrize("rows", [1, 3, 70])
def test_the_librarys_uniforms_are_the_same(rows):
    from ninfer_amd.kernels.build import ensure_built
    rng = random.Random(rows)
    made = [SampleRow(SamplingParams(), History([1]), rng.choice([-1, rng.getrandbits(64), 2 ** 64]),
                      rng.getrandbits(20), rng.getrandbits(66)) for _ in range(rows)]
    streams = _streams(made)
    at = [v.buffer_info()[0] for v in streams]
    out = np.full(rows + 1, 7, np.float32)
    ctypes.CDLL(ensure_built()).ninfer_uniforms(*map(ctypes.c_void_p, at), rows, ctypes.c_void_p(out.ctypes.data))
    assert out[:rows].tolist() == [uniform(r.seed, r.key, r.draw) for r in made] and out[rows] == 7


@pytest.mark.parametrize("rows", [1, 2, 30])
@pytest.mark.parametrize("temperatures", [(0.0,), (0.7,), (0.7, 0.0, -1.0)])
@pytest.mark.parametrize("penalties", [(1.0,), (1.1,), (1.0, 1.1, 0.9)])
def test_what_the_kernel_is_given(rows, temperatures, penalties):
    class Asked:
        FEW_TOKENS = 64

        def sample(self, logits, temperature, uniform, out, **rest):
            self.got = dict(temperature=temperature, uniform=uniform, **rest)
            out.zero_()

    rng = random.Random(rows)
    made = []
    for i in range(rows):
        history = History(rng.choices(range(50), k=rng.randint(0, 90)))
        for t in rng.choices(range(100), k=80):
            history.add(t)
        made.append(SampleRow(SamplingParams(temperature=temperatures[i % len(temperatures)], top_k=i % 60 + 1,
                                             top_p=0.5 + i / 100, repetition_penalty=penalties[i % len(penalties)]),
                              history, key=i, draw=3, seed=5 - i))
    asked = Asked()
    assert Sampler(asked, torch.device("cpu")).sample(torch.zeros(rows, 100), made) == [0] * rows
    got = asked.got
    for name, key in (("temperature", "temperature"), ("top_p", "top_p"), ("repetition_penalty", "rep_penalty"),
                      ("top_k", "top_k")):
        assert got[key].tolist() == [np.float32(getattr(r.params, name)) for r in made]
    assert got["uniform"].tolist() == [uniform(r.seed, r.key, r.draw) if r.params.temperature > 0 else 0 for r in made]
    assert got.get("few", False) == any(r.params.temperature > 0 for r in made)
    at = 0
    for i, r in enumerate(made):
        toks, counts = (a.tolist() for a in r.history.arrays())
        if r.params.repetition_penalty == 1.0:
            toks, counts = [], []
        if "pen_offsets" not in got:
            assert not toks
            continue
        assert got["pen_offsets"][i:i + 2].tolist() == [at, at + len(toks)]
        assert got["pen_tokens"][at:at + len(toks)].tolist() == toks
        assert got["pen_counts"][at:at + len(toks)].tolist() == counts
        at += len(toks)


@pytest.mark.parametrize("rows,arrays", [(1, False), (20, False), (21, True)])
def test_few_rows_draw_one_by_one(monkeypatch, rows, arrays):
    """The numbers of few rows do not pay for the arrays that those of many are laid out in."""
    import ninfer_amd.sampling.sampler as sampler
    asked = []
    monkeypatch.setattr(sampler, "uniforms", lambda drawn: (asked.append(len(drawn)), uniforms(drawn))[1])

    class Asked:
        def sample(self, logits, temperature, uniform, out, **rest):
            self.got = uniform.tolist()
            out.zero_()

    made = [SampleRow(SamplingParams(temperature=0.7 if i != 3 else 0.0), History([1]), key=i, draw=2, seed=9) for i in range(rows + (rows > 3))]
    ops = Asked()
    Sampler(ops, torch.device("cpu")).sample(torch.zeros(len(made), 10), made)
    assert asked == [rows] * arrays
    assert ops.got == [uniform(r.seed, r.key, r.draw) if r.params.temperature > 0 else 0 for r in made]
