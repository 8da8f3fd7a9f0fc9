"""What the sampler hands to the kernel: the random numbers of many rows at once are those of the
rows one by one."""
import random

import numpy as np
import pytest

from ninfer_amd.sampling import SampleRow, SamplingParams
from ninfer_amd.sampling.sampler import History, uniform, uniforms


@pytest.mark.parametrize("rows", [1, 8, 9, 300])
def test_uniforms_are_the_rows_own(rows):
    rng = random.Random(rows)
    made = [SampleRow(SamplingParams(), History([1]), rng.choice([0, -3, rng.getrandbits(64), rng.getrandbits(70)]),
                      rng.randrange(10 ** 6), rng.getrandbits(64)) for _ in range(rows)]
    assert uniforms(made).tolist() == [uniform(r.seed, r.key, r.draw) for r in made]
