"""The uniform numbers of many rows at once are the ones of each row, bit for bit."""
import random

import numpy as np
import pytest

from alice_llm_amd.sampling.sampler import uniform, uniforms


@pytest.mark.parametrize("n", [1, 23, 24, 100])
@pytest.mark.parametrize("seed", [0, -3, 2 ** 70 + 5])
@pytest.mark.parametrize("largest", [2 ** 31, 2 ** 64 + 3])
def test_all_at_once_as_one_by_one(n, seed, largest):
    rng = random.Random(n)
    requests = [rng.randrange(largest) for _ in range(n - 1)] + [-2]
    draws = [rng.randrange(10000) for _ in range(n)]
    assert uniforms(seed, requests, draws).tolist() == [float(np.float32(uniform(seed, r, d))) for r, d in zip(requests, draws)]
