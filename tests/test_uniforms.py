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


def test_what_one_by_one_takes_and_refuses():
    """Generators, lists of unequal length (as many as the shorter has) and integers of any kind are taken; what is no integer is not."""
    n = 30
    want = [float(np.float32(uniform(5, r, 7))) for r in range(n)]
    assert uniforms(5, iter(range(n)), [7] * n).tolist() == want
    assert uniforms(5, range(n), [7] * (n + 4)).tolist() == want and uniforms(5, range(n + 9), [7] * n).tolist() == want
    assert uniforms(5, range(n), [7]).tolist() == want[:1]
    assert uniforms(5, [False, True] + list(range(2, n)), [7] * n).tolist() == want
    for m in (3, n):
        for bad in (1.5, None):
            with pytest.raises(TypeError):
                uniforms(5, [1] * m, [bad] + [7] * (m - 1))
            with pytest.raises(TypeError):
                uniforms(5, [bad] + [1] * (m - 1), [7] * m)
