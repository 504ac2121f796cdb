"""The hadron list's read-back: every byte arrives, at the list sizes where
the staged copy changes its shape (one copy, one chunk more or less, rings of
1, 2 and 4 MB chunks), into fresh and reused buffers."""
import numpy as np
import pytest

import iss_amd

pytestmark = pytest.mark.gpu

MB = 1 << 20
BYTES = [0, 40, 4 * MB // 40 * 40, 4 * MB // 40 * 40 + 40, 5 * MB // 40 * 40, 16 * MB // 40 * 40 + 80,
         17 * MB // 40 * 40, 33 * MB // 40 * 40 + 40, 101 * MB // 40 * 40]


@pytest.fixture(scope="module")
def ctx():
    c = iss_amd.Context(0)
    yield c
    c.close()


@pytest.mark.parametrize("nbytes", BYTES)
def test_list_comes_back_whole(ctx, nbytes):
    n = nbytes // 40
    words = np.random.default_rng(n).integers(0, 2 ** 31 - 1, 10 * n, dtype=np.int32)
    h = words.view(iss_amd.HADRON_DTYPE)
    ctx.set_hadrons([n // 3, n - n // 3], h)
    for _ in range(2):
        assert np.array_equal(ctx.hadrons().view(np.int32), words)
    assert ctx.event_counts().tolist() == [n // 3, n - n // 3]
