"""The hadron list's read-back by the kind of memory and by the context's
earlier lists: page-locked destinations (the runtime's direct copy), also
inside a larger page-locked buffer, short pageable lists before and after the
staging slots exist.  The same bytes everywhere."""
import ctypes

import numpy as np
import pytest
import torch

import iss_amd

pytestmark = pytest.mark.gpu

MB = 1 << 20


@pytest.mark.parametrize("nbytes", [40, 4 * MB // 40 * 40 + 40, 33 * MB // 40 * 40])
def test_pinned_and_pageable_lists_agree(nbytes):
    ctx = iss_amd.Context(0)
    words = np.random.default_rng(nbytes).integers(0, 2 ** 31 - 1, nbytes // 4, dtype=np.int32)
    ctx.set_hadrons([nbytes // 40], words.view(iss_amd.HADRON_DTYPE))
    pinned = torch.zeros(nbytes + 8192, dtype=torch.uint8).pin_memory()
    for at in (0, 4096, 8192):
        pinned.zero_()
        assert ctx.lib.iss_get_hadrons(ctx.h, ctypes.c_void_p(pinned.data_ptr() + at), nbytes // 40) == 0
        got = pinned.numpy()
        assert np.array_equal(got[at:at + nbytes], words.view(np.uint8))
        assert not got[:at].any() and not got[at + nbytes:].any()
    assert np.array_equal(ctx.hadrons().view(np.int32), words)
    ctx.close()


@pytest.mark.parametrize("first", [0, 33 * MB // 40 * 40])
@pytest.mark.parametrize("nbytes", [4 * MB // 40 * 40 + 40, 5 * MB // 40 * 40, 16 * MB // 40 * 40 + 80])
def test_short_lists_before_and_after_the_slots(first, nbytes):
    ctx = iss_amd.Context(0)
    for n in (first, nbytes):
        words = np.random.default_rng(n).integers(0, 2 ** 31 - 1, n // 4, dtype=np.int32)
        ctx.set_hadrons([n // 40], words.view(iss_amd.HADRON_DTYPE))
        for _ in range(7 if n == nbytes else 1):
            assert np.array_equal(ctx.hadrons().view(np.int32), words)
    ctx.close()
