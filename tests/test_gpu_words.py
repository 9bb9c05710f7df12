"""Words of a step that travel as launch arguments and come back through pinned memory."""
import numpy as np
import pytest
import torch

from doppler_amd import capi

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 3, 16])
def test_words_there_and_back(n):
    """In order with the work around them, next to words that stay, and again with other values."""
    L = capi.init(torch.cuda.current_device())
    d = torch.full((24,), 7, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    for seed in (1, 2):
        words = np.random.default_rng(seed).integers(0, 1 << 32, n, dtype=np.uint32)
        capi.check(L.dh_fill_zero(d.data_ptr(), 8, 4 * n))
        capi.check(L.dh_set_words(d.data_ptr(), 8, words.ctypes.data, n))
        kept = words.copy()
        words[:] = 0                                # the launch has them already
        got = np.zeros(n, np.uint32)
        capi.check(L.dh_read_words(got.ctypes.data, d.data_ptr(), 8, n))
        assert np.array_equal(got, kept)
        assert np.array_equal(d.cpu().numpy().view(np.uint32), np.concatenate([[7, 7], kept, [7] * (22 - n)]).astype(np.uint32))


def test_words_refusals():
    L = capi.init(torch.cuda.current_device())
    d = torch.zeros(24, dtype=torch.int32, device="cuda")
    w = np.zeros(17, np.uint32)
    for n, p, off, message in ((0, d.data_ptr(), 0, "words"), (17, d.data_ptr(), 0, "words"), (1, None, 0, "null"), (1, d.data_ptr(), 2, "aligned")):
        assert L.dh_set_words(p, off, w.ctypes.data, n) == 1 and message in L.dh_last_error().decode()
        assert L.dh_read_words(w.ctypes.data, p, off, n) == 1 and message in L.dh_last_error().decode()
