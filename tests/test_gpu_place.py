"""Long variable-length blocks placed in the stream (k_place_blocks): fields
that are mostly zeros, so that up to 64 blocks of a bit each start in one
word, beside blocks of many words, at bit offsets whose lower bits belong to
the caller.  The stream equals the oracle's in every word."""
import numpy as np
import pytest

from zfptest import (NP_OF_TYPE, T_DOUBLE, T_FLOAT, T_INT64, make_layout, max_stream_words, oracle_compress,
                     stream_params_accuracy)

CASES = {
    "reversible_3d": (T_DOUBLE, [61, 30, 17], (1, 16658, 64, -1075)),
    "reversible_1d": (T_FLOAT, [4099], (1, 16658, 64, -1075)),
    "accuracy_4d": (T_FLOAT, [37, 14, 9, 7], stream_params_accuracy(1e-5)),
    "precision_4d_int": (T_INT64, [17, 14, 9, 5], (1, 16658, 64, -1074)),
}


@pytest.mark.gpu
@pytest.mark.parametrize("offset", [0, 1, 63, 200])
@pytest.mark.parametrize("share", [0.0, 0.0005, 0.02, 1.0])
@pytest.mark.parametrize("case", list(CASES))
def test_blocks_that_share_words(case, share, offset):
    import torch

    import zfp_amd as Z
    ztype, n, params = CASES[case]
    rng = np.random.default_rng(offset + int(share * 10000))
    a = rng.standard_normal(int(np.prod(n))) * (2.0 ** 40 if ztype == T_INT64 else 1.0)
    a[rng.random(a.size) >= share] = 0.0
    a = a.astype(NP_OF_TYPE[ztype])
    prefix = np.full(offset // 64 + 1, 0x5a5a5a5a5a5a5a5a, np.uint64)
    prefix[-1] &= np.uint64((1 << offset % 64) - 1)
    base, off, s = make_layout(a, n, "as_is")
    want, bits = oracle_compress(base, off, n, s, ztype, params, offset, prefix=prefix)[:2]
    used = (offset + bits + 63) // 64
    words = torch.full((max_stream_words(n, ztype, params, offset),), -1, dtype=torch.int64, device="cuda")
    words[: prefix.size] = torch.from_numpy(prefix.view(np.int64)).cuda()
    data = torch.from_numpy(a).cuda()
    assert Z.encode(ztype, n, None, data.data_ptr(), params, words.data_ptr(), offset=offset) == bits
    got = words.cpu().numpy().view(np.uint64)
    assert np.array_equal(got[:used], np.asarray(want)[:used])
