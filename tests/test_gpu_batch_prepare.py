"""The words a batch compression clears before blocks OR into them
(k_batch_prepare): more jobs than one pass over them holds (256), jobs of one
word and of several pieces of 2048, at bit offsets whose lower bits belong to
the caller, over buffers full of ones.  Every stream equals the one its job
gives alone."""
import numpy as np
import pytest

from zfptest import T_DOUBLE, T_FLOAT, stream_params_accuracy, stream_params_rate

SIZES = {1: [[3]], 255: [[5]], 256: [[70, 9], [4]], 257: [[300, 290], [2]], 700: [[33], [40, 41], [60, 50, 40], [1]]}


@pytest.mark.gpu
@pytest.mark.parametrize("count", list(SIZES))
def test_cleared_words(count):
    import torch

    import zfp_amd as Z
    rng = np.random.default_rng(count)
    jobs, alone, got, keep = [], [], [], []
    for k in range(count):
        n = SIZES[count][k % len(SIZES[count])]
        ztype = T_FLOAT if k % 3 else T_DOUBLE
        params = stream_params_rate(3, ztype, len(n)) if k % 2 else stream_params_accuracy(1e-4)
        offset = int(rng.integers(0, 200))
        a = torch.from_numpy(rng.standard_normal(int(np.prod(n))).astype(np.float32 if ztype == T_FLOAT else np.float64))
        a = a.cuda()
        cap = Z.max_stream_words(ztype, n, params) + 5
        pair = [torch.full((cap,), -1, dtype=torch.int64, device="cuda") for _ in range(2)]
        index = torch.zeros(int(np.prod([(v + 3) // 4 for v in n])) + 1, dtype=torch.int64, device="cuda")
        bits = Z.encode(ztype, n, None, a.data_ptr(), params, pair[0].data_ptr(), offset=offset)
        jobs.append(Z.make_job(ztype, n, None, a.data_ptr(), params, pair[1].data_ptr(), offset, cap,
                               None if params[0] == params[1] else index.data_ptr()))
        keep.append((a, index))
        alone.append((bits, pair[0]))
        got.append(pair[1])
    bits = Z.Batch(jobs, Z.ZFP_HIP_BATCH_COMPRESS).run()
    for k in range(count):
        assert int(bits[k]) == alone[k][0]
        assert torch.equal(got[k], alone[k][1]), k
