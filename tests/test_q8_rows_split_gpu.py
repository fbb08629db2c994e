"""Q8_0 beyond four rows on the matrix cores: every number of activation-row
pairs per workgroup, bit-identical to the oracle (N of 512 tiles and more take
that kernel; a last ragged tile, a ragged last chunk)."""
import numpy as np
import pytest

import zg_oracle as O
from zerogravity_amd import _lib as L
from zerogravity_amd import regions as R
from zerogravity_amd import synth

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("exact_libm")]


@pytest.mark.parametrize("M", [5, 7, 9, 11, 14, 16, 17, 19, 25, 33])
@pytest.mark.parametrize("N,K", [(8201, 352), (20011, 64), (4100, 1024)])
def test_row_pairs_bit_exact(N, K, M):
    import torch
    kern = R.HipMatVecKernel(0)
    rng = np.random.default_rng(N + K + M)
    w = synth.random_q8_0(rng, N, K)
    h = kern.register(830, f"pairs.{N}.{K}", synth.Q8_0, K, N, w.reshape(-1))
    x = rng.standard_normal((M, K)).astype(np.float32)
    xd, yd = torch.from_numpy(x).cuda(), torch.full((M + 1, N), 3.0, device="cuda")
    torch.cuda.synchronize()
    kern.ctx.check(L.lib().zg_gemv_device(kern.ctx.h, h.h, xd.data_ptr(), L.F32, M, None, 1e-6, yd.data_ptr(), None))
    torch.cuda.synchronize()
    got = yd.cpu().numpy()
    ref = np.stack([O.matvec(synth.Q8_0, w.reshape(-1), N, K, x[m]) for m in range(M)]).astype(np.float32)
    assert np.array_equal(got[:M].view(np.uint32), ref.view(np.uint32))
    assert (got[M] == 3.0).all()
    kern.ctx.close()


@pytest.mark.parametrize("N,K,M", [(4090, 3584, 64), (12280, 1056, 32), (12280, 1056, 64), (300, 8192, 64)])
def test_rows_dealt_over_rounds_bit_exact(N, K, M):
    """Several workgroup rows, in one round of 512 workgroups and in more."""
    test_row_pairs_bit_exact(N, K, M)
