"""Q8_0 projections with few row groups (1-4 rows): K split over a workgroup's
waves, the reference's chain handed on between them.  Bit-identical to the
oracle at ragged N and K, at both sides of every chunk count and of the row
group limits, stored and added into a residual."""
import numpy as np
import pytest

import zg_oracle as O
from zerogravity_amd import _lib as L
from zerogravity_amd import regions as R
from zerogravity_amd import synth

pytestmark = [pytest.mark.gpu, pytest.mark.usefixtures("exact_libm")]


@pytest.fixture(scope="module")
def kern():
    k = R.HipMatVecKernel(0)
    yield k
    k.ctx.close()


@pytest.mark.parametrize("N,K", [(1, 32), (9, 96), (777, 1024), (8, 1056), (100, 2048), (1001, 2080), (1024, 3584),
                                 (63, 4096), (40, 4128), (500, 6144), (17, 6176), (24, 8192), (4096, 160),
                                 (4097, 160), (9216, 64), (9217, 64)])
@pytest.mark.parametrize("M", [1, 2, 3, 4])
def test_narrow_rows_bit_exact(kern, N, K, M):
    import torch
    rng = np.random.default_rng(N * 7 + K + M)
    w = synth.random_q8_0(rng, N, K)
    h = kern.register(810, f"narrow.{N}.{K}.{M}", synth.Q8_0, K, N, w.reshape(-1))
    x = rng.standard_normal((M, K)).astype(np.float32)
    y0 = rng.standard_normal((M, N)).astype(np.float32)
    xd, yd = torch.from_numpy(x).cuda(), torch.full((M + 1, N), 3.0, device="cuda")
    torch.cuda.synchronize()
    ref = np.stack([O.matvec(synth.Q8_0, w.reshape(-1), N, K, x[m]) for m in range(M)]).astype(np.float32)
    kern.ctx.check(L.lib().zg_gemv_device(kern.ctx.h, h.h, xd.data_ptr(), L.F32, M, None, 1e-6, yd.data_ptr(), None))
    torch.cuda.synchronize()
    got = yd.cpu().numpy()
    assert np.array_equal(got[:M].view(np.uint32), ref.view(np.uint32))
    assert (got[M] == 3.0).all()
    yd[:M] = torch.from_numpy(y0)
    torch.cuda.synchronize()
    kern.ctx.check(L.lib().zg_gemv_device_fused(kern.ctx.h, h.h, M, 3, 1, xd.data_ptr(), K, None, 0, None, 1e-6, 128,
                                                yd.data_ptr(), N, None, None, None, None, None))
    torch.cuda.synchronize()
    assert np.array_equal(yd[:M].cpu().numpy().view(np.uint32), (y0 + ref).astype(np.float32).view(np.uint32))
    kern.release_source(810)
