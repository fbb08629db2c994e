"""Q4_K projections of 2-8 rows (zg_gemv_device): 8- and 16-row weight tiles,
ragged N, every wave count, one pass and several, against float64 on the
dequantised weight.  The bounds are those of the f16 operands
(test_prompt_gemm_gpu.py): 1e-3 of the outputs' rms in the mean, 6e-3 each."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from zerogravity_amd import _lib as L
from zerogravity_amd import regions as R
from zerogravity_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kern():
    k = R.HipMatVecKernel(0)
    yield k
    k.ctx.close()


@pytest.mark.parametrize("N,K", [(8, 1024), (1001, 1024), (2040, 2048), (2048, 6144), (2049, 2048), (2064, 3072),
                                 (333, 4096), (4100, 5120), (33001, 1024)])
@pytest.mark.parametrize("M", [2, 3, 7, 8, 9])
def test_small_batch_matches_float64(kern, N, K, M):
    rng = np.random.default_rng(N + K + M)
    w = synth.random_q4_k(rng, N, K)
    h = kern.register(720, f"small.{M}.{N}.{K}", synth.Q4_K, K, N, w.reshape(-1))
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).cuda()
    g = torch.from_numpy((1 + 0.1 * rng.standard_normal(K)).astype(np.float32)).cuda()
    y = torch.full((M + 1, N), 7.0, device="cuda")
    torch.cuda.synchronize()
    kern.ctx.check(L.lib().zg_gemv_device(kern.ctx.h, h.h, x.data_ptr(), L.F32, M, g.data_ptr(), 1e-6, y.data_ptr(),
                                          None))
    torch.cuda.synchronize()
    xr = x.double()
    xr = xr / torch.sqrt((xr * xr).mean(1, keepdim=True) + 1e-6) * g.double()
    ref = xr @ torch.from_numpy(h.dequantize()).cuda().double().t().contiguous()
    err, rms = y[:M].double() - ref, ref.square().mean().sqrt().item()
    assert err.square().mean().sqrt().item() <= 1e-3 * rms
    assert err.abs().max().item() <= 6e-3 * rms
    assert bool((y[M] == 7.0).all())
    kern.release_source(720)
