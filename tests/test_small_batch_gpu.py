"""Q4_K projections of 2-8 rows (zg_gemv_device): 8- and 16-row weight tiles,
ragged N, every wave count, one pass and several, against float64 on the
dequantised weight.  The bounds are those of the f16 operands
(test_prompt_gemm_gpu.py): 1e-3 of the outputs' rms in the mean, 6e-3 each."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

import zg_oracle as O
from zerogravity_amd import _lib as L
from zerogravity_amd import gguf, qwen35
from zerogravity_amd import regions as R
from zerogravity_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kern():
    k = R.HipMatVecKernel(0)
    yield k
    k.ctx.close()


@pytest.mark.parametrize("N,K", [(8, 1024), (1001, 1024), (2040, 2048), (2048, 6144), (2049, 2048), (2064, 3072),
                                 (333, 4096), (4096, 5120), (4100, 5120), (8190, 3072), (33001, 1024)])
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


# the residual and SwiGLU forms, which a session's step alone reaches: 8-row
# tiles (hidden 1024, 2048) with the next projection's tiles and sums, 16-row
# tiles (3072) without; 2, 6 and 10 waves in the down projection
@pytest.mark.parametrize("hidden,ffn", [(1024, 3072), (2048, 5120), (3072, 1024)])
@pytest.mark.parametrize("B", [2, 5, 8])
def test_small_batch_steps_match_oracle(kern, hidden, ffn, B):
    """Three steps of B rows of a four-layer model, each row against its own
    oracle session: logits within 2e-2, the end-to-end bound of the f16
    projections, and the same greedy token where the oracle's best two are
    further apart than two logits within that bound can move (4e-2)."""
    g = dict(hidden=hidden, layers=4, ffn=ffn, vocab=1000, gdn_heads=16, gdn_dim=128, q_heads=8, kv_heads=2,
             head_dim=256, full_attention_interval=4, max_context=4096, eps=1e-6)
    t = qwen35.synthetic_tensors(g, gguf.Q4_K, seed=31)
    m = qwen35.QwenModelHip(g, t, kernel=kern)
    s = m.session(max_batch=B, max_context=64, kv_dtype=L.F32)
    toks = np.random.default_rng(B).integers(0, g["vocab"], (3, B)).astype(np.uint32)
    got = [s.step(row)[0] for row in toks]
    om = O.Model(g, t)
    for b in range(B):
        o = om.session()
        for i in range(3):
            ref = o.forward(int(toks[i, b]))
            assert float(np.max(np.abs(got[i][b] - ref))) <= 2e-2, (b, i)
            second, first = np.sort(ref)[-2:]
            assert first - second <= 4e-2 or int(np.argmax(got[i][b])) == int(np.argmax(ref)), (b, i)
    m.close()
