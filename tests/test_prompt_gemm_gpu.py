"""The prompt GEMM (zg_gemv_device, Q4_K, 256 rows and more): workgroup
shapes, K splits and ragged edges against float64 on the dequantised weight.

The bound: a weight is q s - m with s, m and the difference each rounded to
f16, an activation is rounded to f16; a rounding's rms is 2^-11 / sqrt(3) =
2.8e-4 of its operand, q s and m are about 1.5 times the weight, and the
errors are independent over K, so an output's error has an rms of at most
2.8e-4 sqrt(1.5^2 + 1.5^2 + 1 + 1) = 7.2e-4 of the outputs' rms.  1e-3 bounds
the 2-norm, and 6e-3 (8 of those) each of up to 17 million outputs."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")

from zerogravity_amd import _lib as L
from zerogravity_amd import synth

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def kern():
    from zerogravity_amd import regions as R
    k = R.HipMatVecKernel(0)
    yield k
    k.ctx.close()


# one tile and the 256-row threshold, M and N one past and one short of a
# tile, two, three and four K splits and none, a whole chip of each shape
@pytest.mark.parametrize("M,N,K", [(256, 31, 256), (257, 129, 768), (300, 127, 3072), (385, 260, 3328), (601, 2048, 6144),
                                   (700, 2044, 3072), (640, 1030, 3584), (511, 8224, 1024), (1025, 2049, 2048), (2048, 8224, 512),
                                   (4100, 4097, 256)])
@pytest.mark.parametrize("norm", [False, True])
def test_prompt_gemm_matches_float64(kern, M, N, K, norm):
    rng = np.random.default_rng(M + N + K)
    w = synth.random_q4_k(rng, N, K)
    h = kern.register(700, f"prompt.{M}.{N}.{K}.{norm}", synth.Q4_K, K, N, w.reshape(-1))
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).cuda()
    g = torch.from_numpy((1 + 0.1 * rng.standard_normal(K)).astype(np.float32)).cuda()
    y = torch.full((M + 1, N), 7.0, device="cuda")
    torch.cuda.synchronize()
    for _ in range(2):
        kern.ctx.check(L.lib().zg_gemv_device(kern.ctx.h, h.h, x.data_ptr(), L.F32, M, g.data_ptr() if norm else None,
                                              1e-6, y.data_ptr(), None))
    torch.cuda.synchronize()
    xr = x.double()
    if norm:
        xr = xr / torch.sqrt((xr * xr).mean(1, keepdim=True) + 1e-6) * g.double()
    ref = xr @ torch.from_numpy(h.dequantize()).cuda().double().t().contiguous()
    err, rms = y[:M].double() - ref, ref.square().mean().sqrt().item()
    assert err.square().mean().sqrt().item() <= 1e-3 * rms
    assert err.abs().max().item() <= 6e-3 * rms
    assert bool((y[M] == 7.0).all())  # nothing past the last row
    kern.release_source(700)


def test_prompt_call_lays_out_the_allocation_free_rows(kern):
    """A shape whose small batches read the 32-row tiles: the allocation-free
    call finds them after a prompt alone."""
    N, K = 300, 3584
    rng = np.random.default_rng(9)
    h = kern.register(701, "prompt.noalloc", synth.Q4_K, K, N, synth.random_q4_k(rng, N, K).reshape(-1))
    x = torch.from_numpy(rng.standard_normal((256, K)).astype(np.float32)).cuda()
    y = torch.empty(256, N, device="cuda")
    y3, want = torch.empty(3, N, device="cuda"), torch.empty(3, N, device="cuda")
    torch.cuda.synchronize()
    kern.ctx.check(L.lib().zg_gemv_device(kern.ctx.h, h.h, x.data_ptr(), L.F32, 256, None, 1e-6, y.data_ptr(), None))
    kern.ctx.check(L.lib().zg_gemv_device_noalloc(kern.ctx.h, h.h, x.data_ptr(), L.F32, 3, None, 1e-6, y3.data_ptr(),
                                                  None))
    kern.ctx.check(L.lib().zg_gemv_device(kern.ctx.h, h.h, x.data_ptr(), L.F32, 3, None, 1e-6, want.data_ptr(), None))
    torch.cuda.synchronize()
    assert torch.equal(y3, want)
    kern.release_source(701)


@pytest.mark.parametrize("K", [3584, 2048])
@pytest.mark.parametrize("M", [256, 449, 600])
def test_captured_prompt_call_of_a_weight_without_prompt_tiles(K, M):
    """A weight that only smaller calls have used: the captured prompt runs on
    the 32-row tiles those left, or on the weight's own layout where they
    need none.  Its products are the prompt GEMM's, summed in another order."""
    from zerogravity_amd import regions as R
    k = R.HipMatVecKernel(0)
    N = 1000
    rng = np.random.default_rng(K + M)
    h, other = (k.register(704, f"prompt.late.{i}", synth.Q4_K, K, N, synth.random_q4_k(rng, N, K).reshape(-1))
                for i in range(2))
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).cuda()
    y, want = torch.zeros(M + 1, N, device="cuda"), torch.zeros(M, N, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()

    def call(w, m, to):
        k.ctx.check(L.lib().zg_gemv_device(k.ctx.h, w.h, x.data_ptr(), L.F32, m, None, 1e-6, to.data_ptr(),
                                           stream.cuda_stream))

    call(other, M, want)  # the activation buffer's size
    call(h, 200, want)
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        call(h, M, y)
    call(h, M, want)
    for _ in range(3):
        y.fill_(7.0)
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        diff = (y[:M].double() - want.double()).square().mean().sqrt()
        assert diff <= 1e-5 * want.double().square().mean().sqrt()
        assert bool((y[M] == 7.0).all())
    k.ctx.close()


@pytest.mark.parametrize("K", [7168, 4096])
def test_prompt_call_where_the_f16_tiles_do_not_fit(K):
    """With less memory free than the f16 tiles take, a prompt runs on the
    32-row tiles (K = 7168) or the weight's own layout (K = 4096)."""
    from zerogravity_amd import regions as R
    k = R.HipMatVecKernel(0)
    N, M = 65536, 300
    rng = np.random.default_rng(K)
    h = k.register(705, "prompt.full", synth.Q4_K, K, N, np.tile(synth.random_q4_k(rng, 2048, K).reshape(-1), 32))
    x = torch.from_numpy(rng.standard_normal((M, K)).astype(np.float32)).cuda()
    y, want = torch.zeros(M, N, device="cuda"), torch.zeros(M, N, device="cuda")
    torch.cuda.synchronize()

    def call(to):
        k.ctx.check(L.lib().zg_gemv_device(k.ctx.h, h.h, x.data_ptr(), L.F32, M, None, 1e-6, to.data_ptr(), None))
        torch.cuda.synchronize()

    torch.cuda.empty_cache()
    room = N * K * 2 * 7 // 8  # the 32-row tiles and the buffers fit, the f16 tiles do not
    full = []
    for _ in range(4):  # (less is reported free than the first of them leaves)
        left = torch.cuda.mem_get_info()[0] - room
        if left > 1 << 24:
            full.append(torch.empty(left, dtype=torch.uint8, device="cuda"))
    try:
        call(y)
    finally:
        del full
        torch.cuda.empty_cache()
    call(want)  # the prompt GEMM: the same products in another order
    assert (y.double() - want.double()).square().mean().sqrt() <= 1e-5 * want.double().square().mean().sqrt()
    assert not torch.equal(y, want)  # (they were other kernels)
    k.ctx.close()


def test_a_new_layout_is_written_before_another_stream_finds_it(kern):
    """The first prompt of a large weight on one stream builds its 32-row
    tiles; an allocation-free call on another stream reads them at once."""
    N, K = 40000, 3584
    rng = np.random.default_rng(12)
    w = synth.random_q4_k(rng, 2000, K).reshape(-1)
    h = kern.register(703, "prompt.streams", synth.Q4_K, K, N, np.tile(w, 20))
    x = torch.from_numpy(rng.standard_normal((256, K)).astype(np.float32)).cuda()
    y = torch.empty(256, N, device="cuda")
    y3, want = torch.empty(3, N, device="cuda"), torch.empty(3, N, device="cuda")
    one, two = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    kern.ctx.check(L.lib().zg_gemv_device(kern.ctx.h, h.h, x.data_ptr(), L.F32, 256, None, 1e-6, y.data_ptr(),
                                          one.cuda_stream))
    kern.ctx.check(L.lib().zg_gemv_device_noalloc(kern.ctx.h, h.h, x.data_ptr(), L.F32, 3, None, 1e-6, y3.data_ptr(),
                                                  two.cuda_stream))
    torch.cuda.synchronize()
    kern.ctx.check(L.lib().zg_gemv_device_noalloc(kern.ctx.h, h.h, x.data_ptr(), L.F32, 3, None, 1e-6,
                                                  want.data_ptr(), two.cuda_stream))
    torch.cuda.synchronize()
    assert torch.equal(y3, want)
    assert torch.equal(y3[:, :2000], y3[:, 38000:])
    kern.release_source(703)


def test_captured_prompt_call_outlives_later_calls():
    """A captured prompt whose K is split keeps its buffers through later
    ordinary calls: of its own shape, of a shorter prompt (whose sums are
    larger than its own), of one with other sums.  The graph is replayed
    after all of them, bit for bit what the ordinary call gives."""
    from zerogravity_amd import regions as R
    k = R.HipMatVecKernel(0)
    N, K, M = 2048, 6144, 300
    rng = np.random.default_rng(10)
    h = k.register(702, "prompt.capture", synth.Q4_K, K, N, synth.random_q4_k(rng, N, K).reshape(-1))
    x = torch.from_numpy(rng.standard_normal((1025, K)).astype(np.float32)).cuda()
    out = {m: torch.zeros(m, N, device="cuda") for m in (256, M, 601, 1025)}
    y = torch.zeros(M, N, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()

    def call(m, to):
        k.ctx.check(L.lib().zg_gemv_device(k.ctx.h, h.h, x.data_ptr(), L.F32, m, None, 1e-6, to.data_ptr(),
                                           stream.cuda_stream))

    call(1025, out[1025])
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream, capture_error_mode="thread_local"):
        call(M, y)
    for m in (M, 256, 601, 1025, M):
        call(m, out[m])
        stream.synchronize()
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        # the same products as the longer prompt's unsplit rows, in another order of summation
        diff = (y.double() - out[1025][:M].double()).square().mean().sqrt()
        assert diff <= 1e-5 * out[1025][:M].double().square().mean().sqrt()
    assert torch.equal(y, out[M])
    k.ctx.close()
