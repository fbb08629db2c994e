// Batched Q4_K projections of 2..8 activation rows on v_mfma_f32_16x16x32_f16:
// the operands, dequantisation and epilogues of mfma16_q4k_kernel
// (zg_batched.hip) in the one-row GEMV's shape (zg_gemv1.hpp).
//
// Up to 8 rows the activation block is small (a row of K = 2048 is 4 KB), so
// nothing ties a workgroup to a long run of weight tiles: one tile per
// workgroup, K / 512 waves of four units each, about three workgroups to a
// CU whose loads, dequantisation and reductions overlap.  One 8-wave
// workgroup per CU, as beyond 8 rows, passes through those phases in step
// (gate/up at 3 rows: 8.6 us of which 4.2 stream the weights).
//
// R = 8 (projections of at most 2048 outputs, which 16-row tiles would give
// 128 workgroups): lanes n < 8 carry units 0-1 and lanes n >= 8 units 2-3 of
// the same 8 weight rows, the A operand's rows 0-7 the activations of unit p
// and rows 8-15 those of unit p + 2; of the 16 x 16 product the two
// diagonal 8 x 8 blocks are used, and added where the waves' sums are.
//
// Traced in a 3-row step (mfma16_q4k_kernel -> here, us): gate/up 8.6 -> 7.4,
// down 8.3 -> 5.6, input 7.0 -> 6.6, output 5.6 -> 4.7, LM head 48.8 -> 39.1;
// the step of 8 layers 368 -> 304.  A third of that is the finish: with four
// rows per lane of half a wave, as the product lies in the registers, the
// same kernels took 8.4, 6.7, 6.6, 5.0 and 40.9.
#include <algorithm>

#include "zg_decode_common.hpp"

namespace zg {

typedef _Float16 sb_h8 __attribute__((ext_vector_type(8)));
typedef _Float16 sb_h2 __attribute__((ext_vector_type(2)));

// Grid: workgroups over tiles of 16 weight rows (8 gate + 8 up with EPI_GLU)
// or R = 8, further tiles in further passes; 64 W threads, K = 512 W.
template <int EPI, int W, int R>
__global__ __launch_bounds__(64 * W) void small_batch_q4k_kernel(FusedGemvArgs a, const sb_h8* __restrict__ xh) {
    static_assert(R == 16 || (R == 8 && EPI != EPI_GLU), "16-row tiles, or 8-row tiles without the GLU pairing");
    constexpr int K = 512 * W, nunits = K / 128, nbk = K / 256;
    constexpr int U = R == 16 ? 4 : 2, NH = R == 16 ? 2 : 1;  // weight pieces and block headers per lane
    constexpr int TR = EPI == EPI_GLU ? 8 : R;                // outputs per tile
    constexpr int TPR = 8 * W;                                // threads per row of the sums of squares
    __shared__ v4f red[2][W][64];
    __shared__ float inv_s[8];
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, L = lane >> 4, n16 = lane & 15;
    const int N = a.N, nout = EPI == EPI_GLU ? N >> 1 : N, ntiles = (nout + TR - 1) / TR;
    const uint8_t* qs = (const uint8_t*)a.qs;
    const v4u* hdr = (const v4u*)a.hdr;
    auto row_of = [&](int t) {  // past the end: re-read the last row, never stored
        if (EPI == EPI_GLU) {
            const int o = min(t * 8 + (n16 & 7), nout - 1);
            return n16 < 8 ? o : nout + o;
        }
        return min(t * R + (R == 16 ? n16 : (n16 & 7)), nout - 1);
    };
    const int u0 = 4 * w + (R == 16 ? 0 : 2 * (n16 >> 3));  // the lane's first unit
    v4u wq[U], hd[NH];
    auto load_tile = [&](int t) {
        const size_t row = (size_t)row_of(t);
#pragma unroll
        for (int b = 0; b < NH; ++b) hd[b] = __builtin_nontemporal_load(hdr + q4k_hdr_index(row, (u0 >> 1) + b, nbk));
        const uint8_t* rp = qs + (((row >> 4) * nunits + u0) * 64 + (row & 15) + 16 * L) * 16;
#pragma unroll
        for (int u = 0; u < U; ++u) wq[u] = __builtin_nontemporal_load((const v4u*)(rp + 1024 * u));
    };

    // ---- loads in the order of use: the producer's sums of squares, the
    // activations, the weights, the residual outputs of the first tile
    double ssv[8];
    const int srow = tid / TPR, ssub = tid % TPR;
    if (a.rms_ss_in) {
        const int n = a.rms_ss_n;
        const double* ss = a.rms_ss_in + (size_t)min(srow, a.M - 1) * n;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const int c = ssub + TPR * q;
            const double x = ss[min(c, n - 1)];
            ssv[q] = c < n ? x : 0.0;
        }
    }
    // lane l carries activation row l % 16 (R = 8: l % 8, of unit p or p + 2):
    // the rows past M are the tiles' zero padding, taken without a load
    sb_h8 xa[U][4];
    {
        const int m = R == 16 ? n16 : n16 & 7;
        const bool live = m < a.M;
#pragma unroll
        for (int u = 0; u < U; ++u)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                xa[u][i] = sb_h8{0, 0, 0, 0, 0, 0, 0, 0};
                if (live) xa[u][i] = xh[((size_t)(u0 + u) * 4 + i) * 64 + m + 16 * L];
            }
    }
    load_tile(blockIdx.x);
    // finishing lanes: one output each, row fm, column fn of the tile (16-row
    // tiles without the GLU pairing: waves 0 and 1, eight columns each), so
    // that the sums over the waves, the SiLU and the stores are not four
    // in a row on a quarter of the lanes
    constexpr int FW = R == 16 && EPI != EPI_GLU ? 2 : 1;
    const int fr = lane & 3, fL = lane >> 5, fm = 4 * fL + fr, fn = ((lane >> 2) & 7) + 8 * w;
    float yv = 0.0f, gn = 0.0f;
    if (EPI == EPI_RESID && w < FW) {
        const int o = min((int)blockIdx.x * R + fn, nout - 1);
        yv = a.y[(size_t)min(fm, a.M - 1) * a.ldy + o];
        if (a.rms_tiles_out) gn = a.rms_gamma[o];
    }
    __builtin_amdgcn_sched_barrier(0);  // every load above is in flight before the first product
    if (a.rms_ss_in) {
        double tot = 0.0;
#pragma unroll
        for (int q = 0; q < 8; ++q) tot += ssv[q];
        // TPR threads per row, in a fixed order: 8 lanes, then the row's W groups of 8
        __shared__ double part[8][W];
        tot = group8_sum_all(tot);
        if ((lane & 7) == 0) part[srow][ssub >> 3] = tot;
        lds_barrier();  // the weight loads stay in flight
        if (tid < 8) {
            double s = 0.0;
#pragma unroll
            for (int q = 0; q < W; ++q) s += part[tid][q];
            inv_s[tid] = rms_inv(s, K, a.eps);  // (the first tile's barrier orders it)
        }
    }

    const sb_h2 bias = sb_h2{(_Float16)1024.0f, (_Float16)1024.0f};
    int pb = 0;
    for (int t = blockIdx.x; t < ntiles; t += gridDim.x) {
        v4f acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const v4u hh = hd[NH == 1 ? 0 : u >> 1];
            const float d = f16_to_f32((uint16_t)(hh.x & 0xffffu)), dm = f16_to_f32((uint16_t)(hh.x >> 16));
            const int gl = 2 * (2 * (u & 1) + (L >> 1));  // low-nibble group of the lane's run in its block
            sb_h2 sc2[2], nm2[2];
#pragma unroll
            for (int nib = 0; nib < 2; ++nib) {
                uint32_t sc, mn;
                q4k_dev_scale_min(hh, gl + nib, sc, mn);
                const _Float16 sh = (_Float16)(d * (float)sc), mh = (_Float16)(dm * (float)mn);
                sc2[nib] = sb_h2{sh, sh};
                nm2[nib] = sb_h2{-mh, -mh};
            }
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int nib = i >> 1;
                const uint32_t d0 = i & 1 ? wq[u].z : wq[u].x, d1 = i & 1 ? wq[u].w : wq[u].y;
                const uint32_t w0 = (nib ? (d0 >> 4) : d0) & 0x0f0f0f0fu, w1 = (nib ? (d1 >> 4) : d1) & 0x0f0f0f0fu;
                sb_h8 wb;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    // bytes (q, 0x64) pairs: the f16 bit patterns of 1024 + q
                    const uint32_t p = __builtin_amdgcn_perm(0x64646464u, e < 2 ? w0 : w1, e & 1 ? 0x04030402u : 0x04010400u);
                    const sb_h2 v = __builtin_elementwise_fma(__builtin_bit_cast(sb_h2, p) - bias, sc2[nib], nm2[nib]);
                    wb[2 * e] = v[0];
                    wb[2 * e + 1] = v[1];
                }
                acc = __builtin_amdgcn_mfma_f32_16x16x32_f16(xa[u][i], wb, acc, 0, 0, 0);
            }
        }
        const int next = t + gridDim.x;
        if (next < ntiles) load_tile(next);
        red[pb][w][lane] = acc;
        lds_barrier();
        if (w < FW) {
            // element (column c, row fm) of wave q's product; R = 8: the other
            // diagonal block (column c + 8, rows 8 on) joins
            const float* base = (const float*)red[pb];
            auto sum = [&](int c) {
                float v = 0.0f;
#pragma unroll
                for (int q = 0; q < W; ++q) {
                    v += base[(q * 64 + c + 16 * fL) * 4 + fr];
                    if (R == 8) v += base[(q * 64 + c + 8 + 16 * (fL + 2)) * 4 + fr];
                }
                return a.rms_ss_in ? v * inv_s[fm] : v;
            };
            const float v = sum(fn);
            const int o = t * TR + fn;
            const bool live = o < nout && fm < a.M;
            if (EPI == EPI_GLU) {
                // up * silu(gate), rounded to f16 into the down projection's
                // activation tiles (K2 = N/2 columns)
                const float pr = fm < a.M ? sum(fn + 8) * ggml_silu(v) : 0.0f;
                if (live) {
                    if (a.status && !(fabsf(pr) <= 65504.0f)) atomicOr(a.status, 16);
                    ((_Float16*)a.xh_out)[xh_tile_index(fm, o, nout, a.M)] = (_Float16)pr;
                }
            } else if (EPI == EPI_RESID) {
                const bool first = t == (int)blockIdx.x;
                float xn = 0.0f;
                if (live) {
                    float* p = a.y + (size_t)fm * a.ldy + o;
                    xn = (first ? yv : *p) + v;  // source_binary Add, lib.rs:1258-1271
                    *p = xn;
                    if (!finite_f32(xn)) atomicOr(a.status, 1);
                }
                if (a.rms_tiles_out) {
                    // the next RMS projection's A tile element, as
                    // mfma16_q4k_kernel's, and the sum of squares of the
                    // eight columns
                    if (live) {
                        const float tv = xn * (first ? gn : a.rms_gamma[o]);
                        if (!(fabsf(tv) <= 65504.0f)) atomicOr(a.status, 16);
                        a.rms_tiles_out[xh_tile_index(fm, o, N, a.M)] = (_Float16)tv;
                    }
                    const float sq = xn * xn;
                    double tot = (double)sq;
#pragma unroll
                    for (int off = 4; off < 32; off <<= 1) tot += __shfl_xor(tot, off, 64);
                    if (live && (o & 7) == 0) a.rms_ss_out[(size_t)fm * (N >> 3) + (o >> 3)] = tot;
                }
            } else if (live) {
                a.y[(size_t)fm * a.ldy + o] = v;
            }
        }
        pb ^= 1;
    }
}

// 8-row tiles where 16-row ones would leave CUs without a workgroup.
static int tile_rows(size_t N, int epi) { return epi != EPI_GLU && N <= 2048 && N % 8 == 0 ? 8 : 16; }

// A CU holds 16 of the kernel's waves, of which 6, 10 or 12 to a workgroup
// leave some empty: beyond one round of those, mfma16_q4k_kernel (8 waves).
// At 3 rows, us, there against here: 16384 x 3072 13.7, 15.6; 8224 x 5120
// 15.1, 16.1; 8224 x 6144 16.0, 17.1; within a round 4096 x 5120 11.1, 10.6,
// 4096 x 6144 12.5, 11.2.
bool small_batch_fits(size_t M, size_t K, size_t N, int epi) {
    if (M > 8 || !batched16_supported(M, K, N, epi) || (epi == EPI_GLU && (N / 2) % 8)) return false;
    const size_t W = K / 512, tr = tile_rows(N, epi), tiles = epi == EPI_GLU ? N / 16 : (N + tr - 1) / tr;
    return 16 % W == 0 || tiles <= 256 * (16 / W);
}

int rms_ss_columns(size_t M, size_t K, size_t N) {
    if (small_batch_fits(M, K, N, EPI_RESID)) return 8;
    return batched16_supported(M, K, N, EPI_RESID) ? 16 : 32;
}

template <int EPI, int W>
static hipError_t launch_w(const FusedGemvArgs& a, const sb_h8* xh, hipStream_t s) {
    const int nout = EPI == EPI_GLU ? a.N / 2 : a.N, r = tile_rows(a.N, EPI), tr = EPI == EPI_GLU ? 8 : r;
    const dim3 g((unsigned)std::min((nout + tr - 1) / tr, 2048));
    if constexpr (EPI != EPI_GLU) {
        if (r == 8) {
            hipLaunchKernelGGL((small_batch_q4k_kernel<EPI, W, 8>), g, dim3(64 * W), 0, s, a, xh);
            return hipGetLastError();
        }
    }
    hipLaunchKernelGGL((small_batch_q4k_kernel<EPI, W, 16>), g, dim3(64 * W), 0, s, a, xh);
    return hipGetLastError();
}

template <int EPI>
static hipError_t launch_epi(const FusedGemvArgs& a, const sb_h8* xh, hipStream_t s) {
    switch (a.K / 512) {
    case 2: return launch_w<EPI, 2>(a, xh, s);
    case 4: return launch_w<EPI, 4>(a, xh, s);
    case 6: return launch_w<EPI, 6>(a, xh, s);
    case 8: return launch_w<EPI, 8>(a, xh, s);
    case 10: return launch_w<EPI, 10>(a, xh, s);
    case 12: return launch_w<EPI, 12>(a, xh, s);
    default: return hipErrorInvalidValue;
    }
}

hipError_t launch_small_batch(const FusedGemvArgs& a, const void* xh, hipStream_t s) {
    if (!small_batch_fits(a.M, a.K, a.N, a.epi) || a.M <= 0) return hipErrorInvalidValue;
    // eight sums of squares per thread, 8 W threads per row
    if (a.rms_ss_in && a.rms_ss_n > a.K / 8) return hipErrorInvalidValue;
    switch (a.epi) {
    case EPI_GLU: return launch_epi<EPI_GLU>(a, (const sb_h8*)xh, s);
    case EPI_RESID: return launch_epi<EPI_RESID>(a, (const sb_h8*)xh, s);
    default: return launch_epi<EPI_STORE>(a, (const sb_h8*)xh, s);
    }
}

}  // namespace zg
