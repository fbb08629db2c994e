// Prompt-sized projections (M >= kGemmRows rows): Y[m][n] (+)= sum_k X[m][k] W[n][k]
// with X the f16 activation tiles act16_kernel writes and W the Q4_K weight
// dequantized once to f16 tiles of the same order (ensure_f16_tiles).
//
// gemm_f16_kernel: v_mfma_f32_32x32x16_f16 on operands staged in LDS by
// direct buffer_load ... lds copies.  Both operands lie in memory as 1 KB
// fragments (32 rows x 16 columns, the 64 lanes' 16-byte words in lane
// order), so a fragment is one wave instruction from memory to LDS and one
// conflict-free ds_read_b128 from LDS to registers.  A workgroup of 8 waves
// owns (MT WM) x (NT WN) tiles of 32 x 32, each wave MT x NT; ST stages of
// 32 columns rotate in LDS, ST - 1 of them in flight while one is
// multiplied, and each wave reads the next 16 columns' fragments before the
// current ones' products, across the stage barrier too.
//
// What bounds it: power.  At M = 2048, N = 12288, K = 2048 the GEMM alone
// runs 101 us = 1021 TFLOP/s on random operands and 78 us = 1318 TFLOP/s on
// zeros (same instructions), the library's f16 product 106 us.  The kernel
// this replaces dequantized the weights in every workgroup (5 VALU
// operations per two weights before each operand's products): 135 us for
// the same projection.  The f16 copy costs N K 2 bytes per weight; reading
// four times the bytes of the codec's own payload is hidden from 256 rows on.
#include <algorithm>

#include "zg_decode_common.hpp"

namespace zg {

namespace {

typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef float f16v __attribute__((ext_vector_type(16)));

constexpr float kF16Max = 65504.0f;
constexpr int kFrags = 2;  // 16-column fragments per tile and stage

}  // namespace

// One 1 KB fragment from memory into LDS: lane l's 16 bytes at byte
// `offset` + 16 l of a strip of `bytes` bytes go to `lds` + 16 l.
__device__ __forceinline__ void copy_frag(const _Float16* strip, int bytes, int offset, int lane, char* lds) {
    const __amdgpu_buffer_rsrc_t r = __builtin_amdgcn_make_buffer_rsrc((void*)strip, 0, bytes, 0x00020000);
    __builtin_amdgcn_raw_ptr_buffer_load_lds(r, (__attribute__((address_space(3))) void*)lds, 16, lane * 16, offset, 0,
                                             0);
}

// up * silu(gate) of values the fast form covers (|gate| < 80: the exponent
// stays in range, so ggml_exp's scaling branches and its finite check drop
// out and its bits stay); the quotient by a reciprocal with one Newton step
// and one residual correction instead of the scaled division.  The 16 values
// of a lane's tile in ggml_silu took about 50 VALU instructions each, 19 us
// of the 2048 x 12288 projection's 124.
// Over every |gate| < 80 the bits are those of up * ggml_silu(gate), but for
// the sign of a zero gate's product, so a tile may take either form.
__device__ __forceinline__ float silu_product(float g, float up) {
    const float x = 0.0f - g, r = __uint_as_float(0x4b400000u);
    const float z = fmaf(x, __uint_as_float(0x3fb8aa3bu), r), n = z - r;
    const float b = fmaf(-n, __uint_as_float(0x35bfbe8eu), fmaf(-n, __uint_as_float(0x3f317200u), x));
    const float k = __uint_as_float((__float_as_uint(z) << 23) + 0x3f800000u), u = b * b;
    const float j = fmaf(fmaf(fmaf(__uint_as_float(0x3c072010u), b, __uint_as_float(0x3d2b9f17u)), u,
                              fmaf(__uint_as_float(0x3e2aaf33u), b, __uint_as_float(0x3efffedbu))),
                         u, __uint_as_float(0x3f7ffff6u) * b);
    const float d = 1.0f + fmaf(j, k, k);
    float y = __builtin_amdgcn_rcpf(d);
    y = fmaf(fmaf(-d, y, 1.0f), y, y);
    float q = g * y;
    q = fmaf(fmaf(-q, d, g), y, q);
    return up * q;
}

// Grid of mg x ng x S tiles in one dimension, 64 WM WN threads.  Workgroups go
// round-robin to the 8 XCDs: each XCD takes a contiguous run of the tile
// order (bands of 8 tiles along M, M fastest), so its L2 holds the operands
// its 32 CUs share.  S > 1: run z of the K columns into parts[z].
template <int EPI, int MT, int NT, int WM, int WN, int ST>
__global__ __launch_bounds__(64 * WM * WN, 1) void gemm_f16_kernel(FusedGemvArgs a, const _Float16* __restrict__ xh,
                                                                   const _Float16* __restrict__ wh, int mg, int ng) {
    constexpr int W = WM * WN, TA = MT * WM, TB = NT * WN, FR = (TA + TB) * kFrags, LPW = FR / W;
    static_assert(FR % W == 0 && NT == 2, "whole loads per wave; a wave's two weight tiles are a SwiGLU pair");
    __shared__ __attribute__((aligned(16))) char lds[ST][FR * 1024];
    const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int wm = wv / WN, wn = wv - wm * WN;
    const int S = EPI != EPI_GLU && a.splits > 1 ? a.splits : 1;
    const int total = mg * ng * S, xc = blockIdx.x & 7, li = blockIdx.x >> 3;
    const int per = total >> 3, rem = total & 7, lt = xc * per + min(xc, rem) + li;
    const int z = lt / (mg * ng), t = lt - z * mg * ng;
    const int band = t / (8 * ng), bw = min(8, mg - 8 * band), tb = t - band * 8 * ng;
    const int bm = 8 * band + tb % bw, bn = tb / bw;
    const int N = a.N, kf = a.K >> 4, mtiles = (a.M + 31) >> 5, ntiles = (N + 31) >> 5;
    // stage s covers fragments kFrags s ..; this run's stages [s0, s0 + ns)
    const int s0 = z * (kf / kFrags) / S;
    int ns = (z + 1) * (kf / kFrags) / S - s0;
    // Opaque: with SwiGLU, where S is 1, the compiler otherwise peels the loop
    // below and keeps two copies of the sums (registers of the 256 x 256,
    // 128 x 256 and 128 x 128 shapes: 256 and 254 spilled, 182, 104; with
    // this 184, 102, 60).  8192 x 12288 x 2048: 2379 -> 385 us.
    asm volatile("" : "+s"(ns));

    // Weight tile of slot b of this workgroup: wave wn's slots are 2 wn and
    // 2 wn + 1; with SwiGLU slot 2 wn is a gate tile and 2 wn + 1 the up tile
    // N/64 tiles later (rows j and N/2 + j pair up).
    auto wtile = [&](int b) { return EPI == EPI_GLU ? bn * (TB / 2) + (b >> 1) + (b & 1) * (N >> 6) : bn * TB + b; };
    // the K strip of each of this wave's loads (tiles past the end read the
    // last one; their results are dropped)
    const _Float16* strip[LPW];
#pragma unroll
    for (int i = 0; i < LPW; ++i) {
        const int f = wv + i * W, tile = f / kFrags;
        strip[i] = tile < TA ? xh + (size_t)min(bm * TA + tile, mtiles - 1) * kf * 512
                             : wh + (size_t)min(wtile(tile - TA), ntiles - 1) * kf * 512;
    }
    auto load = [&](int s, int buf) {
#pragma unroll
        for (int i = 0; i < LPW; ++i) {
            const int f = wv + i * W;
            copy_frag(strip[i], kf * 1024, ((s0 + s) * kFrags + f % kFrags) * 1024, lane, &lds[buf][f * 1024]);
        }
    };
    h8v fa[2][MT], fb[2][NT];
    auto frags = [&](int buf, int k, int slot) {
#pragma unroll
        for (int i = 0; i < MT; ++i)
            fa[slot][i] = *(const h8v*)&lds[buf][(((wm * MT + i) * kFrags + k) * 64 + lane) * 16];
#pragma unroll
        for (int j = 0; j < NT; ++j)
            fb[slot][j] = *(const h8v*)&lds[buf][(((TA + wn * NT + j) * kFrags + k) * 64 + lane) * 16];
    };
    f16v acc[MT][NT];
#pragma unroll
    for (int i = 0; i < MT; ++i)
#pragma unroll
        for (int j = 0; j < NT; ++j) acc[i][j] = f16v{};

    // K >= 256 gives ns >= 2 stages per run (K >= 3072 with splits), ST - 1 <= 3
#pragma unroll
    for (int s = 0; s < ST - 1; ++s) load(min(s, ns - 1), s);
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(LPW * (ST - 2)) : "memory");
    frags(0, 0, 0);
    load(min(ST - 1, ns - 1), ST - 1);
    for (int sb = 0; sb < ns; sb += ST) {
#pragma unroll
        for (int u = 0; u < ST; ++u) {
            const int s = sb + u;
            if (s >= ns) break;
            frags(u, 1, 1);
            __builtin_amdgcn_sched_barrier(0);  // the reads go out before the products they overlap
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[0][i], fb[0][j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
            // stage s + 1 has landed (each wave waits for its own copies, the
            // barrier for the others'), and every wave has read stage s, whose
            // buffer then takes stage s + ST.  Every pass issues the same
            // LPW copies (past the end: the last stage again), so the count
            // left in flight is a constant.
            asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(LPW * (ST - 2)) : "memory");
            frags((u + 1) % ST, 0, 0);
            load(min(s + ST, ns - 1), u);
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int j = 0; j < NT; ++j)
#pragma unroll
                for (int i = 0; i < MT; ++i)
                    acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_f16(fa[1][i], fb[1][j], acc[i][j], 0, 0, 0);
            __builtin_amdgcn_sched_barrier(0);
        }
    }
    // no copy into LDS outlives its use below, or the workgroup
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    // D register r of tile (i, j) is row (r%4) + 8*(r/4) + 4*(lane/32) of the
    // activation tile, column lane%32 of the weight tile
    const int hsel = lane >> 5, r32 = lane & 31;
    bool over = false;
#pragma unroll
    for (int i = 0; i < MT; ++i) {
        const int tm = bm * TA + wm * MT + i;
        if (tm >= mtiles) continue;
        if constexpr (EPI == EPI_GLU) {
            // up * silu(gate) in f32, rounded once to f16 into the down
            // projection's A tiles (K = N/2 columns); a value past the f16
            // range raises status bit 4.  The 32 x 32 products are two of
            // those fragments: turned in the wave's own LDS (2 KB), stored as
            // whole 16-byte words.
            _Float16* turn = (_Float16*)lds + wv * 1024;
            bool small = true;  // (false for a NaN gate)
#pragma unroll
            for (int r = 0; r < 16; ++r) small &= fabsf(acc[i][0][r]) < 80.0f;
            const bool fast = __all(small);
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m32 = (r & 3) + 8 * (r >> 2) + 4 * hsel;
                float v = fast ? silu_product(acc[i][0][r], acc[i][1][r]) : acc[i][1][r] * ggml_silu(acc[i][0][r]);
                if (tm * 32 + m32 >= a.M) v = 0.0f;
                over |= !(fabsf(v) <= kF16Max);
                turn[((r32 >> 4) * 64 + ((r32 & 15) >> 3) * 32 + m32) * 8 + (r32 & 7)] = (_Float16)v;
            }
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            const h8v o0 = *(const h8v*)(turn + lane * 8), o1 = *(const h8v*)(turn + 512 + lane * 8);
            _Float16* dst = (_Float16*)a.xh_out + ((size_t)tm * (N >> 5) + 2 * (bn * (TB / 2) + wn)) * 512;
            *(h8v*)(dst + lane * 8) = o0;
            *(h8v*)(dst + 512 + lane * 8) = o1;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // both words read before the next tile turns
        } else {
            const int m0 = tm * 32 + 4 * hsel, n0 = (bn * TB + wn * NT) * 32 + r32;
            auto row = [](int r) { return (r & 3) + 8 * (r >> 2); };
            // the residual rows are all requested before the first is used
            // (read and written element by element, each add waited on a
            // load: 35 us of a 2048 x 2048 x 2048 projection, 21 without)
            float old[EPI == EPI_RESID ? 16 : 1][NT];
            if constexpr (EPI == EPI_RESID) {
#pragma unroll
                for (int r = 0; r < 16; ++r)
#pragma unroll
                    for (int j = 0; j < NT; ++j)
                        old[r][j] = m0 + row(r) < a.M && n0 + 32 * j < N
                                        ? a.y[(size_t)(m0 + row(r)) * a.ldy + n0 + 32 * j]
                                        : 0.0f;
            }
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int m = m0 + row(r);
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    const int n = n0 + 32 * j;
                    if (m >= a.M || n >= N) continue;
                    if constexpr (EPI == EPI_RESID) {
                        const float v = old[r][j] + acc[i][j][r];
                        over |= !finite_f32(v);
                        a.y[(size_t)m * a.ldy + n] = v;
                    } else if (S > 1) {
                        a.parts[((size_t)z * a.M + m) * N + n] = acc[i][j][r];
                    } else {
                        a.y[(size_t)m * a.ldy + n] = acc[i][j][r];
                    }
                }
            }
        }
    }
    // SwiGLU: past the f16 range; residual: nonfinite
    if (over && a.status) atomicOr(a.status, EPI == EPI_GLU ? 16 : 1);
}

// Grid (tiles, K/256), 256 threads: columns 256 kb.. of the 32 rows of tile
// `tile`, dequantized to f16 fragments.  Thread (c4, lane) holds row lane%32,
// columns 64 c4 + 32 half + 16 piece + 8 (lane/32) .. +7 of the four
// fragments (half, piece); scale and min of a 32-group rounded once to f16,
// the weight q s - m as one f16 fma.  Rows past N are zero.
__global__ __launch_bounds__(256) void f16_tile_q4k_kernel(const uint8_t* __restrict__ qs, const v4u* __restrict__ hdr,
                                                           int N, int K, _Float16* __restrict__ wh) {
    const int tile = blockIdx.x, kb = blockIdx.y, nbk = K >> 8;
    const int c4 = threadIdx.x >> 6, lane = threadIdx.x & 63, row = tile * 32 + (lane & 31);
    uint2 p[2] = {};
    v4u hd = v4u{0u, 0u, 0u, 0u};
    if (row < N) {
        const uint8_t* b = qs + q4k_chunk_offset(row, 4 * kb + c4, K) + 8 * (lane >> 5);
        p[0] = *(const uint2*)b;
        p[1] = *(const uint2*)(b + 256);
        hd = hdr[q4k_hdr_index(row, kb, nbk)];
    }
    const float d = f16_to_f32((uint16_t)(hd.x & 0xffffu)), dmin = f16_to_f32((uint16_t)(hd.x >> 16));
    const h2v bias = h2v{(_Float16)1024.0f, (_Float16)1024.0f};
    _Float16* dst = wh + (((size_t)tile * (K >> 4) + 16 * kb + 4 * c4) * 64 + lane) * 8;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        uint32_t s, mn;
        q4k_dev_scale_min(hd, 2 * c4 + h, s, mn);
        const _Float16 sh = (_Float16)(d * (float)s), mh = (_Float16)(dmin * (float)mn);
        const h2v s2 = h2v{sh, sh}, n2 = h2v{-mh, -mh};
#pragma unroll
        for (int q = 0; q < 2; ++q) {
            const uint32_t w0 = (p[q].x >> (4 * h)) & 0x0f0f0f0fu, w1 = (p[q].y >> (4 * h)) & 0x0f0f0f0fu;
            h8v o;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                // bytes (q, 0x64) pairs: the f16 bit patterns of 1024 + q
                const uint32_t pr = __builtin_amdgcn_perm(0x64646464u, e < 2 ? w0 : w1, e & 1 ? 0x04030402u : 0x04010400u);
                const h2v v = __builtin_elementwise_fma(__builtin_bit_cast(h2v, pr) - bias, s2, n2);
                o[2 * e] = v[0];
                o[2 * e + 1] = v[1];
            }
            *(h8v*)(dst + (size_t)(2 * h + q) * 512) = o;
        }
    }
}

// y[m][n] (+)= (parts[0] + parts[1]) (+ parts[2]) (+ parts[3]) at (m, n), the
// splits summed in order, float4 per thread; with ADD (residual) a
// non-finite sum raises status bit 1 as the residual epilogue does.
template <int S, bool ADD>
__global__ __launch_bounds__(256) void split_sum_kernel(FusedGemvArgs a) {
    const size_t i4 = (size_t)blockIdx.x * 256 + threadIdx.x, n4 = (size_t)a.M * a.N / 4;
    if (i4 >= n4) return;
    const size_t e = 4 * i4, m = e / a.N, n = e % a.N, mn = (size_t)a.M * a.N;
    v4f p[S];
#pragma unroll
    for (int z = 0; z < S; ++z) p[z] = *(const v4f*)(a.parts + z * mn + e);
    float* yp = a.y + m * a.ldy + n;
    v4f r = ADD ? *(const v4f*)yp : v4f{0.0f, 0.0f, 0.0f, 0.0f};
    bool bad = false;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        float acc = p[0][q];
#pragma unroll
        for (int z = 1; z < S; ++z) acc = acc + p[z][q];
        r[q] = ADD ? r[q] + acc : acc;
        bad |= !finite_f32(r[q]);
    }
    *(v4f*)yp = r;
    if (ADD && bad) atomicOr(a.status, 1);
}

namespace {

// Workgroup shapes, rows x columns: 256 x 256 (one per CU: 128 KB of LDS),
// 128 x 256 and 128 x 128 (two per CU).
enum { SHAPE_256x256, SHAPE_128x256, SHAPE_128x128 };

long tiles_of(size_t n, size_t w) { return (long)((n + w - 1) / w); }

// The shape with the least time by measured rates: full chips of workgroups
// (512, or 256 of 256 x 256) and the tail by its size.  In us at K = 2048,
// the weights read from HBM as a model's are: 256 workgroups of 256 x 256
// 66 (64 alone: 45), 512 of 128 x 256 70 (256: 36, 64: 26), 512 of
// 128 x 128 44 (256: 19-21, 64: 13); with the weights in the Infinity Cache
// the 128-wide shapes are 67 and 38, which moves no choice by more than 5%.
int choose_shape(size_t M, size_t N) {
    const long l = tiles_of(M, 256) * tiles_of(N, 256), b = tiles_of(M, 128) * tiles_of(N, 256),
               c = tiles_of(M, 128) * tiles_of(N, 128);
    auto tail = [](long r, double few, double some, double many) {
        return r == 0 ? 0.0 : r <= 64 ? few : r <= 256 ? some : many;
    };
    const double tl = (l / 256) * 66.0 + tail(l % 256, 45.0, 62.0, 62.0);
    const double tb = (b / 512) * 70.0 + tail(b % 512, 26.0, 36.0, 70.0);
    const double tc = (c / 512) * 44.0 + tail(c % 512, 13.5, 19.0, 44.0);
    return tc <= tb && tc <= tl ? SHAPE_128x128 : tb <= tl ? SHAPE_128x256 : SHAPE_256x256;
}

template <int EPI>
hipError_t launch_gemm(const FusedGemvArgs& a, int shape, const _Float16* xh, const _Float16* wh, hipStream_t s) {
    const int S = EPI != EPI_GLU && a.splits > 1 ? a.splits : 1;
    const int mg = (int)tiles_of(a.M, shape == SHAPE_256x256 ? 256 : 128);
    const int ng = (int)tiles_of(a.N, shape == SHAPE_128x128 ? 128 : 256);
    const dim3 g((unsigned)(mg * ng * S));
    if (shape == SHAPE_256x256)
        hipLaunchKernelGGL((gemm_f16_kernel<EPI, 4, 2, 2, 4, 4>), g, dim3(512), 0, s, a, xh, wh, mg, ng);
    else if (shape == SHAPE_128x256)
        hipLaunchKernelGGL((gemm_f16_kernel<EPI, 2, 2, 2, 4, 3>), g, dim3(512), 0, s, a, xh, wh, mg, ng);
    else
        hipLaunchKernelGGL((gemm_f16_kernel<EPI, 1, 2, 4, 2, 4>), g, dim3(512), 0, s, a, xh, wh, mg, ng);
    return hipGetLastError();
}

}  // namespace

hipError_t ensure_f16_tiles(DeviceWeight& w, hipStream_t s) {
    if (w.type != kQ4_K || w.K % 256 || w.N == 0) return hipErrorInvalidValue;
    if (w.wh) return hipSuccess;
    const size_t tiles = (w.N + 31) / 32;
    void* p = nullptr;
    hipError_t e = hipMalloc(&p, f16_tile_bytes(w.N, w.K));
    if (e != hipSuccess) {
        (void)hipGetLastError();  // (the caller may go on without)
        return e;
    }
    hipLaunchKernelGGL(f16_tile_q4k_kernel, dim3((unsigned)tiles, (unsigned)(w.K / 256)), dim3(256), 0, s,
                       (const uint8_t*)w.qs, (const v4u*)w.hdr, (int)w.N, (int)w.K, (_Float16*)p);
    e = hipGetLastError();
    // written before any stream can find it
    if (e == hipSuccess) e = hipStreamSynchronize(s);
    if (e != hipSuccess) {
        (void)hipFree(p);
        return e;
    }
    w.wh = p;
    return hipSuccess;
}

// What a prompt is refused by, at 4 GiB or more: the bytes of its f16
// activation tiles (32 rows x K per tile) and of the weight's 32-row tiles and
// headers.  No kernel needs the bound any more (offsets within a K strip, at
// most 512 KB, are what is left in 32 bits); the f16 weight tiles, which it
// does not count, may pass it.
uint64_t prompt_gemm_bytes(size_t M, size_t K, size_t N) {
    const uint64_t mt = (M + 31) / 32, nt = (N + 31) / 32, nbk = K / 256;
    return std::max({mt * K * 64, nt * nbk * 4096, nt * nbk * 512});
}

bool prompt_gemm_supported(int type, size_t K, size_t N, int epi) {
    if (type != kQ4_K || K % 256 || K > 8192 || N == 0) return false;
    if (epi == EPI_GLU) return N % 64 == 0 && (N / 2) % 256 == 0;
    return true;
}

// K splits: 128 x 128 tiles that fill at most half the CUs, with K long
// enough that the shorter runs outweigh the second launch (M = 601, N = 2048,
// K = 6144: 36 us unsplit, 21 us in three runs plus about 5 us for the sum;
// M = 1024: 39 us, 29 us in two).  At most 256 tiles of partial sums, 4 Mi floats.
int prompt_splits(size_t M, size_t K, size_t N) {
    const long c = tiles_of(M, 128) * tiles_of(N, 128);
    return K >= 3072 && N % 4 == 0 && c <= 128 ? (int)std::min<long>(4, 256 / c) : 1;
}

hipError_t prompt_gemm(const DeviceWeight& w, const FusedGemvArgs& args, const _Float16* xh, hipStream_t s) {
    if (!prompt_gemm_supported(w.type, w.K, w.N, args.epi) || !w.wh || args.M <= 0) return hipErrorInvalidValue;
    if (args.epi == EPI_GLU && !args.xh_out) return hipErrorInvalidValue;
    FusedGemvArgs a = args;
    a.K = (int)w.K;
    a.N = (int)w.N;
    a.splits = 0;
    const _Float16* wh = (const _Float16*)w.wh;
    if (a.epi == EPI_GLU) return launch_gemm<EPI_GLU>(a, choose_shape(a.M, a.N), xh, wh, s);
    int S = a.prompt_parts && a.ldy % 4 == 0 && (uintptr_t)a.y % 16 == 0 ? prompt_splits(a.M, w.K, w.N) : 1;
    if ((size_t)S * a.M * a.N > a.prompt_parts_n) S = 1;
    if (S > 1) {
        a.splits = S;
        a.parts = a.prompt_parts;
        const hipError_t e = launch_gemm<EPI_STORE>(a, SHAPE_128x128, xh, wh, s);
        if (e != hipSuccess) return e;
        const dim3 g((unsigned)(((size_t)a.M * a.N / 4 + 255) / 256));
#define ZG_SUM(SV)                                                                                               \
    if (a.epi == EPI_RESID) hipLaunchKernelGGL((split_sum_kernel<SV, true>), g, dim3(256), 0, s, a);               \
    else hipLaunchKernelGGL((split_sum_kernel<SV, false>), g, dim3(256), 0, s, a);
        if (S == 4) {
            ZG_SUM(4)
        } else if (S == 3) {
            ZG_SUM(3)
        } else {
            ZG_SUM(2)
        }
#undef ZG_SUM
        return hipGetLastError();
    }
    const int shape = choose_shape(a.M, a.N);
    return a.epi == EPI_RESID ? launch_gemm<EPI_RESID>(a, shape, xh, wh, s) : launch_gemm<EPI_STORE>(a, shape, xh, wh, s);
}

}  // namespace zg
