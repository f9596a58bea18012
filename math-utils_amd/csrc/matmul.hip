// matmul.hip - out[m][n] = a[m][k] . w[n][k] (+ bias[n]) (+ out), the
// projection every mixer and MLP applies (LocalModel.hpp:1044-1078 apply,
// behind gpu::matmulNT*), for the reference's four weight encodings:
//   F32    [n][k] fp32
//   BF16   [n][k] bf16 (widened by a 16-bit shift, Kernels.hip widenBF16)
//   Q8     [n][k] int8 codes, one fp32 scale per 32 codes (Quant.hpp:528-538)
//   Q4     [n][k/2] bytes, one fp32 scale per 32 codes; byte j of a block
//          holds code j in its low nibble and code j+16 in its high nibble,
//          each offset by 8 (Quant.hpp:540-549)
//
// gemv_kernel serves up to 8 rows of a (decode, small batches): it is bound
// by the weight bytes, so every lane streams 16-byte pieces of a weight row
// (4, 8, 16 or 32 weights), one wave owns GEMV_ROWS weight rows and keeps an
// fp32 accumulator per (weight row, a row), and a shuffle tree reduces the
// lanes. Up to GEMM_MIN_M - 1 rows of a run as blocks of 8 along grid.y;
// more rows take split_a_kernel and gemm_dma_kernel on MFMA, or gemm_kernel
// where k is not whole 32-wide steps (128 for Q8 and Q4).
#include <type_traits>
#include "context.hpp"
#include "device.hpp"
#include "gemv.hpp"
#include "kernels.hpp"

namespace aigpu {

namespace {

constexpr int GEMV_ROWS = 2;   // weight rows per wave
constexpr int GEMV_MAX_M = 8;  // rows of a per launch block
constexpr uint32_t GEMM_MIN_M = 16;   // from here on the MFMA GEMM

template <int TYPE, int M>
__global__ __launch_bounds__(256) void gemv_kernel(GemvParams p) {
    constexpr int E = piece_elems<TYPE>();
    const int lane = threadIdx.x & 63;
    const uint32_t row0 = (blockIdx.x * 4 + (threadIdx.x >> 6)) * GEMV_ROWS;
    if (row0 >= p.n) return;   // whole wave leaves; no block barriers below
    const uint32_t m0 = blockIdx.y * M;
    const uint32_t pieces = p.k / E;
    const size_t rowBytes = size_t(p.k) * row_bytes_per_k_x2<TYPE>() / 2;
    const uint32_t blocks = p.k / 32;

    const char* wrow[GEMV_ROWS];
    const float* srow[GEMV_ROWS];
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r) {
        const uint32_t rr = row0 + r < p.n ? row0 + r : p.n - 1;
        wrow[r] = static_cast<const char*>(p.w) + rr * rowBytes;
        srow[r] = TYPE >= 2 ? p.scales + size_t(rr) * blocks : nullptr;
    }
    float acc[GEMV_ROWS][M];
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r)
#pragma unroll
        for (int i = 0; i < M; ++i) acc[r][i] = 0.0f;

#pragma unroll 2
    for (uint32_t c = lane; c < pieces; c += WAVE) {
        u32x4 wv[GEMV_ROWS];
#pragma unroll
        for (int r = 0; r < GEMV_ROWS; ++r) wv[r] = *reinterpret_cast<const u32x4*>(wrow[r] + size_t(c) * 16);
        float sc[GEMV_ROWS];
#pragma unroll
        for (int r = 0; r < GEMV_ROWS; ++r) sc[r] = TYPE == 2 ? srow[r][c >> 1] : (TYPE == 3 ? srow[r][c] : 1.0f);
#pragma unroll
        for (int i = 0; i < M; ++i) {
            if (m0 + i < p.m) {
                const float* x = p.a + size_t(m0 + i) * p.k + size_t(c) * E;
#pragma unroll
                for (int r = 0; r < GEMV_ROWS; ++r) {
                    const float d = piece_dot<TYPE>(wv[r], x);
                    acc[r][i] = TYPE >= 2 ? fmaf(d, sc[r], acc[r][i]) : acc[r][i] + d;
                }
            }
        }
    }
#pragma unroll
    for (int r = 0; r < GEMV_ROWS; ++r)
#pragma unroll
        for (int i = 0; i < M; ++i) acc[r][i] = wave_sum(acc[r][i]);
    if (lane == 0) {
#pragma unroll
        for (int r = 0; r < GEMV_ROWS; ++r) {
            const uint32_t n = row0 + r;
            if (n >= p.n) continue;
            const float b = p.bias ? p.bias[n] : 0.0f;
#pragma unroll
            for (int i = 0; i < M; ++i) {
                if (m0 + i >= p.m) continue;
                float* o = p.out + size_t(m0 + i) * p.ldo + n;
                *o = (p.accumulate ? *o : 0.0f) + acc[r][i] + b;
            }
        }
    }
}

/*
    gemm_kernel: many rows of a (prefill), on v_mfma_f32_16x16x32_bf16, for
    the shapes gemm_dma_kernel does not take.
    A stays fp32 at the boundary; each value is split into a bf16 high part
    and the bf16 residual, and hi.B + lo.B keeps about 16 bits of it. BF16
    weights and the Q8/Q4 codes are exact in bf16; fp32 weights are split
    the same way (a third product, hi_a.lo_w). For Q8/Q4 one 32-wide K step
    is one scale block, so each step's products go through a scratch
    accumulator and are added in times the column's block scale.
    Tile 128 x 128 x 32 over four waves of 64 x 64 (4 x 4 MFMA tiles); the
    next K step is loaded into registers while the current one computes.
    LDS rows are padded to 40 bf16 (80 bytes), so the 16 lanes of each 16-byte
    operand read land on distinct banks.
*/
constexpr int GM_BM = 128, GM_BN = 128, GM_BK = 32, GM_AS = GM_BK + 8;
constexpr int GM_OP = GM_BM * GM_AS;   // bf16 elements of one operand buffer

template <int TYPE>
__global__ __launch_bounds__(256) void gemm_kernel(GemvParams p, uint32_t kSlice) {
    constexpr bool SPLIT_W = TYPE == 0, QUANT = TYPE >= 2;
    __shared__ __align__(16) __bf16 smem[(SPLIT_W ? 4 : 3) * GM_OP];   // Ah, Al, Bh (, Bl)
    __bf16* const Ah = smem;
    __bf16* const Al = smem + GM_OP;
    __bf16* const Bh = smem + 2 * GM_OP;
    __bf16* const Bl = smem + 3 * GM_OP;   // SPLIT_W only
    __shared__ float Sc[QUANT ? GM_BN : 1];

    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6, wm = w >> 1, wn = w & 1;
    const uint32_t m0 = blockIdx.y * GM_BM, n0 = blockIdx.x * GM_BN;
    const uint32_t K = p.k, M = p.m, N = p.n;
    const int srow = tid >> 1, shalf = tid & 1;   // staging: row and 16-element half of the K step

    floatx4 acc[4][4];
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};

    floatx4 ra[4];                   // a: 16 floats
    u32x4 rw[SPLIT_W ? 4 : 2];       // w: 16 fp32 / 16 bf16 / 16 Q8 codes / a Q4 block
    float rs = 0.0f;
    auto load = [&](uint32_t k0) {
        const uint32_t gm = m0 + srow, kk = k0 + 16 * shalf;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            ra[e] = (gm < M && kk + 4 * e < K) ? *reinterpret_cast<const floatx4*>(p.a + size_t(gm) * K + kk + 4 * e)
                                               : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        const uint32_t gn = n0 + srow;
        if constexpr (TYPE == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e)
                rw[e] = (gn < N && kk + 4 * e < K)
                            ? *reinterpret_cast<const u32x4*>(static_cast<const float*>(p.w) + size_t(gn) * K + kk + 4 * e)
                            : u32x4{0u, 0u, 0u, 0u};
        } else if constexpr (TYPE == 1) {
#pragma unroll
            for (int e = 0; e < 2; ++e)
                rw[e] = (gn < N && kk + 8 * e < K)
                            ? *reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.w) + size_t(gn) * K + kk + 8 * e)
                            : u32x4{0u, 0u, 0u, 0u};
        } else if constexpr (TYPE == 2) {
            rw[0] = gn < N ? *reinterpret_cast<const u32x4*>(static_cast<const int8_t*>(p.w) + size_t(gn) * K + kk)
                           : u32x4{0u, 0u, 0u, 0u};
        } else {
            // a Q4 block is 16 bytes: threads 0..127 take one row's block each
            const uint32_t qn = n0 + uint32_t(tid & 127);
            rw[0] = (tid < 128 && qn < N)
                        ? *reinterpret_cast<const u32x4*>(static_cast<const uint8_t*>(p.w) + size_t(qn) * (K / 2) + k0 / 2)
                        : u32x4{0x88888888u, 0x88888888u, 0x88888888u, 0x88888888u};
        }
        if constexpr (QUANT) rs = (tid < 128 && n0 + tid < N) ? p.scales[size_t(n0 + tid) * (K / 32) + k0 / 32] : 0.0f;
    };
    auto split_store = [&](__bf16* hi, __bf16* lo, const float (&x)[16]) {
        bf16x8 h0, h1, l0, l1;
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            h0[e] = __bf16(x[e]);
            h1[e] = __bf16(x[8 + e]);
            l0[e] = __bf16(x[e] - float(h0[e]));
            l1[e] = __bf16(x[8 + e] - float(h1[e]));
        }
        *reinterpret_cast<bf16x8*>(hi) = h0;
        *reinterpret_cast<bf16x8*>(hi + 8) = h1;
        *reinterpret_cast<bf16x8*>(lo) = l0;
        *reinterpret_cast<bf16x8*>(lo + 8) = l1;
    };
    auto store = [&]() {
        float x[16];
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int c = 0; c < 4; ++c) x[4 * e + c] = ra[e][c];
        split_store(&Ah[srow * GM_AS + 16 * shalf], &Al[srow * GM_AS + 16 * shalf], x);
        if constexpr (TYPE == 0) {
            float y[16];
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int c = 0; c < 4; ++c) y[4 * e + c] = __uint_as_float(rw[e][c]);
            split_store(&Bh[srow * GM_AS + 16 * shalf], &Bl[srow * GM_AS + 16 * shalf], y);
        } else if constexpr (TYPE == 1) {
            *reinterpret_cast<u32x4*>(&Bh[srow * GM_AS + 16 * shalf]) = rw[0];
            *reinterpret_cast<u32x4*>(&Bh[srow * GM_AS + 16 * shalf + 8]) = rw[1];
        } else if constexpr (TYPE == 2) {
            bf16x8 b0, b1;
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int j = 0; j < 4; ++j) {
                    const float c = float(int32_t(rw[0][e] << (24 - 8 * j)) >> 24);
                    if (e < 2) b0[4 * e + j] = __bf16(c);
                    else b1[4 * (e - 2) + j] = __bf16(c);
                }
            *reinterpret_cast<bf16x8*>(&Bh[srow * GM_AS + 16 * shalf]) = b0;
            *reinterpret_cast<bf16x8*>(&Bh[srow * GM_AS + 16 * shalf + 8]) = b1;
        } else {
            if (tid < 128) {
                __bf16* row = &Bh[tid * GM_AS];
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    bf16x8 lo4, hi4;   // codes 4e..4e+3 and 16+4e..16+4e+3, two bytes at a time
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        const uint32_t byte = (rw[0][e] >> (8 * j)) & 0xFFu;
                        lo4[j] = __bf16(float(int(byte & 0xFu) - 8));
                        hi4[j] = __bf16(float(int(byte >> 4) - 8));
                    }
#pragma unroll
                    for (int j = 0; j < 4; ++j) {
                        row[4 * e + j] = lo4[j];
                        row[16 + 4 * e + j] = hi4[j];
                    }
                }
            }
        }
        if constexpr (QUANT)
            if (tid < 128) Sc[tid] = rs;
    };

    // split K: slice blockIdx.z of kSlice (a multiple of GM_BK) columns
    const uint32_t kBegin = blockIdx.z * kSlice, kEnd = kBegin + kSlice < K ? kBegin + kSlice : K;
    load(kBegin);
    for (uint32_t k0 = kBegin; k0 < kEnd; k0 += GM_BK) {
        __syncthreads();   // the previous step's operand reads are done
        store();
        __syncthreads();
        if (k0 + GM_BK < kEnd) load(k0 + GM_BK);
        bf16x8 ah[4], al[4], bh[4], bl[4];
        const int fr = lane & 15, fk = 8 * (lane >> 4);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            ah[i] = *reinterpret_cast<const bf16x8*>(&Ah[(64 * wm + 16 * i + fr) * GM_AS + fk]);
            al[i] = *reinterpret_cast<const bf16x8*>(&Al[(64 * wm + 16 * i + fr) * GM_AS + fk]);
            bh[i] = *reinterpret_cast<const bf16x8*>(&Bh[(64 * wn + 16 * i + fr) * GM_AS + fk]);
            if constexpr (SPLIT_W) bl[i] = *reinterpret_cast<const bf16x8*>(&Bl[(64 * wn + 16 * i + fr) * GM_AS + fk]);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i)
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                if constexpr (QUANT) {
                    floatx4 t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh[j], floatx4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh[j], t, 0, 0, 0);
                    const float sc = Sc[64 * wn + 16 * j + fr];
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(sc, t[r], acc[i][j][r]);
                } else {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bh[j], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al[i], bh[j], acc[i][j], 0, 0, 0);
                    if constexpr (SPLIT_W) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah[i], bl[j], acc[i][j], 0, 0, 0);
                }
            }
    }
    // the accumulator layout: lane holds rows 4 (lane / 16) + r of column lane % 16
#pragma unroll
    for (int i = 0; i < 4; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            const uint32_t n = n0 + 64 * wn + 16 * j + (lane & 15);
            if (n >= N) continue;
            const float b = p.bias ? p.bias[n] : 0.0f;
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t m = m0 + 64 * wm + 16 * i + 4 * (lane >> 4) + r;
                if (m >= M) continue;
                // a K slice writes its own partial tile (no bias, no accumulate)
                float* o = p.out + size_t(blockIdx.z) * M * p.ldo + size_t(m) * p.ldo + n;
                *o = (p.accumulate ? *o : 0.0f) + acc[i][j][r] + b;
            }
        }
}

/*
    gemm_dma_kernel: the MFMA GEMM of every aligned shape (K whole steps of
    32; whole groups of four for Q8 and Q4), after split_a_kernel has split a
    into bf16 high parts and residuals ([M][K] each). Every operand comes in
    by DMA (global_load_lds, 1 KB blocks) into a three-stage LDS ring, step
    t + 2 issued between step t's MFMAs, so nothing passes through registers
    or the VALU on its way in and each step's loads have two steps of compute
    to land; one barrier per step. 2 x WN waves of BM/2 x BN/WN outputs, two
    waves on a SIMD wherever the tile allows, so that one's operand reads
    after the barrier hide behind the other's MFMAs (256 x 256 tiles: 450 us
    with eight waves, 453 with four at 8192 x 4096 -> 4096, 170 and 187 on a
    cool chip at 500 rows; reading the next step's operands before the last
    row tile instead measured 20% slower). It is bound by the MFMA rate at the
    clock the chip holds: 1999 x 4096 -> 4096 in bf16, 128 x 256 tiles, 127 us
    (gemm_kernel, which splits a in registers and stores it to LDS behind two
    barriers a step: 190); Q8 500 x 4096 -> 12288, the whole call with the
    split of a, 140 us (217; this kernel alone 151-155 under the tracer).
      BF16  up to 256 x 256 tiles
      F32   w in fp32 in LDS, split on its way into the operand registers
            (a third product, hi_a.lo_w)
      Q8/Q4 the codes in LDS as stored, widened to bf16 (exactly) on their
            way into the operand registers; one 32-wide step is one scale
            block: its products go through a scratch accumulator and are
            added in times the column's scale. The scales come in by DMA too,
            four steps at a time.
    In LDS, a 1 KB block of bf16 is 16 rows of 64 bytes; row r keeps its
    16-byte chunk c at position c ^ s(r % 16), s(x) = ((x / 2) % 4) ^ (x / 8):
    the 16 rows of an operand read fall on distinct banks both as one
    256-byte access and as two 128-byte halves. A block of fp32 is 8 rows of
    128 bytes, chunk c at c ^ ((r / 2) % 8), for the same reason; Q8 (32 rows
    of 32 bytes) and Q4 (64 rows of 16) need no swizzle.
*/
constexpr int GD_BK = 32, GD_STAGES = 3;

__global__ __launch_bounds__(256) void split_a_kernel(const float* a, bf16x8* hi, bf16x8* lo, uint64_t pieces) {
    for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < pieces; i += uint64_t(gridDim.x) * 256) {
        const floatx4 x0 = reinterpret_cast<const floatx4*>(a)[2 * i];
        const floatx4 x1 = reinterpret_cast<const floatx4*>(a)[2 * i + 1];
        bf16x8 h, l;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
            h[t] = __bf16(x0[t]);
            l[t] = __bf16(x0[t] - float(h[t]));
            h[4 + t] = __bf16(x1[t]);
            l[4 + t] = __bf16(x1[t] - float(h[4 + t]));
        }
        hi[i] = h;
        lo[i] = l;
    }
}

/* s_waitcnt vmcnt(N) alone (N < 64) */
template <int N>
__device__ __forceinline__ void gd_wait_vmcnt() {
    static_assert(N >= 0 && N < 64, "vmcnt is 6 bits");
    __builtin_amdgcn_s_waitcnt((N & 15) | (7 << 4) | (15 << 8) | ((N >> 4) << 14));
}

/* up to three weights over the same rows of a share a launch: segment s has
   the tile columns from `start` (in columns, a multiple of the tile's) on */
constexpr int GD_SEGS = 3;
struct GemmSeg {
    const void* w;
    const float *scales, *bias;
    float* out;
    uint32_t n, ldo, start;
};
struct GemmArgs {
    const __bf16 *ahi, *alo;
    GemmSeg seg[GD_SEGS];
    uint32_t nseg, m, k, accumulate;
    uint32_t columns;      // of all segments, each padded to whole tiles
    uint32_t sliceSteps;   // K steps per slice (blockIdx.y)
    float* part;           // with K slices: their partial tiles, [slice][m][columns]
};

__device__ __forceinline__ int segment_of(const GemmArgs& a, uint32_t n) {
    int s = 0;
#pragma unroll
    for (int i = 1; i < GD_SEGS; ++i)
        if (uint32_t(i) < a.nseg && n >= a.seg[i].start) s = i;
    return s;
}

template <int TYPE> constexpr int gd_row_bytes() { return TYPE == 0 ? 128 : (TYPE == 1 ? 64 : (TYPE == 2 ? 32 : 16)); }
template <int TYPE, int BM, int BN> constexpr int gd_stage() { return 2 * BM * 64 + BN * gd_row_bytes<TYPE>(); }
/* eight Q8 codes to bf16, exactly */
__device__ __forceinline__ bf16x8 widen_q8(u32x2 c) {
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = __bf16(float(int32_t(c[e / 4] << (24 - 8 * (e % 4))) >> 24));
    return r;
}
/* the low nibbles of eight bytes, less 8, to bf16, exactly */
__device__ __forceinline__ bf16x8 widen_q4(u32x2 c) {
    bf16x8 r;
#pragma unroll
    for (int e = 0; e < 8; ++e) r[e] = __bf16(float((c[e / 4] >> (8 * (e % 4))) & 0xFu) - 8.0f);
    return r;
}

template <int TYPE, int BM, int BN, int WN>
__global__ __launch_bounds__(128 * WN, 2) void gemm_dma_kernel(GemmArgs a) {
    constexpr bool QUANT = TYPE >= 2;
    constexpr int W = 2 * WN;                           // waves, 2 x WN
    constexpr int TI = BM / 32, TJ = BN / WN / 16;     // 16 x 16 tiles of a wave's BM/2 x BN/WN
    constexpr int AOP = BM * 64;                        // bytes of one image of a per step
    constexpr int RB = gd_row_bytes<TYPE>();            // bytes of a w row per step
    constexpr int BROWS = 1024 / RB;                    // w rows per DMA block
    constexpr int STAGE = gd_stage<TYPE, BM, BN>();
    constexpr int AJ = BM / 16 / W;                       // DMA blocks of one image of a per wave and step
    constexpr int BJ = BN / BROWS >= W ? BN / BROWS / W : 1;   // of w (fewer blocks than waves: some are loaded twice)
    constexpr int NB = 2 * AJ + BJ;
    __shared__ __align__(16) uint8_t smem[GD_STAGES * STAGE + (QUANT ? 2 * BN * 16 : 0)];
    const int tid = threadIdx.x, lane = tid & 63, wm = (tid >> 6) / WN, wn = (tid >> 6) % WN;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);   // uniform: DMA targets are scalar
    const uint32_t K = a.k, M = a.m;
    const uint32_t ntM = (M + BM - 1) / BM, ntN = a.columns / BN;
    // consecutive workgroups go to different XCDs: remap them so that each XCD
    // takes a run of tiles, when they split evenly over the eight; runs go
    // down four tile rows before the next tile column, so that the tiles an
    // XCD holds at once share both their rows of a and their rows of w in its L2
    uint32_t lg = blockIdx.x;
    if (gridDim.x % 8 == 0) lg = (lg % 8) * (gridDim.x / 8) + lg / 8;
    const uint32_t band = lg / (4 * ntN), inBand = lg % (4 * ntN);
    const uint32_t bandRows = ntM - 4 * band < 4 ? ntM - 4 * band : 4;
    const uint32_t m0 = (4 * band + inBand % bandRows) * BM, n0 = (inBand / bandRows) * BN;
    const uint32_t ldsBase = lds_address(smem);
    const uint32_t kBegin = blockIdx.y * a.sliceSteps;
    const uint32_t kSteps = K / GD_BK - kBegin < a.sliceSteps ? K / GD_BK - kBegin : a.sliceSteps;

    // this wave's DMA blocks of a step. Rows past M or N read the last row:
    // they only reach outputs past M or N, which are not stored.
    const GemmSeg& S = a.seg[segment_of(a, n0)];
    const uint32_t wn0 = n0 - S.start;
    const uint8_t* const wBase = static_cast<const uint8_t*>(S.w) + size_t(kBegin) * RB;
    const uint8_t* const hiBase = reinterpret_cast<const uint8_t*>(a.ahi) + size_t(kBegin) * 64;
    const uint8_t* const loBase = reinterpret_cast<const uint8_t*>(a.alo) + size_t(kBegin) * 64;
    const uint32_t rowStride = K / GD_BK * RB;          // bytes of a w row
    uint32_t aoff[AJ], woff[BJ];
#pragma unroll
    for (int j = 0; j < AJ; ++j) {   // lane l: row l / 4, LDS chunk l % 4, which holds chunk (l % 4) ^ s(l / 4)
        const uint32_t row = m0 + 16u * (AJ * uint32_t(w) + j) + uint32_t(lane >> 2);
        const uint32_t chunk = uint32_t(lane & 3) ^ uint32_t(((lane >> 3) & 3) ^ (lane >> 5));
        aoff[j] = ((row < M ? row : M - 1) * K + 8 * chunk) * 2;
    }
    const uint32_t wblk = BN / BROWS >= W ? uint32_t(BJ) * w : uint32_t(w) % (BN / BROWS);
#pragma unroll
    for (int j = 0; j < BJ; ++j) {
        constexpr int CPR = RB / 16;   // 16-byte chunks per row
        const uint32_t r = uint32_t(lane) / CPR, c = uint32_t(lane) % CPR;
        const uint32_t chunk = TYPE == 0 ? c ^ ((r >> 1) & 3) ^ (4 * ((wblk + j) & 1)) : (TYPE == 1 ? c ^ (((r >> 1) & 3) ^ (r >> 3)) : c);
        const uint32_t row = wn0 + (wblk + j) * BROWS + r;
        woff[j] = (row < S.n ? row : S.n - 1) * rowStride + 16 * chunk;
    }
    uint32_t soff = 0;
    const uint8_t* sBase = nullptr;
    constexpr int SB = BN / 64;   // DMA blocks of four steps' scales: 64 rows each
    const uint32_t scaleLds = ldsBase + GD_STAGES * STAGE + (w % SB) * 1024;
    if constexpr (QUANT) {
        const uint32_t row = wn0 + 64 * (w % SB) + lane;
        soff = (row < S.n ? row : S.n - 1) * (K / 8);   // K / 32 floats per row
        sBase = reinterpret_cast<const uint8_t*>(S.scales) + size_t(kBegin) * 4;
    }
    auto dma = [&](uint32_t kt, int j) __attribute__((always_inline)) {   // block j of step kt
        const uint32_t stage = ldsBase + (kt % GD_STAGES) * STAGE;
        if (j < AJ) dma_block(hiBase + size_t(kt) * 64, aoff[j], stage + (AJ * w + j) * 1024);
        else if (j < 2 * AJ) dma_block(loBase + size_t(kt) * 64, aoff[j - AJ], stage + AOP + (AJ * w + j - AJ) * 1024);
        else dma_block(wBase + size_t(kt) * RB, woff[j - 2 * AJ], stage + 2 * AOP + (wblk + j - 2 * AJ) * 1024);
    };
    auto dma_scales = [&](uint32_t group) __attribute__((always_inline)) {   // four steps' scales: [BN rows][4]
        dma_block(sBase + size_t(group) * 16, soff, scaleLds + (group & 1) * (BN * 16));
    };

    floatx4 acc[TI][TJ];
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
        for (int j = 0; j < TJ; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    const int g = lane >> 4, fr = lane & 15, sw = 16 * (g ^ ((fr >> 1) & 3) ^ (fr >> 3));   // swizzled chunk of k 8 g ..
    if constexpr (QUANT) dma_scales(0);
#pragma unroll
    for (int j = 0; j < NB; ++j) dma(0, j);
    if (kSteps > 1) {
#pragma unroll
        for (int j = 0; j < NB; ++j) dma(1, j);
    }
    // step kt; MORE: step kt + 2's DMA goes out between its row tiles, and step
    // 1 of a group of four also requests the next group's scales (Q8, Q4)
    auto step = [&](uint32_t kt, auto MORE) __attribute__((always_inline)) {
        constexpr bool more = decltype(MORE)::value;
        // step kt's blocks have landed (in order: step kt + 1's, and the
        // scales requested with them, may still be in flight); after the
        // barrier every wave's have, and every read of the stage step kt + 2
        // goes into (that of step kt - 1) is done. Not __syncthreads(): its
        // fence would wait for step kt + 1's blocks too.
        if (QUANT && kt % 4 == 2 && kt + 2 < kSteps) gd_wait_vmcnt<NB + 1>();
        else if (kt + 1 < kSteps) gd_wait_vmcnt<NB>();
        else gd_wait_vmcnt<0>();
        lds_barrier();
        const uint8_t* st = smem + (kt % GD_STAGES) * STAGE;
        if (QUANT && more && kt % 4 == 1 && kt + 3 < kSteps) dma_scales(kt / 4 + 1);
        const int bw = BN / WN * wn;   // the wave's first column
        bf16x8 bh[TJ], bl[TYPE == 0 ? TJ : 1];
        float sc[QUANT ? TJ : 1];
#pragma unroll
        for (int j = 0; j < TJ; ++j) {
            const int row = bw + 16 * j + fr;
            const uint8_t* br = st + 2 * AOP + row * RB;
            if constexpr (TYPE == 1) {
                bh[j] = *reinterpret_cast<const bf16x8*>(br + sw);
            } else if constexpr (TYPE == 0) {
                const int x = (row >> 1) & 7;   // chunks 2 g and 2 g + 1
                const floatx4 x0 = *reinterpret_cast<const floatx4*>(br + 16 * ((2 * g) ^ x));
                const floatx4 x1 = *reinterpret_cast<const floatx4*>(br + 16 * ((2 * g + 1) ^ x));
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    bh[j][e] = __bf16(x0[e]);
                    bl[j][e] = __bf16(x0[e] - float(bh[j][e]));
                    bh[j][4 + e] = __bf16(x1[e]);
                    bl[j][4 + e] = __bf16(x1[e] - float(bh[j][4 + e]));
                }
            } else if constexpr (TYPE == 2) {
                bh[j] = widen_q8(*reinterpret_cast<const u32x2*>(br + 8 * g));
            } else {   // byte t of a block: code t low, code t + 16 high
                const u32x2 c = *reinterpret_cast<const u32x2*>(br + 8 * (g & 1));
                bh[j] = widen_q4(u32x2{c[0] >> (4 * (g >> 1)), c[1] >> (4 * (g >> 1))});
            }
            if constexpr (QUANT)
                sc[j] = *reinterpret_cast<const float*>(smem + GD_STAGES * STAGE + ((kt / 4) & 1) * (BN * 16) + row * 16 + 4 * (kt % 4));
        }
        const int ro = (BM / 2 * wm + fr) * 64 + sw;
        bf16x8 ah = *reinterpret_cast<const bf16x8*>(st + ro);
        bf16x8 al = *reinterpret_cast<const bf16x8*>(st + AOP + ro);
#pragma unroll
        for (int i = 0; i < TI; ++i) {   // row tile i + 1's a operands are read while tile i computes
            bf16x8 nh = ah, nl = al;
            if (i + 1 < TI) {
                nh = *reinterpret_cast<const bf16x8*>(st + ro + (i + 1) * 1024);
                nl = *reinterpret_cast<const bf16x8*>(st + AOP + ro + (i + 1) * 1024);
            }
            if constexpr (more) {   // the NB blocks spread over the TI row tiles
#pragma unroll
                for (int b = i * NB / TI; b < (i + 1) * NB / TI; ++b) dma(kt + 2, b);
            }
#pragma unroll
            for (int j = 0; j < TJ; ++j) {
                if constexpr (QUANT) {
                    floatx4 t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[j], floatx4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
                    t = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[j], t, 0, 0, 0);
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][r] = fmaf(sc[j], t[r], acc[i][j][r]);
                } else {
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bh[j], acc[i][j], 0, 0, 0);
                    acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(al, bh[j], acc[i][j], 0, 0, 0);
                    if constexpr (TYPE == 0) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(ah, bl[j], acc[i][j], 0, 0, 0);
                }
            }
            ah = nh;
            al = nl;
        }
    };
    uint32_t kt = 0;
    for (; kt + 2 < kSteps; ++kt) step(kt, std::bool_constant<true>{});
    for (; kt < kSteps; ++kt) step(kt, std::bool_constant<false>{});
    // the accumulator layout: lane holds rows 4 (lane / 16) + r of column lane % 16
    float* const out = a.part ? a.part + size_t(blockIdx.y) * M * a.columns + n0 : S.out + wn0;
    const uint32_t ldo = a.part ? a.columns : S.ldo;
    const bool add = a.accumulate && !a.part;   // a K slice: its own partial (no bias, no accumulate)
#pragma unroll
    for (int j = 0; j < TJ; ++j) {
        const uint32_t c = BN / WN * wn + 16 * j + fr;
        if (wn0 + c >= S.n) continue;
        const float b = S.bias && !a.part ? S.bias[wn0 + c] : 0.0f;
#pragma unroll
        for (int i = 0; i < TI; ++i)
#pragma unroll
            for (int r = 0; r < 4; ++r) {
                const uint32_t m = m0 + BM / 2 * wm + 16 * i + 4 * g + r;
                if (m >= M) continue;
                float* o = out + size_t(m) * ldo + c;
                *o = (add ? *o : 0.0f) + acc[i][j][r] + b;
            }
    }
}

/* the K slices' partial tiles added in slice order, then the bias and the
   accumulate */
__global__ __launch_bounds__(256) void gemm_reduce_kernel(GemmArgs a, uint32_t slices) {
    const uint64_t quads = uint64_t(a.m) * a.columns / 4, slice = uint64_t(a.m) * a.columns;
    for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < quads; i += uint64_t(gridDim.x) * 256) {
        const uint32_t m = uint32_t(4 * i / a.columns), n = uint32_t(4 * i % a.columns);
        const GemmSeg& S = a.seg[segment_of(a, n)];
        const uint32_t c = n - S.start;
        if (c >= S.n) continue;
        floatx4 v = {0.0f, 0.0f, 0.0f, 0.0f};   // columns past n were not written: not used below
        for (uint32_t sl = 0; sl < slices; ++sl) {
            const floatx4 x = *reinterpret_cast<const floatx4*>(a.part + sl * slice + 4 * i);
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] += x[e];
        }
        float* o = S.out + size_t(m) * S.ldo + c;
#pragma unroll
        for (int e = 0; e < 4; ++e)
            if (c + e < S.n) o[e] = (a.accumulate ? o[e] : 0.0f) + v[e] + (S.bias ? S.bias[c + e] : 0.0f);
    }
}

/* The k and v projections' per-token work after one GEMM over both
   (kv[m][0 .. N1) k, [N1 .. 2 N1) v, fp32): the bias, then for k RMSNorm
   (gamma) and rotate-half RoPE (freqs) as norm_rope_row does them, and each
   row appended to its bf16 cache and to the flash kernel's fp16 copy (the
   rows the prep kernel would write). One workgroup per token: the token's
   rotation angles float(pos) * freq go through sincosf
   once into LDS, then the four waves take its 2 * heads rows (k and v of
   each kv head) in turn, a row staged in LDS for the RoPE partner. A lane
   holds D / 64 consecutive elements. With rope set, the angles' cos and sin
   also go to the flash kernel's table (rope_at);
   with padK / padV set, workgroup 0 zeroes pad16 16-byte pieces of each
   (the working copies' pad rows). */
__global__ __launch_bounds__(256) void kv_epilogue_kernel(const float* kv, const float* kBias, const float* vBias,
                                                          KvEpilogue ek, KvEpilogue ev, uint32_t heads, float* rope,
                                                          uint4* padK, uint4* padV, uint32_t pad16) {
    __shared__ float row[4][128];
    __shared__ float sinT[64], cosT[64];
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const uint32_t t = blockIdx.x, pos = ek.start + t;
    const uint32_t half = ek.freqs ? ek.rot / 2 : 0;   // rot <= D <= 128
    if (w == 0 && uint32_t(lane) < half) {
        float sn, cs;
        sincosf(float(pos) * ek.freqs[lane], &sn, &cs);
        sinT[lane] = sn;
        cosT[lane] = cs;
        if (rope) {
            rope[rope_at(t, 0, uint32_t(lane), half, gridDim.x)] = cs;
            rope[rope_at(t, 1, uint32_t(lane), half, gridDim.x)] = sn;
        }
    }
    if (padK && t == 0)
        for (uint32_t i = threadIdx.x; i < pad16; i += 256) {
            padK[i] = uint4{0u, 0u, 0u, 0u};
            padV[i] = uint4{0u, 0u, 0u, 0u};
        }
    __syncthreads();
    const uint32_t D = ek.dim, N1 = heads * D, EPL = D / 64;   // D 64 or 128
    const uint32_t d0 = uint32_t(lane) * EPL;
    for (uint32_t r = uint32_t(w); r < 2 * heads; r += 4) {
        const uint32_t which = r & 1, h = r >> 1;
        const KvEpilogue& e = which ? ev : ek;
        const float* bias = which ? vBias : kBias;
        const float* src = kv + (size_t(t) * 2 + which) * N1 + size_t(h) * D + d0;
        float x[2] = {0.0f, 0.0f};
        if (EPL == 2) {
            const float2 v2 = *reinterpret_cast<const float2*>(src);   // kv rows are 8-byte aligned
            x[0] = v2.x;
            x[1] = v2.y;
        } else {
            x[0] = src[0];
        }
        float ss = 0.0f;
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            if (bias && uint32_t(i) < EPL) x[i] += bias[size_t(h) * D + d0 + i];
            ss = fmaf(x[i], x[i], ss);
        }
        float inv = 1.0f;
        if (e.gamma) inv = 1.0f / sqrtf(wave_sum(ss) / float(D) + e.eps);
        float y[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            y[i] = e.gamma && uint32_t(i) < EPL ? x[i] * inv * (e.gamma[d0 + i] + e.offset) : x[i];
            if (uint32_t(i) < EPL) row[w][d0 + i] = y[i];
        }
        wave_sync();
        const uint32_t hf = e.freqs ? half : 0;
        bool bad = false;
        uint16_t cb[2];
        _Float16 wb[2];
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            const uint32_t d = d0 + i;
            float v = y[i];
            if (d < 2 * hf) {   // rotate-half pairs (LocalModel.hpp:2624-2641)
                const bool low = d < hf;
                const uint32_t j = low ? d : d - hf, dp = low ? d + hf : d - hf;
                v = low ? y[i] * cosT[j] - row[w][dp] * sinT[j] : y[i] * cosT[j] + row[w][dp] * sinT[j];
            }
            cb[i] = float_to_bf16_bits(v);
            wb[i] = to_f16_checked(v, bad);
        }
        uint16_t* cdst = e.cache + (size_t(h) * e.capacity + pos) * D + d0;
        _Float16* wdst = static_cast<_Float16*>(e.work) + (size_t(h) * e.T + pos) * D + d0;
        if (EPL == 2) {   // 4-byte stores: rows are 16-byte aligned, d0 even
            *reinterpret_cast<uint32_t*>(cdst) = uint32_t(cb[0]) | (uint32_t(cb[1]) << 16);
            _Float16 __attribute__((ext_vector_type(2))) w2 = {wb[0], wb[1]};
            *reinterpret_cast<decltype(w2)*>(wdst) = w2;
        } else {
            cdst[0] = cb[0];
            wdst[0] = wb[0];
        }
        raise_range_flag(e.rangeFlag, bad);
        wave_sync();   // the row's partner reads are done before the next row is staged
    }
}

/* the K slices' partial tiles added in slice order, then the bias and the
   accumulate: out[m][n] (+)= sum_s part[s][m][n] + bias[n] */
__global__ __launch_bounds__(256) void split_reduce_kernel(GemvParams p, const float* part, uint32_t slices) {
    const uint64_t outs = uint64_t(p.m) * p.n;
    for (uint64_t i = uint64_t(blockIdx.x) * 256 + threadIdx.x; i < outs; i += uint64_t(gridDim.x) * 256) {
        float v = 0.0f;
        for (uint32_t sl = 0; sl < slices; ++sl) v += part[uint64_t(sl) * outs + i];
        const uint32_t m = uint32_t(i / p.n), n = uint32_t(i % p.n);
        float* o = p.out + size_t(m) * p.ldo + n;
        *o = (p.accumulate ? *o : 0.0f) + v + (p.bias ? p.bias[n] : 0.0f);
    }
}

/* any k for F32 and BF16 (rows not on 16-byte boundaries): one wave per
   weight row and a row of a, element by element */
template <int TYPE>
__global__ __launch_bounds__(256) void gemv_scalar_kernel(GemvParams p) {
    const int lane = threadIdx.x & 63;
    const uint64_t task = uint64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (task >= uint64_t(p.n) * p.m) return;
    const uint32_t n = uint32_t(task % p.n), i = uint32_t(task / p.n);
    const float* x = p.a + size_t(i) * p.k;
    float s = 0.0f;
    for (uint32_t t = lane; t < p.k; t += WAVE) {
        const float wv = TYPE == 0 ? static_cast<const float*>(p.w)[size_t(n) * p.k + t]
                                   : bf16_bits_to_float(static_cast<const uint16_t*>(p.w)[size_t(n) * p.k + t]);
        s = fmaf(x[t], wv, s);
    }
    s = wave_sum(s);
    if (lane == 0) {
        float* o = p.out + size_t(i) * p.ldo + n;
        *o = (p.accumulate ? *o : 0.0f) + s + (p.bias ? p.bias[n] : 0.0f);
    }
}

constexpr uint32_t CUS = 256;

/* shapes gemm_dma_kernel takes: K in whole steps (of four for Q8 and Q4, whose
   scales come in four at a time), 16-byte aligned rows, 32-bit byte offsets */
bool dma_eligible(const GemvParams& p) {
    auto aligned = [](const void* ptr) { return (reinterpret_cast<uintptr_t>(ptr) % 16) == 0; };
    if (p.m < GEMM_MIN_M || p.k == 0 || p.k % (p.type >= 2 ? 4 * GD_BK : GD_BK) || !aligned(p.w) || !aligned(p.a) ||
        (p.type >= 2 && !aligned(p.scales)))
        return false;
    const uint64_t rowBytes = uint64_t(p.k) / GD_BK * (p.type == 0 ? 128 : (p.type == 1 ? 64 : (p.type == 2 ? 32 : 16)));
    return uint64_t(p.m) * p.k * 2 < (1ull << 32) && uint64_t(p.n) * rowBytes < (1ull << 32) && p.m <= 0x7FFFFFFFu / 2;
}

struct GemmPlan {
    int bm, bn;
    uint32_t tiles, slices, sliceSteps, columns;
};

/* The tile and the number of K slices by estimated time, from what each tile
   costs per 32-wide K step (microseconds, measured at k = 4096, m 16 to 8192,
   n 2048 to 12288): `alone` on its CU with the others idle, `shared` for each
   of several on one CU, or with every CU busy (the clock falls, L2 fills up).
   Small tiles and K slices win while the tiles of one shape do not fill 256
   CUs (m = 500, k = n = 4096, bf16: 256 x 256 tiles 169 us, 128 x 128 71, two
   K slices 57), large ones by their reuse when they do (m = 8192: 450, 128 x
   256 502, 128 x 128 557). Slices cost their partial tiles' round trip. */
struct TileCost {
    int type, bm, bn, resident;   // workgroups of this tile a CU's LDS holds
    float alone, shared;
};
constexpr TileCost TILE_COSTS[] = {
    {0, 128, 256, 1, 1.22f, 1.43f}, {0, 128, 128, 1, 0.68f, 0.80f}, {0, 64, 128, 2, 0.62f, 0.55f},
    {1, 256, 256, 1, 1.26f, 1.66f}, {1, 128, 256, 1, 0.77f, 0.93f}, {1, 128, 128, 2, 0.49f, 0.51f}, {1, 64, 128, 3, 0.30f, 0.31f},
    {2, 128, 256, 1, 0.98f, 1.10f}, {2, 128, 128, 2, 0.72f, 0.58f}, {2, 64, 128, 3, 0.53f, 0.39f},
    {3, 128, 128, 2, 0.82f, 0.64f}, {3, 64, 128, 4, 0.62f, 0.46f},
};

GemmPlan plan_gemm(const GemvParams* ps, int count) {
    const GemvParams& p = ps[0];
    GemmPlan best{};
    float bestCost = 0.0f;
    const uint32_t steps = p.k / GD_BK, group = p.type >= 2 ? 4 : 1;
    for (const TileCost& t : TILE_COSTS) {
        if (t.type != p.type) continue;
        uint64_t columns = 0;
        for (int i = 0; i < count; ++i) columns += (ps[i].n + t.bn - 1) / t.bn;
        const uint64_t tiles = uint64_t((p.m + t.bm - 1) / t.bm) * columns;
        columns *= t.bn;
        if (tiles > 0x7FFFFFFFull || columns > 0x7FFFFFFFull) continue;
        for (uint32_t want = 1; want <= 16; want = want < 4 ? want + 1 : want + 2) {
            const uint32_t per = ((steps + want - 1) / want + group - 1) / group * group;   // whole scale groups
            if ((steps + per - 1) / per != want || (want > 1 && per < 8)) continue;
            // rounds of `resident` tiles a CU; a last round's tiles land where
            // CUs fall free, several on one while others have none
            const uint64_t items = tiles * want, round = uint64_t(CUS) * t.resident;
            const uint64_t rounds = (items + round - 1) / round, most = (items + CUS - 1) / CUS;
            const float full = items < CUS ? float(items) / CUS : 1.0f;
            const float lastFill = float(items - (rounds - 1) * round) / float(round);
            float step = t.alone + (t.shared > t.alone ? (t.shared - t.alone) * full : 0.0f);
            if (rounds == 1 && most > 1) step = fmaxf(t.alone, float(most) * t.shared);
            if (rounds > 1) step = (float(rounds - 1) + (t.resident == 1 ? 1.0f : 0.6f + 0.4f * lastFill)) * float(t.resident) * t.shared;
            float cost = step * per + 1.5f * float(rounds);
            if (want > 1) cost += 4.0f + float(want) * float(p.m) * float(columns) * 8.0f / 6e6f;
            if (best.bm == 0 || cost < bestCost) {
                best = GemmPlan{t.bm, t.bn, uint32_t(tiles), want, per, uint32_t(columns)};
                bestCost = cost;
            }
        }
    }
    return best;
}

/* the products of one a with `count` weights (same a, m, k, type and
   accumulate): a split into its bf16 high parts and residuals (scratch slot
   SLOT_GEMM_A), unless `split` says the slot already holds them, then the DMA
   GEMM. A plan with K slices writes partial tiles that gemm_reduce_kernel adds
   in order. */
bool launch_dma(Context& ctx, const GemvParams* ps, int count, bool split, hipStream_t stream) {
    const GemvParams& p = ps[0];
    const uint64_t aBytes = uint64_t(p.m) * p.k * 2;   // one bf16 image of a
    uint8_t* img = static_cast<uint8_t*>(ctx.grow(SLOT_GEMM_A, 2 * aBytes));
    if (!img) return false;
    bf16x8* hi = reinterpret_cast<bf16x8*>(img);
    bf16x8* lo = reinterpret_cast<bf16x8*>(img + aBytes);
    const GemmPlan plan = plan_gemm(ps, count);
    if (plan.bm == 0) return ctx.fail("matmul: too many tiles");
    GemmArgs a{};
    a.ahi = reinterpret_cast<const __bf16*>(hi);
    a.alo = reinterpret_cast<const __bf16*>(lo);
    uint32_t start = 0;
    for (int i = 0; i < count; ++i) {
        a.seg[i] = GemmSeg{ps[i].w, ps[i].scales, ps[i].bias, ps[i].out, ps[i].n, ps[i].ldo, start};
        start += (ps[i].n + plan.bn - 1) / plan.bn * plan.bn;
    }
    a.nseg = uint32_t(count);
    a.m = p.m;
    a.k = p.k;
    a.accumulate = p.accumulate ? 1u : 0u;
    a.columns = plan.columns;
    a.sliceSteps = plan.sliceSteps;
    if (plan.slices > 1) {
        a.part = static_cast<float*>(ctx.grow(SLOT_GEMM_SPLIT, size_t(plan.slices) * p.m * plan.columns * sizeof(float)));
        if (!a.part) return false;
    }
    if (!split) {
        const uint64_t pieces = aBytes / 16;
        const unsigned sg = unsigned((pieces + 255) / 256 < 8192 ? (pieces + 255) / 256 : 8192);
        if (!ctx.launch("split_a_kernel", stream, [&] {
                hipLaunchKernelGGL(split_a_kernel, dim3(sg), dim3(256), 0, stream, p.a, hi, lo, pieces);
            }))
            return false;
    }
    const dim3 grid(plan.tiles, plan.slices);
#define AIGPU_GD(T, BM, BN, WN)                                                                              \
    if (p.type == T && plan.bm == BM && plan.bn == BN &&                                                     \
        !ctx.launch("gemm_dma_kernel<" #T ", " #BM ", " #BN ">", stream, [&] {                               \
            hipLaunchKernelGGL((gemm_dma_kernel<T, BM, BN, WN>), grid, dim3(128 * WN), 0, stream, a);        \
        }))                                                                                                  \
        return false
    AIGPU_GD(0, 128, 256, 4);
    AIGPU_GD(0, 128, 128, 4);
    AIGPU_GD(0, 64, 128, 2);
    AIGPU_GD(1, 256, 256, 4);
    AIGPU_GD(1, 128, 256, 4);
    AIGPU_GD(1, 128, 128, 2);
    AIGPU_GD(1, 64, 128, 2);
    AIGPU_GD(2, 128, 256, 4);
    AIGPU_GD(2, 128, 128, 2);
    AIGPU_GD(2, 64, 128, 2);
    AIGPU_GD(3, 128, 128, 2);
    AIGPU_GD(3, 64, 128, 2);
#undef AIGPU_GD
    if (plan.slices == 1) return true;
    const uint64_t quads = uint64_t(p.m) * plan.columns / 4;
    const unsigned rg = unsigned((quads + 255) / 256 < 65536 ? (quads + 255) / 256 : 65536);
    return ctx.launch("gemm_reduce_kernel", stream, [&] {
        hipLaunchKernelGGL(gemm_reduce_kernel, dim3(rg), dim3(256), 0, stream, a, plan.slices);
    });
}

template <int TYPE>
bool launch_type(Context& ctx, const GemvParams& p, hipStream_t stream) {
    constexpr int E = piece_elems<TYPE>();
    if (p.k % E || (reinterpret_cast<uintptr_t>(p.w) % 16) || (reinterpret_cast<uintptr_t>(p.a) % 16)) {
        if constexpr (TYPE <= 1) {
            const uint64_t tasks = uint64_t(p.n) * p.m;
            if ((tasks + 3) / 4 > 0x7FFFFFFFull) return ctx.fail("matmul: too many outputs");
            return ctx.launch("gemv_scalar_kernel", stream, [&] {
                hipLaunchKernelGGL((gemv_scalar_kernel<TYPE>), dim3(unsigned((tasks + 3) / 4)), dim3(256), 0, stream, p);
            });
        }
        return ctx.fail("matmul: quantised weights need k a multiple of 32 and 16-byte aligned rows");
    }
    if (dma_eligible(p)) return launch_dma(ctx, &p, 1, false, stream);
    if (p.m >= GEMM_MIN_M) {
        const uint32_t tiles = ((p.n + GM_BN - 1) / GM_BN) * ((p.m + GM_BM - 1) / GM_BM);
        // fewer tiles than CUs and a long K: split K into slices of at least
        // 256 (multiples of a 32-wide step, so Q8/Q4 scale blocks stay whole),
        // each writing a partial tile; split_reduce_kernel adds them in order
        uint32_t slices = 1;
        if (tiles < 256 && p.k >= 512) {
            slices = (512 + tiles - 1) / tiles;
            if (slices > p.k / 256) slices = p.k / 256;
            if (slices > 64) slices = 64;
        }
        const uint32_t kSlice = ((p.k + slices - 1) / slices + GM_BK - 1) / GM_BK * GM_BK;
        slices = (p.k + kSlice - 1) / kSlice;
        const dim3 grid(unsigned((p.n + GM_BN - 1) / GM_BN), unsigned((p.m + GM_BM - 1) / GM_BM), slices);
        if (grid.y > 65535u) return ctx.fail("matmul: too many rows of a");
        if (slices == 1)
            return ctx.launch("gemm_kernel", stream, [&] {
                hipLaunchKernelGGL((gemm_kernel<TYPE>), grid, dim3(256), 0, stream, p, kSlice);
            });
        float* part = static_cast<float*>(ctx.grow(SLOT_GEMM_SPLIT, size_t(slices) * p.m * p.n * sizeof(float)));
        if (!part) return false;
        GemvParams q = p;
        q.out = part;
        q.ldo = p.n;
        q.bias = nullptr;
        q.accumulate = 0;
        if (!ctx.launch("gemm_kernel", stream, [&] {
                hipLaunchKernelGGL((gemm_kernel<TYPE>), grid, dim3(256), 0, stream, q, kSlice);
            }))
            return false;
        const uint64_t outs = uint64_t(p.m) * p.n;
        const unsigned rg = unsigned((outs + 255) / 256 < 65536 ? (outs + 255) / 256 : 65536);
        return ctx.launch("split_reduce_kernel", stream, [&] {
            hipLaunchKernelGGL(split_reduce_kernel, dim3(rg), dim3(256), 0, stream, p, part, slices);
        });
    }
    const unsigned gx = unsigned((p.n + 4 * GEMV_ROWS - 1) / (4 * GEMV_ROWS));
    const int M = p.m <= 1 ? 1 : (p.m <= 2 ? 2 : (p.m <= 4 ? 4 : GEMV_MAX_M));
    const unsigned gy = unsigned((p.m + M - 1) / M);
    if (gy > 65535u) return ctx.fail("matmul: too many rows of a");
    return ctx.launch("gemv_kernel", stream, [&] {
        const dim3 grid(gx, gy);
        if (M == 1) hipLaunchKernelGGL((gemv_kernel<TYPE, 1>), grid, dim3(256), 0, stream, p);
        else if (M == 2) hipLaunchKernelGGL((gemv_kernel<TYPE, 2>), grid, dim3(256), 0, stream, p);
        else if (M == 4) hipLaunchKernelGGL((gemv_kernel<TYPE, 4>), grid, dim3(256), 0, stream, p);
        else hipLaunchKernelGGL((gemv_kernel<TYPE, 8>), grid, dim3(256), 0, stream, p);
    });
}

} // namespace

bool launch_gemvs(const GemvParams* ps, int count, bool split, hipStream_t stream) {
    Context& ctx = Context::instance();
    bool together = count <= GD_SEGS;
    for (int i = 0; i < count; ++i) {
        const GemvParams &p = ps[i], &f = ps[0];
        together = together && p.a == f.a && p.m == f.m && p.k == f.k && p.type == f.type &&
                   (p.accumulate != 0) == (f.accumulate != 0) && p.n > 0 && p.ldo >= p.n && p.w && p.out &&
                   (p.type < 2 || p.scales) && p.type >= 0 && p.type <= 3 && p.a && dma_eligible(p);
    }
    if (together && count > 0) return launch_dma(ctx, ps, count, split, stream);
    for (int i = 0; i < count; ++i)
        if (!launch_gemv(ps[i], stream)) return false;
    return true;
}

bool launch_gemv(const GemvParams& p, hipStream_t stream) {
    Context& ctx = Context::instance();
    if (p.m == 0 || p.n == 0) return true;
    if (!p.a || !p.w || !p.out) return ctx.fail("matmul: null tensor");
    if (p.k == 0) return ctx.fail("matmul: k must be positive");
    if (p.ldo < p.n) return ctx.fail("matmul: output row stride below n");
    if (p.type >= 2 && !p.scales) return ctx.fail("matmul: quantised weights need scales");
    if (p.type >= 2 && p.k % 32) return ctx.fail("matmul: quantised weights need k a multiple of 32");
    switch (p.type) {
        case 0: return launch_type<0>(ctx, p, stream);
        case 1: return launch_type<1>(ctx, p, stream);
        case 2: return launch_type<2>(ctx, p, stream);
        case 3: return launch_type<3>(ctx, p, stream);
        default: return ctx.fail("matmul: unknown weight type");
    }
}

static bool kv_checks(Context& ctx, const GemvParams& p, const KvEpilogue& e);

bool gemm_splits_a(const GemvParams& p) { return dma_eligible(p); }

uint16_t* gemm_split_image(const GemvParams& p) {
    if (!dma_eligible(p)) return nullptr;
    return static_cast<uint16_t*>(Context::instance().grow(SLOT_GEMM_A, 2 * uint64_t(p.m) * p.k * 2));
}

bool launch_gemv_presplit(const GemvParams& p, hipStream_t stream) {
    Context& ctx = Context::instance();
    if (p.m == 0 || p.n == 0) return true;
    if (!p.w || !p.out || p.ldo < p.n || !dma_eligible(p)) return ctx.fail("matmul: no presplit GEMM for this shape");
    return launch_dma(ctx, &p, 1, true, stream);
}

bool launch_gemm_kv_pair(const GemvParams& pk, const GemvParams& pv, const KvEpilogue& ek, const KvEpilogue& ev,
                         bool aSplit, bool fold, float* rope, hipStream_t stream) {
    Context& ctx = Context::instance();
    if (pk.m == 0) return true;
    if (!kv_checks(ctx, pk, ek) || !kv_checks(ctx, pv, ev)) return false;
    if (pk.n != pv.n || pk.m != pv.m || pk.a != pv.a || ek.dim != ev.dim)
        return ctx.fail("projection epilogue: k and v differ in shape");
    // k and v side by side, [m][k's columns, v's]
    float* kv = static_cast<float*>(ctx.grow(SLOT_MIXER_KV, size_t(pk.m) * 2 * pk.n * sizeof(float)));
    if (!kv) return false;
    GemvParams both[2] = {pk, pv};
    for (int i = 0; i < 2; ++i) {
        both[i].out = kv + i * pk.n;
        both[i].ldo = 2 * pk.n;
        both[i].bias = nullptr;
        both[i].accumulate = 0;
    }
    if (!launch_gemvs(both, 2, aSplit, stream)) return false;
    const uint32_t heads = pk.n / ek.dim;
    if (fold && rope && !ek.freqs) return ctx.fail("projection epilogue: a cos/sin table needs RoPE");
    // the pad rows start past the last head's T rows (16-byte aligned: dim is 64 or 128)
    const size_t padAt = size_t(heads) * ek.T * ek.dim * 2;
    uint4* padK = fold ? reinterpret_cast<uint4*>(static_cast<uint8_t*>(ek.work) + padAt) : nullptr;
    uint4* padV = fold ? reinterpret_cast<uint4*>(static_cast<uint8_t*>(ev.work) + padAt) : nullptr;
    const uint32_t pad16 = PREFILL_PAD_ROWS * ek.dim * 2 / 16;
    return ctx.launch("kv_epilogue_kernel", stream, [&] {
        hipLaunchKernelGGL(kv_epilogue_kernel, dim3(pk.m), dim3(256), 0, stream, kv, pk.bias, pv.bias, ek, ev, heads,
                           fold ? rope : nullptr, padK, padV, pad16);
    });
}

/* the shapes and alignments a k or v projection with its epilogue needs */
static bool kv_checks(Context& ctx, const GemvParams& p, const KvEpilogue& e) {
    if (!p.a || !p.w || !e.cache || !e.work) return ctx.fail("projection epilogue: null tensor");
    if (e.dim != 64 && e.dim != 128) return ctx.fail("projection epilogue: dim must be 64 or 128");
    if (p.n == 0 || p.n % e.dim) return ctx.fail("projection epilogue: n must be a multiple of dim");
    if (e.freqs && (e.rot == 0 || e.rot > e.dim || e.rot % 2)) return ctx.fail("projection epilogue: bad rotaryDims");
    if (uint64_t(e.start) + p.m > e.T || e.T > e.capacity) return ctx.fail("projection epilogue: rows past the cache");
    if (p.k == 0) return ctx.fail("matmul: k must be positive");
    if (p.type >= 2 && (!p.scales || p.k % 32)) return ctx.fail("matmul: quantised weights need scales and k % 32");
    const int E = p.type == 0 ? 4 : (p.type == 1 ? 8 : (p.type == 2 ? 16 : 32));
    if (p.k % E || (reinterpret_cast<uintptr_t>(p.w) % 16) || (reinterpret_cast<uintptr_t>(p.a) % 16) ||
        (reinterpret_cast<uintptr_t>(e.cache) % 16) || (reinterpret_cast<uintptr_t>(e.work) % 16))
        return ctx.fail("projection epilogue: rows of a, w and the caches must be 16-byte aligned");
    return true;
}

} // namespace aigpu
