// attention_f32.hip - fp32 causal GQA attention with kernels::attention's
// semantics (include/ai/Kernels.hpp:130-168): for token t and head h at
// position start+t, keys [first, start+t] of kv head h/(heads/kvHeads), with
// first = start+t+1-window when a window is set; out = softmax(q.K/sqrt(D)) V.
//
// This is the exact-arithmetic path behind the drop-in aigpu_attention, in
// these forms. fp32 q and KV of dim 64 or 128 on 16-byte boundaries take the
// fp32 matrix cores, in tiles of 128 tokens or, where those leave the chip
// idle, in groups of 16 query rows (attention_f32_tile_kernel and
// attention_f32_narrow_kernel, described at them); every other call (bf16 KV, other dims, unaligned rows) takes the
// scalar form: fp32 loads, fp32 FMAs, expf. There one wave owns one (token,
// head) and walks the keys in blocks of 64 with an online softmax: lane j
// scores key j of the block, then the lanes switch to owning dimensions for
// the P.V accumulation. Both loops issue their loads in batches before using
// them (a key row as up to 16 16-byte pieces per lane with four partial sums
// when rows are 16-byte aligned; value rows as 16-byte pieces, several rows
// per load instruction, or else eight rows at a time), so that a block costs
// a few memory round trips rather than one per dimension or per key.
#include "context.hpp"
#include "device.hpp"
#include "kernels.hpp"

namespace aigpu {

namespace {

constexpr int MAX_DIM = 256;

__global__ __launch_bounds__(256) void attention_f32_kernel(AttentionF32Params p) {
    __shared__ __align__(16) float qs[4][MAX_DIM];
    __shared__ float ps[4][WAVE];

    const int lane = threadIdx.x & (WAVE - 1);
    const int w = threadIdx.x / WAVE;
    const uint64_t task = uint64_t(blockIdx.x) * 4 + w;
    if (task >= p.count * p.heads) return;  // whole wave leaves; no block barriers below

    const uint64_t token = task / p.heads, head = task % p.heads;
    const uint64_t position = p.start + token;
    const uint64_t first = p.window && position + 1 > p.window ? position + 1 - p.window : 0;
    const uint64_t kv = head / (p.heads / p.kvHeads);
    const int dim = int(p.dim);
    const float scale = 1.0f / sqrtf(float(dim));

    for (int d = lane; d < dim; d += WAVE)
        qs[w][d] = load_elem(p.q, (token * p.heads + head) * p.qStride + d, p.qType);
    wave_sync();

    const size_t kvBase = kv * p.headStride;
    float m = -INFINITY, l = 0.0f;
    float acc[MAX_DIM / WAVE] = {0.0f, 0.0f, 0.0f, 0.0f};
    // key rows in 16-byte pieces: every row start (and q's copy in LDS) on a
    // 16-byte boundary, which fp32 rows with dim % 4 == 0 and bf16 rows with
    // dim % 8 == 0 and strides to match give
    const size_t esz = p.kvType == 0 ? 4 : 2, per = 16 / esz;
    const bool vec = dim % int(per) == 0 && (reinterpret_cast<uintptr_t>(p.keys) % 16) == 0 &&
                     (kvBase * esz) % 16 == 0 && (p.posStride * esz) % 16 == 0;
    // fp32 value rows of dim / 4 16-byte pieces, a power of two: LPR lanes per
    // row, RPI = 64 / LPR rows per load instruction, each lane a four-float
    // accumulator for its piece and its group of rows (summed across the
    // groups at the end); up to 16 pieces per lane in flight
    const int LPR = dim / 4;
    const bool vecv = p.kvType == 0 && dim % 4 == 0 && (LPR & (LPR - 1)) == 0 &&
                      (reinterpret_cast<uintptr_t>(p.values) % 16) == 0 && (kvBase * 4) % 16 == 0 &&
                      (p.posStride * 4) % 16 == 0;
    const int RPI = vecv ? WAVE / LPR : 1, vg = vecv ? lane / LPR : 0, vc = vecv ? lane % LPR : 0;
    floatx4 acc2 = {0.0f, 0.0f, 0.0f, 0.0f};

    for (uint64_t j0 = first; j0 <= position; j0 += WAVE) {
        const uint64_t j = j0 + lane;
        const bool ok = j <= position;
        float s = -INFINITY;
        if (ok) {
            const size_t row = kvBase + j * p.posStride;
            float dot = 0.0f;
            if (vec && p.kvType == 0) {
                // up to 64 dimensions per batch: 16 pieces in flight, four partial sums
                const floatx4* kr = reinterpret_cast<const floatx4*>(static_cast<const float*>(p.keys) + row);
                const floatx4* q4 = reinterpret_cast<const floatx4*>(qs[w]);
                floatx4 part = {0.0f, 0.0f, 0.0f, 0.0f};
                for (int c0 = 0; c0 < dim / 4; c0 += 16) {
                    floatx4 kp[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (c0 + i < dim / 4) kp[i] = kr[c0 + i];
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (c0 + i < dim / 4) {
                            const floatx4 qv = q4[c0 + i];
#pragma unroll
                            for (int e = 0; e < 4; ++e) part[e] = fmaf(qv[e], kp[i][e], part[e]);
                        }
                }
                dot = (part[0] + part[1]) + (part[2] + part[3]);
            } else if (vec) {
                // bf16: eight elements per piece, up to 128 dimensions per batch
                const u32x4* kr = reinterpret_cast<const u32x4*>(static_cast<const uint16_t*>(p.keys) + row);
                const floatx4* q4 = reinterpret_cast<const floatx4*>(qs[w]);
                floatx4 part = {0.0f, 0.0f, 0.0f, 0.0f};
                for (int c0 = 0; c0 < dim / 8; c0 += 16) {
                    u32x4 kp[16];
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (c0 + i < dim / 8) kp[i] = kr[c0 + i];
#pragma unroll
                    for (int i = 0; i < 16; ++i)
                        if (c0 + i < dim / 8) {
                            const floatx4 qa = q4[2 * (c0 + i)], qb = q4[2 * (c0 + i) + 1];
#pragma unroll
                            for (int e = 0; e < 4; ++e) {
                                const uint32_t wv = kp[i][e];
                                const float lo = __uint_as_float(wv << 16), hi = __uint_as_float(wv & 0xFFFF0000u);
                                const float q0 = e < 2 ? qa[2 * e] : qb[2 * e - 4];
                                const float q1 = e < 2 ? qa[2 * e + 1] : qb[2 * e - 3];
                                part[e] = fmaf(q1, hi, fmaf(q0, lo, part[e]));
                            }
                        }
                }
                dot = (part[0] + part[1]) + (part[2] + part[3]);
            } else if (p.kvType == 0) {
                const float* kr = static_cast<const float*>(p.keys) + row;
                for (int d = 0; d < dim; ++d) dot = fmaf(qs[w][d], kr[d], dot);
            } else {
                const uint16_t* kr = static_cast<const uint16_t*>(p.keys) + row;
                for (int d = 0; d < dim; ++d) dot = fmaf(qs[w][d], bf16_bits_to_float(kr[d]), dot);
            }
            s = dot * scale;
        }
        const float mn = fmaxf(m, wave_max(s));  // finite: the block holds key j0
        const float alpha = expf(m - mn);
        const float pj = ok ? expf(s - mn) : 0.0f;
        l = l * alpha + wave_sum(pj);
        m = mn;
#pragma unroll
        for (int i = 0; i < MAX_DIM / WAVE; ++i) acc[i] *= alpha;
#pragma unroll
        for (int e = 0; e < 4; ++e) acc2[e] *= alpha;

        ps[w][lane] = pj;
        wave_sync();
        const int nb = int(position + 1 - j0 < WAVE ? position + 1 - j0 : WAVE);
        if (vecv) {
            const floatx4* vb = reinterpret_cast<const floatx4*>(static_cast<const float*>(p.values) + kvBase) + vc;
            const size_t rs = p.posStride / 4;
            for (int t0 = 0; t0 < LPR; t0 += 16) {
                floatx4 vp[16];
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    const int r = (t0 + u) * RPI + vg;
                    vp[u] = t0 + u < LPR && r < nb ? vb[(j0 + uint64_t(r)) * rs] : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
                for (int u = 0; u < 16; ++u) {
                    const int r = (t0 + u) * RPI + vg;
                    if (t0 + u < LPR && r < nb) {
                        const float pv = ps[w][r];
#pragma unroll
                        for (int e = 0; e < 4; ++e) acc2[e] = fmaf(pv, vp[u][e], acc2[e]);
                    }
                }
            }
        }
        for (int jb = 0; !vecv && jb < nb; jb += 8) {   // eight value rows' loads in flight
            float vr[8][MAX_DIM / WAVE];
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                const size_t row = kvBase + (j0 + jb + u) * p.posStride;
#pragma unroll
                for (int i = 0; i < MAX_DIM / WAVE; ++i) {
                    const int d = lane + i * WAVE;
                    vr[u][i] = jb + u < nb && d < dim ? load_elem(p.values, row + d, p.kvType) : 0.0f;
                }
            }
#pragma unroll
            for (int u = 0; u < 8; ++u) {
                if (jb + u >= nb) break;   // uniform
                const float pv = ps[w][jb + u];
#pragma unroll
                for (int i = 0; i < MAX_DIM / WAVE; ++i) acc[i] = fmaf(pv, vr[u][i], acc[i]);
            }
        }
        wave_sync();
    }

    const float inv = 1.0f / l;
    float* dst = p.out + task * p.dim;
    if (vecv) {
        for (int off = LPR; off < WAVE; off <<= 1)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc2[e] += __shfl_xor(acc2[e], off, WAVE);
        if (vg == 0) {
#pragma unroll
            for (int e = 0; e < 4; ++e) dst[4 * vc + e] = acc2[e] * inv;
        }
        return;
    }
#pragma unroll
    for (int i = 0; i < MAX_DIM / WAVE; ++i) {
        const int d = lane + i * WAVE;
        if (d < dim) dst[d] = acc[i] * inv;
    }
}

/*
    The tiled form, for fp32 q and KV of dim 64 or 128 with 16-byte aligned
    rows: the products run on the fp32 matrix cores (v_mfma_f32_32x32x2_f32
    multiplies and accumulates in fp32) and the softmax in fp32 with expf, so
    it differs from the form above only in summation order.

    A workgroup is 4 waves x 32 query tokens (TQ = 128 tokens) of one head;
    it walks key tiles of TK = 64 keys, K and V staged in LDS by DMA in two
    stages, so every K and V element a tile brings in serves 128 queries. A
    long key range is split over `splits` workgroups of `tilesPerSplit`
    tiles each; they write unnormalised partial records (o, running max m,
    sum l) that attention_f32_merge_kernel combines.

    Per wave and tile, S^T (64 keys x 32 queries) = K Q^T as two 32 x 32
    blocks of D/2 products, each over two dims: lanes 0-31 supply dim s and
    lanes 32-63 dim D/2 + s, so a lane's B operands are its query's half row,
    held in registers. Register r of a score block holds key
    8 (r / 4) + 4 (lane / 32) + r % 4 of the block for query lane % 32; that
    register is directly the B operand of one P.V product, O^T (D x 32) +=
    V^T P^T, whose A operand is then the V row of that key. The operand reads
    of both products run AH steps ahead of their MFMAs, and the two score
    blocks (and the D/32 output tiles) are independent accumulator chains.

    LDS K rows keep 16-byte block c at c ^ (row % 16), so the 16 rows one
    A-operand read touches hit distinct banks; V rows are natural.
*/
constexpr int TK = 64;     // keys per tile
constexpr int TQ = 128;    // query tokens per workgroup

/* s_waitcnt vmcnt(0), the other counters left alone */
__device__ __forceinline__ void wait_vmcnt_all() {
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));
}

struct TileArgs {
    AttentionF32Params p;
    float* acc;              // split records [split][head][token][dim]
    float2* ml;              // their (m, l) [split][head][token]
    uint32_t groups;         // token groups of TQ (narrow: row groups of NR)
    uint32_t splits;         // workgroups per (token group, head) (narrow: per (row group, kv head))
    uint32_t tilesPerSplit;  // key tiles per workgroup when splits > 1; 0: the narrow form
};

/* the key tiles of token group `grp`: every key a token of the group sees
   lies in [kbeg, kbeg + TK * ntiles) */
__host__ __device__ inline void group_tiles(uint64_t count, uint64_t start, uint64_t window, uint64_t grp,
                                            uint64_t& kbeg, uint32_t& ntiles) {
    const uint64_t t0 = grp * TQ;
    const uint64_t tLast = (t0 + TQ < count ? t0 + TQ : count) - 1;
    const uint64_t p0 = start + t0, p1 = start + tLast;
    const uint64_t first = window && p0 + 1 > window ? p0 + 1 - window : 0;
    kbeg = first / TK * TK;
    ntiles = uint32_t((p1 + 1 - kbeg + TK - 1) / TK);
}

template <int D>
__global__ __launch_bounds__(256) void attention_f32_tile_kernel(TileArgs a) {
    constexpr int DT = D / 32;             // 32-dim tiles of O^T
    constexpr int HALF = D / 2;            // q elements per lane
    constexpr int NI = HALF / 4;           // 16-byte q pieces per lane
    constexpr int CPR = D / 4;             // 16-byte blocks per row
    constexpr int TILE = TK * D;           // floats per K or V tile
    constexpr int BPW = TILE * 4 / 1024 / 4;   // 1 KB DMA blocks per wave per tile (K or V)
    constexpr int AH = 2;                  // operand reads in flight ahead of their products
    __shared__ __attribute__((aligned(16))) float Ks[2 * TILE];
    __shared__ __attribute__((aligned(16))) float Vs[2 * TILE];

    const AttentionF32Params& p = a.p;
    const int lane = threadIdx.x & 63, h = lane >> 5, j = lane & 31;
    const uint32_t w = __builtin_amdgcn_readfirstlane(uint32_t(threadIdx.x >> 6));
    uint32_t bid = blockIdx.x;
    const uint32_t sigma = bid % a.splits;
    bid /= a.splits;
    const uint64_t head = bid % uint32_t(p.heads);
    const uint64_t grp = a.groups - 1 - bid / uint32_t(p.heads);   // the longest groups first
    uint64_t kbeg;
    uint32_t ntiles;
    group_tiles(p.count, p.start, p.window, grp, kbeg, ntiles);
    const uint32_t tBegin = a.splits > 1 ? sigma * a.tilesPerSplit : 0u;
    if (tBegin >= ntiles) return;   // the whole workgroup: no split here
    const uint32_t tEnd = a.splits > 1 && tBegin + a.tilesPerSplit < ntiles ? tBegin + a.tilesPerSplit : ntiles;

    const uint64_t kv = head / (p.heads / p.kvHeads);
    const uint64_t lastKey = p.start + p.count - 1;
    const uint64_t tw0 = grp * TQ + 32 * w;
    const bool waveRows = tw0 < p.count;
    const uint64_t t = tw0 + j;
    const bool rowValid = t < p.count;
    const uint64_t P = p.start + t;
    const uint64_t first = p.window && P + 1 > p.window ? P + 1 - p.window : 0;
    // keys any row of the wave sees: [wFirst, wLast]
    const uint64_t wLast = p.start + (tw0 + 31 < p.count ? tw0 + 31 : p.count - 1);
    const uint64_t wFirst = p.window && p.start + tw0 + 1 > p.window ? p.start + tw0 + 1 - p.window : 0;

    float qh[HALF];
    {
        const float* qrow = static_cast<const float*>(p.q) + (t * p.heads + head) * p.qStride + HALF * h;
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const floatx4 v = rowValid ? *reinterpret_cast<const floatx4*>(qrow + 4 * i) : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
            for (int e = 0; e < 4; ++e) qh[4 * i + e] = v[e];
        }
    }

    // DMA of the tile at key k0 into stage st: block n of this wave covers
    // 16-byte slots 64 (BPW w + n) + lane, row slot / CPR; K row r takes its
    // block (slot % CPR) ^ (r % 16) from memory. Rows past the last key
    // repeat it (their scores are masked and their P is 0).
    const char* kbase = reinterpret_cast<const char*>(static_cast<const float*>(p.keys) + kv * p.headStride);
    const char* vbase = reinterpret_cast<const char*>(static_cast<const float*>(p.values) + kv * p.headStride);
    const uint32_t ldsK = lds_address(Ks), ldsV = lds_address(Vs);
    const uint32_t rowBytes = uint32_t(p.posStride) * 4;
    auto issue = [&](uint64_t k0, uint32_t st) __attribute__((always_inline)) {
        const uint32_t lim = uint32_t(lastKey - k0 < TK - 1 ? lastKey - k0 : TK - 1);
        const char* kt = kbase + k0 * rowBytes;
        const char* vt = vbase + k0 * rowBytes;
#pragma unroll
        for (int n = 0; n < BPW; ++n) {
            const uint32_t blk = w * BPW + n;
            const uint32_t slot = blk * 64 + lane, r = slot / CPR, cp = slot % CPR;
            const uint32_t rowOff = (r < lim ? r : lim) * rowBytes;
            const uint32_t lds = __builtin_amdgcn_readfirstlane(st * TILE * 4 + blk * 1024);
            dma_block(kt, rowOff + 16 * (cp ^ (r & 15)), ldsK + lds);
            dma_block(vt, rowOff + 16 * cp, ldsV + lds);
        }
    };

    floatx16 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.0f;
    float m = -INFINITY, lsum = 0.0f;
    const float scale = 1.0f / sqrtf(float(D));

    issue(kbeg + uint64_t(tBegin) * TK, 0);
    for (uint32_t it = tBegin; it < tEnd; ++it) {
        const uint32_t st = (it - tBegin) & 1;
        const uint64_t k0 = kbeg + uint64_t(it) * TK;
        // tile `it` (and, the first time, q) has landed for every wave, and
        // every wave is done with the other stage
        wait_vmcnt_all();
        lds_barrier();
        if (it + 1 < tEnd) issue(k0 + TK, st ^ 1);
        if (!waveRows || k0 > wLast || k0 + TK - 1 < wFirst) continue;   // uniform over the wave
        const float* ks = Ks + st * TILE;
        const float* vs = Vs + st * TILE;

        // S^T: step i takes dims HALF h + 4 i .. + 3 of both key blocks, its
        // K operands read AH steps ahead into a ring; the two blocks' chains
        // alternate, and the scheduling groups pin that order
        floatx16 s[2];
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) s[b][r] = 0.0f;
        {
            auto kfrag = [&](int i, int b) __attribute__((always_inline)) {
                const int c = NI * h + i;
                return *reinterpret_cast<const floatx4*>(ks + (32 * b + j) * D + 4 * (c ^ (j & 15)));
            };
            floatx4 f[AH + 1][2];
#pragma unroll
            for (int i = 0; i < AH; ++i)
#pragma unroll
                for (int b = 0; b < 2; ++b) f[i][b] = kfrag(i, b);
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                if (i + AH < NI)
#pragma unroll
                    for (int b = 0; b < 2; ++b) f[(i + AH) % (AH + 1)][b] = kfrag(i + AH, b);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int b = 0; b < 2; ++b)
                        s[b] = __builtin_amdgcn_mfma_f32_32x32x2f32(f[i % (AH + 1)][b][e], qh[4 * i + e], s[b], 0, 0, 0);
            }
            __builtin_amdgcn_sched_group_barrier(0x100, 2 * AH, 0);
#pragma unroll
            for (int i = 0; i < NI; ++i) {
                if (i + AH < NI) __builtin_amdgcn_sched_group_barrier(0x100, 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, 8, 0);
            }
        }
        // keys of the tile this row sees: offsets [lo, hi] from k0
        const int64_t hi64 = int64_t(P) - int64_t(k0), lo64 = int64_t(first) - int64_t(k0);
        const int hi = rowValid ? int(hi64 < TK ? hi64 : TK) : -1;
        const int lo = int(lo64 > TK ? TK + 1 : (lo64 > 0 ? lo64 : 0));
        float mx = -INFINITY;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const int key = 32 * b + 8 * (r >> 2) + 4 * h + (r & 3);
                s[b][r] = key >= lo && key <= hi ? s[b][r] * scale : -INFINITY;
                mx = fmaxf(mx, s[b][r]);
            }
        mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
        const float mn = fmaxf(m, mx);
        float alpha = 1.0f, psum = 0.0f;
        if (mn == -INFINITY) {   // no key of this row so far
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) s[b][r] = 0.0f;
        } else {
            alpha = expf(m - mn);
#pragma unroll
            for (int b = 0; b < 2; ++b)
#pragma unroll
                for (int r = 0; r < 16; ++r) {
                    s[b][r] = expf(s[b][r] - mn);
                    psum += s[b][r];
                }
        }
        psum += __shfl_xor(psum, 32, WAVE);
        lsum = lsum * alpha + psum;
        m = mn;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;

        // P.V: step n = (b, r) takes key row 32 b + 8 (r / 4) + 4 h + r % 4 of
        // every d tile (DT independent chains), its V operands AH steps ahead
        {
            auto vfrag = [&](int n, int dt) __attribute__((always_inline)) {
                const int b = n >> 4, r = n & 15;
                return vs[(32 * b + 8 * (r >> 2) + 4 * h + (r & 3)) * D + 32 * dt + j];
            };
            float f[AH + 1][DT];
#pragma unroll
            for (int n = 0; n < AH; ++n)
#pragma unroll
                for (int dt = 0; dt < DT; ++dt) f[n][dt] = vfrag(n, dt);
#pragma unroll
            for (int n = 0; n < 32; ++n) {
                if (n + AH < 32)
#pragma unroll
                    for (int dt = 0; dt < DT; ++dt) f[(n + AH) % (AH + 1)][dt] = vfrag(n + AH, dt);
#pragma unroll
                for (int dt = 0; dt < DT; ++dt)
                    o[dt] = __builtin_amdgcn_mfma_f32_32x32x2f32(f[n % (AH + 1)][dt], s[n >> 4][n & 15], o[dt], 0, 0, 0);
            }
            // the reads of a step pair up into DT / 2 two-address reads
            __builtin_amdgcn_sched_group_barrier(0x100, AH * DT / 2, 0);
#pragma unroll
            for (int n = 0; n < 32; ++n) {
                if (n + AH < 32) __builtin_amdgcn_sched_group_barrier(0x100, DT / 2, 0);
                __builtin_amdgcn_sched_group_barrier(0x008, DT, 0);
            }
        }
    }
    if (!rowValid) return;

    // O^T register r of d tile dt holds dim 32 dt + 8 (r / 4) + 4 (lane / 32) + r % 4
    if (a.splits == 1) {
        const float inv = 1.0f / lsum;
        float* dst = p.out + (t * p.heads + head) * D;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int g = 0; g < 4; ++g)
                *reinterpret_cast<floatx4*>(dst + 32 * dt + 8 * g + 4 * h) =
                    floatx4{o[dt][4 * g] * inv, o[dt][4 * g + 1] * inv, o[dt][4 * g + 2] * inv, o[dt][4 * g + 3] * inv};
        return;
    }
    const size_t rec = (size_t(sigma) * p.heads + head) * p.count + t;
    float* dst = a.acc + rec * D;
#pragma unroll
    for (int dt = 0; dt < DT; ++dt)
#pragma unroll
        for (int g = 0; g < 4; ++g)
            *reinterpret_cast<floatx4*>(dst + 32 * dt + 8 * g + 4 * h) =
                floatx4{o[dt][4 * g], o[dt][4 * g + 1], o[dt][4 * g + 2], o[dt][4 * g + 3]};
    if (h == 0) a.ml[rec] = make_float2(m, lsum);
}

/*
    The narrow form, for calls whose tiles of 128 tokens would leave most of
    the chip idle: a workgroup owns 16 query rows of one kv head (a row is a
    (token, query head) pair, token-major, so a group's heads share the K and
    V they read) and its NW waves take 16-key blocks in turn, each with its
    own softmax state, combined in LDS at the end. K, V and q go from memory
    to the operand registers 16 bytes a lane, a block ahead of its products:
    nothing is shared between waves, so there is nothing to stage.

    S^T (16 keys x 16 rows) = K Q^T on v_mfma_f32_16x16x4_f32: lane group g
    (lane / 16) supplies dims g D/4 + s at step s, so a lane reads D/4
    contiguous floats of key lane % 16. Register r of the block is key
    4 g + r for row lane % 16, which is the B operand of P.V's step r; its A
    operand, row i of d tile dt, is dim i D/16 + dt, so a lane reads D/16
    contiguous floats of that key's value, and O^T leaves it D/4 contiguous
    dims of its row.

    It is bound by its chain of loads, 2 x D/4 products and a softmax a step;
    128 tokens of 12 x 64 heads take it 6.3 us (tiled and merged 10.7 + 3.8).

    A row that saw only scores of -inf keeps m = -inf with l = 0; NaN scores
    stay NaN in l and o, whatever m is.
*/
constexpr int NR = 16;     // query rows per workgroup
constexpr int NB = 16;     // keys per block
constexpr int NW = 8;      // waves per workgroup

template <int D>
__global__ __launch_bounds__(64 * NW, D == 64 ? 4 : 2) void attention_f32_narrow_kernel(TileArgs a) {
    constexpr int KF = D / 16;             // 16-byte K (and q) pieces per lane
    constexpr int VF = D / 64;             // 16-byte V pieces per lane and key
    constexpr int DT = D / 16;             // 16-dim tiles of O^T
    constexpr int OS = D + 4;              // floats per row of Os
    __shared__ __attribute__((aligned(16))) float Os[NW * NR * OS];
    __shared__ float2 Ml[NW][NR];

    const AttentionF32Params& p = a.p;
    const int lane = threadIdx.x & 63, g = lane >> 4, j = lane & 15;
    const uint32_t w = __builtin_amdgcn_readfirstlane(uint32_t(threadIdx.x >> 6));
    // 32 bits hold every row, position and block here (launch_tiled)
    const uint32_t heads = uint32_t(p.heads), kvHeads = uint32_t(p.kvHeads), G = heads / kvHeads;
    const uint32_t count = uint32_t(p.count), start = uint32_t(p.start), rows = count * G;
    uint32_t bid = blockIdx.x;
    const uint32_t sigma = bid % a.splits;
    bid /= a.splits;
    const uint32_t kv = bid % kvHeads, grp = a.groups - 1 - bid / kvHeads;   // the longest groups first
    const uint32_t row0 = grp * NR, rowLast = row0 + NR < rows ? row0 + NR - 1 : rows - 1;
    auto firstKey = [&](uint32_t pos) __attribute__((always_inline)) {
        return p.window && pos + 1 > p.window ? pos + 1 - uint32_t(p.window) : 0u;
    };
    // keys any row sees: [kbeg, kend)
    const uint32_t kbeg = firstKey(start + row0 / G), kend = start + rowLast / G + 1;
    const uint32_t nb = (kend - kbeg + NB - 1) / NB;
    const uint32_t bBegin = uint32_t(uint64_t(nb) * sigma / a.splits), bEnd = uint32_t(uint64_t(nb) * (sigma + 1) / a.splits);

    // rows past the last repeat it and store nothing
    const uint32_t row = row0 + j < rows ? row0 + j : rows - 1, t = row / G, head = kv * G + row % G;
    const uint32_t P = start + t, first = firstKey(P);
    const float* kbase = static_cast<const float*>(p.keys) + kv * p.headStride + g * (D / 4);
    const float* vbase = static_cast<const float*>(p.values) + kv * p.headStride + j * (D / 16);
    const uint32_t posStride = uint32_t(p.posStride);

    floatx4 qf[KF];
    {
        const float* qrow = static_cast<const float*>(p.q) + (uint64_t(t) * heads + head) * p.qStride + g * (D / 4);
#pragma unroll
        for (int i = 0; i < KF; ++i)
            qf[i] = *reinterpret_cast<const floatx4*>(qrow + 4 * i);
    }
    // keys past the group's last repeat it (their scores are masked, their P is 0)
    auto load = [&](uint32_t b, floatx4 (&kf)[KF], floatx4 (&vf)[4][VF]) __attribute__((always_inline)) {
        const uint32_t k0 = kbeg + b * NB;
        const float* kr = kbase + uint64_t(k0 + j < kend ? k0 + j : kend - 1) * posStride;
#pragma unroll
        for (int i = 0; i < KF; ++i) kf[i] = *reinterpret_cast<const floatx4*>(kr + 4 * i);
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t vk = k0 + 4 * g + r;
            const float* vr = vbase + uint64_t(vk < kend ? vk : kend - 1) * posStride;
#pragma unroll
            for (int i = 0; i < VF; ++i) vf[r][i] = *reinterpret_cast<const floatx4*>(vr + 4 * i);
        }
    };

    floatx4 o[DT];
#pragma unroll
    for (int dt = 0; dt < DT; ++dt) o[dt] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    float m = -INFINITY, lsum = 0.0f;
    const float scale = 1.0f / sqrtf(float(D));

    floatx4 kf[KF], vf[4][VF];
    if (bBegin + w < bEnd) load(bBegin + w, kf, vf);
    for (uint32_t b = bBegin + w; b < bEnd; b += NW) {
        floatx4 kn[KF], vn[4][VF];
        if (b + NW < bEnd) load(b + NW, kn, vn);
        floatx4 s = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int i = 0; i < KF; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) s = __builtin_amdgcn_mfma_f32_16x16x4f32(kf[i][e], qf[i][e], s, 0, 0, 0);
        const uint32_t k0 = kbeg + b * NB + 4 * g;
        float mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = k0 + r >= first && k0 + r <= P ? s[r] * scale : -INFINITY;
            mx = fmaxf(mx, s[r]);
        }
        mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
        mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
        const float mn = fmaxf(m, mx), mz = mn == -INFINITY ? 0.0f : mn;   // all -inf so far: zeros (or NaN)
        const float alpha = expf(m - mz);
        float psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            s[r] = expf(s[r] - mz);
            psum += s[r];
        }
        psum += __shfl_xor(psum, 16, WAVE);
        psum += __shfl_xor(psum, 32, WAVE);
        lsum = lsum * alpha + psum;
        m = mn;
#pragma unroll
        for (int dt = 0; dt < DT; ++dt)
#pragma unroll
            for (int r = 0; r < 4; ++r) o[dt][r] *= alpha;
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int dt = 0; dt < DT; ++dt)
                o[dt] = __builtin_amdgcn_mfma_f32_16x16x4f32(vf[r][dt / 4][dt % 4], s[r], o[dt], 0, 0, 0);
        if (b + NW < bEnd) {
#pragma unroll
            for (int i = 0; i < KF; ++i) kf[i] = kn[i];
#pragma unroll
            for (int r = 0; r < 4; ++r)
#pragma unroll
                for (int i = 0; i < VF; ++i) vf[r][i] = vn[r][i];
        }
    }

    // O^T register r of d tile dt is dim (4 g + r) D/16 + dt: a lane's D/4
    // dims from g D/4 on, in the order (r, dt)
    float* ow = Os + (w * NR + j) * OS + g * (D / 4);
#pragma unroll
    for (int i = 0; i < D / 16; ++i) {
        floatx4 v;
#pragma unroll
        for (int e = 0; e < 4; ++e) v[e] = o[(4 * i + e) % DT][(4 * i + e) / DT];
        *reinterpret_cast<floatx4*>(ow + 4 * i) = v;
    }
    if (g == 0) Ml[w][j] = make_float2(m, lsum);
    __syncthreads();

    // one 16-byte piece of a row per thread; a wave without a block left m =
    // -inf with zeros, and m = -inf weighs 0 (its l and o are zeros, or NaN)
    constexpr int PIECES = D / 4;
    const uint32_t r = threadIdx.x / PIECES, c = threadIdx.x % PIECES;
    if (r >= NR || row0 + r >= rows) return;
    const uint32_t ot = (row0 + r) / G, oh = kv * G + (row0 + r) % G;
    float M = -INFINITY, L = 0.0f;
#pragma unroll
    for (int u = 0; u < NW; ++u) M = fmaxf(M, Ml[u][r].x);
    const float Mz = M == -INFINITY ? 0.0f : M;
    floatx4 acc = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int u = 0; u < NW; ++u) {
        const float2 ml = Ml[u][r];
        const float e = expf(ml.x - Mz);
        const floatx4 v = *reinterpret_cast<const floatx4*>(Os + (u * NR + r) * OS + 4 * c);
        L += ml.y * e;
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[i] += v[i] * e;
    }
    if (a.splits == 1) {
        const float inv = 1.0f / L;
        *reinterpret_cast<floatx4*>(p.out + (uint64_t(ot) * heads + oh) * D + 4 * c) =
            floatx4{acc[0] * inv, acc[1] * inv, acc[2] * inv, acc[3] * inv};
        return;
    }
    const size_t rec = (size_t(sigma) * heads + oh) * count + ot;
    *reinterpret_cast<floatx4*>(a.acc + rec * D + 4 * c) = acc;
    // the merge leaves out records of m = -inf: one that holds NaN keeps it
    if (c == 0) a.ml[rec] = make_float2(M == -INFINITY && L != L ? 0.0f : M, L);
}

/* one wave per (token, head): out = sum_s e^(m_s - M) o_s / sum_s e^(m_s - M) l_s
   over the splits that cover the token's group (a split in which the row
   saw no key has m = -inf and adds nothing); the records of up to MB splits
   are loaded together, one memory round trip per MB splits */
template <int D>
__global__ __launch_bounds__(256) void attention_f32_merge_kernel(TileArgs a) {
    constexpr int MB = 16, NE = D / 64;
    const AttentionF32Params& p = a.p;
    const int lane = threadIdx.x & 63;
    const uint64_t task = uint64_t(blockIdx.x) * 4 + (threadIdx.x >> 6);
    if (task >= p.count * p.heads) return;
    const uint64_t t = task / p.heads, head = task % p.heads;
    uint32_t n = a.splits;           // the narrow form's splits all leave a record
    if (a.tilesPerSplit) {
        uint64_t kbeg;
        uint32_t ntiles;
        group_tiles(p.count, p.start, p.window, t / TQ, kbeg, ntiles);
        n = (ntiles + a.tilesPerSplit - 1) / a.tilesPerSplit;
    }
    float M = -INFINITY, L = 0.0f, acc[NE] = {};
    for (uint32_t s0 = 0; s0 < n; s0 += MB) {
        float2 ml[MB];
        float av[MB][NE];
#pragma unroll
        for (int u = 0; u < MB; ++u) {
            const bool ok = s0 + u < n;
            const size_t rec = ((size_t(s0) + u) * p.heads + head) * p.count + t;
            ml[u] = ok ? a.ml[rec] : make_float2(-INFINITY, 0.0f);
#pragma unroll
            for (int i = 0; i < NE; ++i) av[u][i] = ok ? a.acc[rec * D + lane + 64 * i] : 0.0f;
        }
        float bm = M;
#pragma unroll
        for (int u = 0; u < MB; ++u) bm = fmaxf(bm, ml[u].x);
        if (bm == -INFINITY) continue;
        const float sc = expf(M - bm);   // 0 while nothing is merged
        L *= sc;
#pragma unroll
        for (int i = 0; i < NE; ++i) acc[i] *= sc;
#pragma unroll
        for (int u = 0; u < MB; ++u) {
            if (ml[u].x == -INFINITY) continue;
            const float e = expf(ml[u].x - bm);
            L += ml[u].y * e;
#pragma unroll
            for (int i = 0; i < NE; ++i) acc[i] += e * av[u][i];
        }
        M = bm;
    }
    const float inv = 1.0f / L;
    float* dst = p.out + task * D;
#pragma unroll
    for (int i = 0; i < NE; ++i) dst[lane + 64 * i] = acc[i] * inv;
}

/* whether the tiled form takes this call: fp32 q and KV, dim 64 or 128,
   every row and the output on 16-byte boundaries, a tile's rows within a
   32-bit byte offset */
bool tile_eligible(const AttentionF32Params& p) {
    auto aligned = [](const void* x) { return (reinterpret_cast<uintptr_t>(x) & 15) == 0; };
    return p.qType == 0 && p.kvType == 0 && (p.dim == 64 || p.dim == 128) && aligned(p.q) && aligned(p.keys) &&
           aligned(p.values) && aligned(p.out) && p.qStride % 4 == 0 && p.posStride % 4 == 0 &&
           p.headStride % 4 == 0 && p.posStride < (uint64_t(1) << 22);
}

/* room for a.splits records of every row */
bool split_records(TileArgs& a) {
    const AttentionF32Params& p = a.p;
    const size_t accBytes = size_t(a.splits) * p.heads * p.count * p.dim * 4;
    char* parts = static_cast<char*>(
        Context::instance().grow(SLOT_ATTN_PARTS, accBytes + size_t(a.splits) * p.heads * p.count * 8));
    if (!parts) return false;
    a.acc = reinterpret_cast<float*>(parts);
    a.ml = reinterpret_cast<float2*>(parts + accBytes);
    return true;
}

bool launch_merge(const TileArgs& a, hipStream_t stream) {
    const bool d64 = a.p.dim == 64;
    const uint64_t mblocks = (a.p.count * a.p.heads + 3) / 4;
    return Context::instance().launch("attention_f32_merge_kernel", stream, [&] {
        if (d64) hipLaunchKernelGGL(attention_f32_merge_kernel<64>, dim3(unsigned(mblocks)), dim3(256), 0, stream, a);
        else hipLaunchKernelGGL(attention_f32_merge_kernel<128>, dim3(unsigned(mblocks)), dim3(256), 0, stream, a);
    });
}

/*
    Tiled or narrow, and the narrow form's splits: by the modelled time (us)
    of each. A workgroup's serial chain sets both: `rounds` workgroups per
    CU, each walking its longest key range. A tile of 64 keys x 128 tokens
    takes 9 us of a CU at dim 128 (two workgroups of dim 64 share one); a
    narrow step, a block of 16 keys in each of NW waves, 3.2 us at dim 128 and
    1.5 at 64; a merge launch 2.8 to 3.8 us and its records. The constants
    are fitted to 140 shapes, 1 to 512 tokens behind 0 to 2000 positions at
    five head counts (7% rms); 8% closer than that, the tiled form keeps the
    call. 128 tokens from empty at 12 x 64: 15.9 -> 10.3 us, at 32q/8kv x 128
    24.3 -> 11.8; one token after 2000 at 32q/8kv x 128 48.5 -> 14.9; 64
    tokens after 2000 62.5 -> 42.3. Where tiles fill the chip they read K and
    V for eight times the rows: 256 tokens after 2000 at 32q/8kv x 128 take
    108 us tiled, 118 narrow; 700 from empty at 64 x 128, window 256, 101 and
    126.
*/
double merge_cost(bool d64, bool narrow, double recordBytes) {
    return narrow ? 2.8 + recordBytes * (d64 ? 0.3e-6 : 1.2e-6) : 3.8 + recordBytes * 0.9e-6;
}

double rounds(uint64_t blocks, uint64_t slots) { return double((blocks + slots - 1) / slots); }

/* the narrow form's splits for this call, or 0 where the tiled form's
   `tiled` us are less */
uint32_t narrow_splits(const AttentionF32Params& p, double tiled) {
    // rows and positions in 32 bits
    if (p.count >= (1u << 30) || p.start >= (1u << 30) || p.heads >= (1u << 20) ||
        p.count * p.heads >= (uint64_t(1) << 30))
        return 0;
    const bool d64 = p.dim == 64;
    const uint64_t G = p.heads / p.kvHeads, wgs = (p.count * G + NR - 1) / NR * p.kvHeads;
    uint64_t keys = p.start + p.count;                       // the longest row group's
    const uint64_t span = (NR + G - 1) / G;                  // tokens of a row group, less one
    if (p.window && p.window + span < keys) keys = p.window + span;
    const uint64_t nb = (keys + NB - 1) / NB;
    const uint64_t rowBytes = p.count * p.heads * (p.dim * 4 + 8);
    uint32_t best = 0;
    for (uint32_t sp = 1; sp == 1 || (4 * sp <= nb && sp <= 64 && sp * rowBytes <= (uint64_t(256) << 20)); sp *= 2) {
        const double steps = double((nb + uint64_t(NW) * sp - 1) / (uint64_t(NW) * sp));
        const double us = 8.0 + rounds(wgs * sp, 256) * (d64 ? 1.5 * steps + 0.4 : 3.2 * steps) +
                          (sp > 1 ? merge_cost(d64, true, double(sp * rowBytes)) : 0.0);
        if (us < tiled) tiled = us, best = sp;
    }
    return best;
}

bool launch_narrow(TileArgs a, hipStream_t stream, uint32_t splits) {
    Context& ctx = Context::instance();
    const AttentionF32Params& p = a.p;
    a.groups = uint32_t((p.count * (p.heads / p.kvHeads) + NR - 1) / NR);
    a.splits = splits;
    a.tilesPerSplit = 0;
    if (a.splits > 1 && !split_records(a)) return false;
    const uint64_t blocks = uint64_t(a.groups) * p.kvHeads * a.splits;
    if (!ctx.launch("attention_f32_narrow_kernel", stream, [&] {
            if (p.dim == 64)
                hipLaunchKernelGGL(attention_f32_narrow_kernel<64>, dim3(unsigned(blocks)), dim3(64 * NW), 0, stream, a);
            else
                hipLaunchKernelGGL(attention_f32_narrow_kernel<128>, dim3(unsigned(blocks)), dim3(64 * NW), 0, stream, a);
        }))
        return false;
    return a.splits == 1 || launch_merge(a, stream);
}

bool launch_tiled(const AttentionF32Params& p, hipStream_t stream) {
    Context& ctx = Context::instance();
    TileArgs a{};
    a.p = p;
    const uint64_t groups = (p.count + TQ - 1) / TQ;
    uint64_t total = 0;
    uint32_t maxTiles = 0;
    for (uint64_t g = 0; g < groups; ++g) {
        uint64_t kbeg;
        uint32_t nt;
        group_tiles(p.count, p.start, p.window, g, kbeg, nt);
        total += nt;
        maxTiles = nt > maxTiles ? nt : maxTiles;
    }
    total *= p.heads;
    // split the key ranges when the (group, head) pairs alone leave workgroup
    // slots of the 256 CUs empty (one workgroup per CU at dim 128, two at 64),
    // and the records stay under 256 MB
    const uint64_t slots = p.dim == 64 ? 512 : 256;
    uint64_t tps = (total + slots - 1) / slots;
    const uint64_t perSplit = p.heads * p.count * (p.dim * 4 + 8);
    while (tps < maxTiles && ((maxTiles + tps - 1) / tps) * perSplit > (uint64_t(256) << 20)) tps *= 2;
    a.groups = uint32_t(groups);
    a.splits = tps < maxTiles ? uint32_t((maxTiles + tps - 1) / tps) : 1u;
    a.tilesPerSplit = a.splits > 1 ? uint32_t(tps) : maxTiles;
    uint64_t live = 0;   // workgroups with tiles
    for (uint64_t g = 0; g < groups; ++g) {
        uint64_t kbeg;
        uint32_t nt;
        group_tiles(p.count, p.start, p.window, g, kbeg, nt);
        live += (nt + a.tilesPerSplit - 1) / a.tilesPerSplit;
    }
    double tiles = rounds(live * p.heads, slots) * a.tilesPerSplit;
    if (a.splits == 1) {   // ranges of all lengths, the longest first: they even out over the CUs
        const double even = double(total) / double(slots) + 0.25 * maxTiles;
        tiles = tiles < even ? tiles : even;
    }
    const double us = (p.dim == 64 ? 2.0 : 7.0) + 9.0 * tiles +
                      (a.splits > 1 ? merge_cost(p.dim == 64, false, double(a.splits * perSplit)) : 0.0);
    if (const uint32_t sp = narrow_splits(p, 0.92 * us)) return launch_narrow(a, stream, sp);
    const uint64_t blocks = groups * p.heads * a.splits;
    if (blocks > 0x7FFFFFFFull) return ctx.fail("attention: too many tasks");
    if (a.splits > 1 && !split_records(a)) return false;
    const bool d64 = p.dim == 64;
    if (!ctx.launch("attention_f32_tile_kernel", stream, [&] {
            if (d64) hipLaunchKernelGGL(attention_f32_tile_kernel<64>, dim3(unsigned(blocks)), dim3(256), 0, stream, a);
            else hipLaunchKernelGGL(attention_f32_tile_kernel<128>, dim3(unsigned(blocks)), dim3(256), 0, stream, a);
        }))
        return false;
    return a.splits == 1 || launch_merge(a, stream);
}

} // namespace

bool launch_attention_f32(const AttentionF32Params& p, hipStream_t stream) {
    Context& ctx = Context::instance();
    if (p.dim == 0 || p.dim > MAX_DIM) return ctx.fail("attention: dim must be 1..256");
    if (p.kvHeads == 0 || p.heads % p.kvHeads) return ctx.fail("attention: heads must be a multiple of kvHeads");
    if (p.qStride < p.dim) return ctx.fail("attention: qStride < dim");
    const uint64_t tasks = p.count * p.heads;
    if (tasks == 0) return true;
    if (tile_eligible(p)) return launch_tiled(p, stream);
    const uint64_t blocks = (tasks + 3) / 4;
    if (blocks > 0x7FFFFFFFull) return ctx.fail("attention: too many tasks");
    return ctx.launch("attention_f32_kernel", stream, [&] {
        hipLaunchKernelGGL(attention_f32_kernel, dim3(unsigned(blocks)), dim3(256), 0, stream, p);
    });
}

} // namespace aigpu
