// latent.hip - multi-head latent attention (latentAttentionMixer,
// LocalModel.hpp:3086-3163; DeepSeek's MLA as GLM-5.3 uses it, without
// positional encoding). Every token's key and value are one kvLoraRank-wide
// latent c; head h's key would be Wk_h c and its value Wv_h c, Wk_h and Wv_h
// its rows of kv_b_proj. Both are linear, so
//   q . (Wk_h c) = (Wk_h^T q) . c         sum_j p_j Wv_h c_j = Wv_h (sum_j p_j c_j)
// and nothing is ever expanded:
//   latent_fold_kernel    folded[t][h] = Wk_h^T q[t][h]
//   latent_attn_kernel    softmax(folded . c_j * scale) over the token's keys
//                         (all positions up to it, or the indexer's sorted
//                         selection), context = sum p_j c_j, on the fp32
//                         matrix cores; every cached latent is read once per
//                         group of 16 or 32 heads
//   latent_unfold_kernel  (decode-sized calls: the key splits combined, then)
//                         out[t][h] = Wv_h context[t][h]
// fp32 throughout, as the reference computes it; kv_b_proj may be fp32 or
// bf16 (widened).
#include "context.hpp"
#include "device.hpp"
#include "kernels.hpp"

namespace aigpu {

namespace {

constexpr int KB = 32;          // keys per block
constexpr int MAX_RANK = 512;   // kvLoraRank
constexpr int MAX_NOPE = 256;
constexpr int RS = MAX_RANK + 4;   // LDS row stride of a block's latents
constexpr int PS = KB + 4;         // and of its scores and probabilities

struct LatentArgs {
    LatentParams p;
    float* folded;    // [count][heads][C]
    float* context;   // [count][heads][C]
    float* partial;   // [count][heads][splits][C + 4]: max, sum, two unused, acc
    uint32_t splits;
};

typedef u32x4 __attribute__((aligned(4))) u32x4_a4;   // kv_b_proj's rows need not be 16-byte aligned

/* 16 bytes of kv_b_proj (8 bf16 or 4 fp32 elements from index i) as fp32 */
template <bool BF16>
__device__ __forceinline__ void wkv_piece(const u32x4 w, float (&x)[BF16 ? 8 : 4]) {
#pragma unroll
    for (int e = 0; e < 4; ++e) {
        if constexpr (BF16) {
            x[2 * e] = __uint_as_float(w[e] << 16);
            x[2 * e + 1] = __uint_as_float(w[e] & 0xFFFF0000u);
        } else {
            x[e] = __uint_as_float(w[e]);
        }
    }
}
template <bool BF16>
__device__ __forceinline__ u32x4 wkv_load(const void* w, size_t i) {
    return *reinterpret_cast<const u32x4_a4*>(static_cast<const char*>(w) + i * (BF16 ? 2 : 4));
}

/* folded[t][h][c] = sum_d q[t][h][d] Wk_h[d][c] (:3124-3129): workgroup
   (head, 256 columns, TT tokens). Bound by reading Wk: each lane takes 16
   bytes of a row, 256 / (256 / E) rows at once, eight of its rows in flight;
   the row slots' sums are added in LDS. One token, 128 heads, nope 128, rank
   512, bf16: 4.9 us (13.6 with 2-byte loads, one row at a time). */
template <bool BF16, int TT>
__global__ __launch_bounds__(256) void latent_fold_kernel(LatentArgs a) {
    constexpr int E = BF16 ? 8 : 4, SLOTS = E;   // 256 columns / E lanes a row: E row slots
    __shared__ float qs[TT][MAX_NOPE];
    __shared__ __align__(16) float part[SLOTS][TT][256];
    const LatentParams& p = a.p;
    const uint32_t tid = threadIdx.x, h = blockIdx.x, slot = tid / (256 / E), cl = E * (tid % (256 / E));
    const uint32_t c = blockIdx.y * 256 + cl;
    const uint64_t t0 = uint64_t(blockIdx.z) * TT;
    const uint32_t Dn = uint32_t(p.nope), C = uint32_t(p.rank);
    const size_t wk = size_t(h) * (p.nope + p.vdim) * C;
    const bool in = c < C;   // C % 16 == 0: a piece is in or out whole
    float acc[TT][E] = {};
    bool staged = false;
    for (uint32_t d0 = slot; d0 < Dn + slot; d0 += 8 * SLOTS) {   // the same passes for every slot
        u32x4 wv[8];
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t d = d0 + SLOTS * u;
            wv[u] = in && d < Dn ? wkv_load<BF16>(p.wkv, wk + size_t(d) * C + c) : u32x4{0u, 0u, 0u, 0u};
        }
        if (!staged) {   // q while the first rows are in flight; zeros past nope
            staged = true;
            for (uint32_t i = tid; i < TT * MAX_NOPE; i += 256) {
                const uint32_t t = i / MAX_NOPE, d = i % MAX_NOPE;
                qs[t][d] = t0 + t < p.count && d < Dn ? p.q[((t0 + t) * p.heads + h) * Dn + d] : 0.0f;
            }
            __syncthreads();
        }
#pragma unroll
        for (int u = 0; u < 8; ++u) {
            const uint32_t d = d0 + SLOTS * u;
            if (d < Dn) {
                float x[E];
                wkv_piece<BF16>(wv[u], x);
#pragma unroll
                for (int t = 0; t < TT; ++t)
#pragma unroll
                    for (int e = 0; e < E; ++e) acc[t][e] = fmaf(qs[t][d], x[e], acc[t][e]);
            }
        }
    }
#pragma unroll
    for (int t = 0; t < TT; ++t)
#pragma unroll
        for (int e = 0; e < E; e += 4)
            *reinterpret_cast<floatx4*>(&part[slot][t][cl + e]) = floatx4{acc[t][e], acc[t][e + 1], acc[t][e + 2], acc[t][e + 3]};
    __syncthreads();
    const uint32_t oc = blockIdx.y * 256 + tid;
    if (oc < C) {
#pragma unroll
        for (int t = 0; t < TT; ++t) {
            if (t0 + t >= p.count) break;
            float s = 0.0f;
#pragma unroll
            for (int i = 0; i < SLOTS; ++i) s += part[i][t][tid];
            a.folded[((t0 + t) * p.heads + h) * C + oc] = s;
        }
    }
}

__device__ __forceinline__ floatx4 mfma4(float a, float b, floatx4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

/* 1 / the sum of a token's probabilities. An empty selection (no key at or
   before the token) leaves the context at zero, as the mixer's job does; keys
   whose scores are all -inf have no softmax: NaN, as a NaN among them gives. */
__device__ __forceinline__ float context_scale(float l, bool empty) {
    return l != 0.0f ? 1.0f / l : (empty ? 0.0f : __builtin_nanf(""));
}

/*
    Workgroup (token, 16 RT heads, key split), eight waves: online softmax over
    blocks of 32 keys. A block's latents come in by DMA (two 1 KB pieces a
    row) into one of two LDS buffers while the other one computes, and serve
    both products, on v_mfma_f32_16x16x4f32:
      scores   KP waves share a 16 x 16 (heads x keys) tile, each a part of the
               rank; its folded queries stay in registers for the whole launch
      context  wave w owns columns 64 w .. + 63 of all 16 RT heads; the k slots
               of step s are keys 16 (s / 4) + 4 g + s % 4, so the
               probabilities are 16-byte reads and the latents' four rows lie
               16 banks apart (row stride 516 floats; the scores' reads, one
               row a lane, then fall on distinct banks too)
    32 heads where there are more than 16: half the reads of the latents per
    head. One token against 4,097 latents, 128 heads, rank 512: 27 us (111 with
    fp32 FMAs from LDS, 16 heads a workgroup): about 10 before the first
    products are done and 5 per block, whose products take 3.7.
*/
template <int RT>
__global__ __launch_bounds__(512, 2) void latent_attn_kernel(LatentArgs a) {
    constexpr int KP = 4 / RT;                 // parts of the rank
    constexpr int KQ = MAX_RANK / KP / 16;     // 16-wide steps of a part
    constexpr int TPR = 512 / (16 * RT), KPT = KB / TPR;   // softmax: threads per head, keys per thread
    __shared__ __align__(16) float cb[2][KB * RS];
    __shared__ __align__(16) float sp[KP][16 * RT * PS];
    __shared__ __align__(16) float pr[16 * RT * PS];
    __shared__ __align__(16) float alpha[16 * RT];

    const LatentParams& p = a.p;
    const uint64_t t = blockIdx.x;
    const uint32_t h0 = blockIdx.y * 16 * RT, s = blockIdx.z;
    const uint32_t C = uint32_t(p.rank);
    const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, c16 = lane & 15;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const uint64_t pos = p.startPos + t;
    const bool dense = !p.selCount || p.selCount[t] == 0xFFFFFFFFu;
    const uint32_t n = dense ? uint32_t(pos + 1) : p.selCount[t];   // keys are 32-bit indices
    const uint32_t* sel = dense ? nullptr : p.selKeys + p.selStart[t];
    // this split's keys [kBegin, kEnd) of the token's n, the splits even to a key
    const uint32_t each = n / a.splits, more = n % a.splits;
    const uint32_t kBegin = s * each + (s < more ? s : more), kEnd = kBegin + each + (s < more ? 1 : 0);

    // rows 4 w .. + 3 of a block; rows past the end repeat the last key (their
    // probability is 0), columns past C the row's first (their query is 0,
    // their context not stored)
    const uint32_t lds0 = lds_address(cb[0]) + 4 * w * RS * 4, lds1 = lds_address(cb[1]) + 4 * w * RS * 4;
    uint32_t keyv = 0;   // lane r (and r + 32): the key of row r of the block to be requested next
    auto find = [&](uint32_t k0) {
        uint32_t i = k0 + (lane & 31);
        if (i >= kEnd) i = kEnd - 1;
        keyv = dense ? i : sel[i];
    };
    uint32_t off[2];
#pragma unroll
    for (int hf = 0; hf < 2; ++hf) {
        const uint32_t c = 256 * hf + 4 * lane;
        off[hf] = (c < C ? c : 0) * 4;
    }
    auto issue = [&](uint32_t lds) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float* row = p.latent + size_t(uint32_t(__builtin_amdgcn_readlane(keyv, 4 * w + r))) * C;
#pragma unroll
            for (int hf = 0; hf < 2; ++hf) dma_block(row, off[hf], lds + r * RS * 4 + hf * 1024);
        }
    };
    if (kBegin < kEnd) {
        find(kBegin);
        issue(lds0);
        find(kBegin + KB);
    }

    // the wave's score tile: heads 16 rb .., keys 16 ct .., rank part kp
    const int rb = RT == 2 ? w & 1 : 0, ct = RT == 2 ? (w >> 1) & 1 : w & 1, kp = RT == 2 ? w >> 2 : w >> 1;
    floatx4 fa[KQ];
    {
        const uint32_t h = h0 + 16 * rb + c16;
        const float* row = a.folded + (t * p.heads + (h < p.heads ? h : p.heads - 1)) * C;
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            const uint32_t c = kp * (MAX_RANK / KP) + 16 * q + 4 * g;
            fa[q] = *reinterpret_cast<const floatx4*>(row + (c < C ? c : 0));   // in flight together: no branch
        }
#pragma unroll
        for (int q = 0; q < KQ; ++q) {
            const bool live = h < p.heads && kp * (MAX_RANK / KP) + 16 * q + 4 * g < C;
#pragma unroll
            for (int e = 0; e < 4; ++e) fa[q][e] = live ? fa[q][e] : 0.0f;
        }
    }
    // the folded queries have landed (with the first block): no wait inside the
    // loop then stands for them and, with them, for the next block's DMA
    __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));   // vmcnt(0)

    floatx4 acc[RT][4];
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < 4; ++j) acc[i][j] = floatx4{0.0f, 0.0f, 0.0f, 0.0f};
    // softmax: thread (head sr, keys sk ..)
    const int sr = tid / TPR, sk = KPT * (tid % TPR);
    float m = -INFINITY, l = 0.0f;
    auto ld4 = [](const float* ptr) { return *reinterpret_cast<const floatx4*>(ptr); };
    int buf = 0;
    for (uint32_t k0 = kBegin; k0 < kEnd; k0 += KB, buf ^= 1) {
        const bool second = kEnd - k0 > 16;   // keys 16 .. 31 of the block: a split's last block may have none
        // the other buffer's reads ended before the last barrier
        if (k0 + KB < kEnd) {
            issue(buf ? lds0 : lds1);
            __builtin_amdgcn_s_waitcnt(8 | (7 << 4) | (15 << 8));   // vmcnt(8): this block's eight have landed
            if (k0 + 2 * KB < kEnd) find(k0 + 2 * KB);
        } else {
            __builtin_amdgcn_s_waitcnt((7 << 4) | (15 << 8));       // vmcnt(0)
        }
        lds_barrier();
        const float* cbuf = cb[buf];
        if (ct == 0 || second) {   // scores
            floatx4 x0 = {0.0f, 0.0f, 0.0f, 0.0f}, x1 = x0;
            const float* row = cbuf + (16 * ct + c16) * RS + kp * (MAX_RANK / KP) + 4 * g;
            constexpr int AHEAD = 8;   // operand reads ahead of their products
            floatx4 kv[AHEAD];
#pragma unroll
            for (int q = 0; q < AHEAD; ++q) kv[q] = ld4(row + 16 * q);
#pragma unroll
            for (int q = 0; q < KQ; q += 2) {
                const floatx4 k0v = kv[q % AHEAD], k1v = kv[(q + 1) % AHEAD];
                if (q + AHEAD < KQ) {
                    kv[q % AHEAD] = ld4(row + 16 * (q + AHEAD));
                    kv[(q + 1) % AHEAD] = ld4(row + 16 * (q + 1 + AHEAD));
                }
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    x0 = mfma4(fa[q][e], k0v[e], x0);
                    x1 = mfma4(fa[q + 1][e], k1v[e], x1);
                }
            }
#pragma unroll
            for (int r = 0; r < 4; ++r) sp[kp][(16 * rb + 4 * g + r) * PS + 16 * ct + c16] = x0[r] + x1[r];
        }
        lds_barrier();
        {   // softmax of the block's 32 keys
            float x[KPT], mx = -INFINITY;
#pragma unroll
            for (int e = 0; e < KPT; ++e) {
                float v = 0.0f;
#pragma unroll
                for (int k = 0; k < KP; ++k) v += sp[k][sr * PS + sk + e];
                x[e] = k0 + sk + e < kEnd ? v * p.scale : -INFINITY;
                mx = fmaxf(mx, x[e]);
            }
#pragma unroll
            for (int o = 1; o < TPR; o <<= 1) mx = fmaxf(mx, __shfl_xor(mx, o, WAVE));
            const float mn = fmaxf(m, mx), mz = mn == -INFINITY ? 0.0f : mn;   // all -inf so far: zeros (or NaN)
            const float f = expf(m - mz);    // 0 on the first block
            m = mn;
            float ps = 0.0f;
#pragma unroll
            for (int e = 0; e < KPT; ++e) {
                const float pe = expf(x[e] - mz);
                pr[sr * PS + sk + e] = pe;
                ps += pe;
            }
            l = l * f + ps;
            if (sk == 0) alpha[sr] = f;
        }
        lds_barrier();
        {   // context
#pragma unroll
            for (int i = 0; i < RT; ++i) {
                const floatx4 f4 = ld4(&alpha[16 * i + 4 * g]);
#pragma unroll
                for (int j = 0; j < 4; ++j)
#pragma unroll
                    for (int r = 0; r < 4; ++r) acc[i][j][r] *= f4[r];
            }
            floatx4 pa[KB / 16][RT];
            float v[KB / 16][4][4];
            auto read = [&](int q) __attribute__((always_inline)) {
#pragma unroll
                for (int i = 0; i < RT; ++i) pa[q][i] = ld4(&pr[(16 * i + c16) * PS + 16 * q + 4 * g]);
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < 4; ++j) v[q][e][j] = cbuf[(16 * q + 4 * g + e) * RS + 64 * w + c16 + 16 * j];
            };
            auto add = [&](int q) __attribute__((always_inline)) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < 4; ++j)
#pragma unroll
                        for (int i = 0; i < RT; ++i) acc[i][j] = mfma4(pa[q][i][e], v[q][e][j], acc[i][j]);
            };
            read(0);
            read(1);   // rows past the end repeat a live key; their probabilities are 0
            add(0);
            if (second) add(1);
        }
        lds_barrier();   // the next block's latents, scores and probabilities go into what this one read
    }
#pragma unroll
    for (int o = 1; o < TPR; o <<= 1) l += __shfl_xor(l, o, WAVE);

    if (a.splits == 1) {
        if (sk == 0) alpha[sr] = context_scale(l, n == 0);
        __syncthreads();
    }
    const size_t rec = size_t(C) + 4;
#pragma unroll
    for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const uint32_t h = h0 + 16 * i + 4 * g + r;
            if (h >= p.heads) continue;
            float* out = a.splits == 1 ? a.context + (t * p.heads + h) * C : a.partial + ((t * p.heads + h) * a.splits + s) * rec + 4;
            const float f = a.splits == 1 ? alpha[16 * i + 4 * g + r] : 1.0f;
#pragma unroll
            for (int j = 0; j < 4; ++j) {
                const uint32_t c = 64 * w + 16 * j + c16;
                if (c < C) out[c] = acc[i][j][r] * f;
            }
        }
    if (a.splits > 1 && sk == 0 && h0 + sr < p.heads) {
        float* out = a.partial + ((t * p.heads + h0 + sr) * a.splits + s) * rec;
        out[0] = m;
        out[1] = l;
    }
}

/* out[t][h][v] = Wv_h[v] . context[t][h] (:3153-3154): workgroup (head, 64 v
   rows, TT tokens), each wave 16 of the rows, the lanes along the rank. Bound
   by reading Wv: the wave's first VB rows are requested before the contexts
   are formed (with splits, from their records: the at most 64 maxima and sums
   with a lane per split, then the accumulators column by column). One token,
   128 heads, 64 splits, v 128, rank 512, bf16: 10.5 us (a merge launch of its
   own 8.5, then 31.9 a row at a time). */
template <bool BF16, int TT>
__global__ __launch_bounds__(256) void latent_unfold_kernel(LatentArgs a) {
    constexpr int E = BF16 ? 8 : 4, PC = MAX_RANK / (E * WAVE);   // pieces per lane and row: 1 or 2
    constexpr int VB = 8;                                         // rows in flight
    __shared__ __align__(16) float cs[TT][MAX_RANK];
    __shared__ __align__(16) float half[128][4];
    const LatentParams& p = a.p;
    const uint32_t h = blockIdx.x;
    const uint64_t t0 = uint64_t(blockIdx.z) * TT;
    const uint32_t C = uint32_t(p.rank), Dv = uint32_t(p.vdim);
    const int tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const size_t wv0 = (size_t(h) * (p.nope + p.vdim) + p.nope) * C;
    const uint32_t v0 = blockIdx.y * 64 + 16 * w;
    u32x4 wr[VB][PC];
    auto fetch = [&](uint32_t v) {
#pragma unroll
        for (int u = 0; u < VB; ++u)
#pragma unroll
            for (int e = 0; e < PC; ++e) {
                const uint32_t c = E * (lane + WAVE * e);
                wr[u][e] = v + u < Dv && c < C ? wkv_load<BF16>(p.wkv, wv0 + size_t(v + u) * C + c) : u32x4{0u, 0u, 0u, 0u};
            }
    };
    fetch(v0);
    const int tn = int(p.count - t0 < uint64_t(TT) ? p.count - t0 : uint64_t(TT));
    if (a.splits == 1) {
        for (uint32_t i = tid; i < TT * MAX_RANK / 4; i += 256) {
            const uint32_t t = i / (MAX_RANK / 4), c = 4 * (i % (MAX_RANK / 4));
            *reinterpret_cast<floatx4*>(&cs[t][c]) =
                int(t) < tn && c < C ? *reinterpret_cast<const floatx4*>(&a.context[((t0 + t) * p.heads + h) * C + c])
                                     : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    } else {
        const size_t rec = size_t(C) + 4;
        const uint32_t c = 4 * (tid & 127), odd = tid >> 7;   // columns c .. + 3 of the even or the odd splits
        for (int t = 0; t < tn; ++t) {
            const float* base = a.partial + ((t0 + t) * p.heads + h) * a.splits * rec;
            const bool mine = lane < int(a.splits);
            const float mi = mine ? base[lane * rec] : -INFINITY;
            const float li = mine ? base[lane * rec + 1] : 0.0f;
            const float M = wave_max(mi);
            const float fi = mi != -INFINITY ? expf(mi - M) : 0.0f;
            const float L = wave_sum(li * fi);
            const float inv = context_scale(L, p.selCount && p.selCount[t0 + t] == 0);
            floatx4 sum = {0.0f, 0.0f, 0.0f, 0.0f};
            for (uint32_t i0 = odd; i0 < a.splits; i0 += 16) {   // eight records in flight
                floatx4 x[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const uint32_t i = i0 + 2 * u;
                    x[u] = i < a.splits && c < C ? *reinterpret_cast<const floatx4*>(base + i * rec + 4 + c)
                                                 : floatx4{0.0f, 0.0f, 0.0f, 0.0f};
                }
#pragma unroll
                for (int u = 0; u < 8; ++u) {
                    const float f = __shfl(fi, int((i0 + 2 * u) & 63), WAVE);   // lanes past the splits hold 0
#pragma unroll
                    for (int e = 0; e < 4; ++e) sum[e] = fmaf(x[u][e], f, sum[e]);
                }
            }
            if (odd) *reinterpret_cast<floatx4*>(half[tid & 127]) = sum;
            __syncthreads();
            if (!odd) {
                const floatx4 o = *reinterpret_cast<const floatx4*>(half[tid]);
#pragma unroll
                for (int e = 0; e < 4; ++e) sum[e] = (sum[e] + o[e]) * inv;
                *reinterpret_cast<floatx4*>(&cs[t][c]) = sum;
            }
            __syncthreads();
        }
    }
    __syncthreads();
    for (uint32_t v = v0; v < v0 + 16 && v < Dv; v += VB) {   // uniform over the wave
        if (v > v0) fetch(v);
        for (int t = 0; t < tn; ++t) {
            float acc[VB] = {};
#pragma unroll
            for (int e = 0; e < PC; ++e) {
                const int c = E * (lane + WAVE * e);
                float x[E];
#pragma unroll
                for (int k = 0; k < E; k += 4) {
                    const floatx4 v4 = *reinterpret_cast<const floatx4*>(&cs[t][c + k]);
#pragma unroll
                    for (int i = 0; i < 4; ++i) x[k + i] = v4[i];
                }
#pragma unroll
                for (int u = 0; u < VB; ++u) {
                    float y[E];
                    wkv_piece<BF16>(wr[u][e], y);
#pragma unroll
                    for (int k = 0; k < E; ++k) acc[u] = fmaf(y[k], x[k], acc[u]);
                }
            }
            // the eight rows' sums over the lanes at once: each exchange halves
            // the rows a lane holds; lane l ends with row (l / 8)'s
#pragma unroll
            for (int k = VB / 2, bit = 32; k > 0; k >>= 1, bit >>= 1) {
                const bool up = lane & bit;
#pragma unroll
                for (int u = 0; u < k; ++u) {
                    const float give = up ? acc[u] : acc[u + k], keep = up ? acc[u + k] : acc[u];
                    acc[u] = keep + __shfl_xor(give, bit, WAVE);
                }
            }
            float r = acc[0];
#pragma unroll
            for (int o = 4; o > 0; o >>= 1) r += __shfl_xor(r, o, WAVE);
            const uint32_t row = v + uint32_t(lane >> 3);
            if ((lane & 7) == 0 && row < Dv) p.out[((t0 + t) * p.heads + h) * Dv + row] = r;
        }
    }
}

} // namespace

bool launch_latent_attention(const LatentParams& p, hipStream_t stream) {
    Context& ctx = Context::instance();
    if (!p.q || !p.latent || !p.wkv || !p.out) return ctx.fail("latent attention: null tensor");
    if (p.selCount && (!p.selStart || !p.selKeys)) return ctx.fail("latent attention: a selection needs start and keys");
    if (p.wType > 1) return ctx.fail("latent attention: kv_b_proj must be fp32 or bf16");
    if (p.rank == 0 || p.rank > uint64_t(MAX_RANK) || p.rank % 16)
        return ctx.fail("latent attention: kvLoraRank must be a multiple of 16 up to 512");
    if (p.nope == 0 || p.nope > uint64_t(MAX_NOPE)) return ctx.fail("latent attention: qk_nope_head_dim must be 1 to 256");
    if (p.vdim == 0 || p.vdim > 256) return ctx.fail("latent attention: v_head_dim must be 1 to 256");
    if (p.heads == 0) return ctx.fail("latent attention: no heads");
    if (reinterpret_cast<uintptr_t>(p.latent) % 16) return ctx.fail("latent attention: latents must be 16-byte aligned");
    if (p.count == 0) return true;
    if (p.count > 0x7FFFFFFFull || p.heads > 65535u) return ctx.fail("latent attention: too many tokens or heads");
    LatentArgs a{};
    a.p = p;
    const uint32_t hg = p.heads > 16 ? 32 : 16;
    const uint32_t groups = uint32_t((p.heads + hg - 1) / hg);
    // decode-sized calls split the keys so that about 256 workgroups run
    const uint64_t maxKeys = p.startPos + p.count;
    const uint64_t maxBlocks = (maxKeys + KB - 1) / KB;
    uint64_t want = 256 / (p.count * groups);
    if (want > maxBlocks) want = maxBlocks;
    if (want < 1) want = 1;
    if (want > 64) want = 64;
    a.splits = uint32_t(want);
    const size_t cells = size_t(p.count) * p.heads * p.rank;
    const size_t bytes = (2 * cells + (a.splits > 1 ? size_t(p.count) * p.heads * a.splits * (p.rank + 4) : 0)) * 4;
    float* work = static_cast<float*>(ctx.grow(SLOT_LATENT, bytes));
    if (!work) return false;
    a.folded = work;
    a.context = work + cells;
    a.partial = work + 2 * cells;
    const bool bf16 = p.wType == 1, one = p.count == 1;
    const unsigned tokens = unsigned((p.count + 7) / 8);
    if (tokens > 65535u) return ctx.fail("latent attention: too many tokens for one call");
    const dim3 fgrid(unsigned(p.heads), unsigned((p.rank + 255) / 256), tokens);
    if (!ctx.launch("latent_fold_kernel", stream, [&] {
            if (bf16 && one) hipLaunchKernelGGL((latent_fold_kernel<true, 1>), fgrid, dim3(256), 0, stream, a);
            else if (bf16) hipLaunchKernelGGL((latent_fold_kernel<true, 8>), fgrid, dim3(256), 0, stream, a);
            else if (one) hipLaunchKernelGGL((latent_fold_kernel<false, 1>), fgrid, dim3(256), 0, stream, a);
            else hipLaunchKernelGGL((latent_fold_kernel<false, 8>), fgrid, dim3(256), 0, stream, a);
        }))
        return false;
    const dim3 agrid(unsigned(p.count), groups, a.splits);
    if (!ctx.launch("latent_attn_kernel", stream, [&] {
            if (hg == 32) hipLaunchKernelGGL(latent_attn_kernel<2>, agrid, dim3(512), 0, stream, a);
            else hipLaunchKernelGGL(latent_attn_kernel<1>, agrid, dim3(512), 0, stream, a);
        }))
        return false;
    const dim3 ugrid(unsigned(p.heads), unsigned((p.vdim + 63) / 64), tokens);
    return ctx.launch("latent_unfold_kernel", stream, [&] {
        if (bf16 && one) hipLaunchKernelGGL((latent_unfold_kernel<true, 1>), ugrid, dim3(256), 0, stream, a);
        else if (bf16) hipLaunchKernelGGL((latent_unfold_kernel<true, 8>), ugrid, dim3(256), 0, stream, a);
        else if (one) hipLaunchKernelGGL((latent_unfold_kernel<false, 1>), ugrid, dim3(256), 0, stream, a);
        else hipLaunchKernelGGL((latent_unfold_kernel<false, 8>), ugrid, dim3(256), 0, stream, a);
    });
}

} // namespace aigpu
