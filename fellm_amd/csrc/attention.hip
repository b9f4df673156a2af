// Paged decode attention over the KV cache the fused RoPE + KV append writes.
//
// Reference: crates/fellm-plugin-abi/src/attention_provider.rs:391-459
//   (reference_attention_paged_f32: per query head, online softmax over the
//   keys 0 .. seq-1, score = (q . k) * scale, keys older than the window
//   skipped when causal; out = sum p v / sum p), driven per batch row as
//   crates/backend-cpu/src/backend.rs:1286-1323 does (seq = row_lengths[row],
//   causal, window = attention_window) and as the CUDA plugin's
//   attention_paged_batch_heads launch (plugins/cuda_kernels/src/launchers.rs
//   :3394-3446) is fed; K/V rows as crates/fellm-plugin-abi/src/paged_ctx.rs
//   :138-174 address them.
//
// Work split.  One workgroup per (key split s, batch row b, KV head g), its
// four wavefronts (or one: one_wave below) taking every fourth pair of cache
// blocks and merging their (max, sum, accumulators) through LDS at the end; the
// G = n_heads / n_kv query heads that share KV head g are processed together
// (as up to 16 head slots), so every K/V byte is read once.  Both products of a
// pair of blocks (2 x 16 tokens) run on the matrix cores:
//  * S^T = K . Q^T by v_mfma_f32_16x16x32: A = a block's K rows (lane = token
//    lane % 16, dims 32c + 8 (lane / 16) .. +7 of step c), B = q.  For an f16
//    cache q is split into f16 high and low parts (two MFMAs per step), which
//    hold f16 values whole and f32 ones to 2^-23 relative where the low part
//    is normal (|q| above 2^-2), to 2^-25 absolute below; |q| above 65504
//    overflows.  A bf16 cache uses bf16 MFMAs and three parts: all 24 bits.
//  * Lane (head slot lane % 16, group lane / 16) then owns the scores of
//    tokens 4 group .. +3 of each block, which is the layout the second
//    product takes its B operand in, so the online softmax runs in f32 with
//    its maximum, rescaling factor and sum per lane, and nothing goes through
//    LDS.
//  * out^T = V^T . P^T: the probabilities in three parts, A = V^T assembled
//    from the lanes' row pieces by byte permutes, f32 accumulation.  Three bf16
//    parts hold all 24 bits.  The f16 parts do so down to p = 2^-28, to 2^-52
//    absolute below, since p is scaled by 2^15 and the second and third part
//    by 2^12 more; their sum is folded in by one FMA.  (Two parts kept 2^-23
//    and 2^-39, and took 0.2 us less for one row of 64 keys, 0.3 of 27.5 for
//    32768, 1 of 37 for 256 rows of 16 .. 256.)  The lower parts of q and p are
//    summed apart from the first, which keeps their bits.
// The next pair's K is requested once Q.K has read the registers, its V once
// P.V has.
//
// Bound by the cache's bytes.  Against the kernel before it (one wavefront per
// workgroup, P.V on the vector ALUs, two blocks ahead): 256 rows of 256 .. 4096
// keys, 64/8 heads of 128, bf16 (2.39 GB) 629 -> 414 us; the same of 4096 keys
// each 747 -> 709 (6.1 TB/s); one row of 32768 keys, 32/8 heads, f16 33.9 -> 27.6.
//
// Splits write unnormalised partial sums with their running max and
// denominator; a second kernel combines them.  A row whose keys fit one split
// is finished by that split and skipped by the combine.  Tokens outside
// [lo, seq) are masked with -inf and their V rows read as zero, so stale
// cache bytes never reach the output.
#include "common.hpp"

#include "fellm_rocm.h"

namespace fellm {
namespace {

typedef _Float16 half8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf8_t __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
using Rsrc = __amdgpu_buffer_rsrc_t;

constexpr uint32_t kBlockTokens = 16;  // tokens per cache block handled by one MFMA tile
// A split's partial record per head slot: HD sums, m, l and two unused
// floats, so that every record starts on a 16-byte boundary.
constexpr uint32_t kRecTail = 4;
// Wavefronts that share a split's blocks.  Measured (kernels of 1 / 2 / 4 / 8,
// f16, two parts of p): 256 rows of 256 .. 4096 keys 445 / 416 / 396 / 462 us, one row of 32768
// keys 31.6 / 26.3 / 27.3 / 31.0, 256 rows of 16 .. 256 keys 36 / 30 / 36 / 67.
constexpr uint32_t kDecodeWaves = 4;
// Cache policies of the K and V reads.  V is read once by whole lines, so it
// bypasses cache retention.  A K load instruction takes 64 bytes of each of
// 16 rows, half a line, and the next one the other half: non-temporal K reads
// fetched lines twice.  Measured (K, V non-temporal or not): 256 rows x 4096
// keys 677 us (V only), 724 (both), 733 (K only), 737 (neither).
constexpr int kKPolicy = 0, kVPolicy = 2;

struct PagedGeom {
    const uint8_t *arena;
    uint64_t arena_len;
    const uint32_t *table;
    uint64_t n_table;
    uint32_t n_logical, n_layers, layer, block_size;
    uint64_t block_bytes;
    uint32_t stride;  // elements per token row (n_kv * head_dim)
};

// Cache element policies: the matrix-core type and the splitting of an f32
// operand into kParts of them.
struct CacheF16 {
    static constexpr int kParts = 2, kPParts = 3;
    static constexpr float kPScale = 32768.0f;  // probabilities times this are split,
    static constexpr float kPLower = 4096.0f;   // the parts after the first times this more
    // Two values rounded to nearest even and packed; the remainders replace them.
    __device__ static uint32_t part(float &x, float &y) {
        typedef _Float16 half2_t __attribute__((ext_vector_type(2)));
        half2_t h;
        h[0] = (_Float16)x;
        h[1] = (_Float16)y;
        x = x - (float)h[0];
        y = y - (float)h[1];
        return __builtin_bit_cast(uint32_t, h);
    }
    __device__ static float widen(uint32_t low16) { return (float)__builtin_bit_cast(_Float16, (uint16_t)low16); }
    __device__ static f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(half8_t, a), __builtin_bit_cast(half8_t, b), c, 0,
                                                      0, 0);
    }
};

struct CacheBF16 {
    static constexpr int kParts = 3, kPParts = 3;
    static constexpr float kPScale = 1.0f, kPLower = 1.0f;
    __device__ static uint32_t part(float &x, float &y) {
        typedef __bf16 bf2_t __attribute__((ext_vector_type(2)));
        bf2_t h;
        h[0] = (__bf16)x;
        h[1] = (__bf16)y;
        const uint32_t u = __builtin_bit_cast(uint32_t, h);
        x = x - __uint_as_float(u << 16);
        y = y - __uint_as_float(u & 0xffff0000u);
        return u;
    }
    __device__ static float widen(uint32_t low16) { return __uint_as_float(low16 << 16); }
    __device__ static f32x4 mfma(u32x4 a, u32x4 b, f32x4 c) {
        return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf8_t, a), __builtin_bit_cast(bf8_t, b), c, 0, 0,
                                                       0);
    }
};

// v[0..7] as N operands, the first remainder times `lower`.
template <typename C, int N>
__device__ __forceinline__ void split8(const float (&v)[8], float lower, u32x4 (&o)[N]) {
    float rem[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) rem[i] = v[i];
#pragma unroll
    for (int p = 0; p < N; ++p)
#pragma unroll
        for (int w = 0; w < 4; ++w) {
            o[p][w] = C::part(rem[2 * w], rem[2 * w + 1]);
            if (p == 0) rem[2 * w] *= lower, rem[2 * w + 1] *= lower;
        }
}

// Keys [lo, seq) of a row: cache blocks [first, last) and how many of the
// launch's splits of bps blocks hold any.
struct RowKeys {
    uint32_t lo, seq, first, last, splits;
};
__device__ __forceinline__ RowKeys row_keys(uint32_t seq, uint32_t causal, uint32_t window, uint32_t bps,
                                            uint32_t splits) {
    RowKeys r;
    r.seq = seq;
    r.lo = (causal && window && seq > window) ? seq - window : 0;
    r.first = r.lo / kBlockTokens;
    r.last = (seq + kBlockTokens - 1) / kBlockTokens;
    r.splits = (r.last - r.first + bps - 1) / bps;
    if (r.splits > splits) r.splits = splits;  // a length past max_seq
    return r;
}

// Maximum over the four 16-lane rows; every lane gets the result.
__device__ __forceinline__ float rows_max(float v) {
    const uint32_t u = __float_as_uint(v);
    const auto a = __builtin_amdgcn_permlane32_swap(u, u, false, false);
    v = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
    const uint32_t w = __float_as_uint(v);
    const auto b = __builtin_amdgcn_permlane16_swap(w, w, false, false);
    return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// Q: query activation policy, O: output policy, C: cache policy, HD: head
// dim (64, 128 or 256), W: wavefronts.  solo: pairs of blocks that one
// wavefront takes alone.  rec_heads: head slots of a partial record.  early:
// the first blocks are requested before the row length is known.
template <typename Q, typename O, typename C, int HD, uint32_t W>
__global__ __launch_bounds__(kWave *W, HD == 64 && C::kParts == 2 ? 4 : 1) void paged_decode_kernel(const typename Q::T *__restrict__ q,
                                                             typename O::T *__restrict__ out,
                                                             float *__restrict__ part, const uint32_t *__restrict__ lens,
                                                             PagedGeom geo, uint32_t batch, uint32_t n_heads,
                                                             uint32_t n_kv, float scale, uint32_t causal,
                                                             uint32_t window, uint32_t splits, uint32_t bps,
                                                             uint32_t rec_heads, uint32_t early, uint32_t solo) {
    constexpr int NC = HD / 32;               // Q.K steps, and 16-byte K loads per lane and block
    constexpr int DP = HD < 128 ? 4 : 8;      // consecutive dims of a lane's V piece
    constexpr int VH = HD / 16 / DP;          // V pieces per token row
    constexpr int NT = HD / 16;               // output tiles
    constexpr float kUnscale = 1.0f / C::kPScale;

    extern __shared__ __align__(16) float merge_lds[];
    const uint32_t lane = threadIdx.x % kWave, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t col = lane % 16, grp = lane / 16;
    // Splits in the outer order: the later ones, which fewer rows reach, come last.
    const uint32_t bg = blockIdx.x % (batch * n_kv), s = blockIdx.x / (batch * n_kv);
    const uint32_t g = bg % n_kv, b = bg / n_kv;
    const uint32_t G = n_heads / n_kv;
    const uint32_t row_bytes = geo.stride * 2;
    const size_t table_base = ((size_t)b * geo.n_layers + geo.layer) * geo.n_logical;

    // This wavefront's pairs of blocks: first + 2 (way + ways n), n = 0, 1, ..
    // Lane l holds the physical block (~0: none, or at or past lim) of block
    // l % 2 of pair tab0 + l / 2; a walk of more than 32 pairs reloads.
    uint32_t tab = ~0u, tab0 = 0, way = wave, ways = W;
    auto pair_block = [&](uint32_t first, uint32_t n) { return first + 2 * (way + ways * n); };
    auto load_table = [&](uint32_t first, uint32_t n, uint32_t lim) {
        tab0 = n;
        const uint32_t blk = pair_block(first, n + lane / 2) + lane % 2;
        const size_t ti = table_base + blk;
        tab = ~0u;
        if (blk < lim && blk < geo.n_logical && ti < geo.n_table) {
            const uint64_t p = geo.table[ti];
            if ((p + 1) * geo.block_bytes <= geo.arena_len) tab = (uint32_t)p;
        }
    };
    // Both blocks are read through buffer resources that span a block: an
    // absent one has range 0 and reads as zeros without memory traffic.
    struct Pair {
        Rsrc rs[2];
        bool ok[2];
    };
    auto pair_at = [&](uint32_t n) -> Pair {
        Pair r;
#pragma unroll
        for (int u = 0; u < 2; ++u) {
            const uint32_t phys = (uint32_t)__builtin_amdgcn_readlane((int)tab, (int)(2 * (n - tab0) + u));
            r.ok[u] = phys != ~0u;
            const uint8_t *base = geo.arena + (r.ok[u] ? phys * geo.block_bytes : 0);
            r.rs[u] = __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(base), 0,
                                                        r.ok[u] ? (int)geo.block_bytes : 0, 0x00020000);
        }
        return r;
    };
    u32x4 kr[2][NC];  // K: token col, dims 32c + 8 grp .. +7
    auto load_k = [&](const Pair &r) {
        const uint32_t off = g * HD * 2 + col * row_bytes + 16 * grp;
#pragma unroll
        for (int u = 0; u < 2; ++u)
#pragma unroll
            for (int c = 0; c < NC; ++c) kr[u][c] = __builtin_amdgcn_raw_buffer_load_b128(r.rs[u], off + 64 * c, 0, kKPolicy);
    };
    uint32_t vr[8][VH][DP / 2];  // V: token 4 grp + i % 4 of block i / 4, dims 128h + DP col .. +DP-1
    auto load_v = [&](const Pair &r) {
#pragma unroll
        for (int i = 0; i < 8; ++i)
#pragma unroll
            for (int h = 0; h < VH; ++h) {
                const uint32_t o = (geo.block_size + 4 * grp + i % 4) * row_bytes + (g * HD + 128 * h + DP * col) * 2;
                if constexpr (DP == 4) {
                    const u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(r.rs[i / 4], o, 0, kVPolicy);
                    vr[i][h][0] = t.x;
                    vr[i][h][1] = t.y;
                } else {
                    const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r.rs[i / 4], o, 0, kVPolicy);
#pragma unroll
                    for (int w = 0; w < 4; ++w) vr[i][h][w] = t[w];
                }
            }
    };

    // Without a sliding window the split's first block is s * bps whatever
    // the row length; `early` requests it before the length arrives (tokens
    // past the length are masked), which a launch of few wavefronts gains
    // from and one of many does not need.
    Pair cur;
    if (early) {
        load_table(s * bps, 0, s * bps + bps);
        cur = pair_at(0);
        load_k(cur);
        load_v(cur);
    }
    const RowKeys row = row_keys(lens[b], causal, window, bps, splits);
    if (s >= (row.splits ? row.splits : 1)) return;
    const uint32_t blk0 = row.first + s * bps;
    const uint32_t blk1 = blk0 + bps < row.last ? blk0 + bps : row.last;
    // Wavefronts without a pair of blocks end here and take no part in the
    // barriers below (256 rows of 30 keys, 32/8 heads of 128, in a launch made
    // for 4096: 23.2 -> 11.5 us).
    const uint32_t has = (blk1 - blk0 + 1) / 2, live = has <= solo ? 1 : has < W ? has : W;
    if (wave >= live) return;
    if (live == 1) ways = 1;
    if (!early) {
        load_table(blk0, 0, blk1);
        cur = pair_at(0);
        load_k(cur);
        load_v(cur);
    }

    // q as the B operand: head slot col (= query head g*G + col), dims 32c + 8 grp .. +7
    u32x4 qb[NC][C::kParts];
    {
        const bool hv = col < G;
        const typename Q::T *qh = q + ((size_t)b * n_heads + (size_t)g * G + (hv ? col : 0)) * HD;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            float v[8];
            load_f32<Q, 8>(qh + 32 * c + 8 * grp, v);
            if (!hv)
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = 0.0f;
            split8<C>(v, 1.0f, qb[c]);
        }
    }

    f32x4 acc[NT];  // tile (h, j) of lane (col, grp): dims 128h + DP (4 grp + e) + j of head slot col
    float m, l;     // running max, this lane's part of the denominator
    auto clear = [&] {
        m = -__builtin_inff();
        l = 0.0f;
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    // p[i]: score of token 4 grp + i % 4 of block i / 4 of pair n with head slot col
    auto scores = [&](float (&p)[8]) {
        f32x4 sc[2], sl[2];
#pragma unroll
        for (int u = 0; u < 2; ++u) sc[u] = sl[u] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int x = 0; x < C::kParts; ++x)
#pragma unroll
                for (int u = 0; u < 2; ++u) {
                    // the parts below the first in a sum of their own
                    f32x4 &d = x ? sl[u] : sc[u];
                    d = C::mfma(kr[u][c], qb[c][x], d);
                }
#pragma unroll
        for (int i = 0; i < 8; ++i) p[i] = (sc[i / 4][i % 4] + sl[i / 4][i % 4]) * scale;
    };
    // Tokens outside the row's keys: -inf scores, zero V.
    auto mask = [&](uint32_t n, float (&p)[8]) {
        const uint32_t t0 = pair_block(blk0, n) * kBlockTokens;
        const bool edge = t0 < row.lo || t0 + 2 * kBlockTokens > row.seq || !cur.ok[0] || !cur.ok[1];
        if (!edge) return;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t t = t0 + (i / 4) * kBlockTokens + 4 * grp + i % 4;
            const bool on = cur.ok[i / 4] && t >= row.lo && t < row.seq;
            if (!on) p[i] = -__builtin_inff();
#pragma unroll
            for (int h = 0; h < VH; ++h)
#pragma unroll
                for (int w = 0; w < DP / 2; ++w) vr[i][h][w] = on ? vr[i][h][w] : 0u;
        }
    };
    // Scores to probabilities times kPScale against the running maximum.
    auto soften = [&](float (&p)[8]) {
        float mx = -__builtin_inff();
#pragma unroll
        for (int i = 0; i < 8; ++i) mx = fmaxf(mx, p[i]);
        const float mn = fmaxf(m, rows_max(mx));
        if (__any(mn > m)) {  // most pairs raise no head's maximum
            const float alpha = m > -__builtin_inff() ? __expf(m - mn) : 0.0f;
            l *= alpha;
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[n] *= alpha;
            m = mn;
        }
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            p[i] = p[i] > -__builtin_inff() ? __expf(p[i] - m) : 0.0f;
            l += p[i];
            p[i] *= C::kPScale;
        }
    };

    clear();
    for (uint32_t n = 0; pair_block(blk0, n) < blk1; ++n) {
        float p[8];
        scores(p);
        if (n + 1 - tab0 == (uint32_t)kWave / 2) load_table(blk0, n + 1, blk1);
        const Pair next = pair_at(n + 1);
        __builtin_amdgcn_sched_barrier(0);  // a second register set of K would cost occupancy
        load_k(next);
        mask(n, p);
        soften(p);
        u32x4 pb[C::kPParts];
        split8<C>(p, C::kPLower, pb);
#pragma unroll
        for (int h = 0; h < VH; ++h)
#pragma unroll
            for (int j = 0; j < DP; ++j) {
                u32x4 a;  // dim DP col + j of the eight tokens
#pragma unroll
                for (int w = 0; w < 4; ++w)
                    a[w] = __builtin_amdgcn_perm(vr[2 * w + 1][h][j / 2], vr[2 * w][h][j / 2],
                                                 j % 2 ? 0x07060302u : 0x05040100u);
                // the pair's sum by itself, smallest part first, then once onto the running one
                f32x4 t = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
                for (int x = C::kPParts - 1; x > 0; --x) t = C::mfma(a, pb[x], t);
                if constexpr (C::kPLower == 1.0f) {
                    t = C::mfma(a, pb[0], t);
                } else {
                    const f32x4 t0 = C::mfma(a, pb[0], f32x4{0.0f, 0.0f, 0.0f, 0.0f});
#pragma unroll
                    for (int e = 0; e < 4; ++e) t[e] = __builtin_fmaf(t[e], 1.0f / C::kPLower, t0[e]);
                }
                acc[h * DP + j] += t;
            }
        __builtin_amdgcn_sched_barrier(0);
        load_v(next);
        cur = next;
    }
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);

    // Merge the wavefronts pairwise through LDS: [half, 2 half) hand theirs to [0, half).
    constexpr uint32_t kMerge = (NT * 4 + 2) * kWave;  // floats per wavefront
#pragma unroll
    for (uint32_t half = W / 2; half > 0; half /= 2) {
        if (half >= live) continue;  // the same in every live wavefront
        float *rec = merge_lds + (size_t)(wave % half) * kMerge + lane;
        __syncthreads();
        if (wave >= half && wave < 2 * half) {
            rec[0] = m;
            rec[kWave] = l;
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) rec[(2 + n * 4 + e) * kWave] = acc[n][e];
        }
        __syncthreads();
        if (wave < half && wave + half < live) {
            const float mo = rec[0], mn = fmaxf(m, mo);
            const float wa = m > -__builtin_inff() ? __expf(m - mn) : 0.0f;
            const float wb = mo > -__builtin_inff() ? __expf(mo - mn) : 0.0f;
            l = l * wa + rec[kWave] * wb;
            m = mn;
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[n][e] = acc[n][e] * wa + rec[(2 + n * 4 + e) * kWave] * wb;
        }
    }
    if (wave != 0) return;
    auto store = [&] {
        if (col >= G) return;
        if (row.splits <= 1) {
            const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
            for (int h = 0; h < VH; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    typename O::T *o =
                        out + ((size_t)b * n_heads + (size_t)g * G + col) * HD + 128 * h + DP * (4 * grp + e);
                    float r[DP];
#pragma unroll
                    for (int j = 0; j < DP; ++j) r[j] = l > 0.0f ? acc[h * DP + j][e] * kUnscale * inv : 0.0f;
                    store_f32<O, DP>(o, r);
                }
        } else {
            // partial record per (b, g, s, head slot): HD sums, then m, l
            float *rec = part + (((size_t)bg * splits + s) * rec_heads + col) * (HD + kRecTail);
#pragma unroll
            for (int h = 0; h < VH; ++h)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int j = 0; j < DP; ++j) rec[128 * h + DP * (4 * grp + e) + j] = acc[h * DP + j][e] * kUnscale;
            if (grp == 0) {
                rec[HD] = m;
                rec[HD + 1] = l;
            }
        }
    };
    uint32_t top = 0;
#pragma unroll
    for (int n = 0; n < NT; ++n)
#pragma unroll
        for (int e = 0; e < 4; ++e) top = max(top, __float_as_uint(acc[n][e]) & 0x7fffffffu);
    store();
    // An infinite V times the parts of p makes NaN (the lower parts are 0 or of
    // either sign).  Where a sum is not finite, this wavefront takes all of the
    // split's keys again, now with f32 matrix products of the widened V and
    // whole p.  The registers of this rare walk are apart from the first's: a
    // second walk before the merge moved every accumulator (0.5 us a launch).
    if (__builtin_expect(__any(top >= 0x7f800000u), 0)) {
        way = 0;
        ways = 1;
        clear();
        for (uint32_t n = 0; pair_block(blk0, n) < blk1; ++n) {
            if (n % (kWave / 2) == 0) load_table(blk0, n, blk1);
            cur = pair_at(n);
            load_k(cur);
            float p[8];
            scores(p);
            load_v(cur);
            mask(n, p);
            soften(p);
#pragma unroll
            for (int h = 0; h < VH; ++h)
#pragma unroll
                for (int j = 0; j < DP; ++j)
#pragma unroll
                    for (int i = 0; i < 8; ++i) {
                        const uint32_t w = vr[i][h][j / 2];
                        f32x4 &d = acc[h * DP + j];
                        d = __builtin_amdgcn_mfma_f32_16x16x4f32(C::widen(j % 2 ? w >> 16 : w), p[i], d, 0, 0, 0);
                    }
        }
        l += __shfl_xor(l, 16, kWave);
        l += __shfl_xor(l, 32, kWave);
        store();
    }
}

// Combine the splits of one (b, query head): M = max m_s, w_s = exp(m_s - M),
// out = sum w_s acc_s / sum w_s l_s.  1024 threads: thread (p, d) owns
// dimension d of splits p, p + kParts, ...  Every load (the partial sums and
// each split's m, l) is issued up front, so the kernel pays one memory
// latency; the maxima, weights and denominators then go through LDS.
constexpr int kCombineThreads = 1024;
constexpr uint32_t kMaxSplits = 256;

template <typename O, int HD, int GM>
__global__ __launch_bounds__(kCombineThreads) void paged_decode_combine(const float *__restrict__ part,
                                                                        typename O::T *__restrict__ out,
                                                                        const uint32_t *__restrict__ lens,
                                                                        uint32_t n_heads, uint32_t n_kv,
                                                                        uint32_t causal, uint32_t window,
                                                                        uint32_t alloc_splits, uint32_t bps) {
    constexpr int kParts = kCombineThreads / HD;
    constexpr int kPer = kMaxSplits / kParts;  // splits per thread at most
    constexpr int kWaves = kCombineThreads / kWave;
    __shared__ float w_lds[kMaxSplits];
    __shared__ float red[kWaves];
    __shared__ float acc_lds[kParts][HD];
    const uint32_t bh = blockIdx.x, h = bh % n_heads, b = bh / n_heads;
    const uint32_t G = n_heads / n_kv, g = h / G, slot = h % G;
    constexpr uint32_t kRec = GM * (HD + kRecTail);
    const float *base = part + ((size_t)(b * n_kv + g) * alloc_splits) * kRec + slot * (HD + kRecTail);
    const uint32_t splits = row_keys(lens[b], causal, window, bps, alloc_splits).splits;
    if (splits <= 1) return;  // finished by its split
    const uint32_t t = threadIdx.x, d = t % HD, p = t / HD;
    float av[kPer];
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const uint32_t sp = p + (uint32_t)i * kParts;
        av[i] = sp < splits ? base[(size_t)sp * kRec + d] : 0.0f;
    }
    const float ms = t < splits ? base[(size_t)t * kRec + HD] : -__builtin_inff();
    const float ls = t < splits ? base[(size_t)t * kRec + HD + 1] : 0.0f;
    float M = wave_max(ms);
    if (t % kWave == 0) red[t / kWave] = M;
    __syncthreads();
    M = red[0];
#pragma unroll
    for (int i = 1; i < kWaves; ++i) M = fmaxf(M, red[i]);
    const float w = (t < splits && ms > -__builtin_inff()) ? __expf(ms - M) : 0.0f;
    if (t < kMaxSplits) w_lds[t] = w;
    float L = wave_sum(w * ls);
    __syncthreads();
    if (t % kWave == 0) red[t / kWave] = L;
    __syncthreads();
    L = 0.0f;
#pragma unroll
    for (int i = 0; i < kWaves; ++i) L += red[i];
    float o = 0.0f;
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
        const uint32_t sp = p + (uint32_t)i * kParts;
        if (sp < splits) o += w_lds[sp] * av[i];
    }
    acc_lds[p][d] = o;
    __syncthreads();
    if (t < (uint32_t)HD) {
        float r = 0.0f;
#pragma unroll
        for (int q = 0; q < kParts; ++q) r += acc_lds[q][t];
        out[((size_t)b * n_heads + h) * HD + t] = O::store(L > 0.0f ? r * (1.0f / L) : 0.0f);
    }
}

// The same combine by one wavefront per (b, query head), for the launches
// where the 1024-thread form's barriers and width cost more than its work:
// lanes take the splits for m and l (wavefront reductions, no barrier); for
// the sums HD/4 lanes cover a record's dims with 16-byte loads and the
// 64 / (HD/4) lane groups take interleaved splits, every load issued before
// the sums.  M, the weights and L as in paged_decode_combine.
template <typename O, int HD, int GM>
__global__ __launch_bounds__(kWave) void paged_decode_combine_wave(const float *__restrict__ part,
                                                                   typename O::T *__restrict__ out,
                                                                   const uint32_t *__restrict__ lens,
                                                                   uint32_t n_heads, uint32_t n_kv,
                                                                   uint32_t causal, uint32_t window,
                                                                   uint32_t alloc_splits, uint32_t bps) {
    constexpr uint32_t kRec = HD + kRecTail;
    constexpr uint32_t LPR = HD / 4, SG = kWave / LPR;  // lanes per record, split groups
    constexpr uint32_t kPerLane = kMaxSplits / kWave;
    __shared__ float w_lds[kMaxSplits];
    const uint32_t bh = blockIdx.x, h = bh % n_heads, b = bh / n_heads;
    const uint32_t G = n_heads / n_kv, g = h / G, slot = h % G;
    const float *base = part + ((size_t)(b * n_kv + g) * alloc_splits * GM + slot) * kRec;  // split s: + s * GM * kRec
    const uint32_t splits = row_keys(lens[b], causal, window, bps, alloc_splits).splits;
    if (splits <= 1) return;  // finished by its split
    const uint32_t lane = threadIdx.x, dq = lane % LPR, sg = lane / LPR;
    // the first batch of record sums first: its latency overlaps the m / l
    // reductions
    constexpr uint32_t kBatch = 16;
    float4 v[kBatch];
    auto load_batch = [&](uint32_t s0) {
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t sp = s0 + sg + j * SG;
            v[j] = sp < splits ? *reinterpret_cast<const float4 *>(base + (size_t)sp * GM * kRec + 4 * dq)
                               : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        }
    };
    load_batch(0);
    float ms[kPerLane], ls[kPerLane];
    float M = -__builtin_inff();
#pragma unroll
    for (uint32_t i = 0; i < kPerLane; ++i) {
        const uint32_t sp = lane + i * kWave;
        ms[i] = sp < splits ? base[(size_t)sp * GM * kRec + HD] : -__builtin_inff();
        ls[i] = sp < splits ? base[(size_t)sp * GM * kRec + HD + 1] : 0.0f;
        M = fmaxf(M, ms[i]);
    }
    M = wave_max(M);
    float Lp = 0.0f;
#pragma unroll
    for (uint32_t i = 0; i < kPerLane; ++i) {
        const uint32_t sp = lane + i * kWave;
        const float w = (sp < splits && ms[i] > -__builtin_inff()) ? __expf(ms[i] - M) : 0.0f;
        w_lds[sp] = w;
        Lp += w * ls[i];
    }
    const float L = wave_sum(Lp);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
    float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    for (uint32_t s0 = 0;;) {
#pragma unroll
        for (uint32_t j = 0; j < kBatch; ++j) {
            const uint32_t sp = s0 + sg + j * SG;
            const float w = sp < splits ? w_lds[sp] : 0.0f;
            o.x += w * v[j].x;
            o.y += w * v[j].y;
            o.z += w * v[j].z;
            o.w += w * v[j].w;
        }
        s0 += kBatch * SG;
        if (s0 >= splits) break;
        load_batch(s0);
    }
#pragma unroll
    for (uint32_t off = LPR; off < kWave; off *= 2) {
        o.x += __shfl_xor(o.x, off, kWave);
        o.y += __shfl_xor(o.y, off, kWave);
        o.z += __shfl_xor(o.z, off, kWave);
        o.w += __shfl_xor(o.w, off, kWave);
    }
    if (sg == 0) {
        const float inv = 1.0f / L;
        const float r[4] = {L > 0.0f ? o.x * inv : 0.0f, L > 0.0f ? o.y * inv : 0.0f, L > 0.0f ? o.z * inv : 0.0f,
                            L > 0.0f ? o.w * inv : 0.0f};
        store_f32<O, 4>(out + ((size_t)b * n_heads + h) * HD + 4 * dq, r);
    }
}

// Splits of a row's keys over workgroups.
//  * Few (row, KV head) pairs: about one workgroup per CU, at least 8 blocks
//    each (a pair of blocks per wavefront); rows of up to 32 blocks stay whole,
//    at heads of 256 of up to 24 (512 keys 17.5 us whole, 13.4 in four splits).
//    A window that fits stays whole too (128 of 4096 keys 7.5 -> 6.3 us).
//    One row at 8 KV heads: 256 keys 6.6 us whole, 8.9 in two splits; 2048 keys
//    9.9 us in 16 splits, 11.3 in 8; 32768 keys 27.3 in 32, 28.4 in 64.
//  * Long rows: splits of 128 blocks (2048 keys) while the launch stays within
//    2048 workgroups, so that a batch of mixed lengths does not wait for its
//    longest rows.  64 rows of 256 .. 4096 keys: 123.7 us against 118.4 with
//    splits of 64 blocks, but 64 rows of 4096 keys each 194 against 202; 256
//    rows of 4096 keys 677 us whole, 740 in two splits.
constexpr uint32_t kSplitTarget = 256, kMinSplitBlocks = 8;
constexpr uint32_t kLongSplitBlocks = 128, kLongSplitMax = 2048;
uint32_t whole_blocks(uint32_t head_dim) { return head_dim == 256 ? 24 : 32; }
uint32_t choose_splits(uint32_t batch, uint32_t n_kv, uint32_t max_seq, uint32_t head_dim) {
    const uint32_t pairs = batch * n_kv;
    const uint32_t blocks = (max_seq + kBlockTokens - 1) / kBlockTokens;
    if (pairs == 0 || blocks <= whole_blocks(head_dim)) return 1;
    uint32_t s = (kSplitTarget + pairs - 1) / pairs;
    if (s > blocks / kMinSplitBlocks) s = blocks / kMinSplitBlocks;
    uint32_t by_length = (blocks + kLongSplitBlocks - 1) / kLongSplitBlocks;
    if (by_length > kLongSplitMax / pairs) by_length = kLongSplitMax / pairs;
    if (s < by_length) s = by_length;
    return s < kMaxSplits ? s : kMaxSplits;
}

// One wavefront a workgroup instead of kDecodeWaves: no merge, and more
// workgroups on a CU.  Where a pair of blocks is all there is (8 rows of 32
// keys, 32/8 heads of 128: 4.2 against 4.5 us), and where the (row, KV head)
// pairs alone fill the chip and no row is long: a row's one wavefront must not
// outlast the others.  At 256 rows of these heads: 32 keys 8.1 us against 10.4,
// 100 keys 22.0 and 32.2, 512 keys 79.5 and 82.9, 16 .. 512 53.0 and 52.9, but
// 16 .. 768 81 and 71.  Heads of 64 turn at half of that (256 rows, 8/8 heads:
// 16 .. 256 keys 18.2 and 18.6, 16 .. 384 26.1 and 23.5); heads of 256 at twice
// (128 rows, 16/8 heads: 16 .. 1024 keys 100 and 106, 16 .. 2048 200 and 193),
// and from half as many pairs (64 rows of 512 keys 43 and 49), where the others
// gain up to head_dim keys (64 rows of 64 keys 5.9 and 6.8, of 200 12.3 and 11.7).
bool fills(uint32_t pairs, uint32_t head_dim) { return pairs >= (head_dim == 256 ? 512u : 1024u); }
bool one_wave(uint32_t pairs, uint32_t blocks, uint32_t bps, uint32_t head_dim) {
    return blocks <= 2 || (pairs >= 512 && blocks <= head_dim / 16) ||
           (fills(pairs, head_dim) && bps <= head_dim / 4);
}

// Launches of at most this many workgroups request their first blocks before
// the row length arrives (one row of 32768 keys 27.9 -> 27.3 us).
constexpr uint32_t kEarlyGrid = 512;
// The one-wavefront combine up to this many splits (32 splits: 27.3 us against
// 28.5 with the 1024-thread one), the 1024-thread combine beyond.
constexpr uint32_t kWaveCombineSplits = 64;

template <typename Q, typename O, typename C, int HD>
int launch_decode(const void *q, void *out, uint32_t batch, uint32_t n_heads, uint32_t n_kv, const uint32_t *lens,
                  uint32_t max_seq, float scale, uint32_t causal, uint32_t window, const PagedGeom &geo,
                  float *ws, uint64_t ws_bytes, hipStream_t st) {
    const uint32_t gm = n_heads / n_kv <= 8 ? 8 : 16;
    const uint32_t blocks = (max_seq + kBlockTokens - 1) / kBlockTokens;
    // Blocks that a row attends at most: a window's keys start anywhere in a block.
    const uint32_t held = causal && window
                              ? (uint32_t)std::min<uint64_t>(blocks, ((uint64_t)window + 2 * kBlockTokens - 2) / kBlockTokens)
                              : blocks;
    uint32_t splits = held <= whole_blocks(HD) ? 1 : choose_splits(batch, n_kv, max_seq, HD);
    const uint64_t need = (uint64_t)batch * n_kv * splits * gm * (HD + kRecTail) * 4;
    if (splits > 1 && (!ws || ws_bytes < need)) splits = 1;
    const uint32_t bps = blocks ? (blocks + splits - 1) / splits : 1;
    const uint32_t grid = batch * n_kv * splits;
    // Short rows of a launch that fills the chip for long ones (128 rows of 100
    // keys, 32/8 heads of 128, made for 4096: 20.6 -> 17.6 us).
    const uint32_t solo = HD < 256 && fills(batch * n_kv, HD) ? 4 : 1;
    const uint32_t early = !(causal && window) && grid <= kEarlyGrid && solo == 1;
    auto decode = [&]<uint32_t W>() {
        const uint32_t lds = W / 2 * (HD / 4 + 2) * kWave * sizeof(float);
        FELLM_LAUNCH((paged_decode_kernel<Q, O, C, HD, W>), dim3(grid), dim3(kWave * W), lds, st,
                     static_cast<const typename Q::T *>(q), static_cast<typename O::T *>(out), ws, lens, geo, batch,
                     n_heads, n_kv, scale, causal, window, splits, bps, gm, early, solo);
    };
    if (one_wave(batch * n_kv, held, std::min(bps, held), HD))
        decode.template operator()<1>();
    else
        decode.template operator()<kDecodeWaves>();
    int rc = launch_status();
    if (rc != FELLM_OK || splits == 1) return rc;
    auto combine = [&]<int GM>() {
        if (splits <= kWaveCombineSplits && aligned_to(ws, 16))
            FELLM_LAUNCH((paged_decode_combine_wave<O, HD, GM>), dim3(batch * n_heads), dim3(kWave), 0, st, ws,
                         static_cast<typename O::T *>(out), lens, n_heads, n_kv, causal, window, splits, bps);
        else
            FELLM_LAUNCH((paged_decode_combine<O, HD, GM>), dim3(batch * n_heads), dim3(kCombineThreads), 0, st, ws,
                         static_cast<typename O::T *>(out), lens, n_heads, n_kv, causal, window, splits, bps);
    };
    if (gm == 8)
        combine.template operator()<8>();
    else
        combine.template operator()<16>();
    return launch_status();
}

template <typename Q, typename O, typename C>
int dispatch_hd(uint32_t hd, const void *q, void *out, uint32_t batch, uint32_t n_heads, uint32_t n_kv,
                const uint32_t *lens, uint32_t max_seq, float scale, uint32_t causal, uint32_t window,
                const PagedGeom &geo, float *ws, uint64_t ws_bytes, hipStream_t st) {
#define FELLM_ATT(HDV)                                                                                              \
    if (hd == HDV)                                                                                                  \
        return launch_decode<Q, O, C, HDV>(q, out, batch, n_heads, n_kv, lens, max_seq, scale, causal, window, geo, \
                                           ws, ws_bytes, st);
    FELLM_ATT(64)
    FELLM_ATT(128)
    FELLM_ATT(256)
#undef FELLM_ATT
    return FELLM_ERR_SHAPE;
}

}  // namespace
}  // namespace fellm

extern "C" uint64_t fellm_rocm_paged_attention_workspace(uint32_t batch, uint32_t n_heads, uint32_t n_kv_heads,
                                                         uint32_t head_dim, uint32_t max_seq) {
    using namespace fellm;
    if (!n_kv_heads || n_heads % n_kv_heads) return 0;
    const uint32_t splits = choose_splits(batch, n_kv_heads, max_seq, head_dim);
    if (splits <= 1) return 0;
    const uint32_t gm = n_heads / n_kv_heads <= 8 ? 8 : 16;
    return (uint64_t)batch * n_kv_heads * splits * gm * (head_dim + kRecTail) * 4;
}

extern "C" int fellm_rocm_paged_attention(const void *q, uint32_t q_dtype, void *out, uint32_t out_dtype,
                                          uint32_t batch, uint32_t n_heads, uint32_t n_kv_heads, uint32_t head_dim,
                                          const uint32_t *row_lengths, uint32_t max_seq, float scale,
                                          uint32_t causal, uint32_t window, const FellmRocmPagedKv *kv,
                                          float *workspace, uint64_t workspace_bytes, void *stream) {
    using namespace fellm;
    if (!q || !out || !row_lengths || !kv || !kv->arena || !kv->block_table) return FELLM_ERR_ARITY;
    if (!n_kv_heads || n_heads % n_kv_heads || n_heads / n_kv_heads > 16) return FELLM_ERR_SHAPE;
    if (kv->stride != n_kv_heads * head_dim || kv->block_size != kBlockTokens) return FELLM_ERR_SHAPE;
    if (kv->block_bytes < 2ull * kv->block_size * kv->stride * 2 || kv->block_bytes % 16) return FELLM_ERR_SHAPE;
    if (kv->layer >= kv->n_layers) return FELLM_ERR_SHAPE;
    if (!aligned_to(kv->arena, 16) || !aligned_to(q, 16) || !aligned_to(out, 16)) return FELLM_ERR_SHAPE;
    if (batch == 0) return FELLM_OK;
    if (!(scale > 0.0f)) scale = 1.0f / sqrtf((float)head_dim);
    const PagedGeom geo{static_cast<const uint8_t *>(kv->arena), kv->arena_len, kv->block_table, kv->n_block_table,
                        kv->n_logical_blocks, kv->n_layers, kv->layer, kv->block_size, kv->block_bytes, kv->stride};
    hipStream_t st = as_stream(stream);
    if (kv->kv_dtype != FELLM_DTYPE_F16 && kv->kv_dtype != FELLM_DTYPE_BF16) return FELLM_ERR_DTYPE;
    const bool bf = kv->kv_dtype == FELLM_DTYPE_BF16;
#define FELLM_ATT_QO(QD, QT, OD, OT)                                                                              \
    if (q_dtype == QD && out_dtype == OD)                                                                         \
        return bf ? dispatch_hd<QT, OT, CacheBF16>(head_dim, q, out, batch, n_heads, n_kv_heads, row_lengths,  \
                                                   max_seq, scale, causal, window, geo, workspace, workspace_bytes, \
                                                   st)                                                            \
                  : dispatch_hd<QT, OT, CacheF16>(head_dim, q, out, batch, n_heads, n_kv_heads, row_lengths,   \
                                                  max_seq, scale, causal, window, geo, workspace, workspace_bytes,  \
                                                  st);
    FELLM_ATT_QO(FELLM_DTYPE_F32, F32, FELLM_DTYPE_F32, F32)
    FELLM_ATT_QO(FELLM_DTYPE_F16, F16, FELLM_DTYPE_F16, F16)
    FELLM_ATT_QO(FELLM_DTYPE_BF16, BF16, FELLM_DTYPE_BF16, BF16)
    FELLM_ATT_QO(FELLM_DTYPE_F16, F16, FELLM_DTYPE_F32, F32)
    FELLM_ATT_QO(FELLM_DTYPE_BF16, BF16, FELLM_DTYPE_F32, F32)
#undef FELLM_ATT_QO
    return FELLM_ERR_DTYPE;
}
