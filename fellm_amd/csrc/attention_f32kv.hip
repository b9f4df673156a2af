// Attention over f32 K/V rows held contiguously ([t, n_kv * head_dim]), the
// non-paged arms of the reference's Attention launch:
//  * decode (backend.rs:1371-1397; CUDA attention_heads, launchers.rs:
//    3719-3760): one query row against keys [max(0, seq - window), seq) of
//    one K/V pair;
//  * rows (attention_provider.rs:251-385): query_len rows, causal or windowed;
//  * canvas (backend.rs:1412-1535; CUDA attention_canvas_heads,
//    launchers.rs:3270-3333): every query row against the prefix keys
//    [prefix_start, past) of one pair and then all `rows` canvas keys of a
//    second pair, with no causal mask.
//
// Work split.  The G query heads of a KV head times the query rows form that
// KV head's slots (slot = row * G + head); a wavefront takes 16 slots and
// walks keys in tiles of 16, both products on the f32 matrix cores
// (v_mfma_f32_16x16x4_f32: f32 products and sums, so the arithmetic is that of
// an f32 FMA chain).
//  * S^T = K . Q^T: A is the K tile (lane = key lane % 16, dims 16j + 4 (lane
//    / 16) .. +3 of piece j), B the slots' q, held in registers for the walk.
//  * Lane (slot lane % 16, group lane / 16) then owns the scores of keys
//    4 group .. +3 of its slot, which is the layout the second product takes
//    its B operand in: the probabilities go from the softmax into
//    out^T = V^T . P^T without leaving their registers.  The running max and
//    the rescaling factors are per lane for the same reason; the sum of
//    probabilities stays a per-lane partial until the end.
//  * Tiles come by consecutive 16-byte loads (1 KB an instruction) a tile
//    ahead, and reach the operand layout through LDS, 16-byte pieces XORed
//    with the row so that neither side conflicts.  Loads in the operand
//    layout itself (16 rows an instruction) measured 37 GB/s per CU against
//    100 for consecutive ones.
// A workgroup is one slot tile: its NW wavefronts take key tiles w, w + NW,
// ..., each with a K buffer of its own (no barrier in the walk), and their
// (max, sum, accumulators) are merged pairwise through LDS at the end.
//
// Measured at 32/8 heads of 128, against one 256-thread workgroup per query
// row and KV head on the vector ALUs:
//  * 512 rows x 2048 keys (15 GFLOP): 1180 -> 180 us, 83 TFLOP/s of the 153 a
//    large f32 matrix product reaches.  The counters show the matrix cores
//    busy half the time and the vector ALUs (softmax with the exact exp) a
//    third, with little overlap between a SIMD's two wavefronts.  Sharing
//    staged tiles between the slot groups of a workgroup (barriers) 202-212,
//    two slot tiles per wavefront 232, the next tile's Q.K issued beside this
//    one's softmax 177.
//  * one row x 4096 keys: 713 -> 72 us.  The C entry points have no scratch
//    for partial results of several workgroups, so a KV head's keys stay in
//    one workgroup per quarter of the output dims, which is bound by its CU's
//    matrix cores (12 of 16 slots are surplus at four heads per KV head).
#include "common.hpp"

#include "fellm_rocm.h"

namespace fellm {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
using Rsrc = __amdgpu_buffer_rsrc_t;

constexpr uint32_t kTileKeys = 16;
constexpr uint32_t kNoLoad = 0x80000000u;  // buffer offset past every range: reads as zero

struct F32kvArgs {
    const float *q;
    float *out;
    const float *k1, *v1, *k2, *v2;
    uint32_t rows, n_heads, n_kv, hd;
    uint32_t b1, e1, n2;
    float scale;
    // 0: keys [b1, e1) then n2 keys of the second pair; 1: causal, the query
    // rows ending at key e1 - 1, the last `window` keys when window > 0;
    // 2: keys within `window` of the row index (all when window == 0).
    uint32_t row_mode, window;
    uint32_t head_major;  // q and out are [head][row][d] instead of [row][head][d]
};

// Keys [lo, hi) of the first pair that query row `row` attends.
__device__ __forceinline__ void row_keys(const F32kvArgs &a, uint32_t row, uint32_t &lo, uint32_t &hi) {
    lo = a.b1;
    hi = a.e1;
    if (a.row_mode == 1) {
        hi = a.e1 - a.rows + row + 1;
        lo = a.window && hi > a.window ? hi - a.window : 0;
    } else if (a.row_mode == 2) {
        lo = a.window && row + 1 > a.window ? row + 1 - a.window : 0;
        if (a.window && row + a.window < a.e1) hi = row + a.window;
    }
    if (lo > hi) lo = hi;
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

template <int N>
__device__ __forceinline__ void buf_load(Rsrc r, uint32_t off, float *v) {
    if constexpr (N == 4) {
        const u32x4 t = __builtin_amdgcn_raw_buffer_load_b128(r, off, 0, 0);
#pragma unroll
        for (int i = 0; i < 4; ++i) v[i] = __uint_as_float(t[i]);
    } else if constexpr (N == 2) {
        const u32x2 t = __builtin_amdgcn_raw_buffer_load_b64(r, off, 0, 0);
        v[0] = __uint_as_float(t[0]);
        v[1] = __uint_as_float(t[1]);
    } else {
        v[0] = __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, 0, 0));
    }
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// HD: head_dim rounded up to 64, 128 or 256 (FULL: equal to it).  NT: 16-dim
// output tiles per workgroup (HD / 16, or a quarter of it).  NW: wavefronts
// (key ways) per workgroup.
template <int HD, int NT, int NW, bool FULL>
__global__ __launch_bounds__(NW *kWave) void attention_f32kv_kernel(F32kvArgs a) {
    constexpr int KJ = HD / 16;           // 16-byte K pieces per lane and tile
    constexpr int VW = NT < 4 ? NT : 4;   // consecutive dims per V load
    constexpr int VH = NT / VW;           // V loads per lane and key
    constexpr int DS = HD / 16 / NT;      // workgroups that share a slot group's output dims
    constexpr uint32_t CPR = HD / 4;      // 16-byte pieces per row
    extern __shared__ __align__(16) float f32kv_lds[];
    __shared__ uint64_t exp_tab[32];
    const uint32_t G = a.n_heads / a.n_kv, slots = a.rows * G;
    const uint32_t lane = threadIdx.x % kWave, col = lane % 16, grp = lane / 16;
    const uint32_t way = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave);
    const uint32_t g = blockIdx.x % a.n_kv, rest = blockIdx.x / a.n_kv;
    const uint32_t d0 = (rest % DS) * (NT * 16);  // first output dim
    // The last rows of a causal launch attend the most keys: they go first.
    const uint32_t n_groups = (slots + 15) / 16;
    const uint32_t slot0 = (n_groups - 1 - rest / DS) * 16;
    if (threadIdx.x < 32) exp_tab[threadIdx.x] = make_expf_table().tab[threadIdx.x];

    const uint32_t hd = FULL ? (uint32_t)HD : a.hd;
    const size_t hstride = a.head_major ? (size_t)a.rows * hd : hd;
    const size_t rstride = a.head_major ? hd : (size_t)a.n_heads * hd;
    // Surplus slots repeat the last one and are not stored.
    auto clamp_slot = [&](uint32_t s) { return s < slots ? s : slots - 1; };
    // q as the B operand, piece j: dims 16j + 4 grp .. +3.  Keys that this
    // lane's slots attend, that any slot of the wavefront does, and that all
    // of them do (the bounds do not decrease with the row).
    float qv[KJ][4];
    uint32_t klo, khi, lo, hi, lo_all, hi_all;
    const uint32_t my_slot = clamp_slot(slot0 + col);
    row_keys(a, my_slot / G, klo, khi);
    const size_t qoff = ((size_t)g * G + my_slot % G) * hstride + my_slot / G * rstride;
#pragma unroll
    for (int j = 0; j < KJ; ++j) {
        const uint32_t d = 16 * j + 4 * grp;
        if (FULL || d < hd) {
            load_f32<F32, 4>(a.q + qoff + d, qv[j]);
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) qv[j][i] = 0.0f;
        }
    }
    row_keys(a, clamp_slot(slot0) / G, lo, hi_all);
    row_keys(a, clamp_slot(slot0 + 15) / G, lo_all, hi);
    const uint32_t kvw = a.n_kv * hd;
    const uint32_t tiles1 = (hi - lo + kTileKeys - 1) / kTileKeys, tiles = tiles1 + (a.n2 + kTileKeys - 1) / kTileKeys;

    // A tile's rows are read through a buffer resource that ends with its
    // last key: keys past it (and dims past hd) read as zeros.
    struct Tile {
        uint32_t first, count;  // keys of its pair
    };
    auto tile_of = [&](uint32_t i) -> Tile {
        const bool p1 = i < tiles1;
        const uint32_t first = p1 ? lo + i * kTileKeys : (i - tiles1) * kTileKeys;
        const uint32_t end = p1 ? hi : a.n2;
        const uint32_t c = i < tiles ? end - first : 0;
        return {first, c < kTileKeys ? c : kTileKeys};
    };
    auto rsrc = [&](const float *p, const Tile &t) {
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(p + (size_t)t.first * kvw + (size_t)g * hd), 0,
                                                 t.count ? (int)(((t.count - 1) * kvw + hd) * 4) : 0, 0x00020000);
    };
    // K on its way to LDS: load j is 1 KB number j of the tile.
    float *const kbuf = f32kv_lds + way * (kTileKeys * HD);
    const uint32_t chunk = lane % CPR;  // CPR divides 64
    auto stage_row = [&](int j) { return (j * kWave + lane) / CPR; };
    float sk[KJ][4];
    auto stage_load = [&](uint32_t i) {
        const Rsrc r = rsrc(i < tiles1 ? a.k1 : a.k2, tile_of(i));
#pragma unroll
        for (int j = 0; j < KJ; ++j)
            buf_load<4>(r, FULL || 4 * chunk < hd ? stage_row(j) * kvw * 4 + 16 * chunk : kNoLoad, sk[j]);
    };
    auto stage_store = [&] {
        wave_lds_sync();
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
            const uint32_t r = stage_row(j);
            *reinterpret_cast<float4 *>(kbuf + r * HD + 4 * (chunk ^ (r & 15))) =
                make_float4(sk[j][0], sk[j][1], sk[j][2], sk[j][3]);
        }
        wave_lds_sync();
    };
    // V of keys 4 grp + e: output tile VW h + x of lane col is dim d0 + 16 VW h + VW col + x.
    float vr[4][VH][VW];
    auto load_v = [&](uint32_t i) {
        const Rsrc r = rsrc(i < tiles1 ? a.v1 : a.v2, tile_of(i));
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int h = 0; h < VH; ++h) {
                const uint32_t d = d0 + 16 * VW * h + VW * col;
                buf_load<VW>(r, FULL || d < hd ? ((4 * grp + e) * kvw + d) * 4 : kNoLoad, vr[e][h]);
            }
    };
    f32x4 acc[NT];
    float m, l;
    bool redo = false;
    auto clear = [&] {
        m = -__builtin_inff();
        l = 0.0f;
#pragma unroll
        for (int n = 0; n < NT; ++n) acc[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
    };
    clear();
    __syncthreads();  // exp_tab

    stage_load(way);
    stage_store();
    for (uint32_t i = way; i < tiles; i += NW) {
        const Tile tl = tile_of(i);
        const bool pair1 = i < tiles1;
        load_v(i);
        stage_load(i + NW);
        f32x4 sc[4];  // partial sums, one per dim of a piece
#pragma unroll
        for (int x = 0; x < 4; ++x) sc[x] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int j = 0; j < KJ; ++j) {
            float k4[4];
            load_f32<F32, 4>(kbuf + col * HD + 4 * ((4 * j + grp) ^ col), k4);
#pragma unroll
            for (int x = 0; x < 4; ++x) sc[x] = __builtin_amdgcn_mfma_f32_16x16x4f32(k4[x], qv[j][x], sc[x], 0, 0, 0);
        }
        float p[4], mx = -__builtin_inff();
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const uint32_t kk = 4 * grp + e, key = tl.first + kk;
            const bool on = kk < tl.count && (!pair1 || (key >= klo && key < khi));
            p[e] = on ? ((sc[0][e] + sc[1][e]) + (sc[2][e] + sc[3][e])) * a.scale : -__builtin_inff();
            mx = fmaxf(mx, p[e]);
        }
        const float mn = fmaxf(m, rows_max(mx));
        // No score above -inf yet: every p is exp(-inf) = 0.
        const float mr = mn > -__builtin_inff() ? mn : 0.0f;
        if (__any(mn > m)) {  // most tiles raise no slot's maximum
            const float alpha = expf_glibc_nonpos(m - mr, exp_tab);
            l *= alpha;
#pragma unroll
            for (int n = 0; n < NT; ++n) acc[n] *= alpha;
            m = mn;
        }
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            p[e] = expf_glibc_nonpos(p[e] - mr, exp_tab);  // 0 for a key not attended (-inf)
            l += p[e];
        }
        // A key that only some of the wavefront's slots attend must not reach
        // the others as 0 * inf: with a non-finite V value in such a tile the
        // wavefront redoes its keys one by one after the walk.
        if (pair1 && (tl.first < lo_all || tl.first + tl.count > hi_all)) {
            float z = 0.0f;
            __asm__ volatile("" : "+v"(z));  // keeps the test inside the branch
#pragma unroll
            for (int e = 0; e < 4; ++e)
#pragma unroll
                for (int h = 0; h < VH; ++h)
#pragma unroll
                    for (int x = 0; x < VW; ++x) z += vr[e][h][x] * 0.0f;
            redo |= __any(z != 0.0f);  // z is NaN where a value is inf or NaN
        }
#pragma unroll
        for (int e = 0; e < 4; ++e)
#pragma unroll
            for (int h = 0; h < VH; ++h)
#pragma unroll
                for (int x = 0; x < VW; ++x)
                    acc[h * VW + x] =
                        __builtin_amdgcn_mfma_f32_16x16x4f32(vr[e][h][x], p[e], acc[h * VW + x], 0, 0, 0);
        stage_store();
    }
    l += __shfl_xor(l, 16, kWave);
    l += __shfl_xor(l, 32, kWave);
    if (redo) {
        clear();
        for (uint32_t i = way; i < tiles; i += NW) {
            const Tile tl = tile_of(i);
            for (uint32_t kk = 0; kk < tl.count; ++kk) {
                const uint32_t key = tl.first + kk;
                const size_t at = (size_t)key * kvw + (size_t)g * hd;
                const float *kp = (i < tiles1 ? a.k1 : a.k2) + at, *vp = (i < tiles1 ? a.v1 : a.v2) + at;
                float s = 0.0f;
#pragma unroll
                for (int j = 0; j < KJ; ++j)
#pragma unroll
                    for (int x = 0; x < 4; ++x) {
                        const uint32_t d = 16 * j + 4 * grp + x;
                        s += qv[j][x] * (FULL || d < hd ? kp[d] : 0.0f);
                    }
                s += __shfl_xor(s, 16, kWave);
                s += __shfl_xor(s, 32, kWave);
                if (i < tiles1 && (key < klo || key >= khi)) continue;
                s *= a.scale;
                const float mn = fmaxf(m, s), mr = mn > -__builtin_inff() ? mn : 0.0f;
                const float alpha = expf_glibc_nonpos(m - mr, exp_tab), pk = expf_glibc_nonpos(s - mr, exp_tab);
                l = l * alpha + pk;
                m = mn;
#pragma unroll
                for (int n = 0; n < NT; ++n)
#pragma unroll
                    for (int e = 0; e < 4; ++e) {
                        const uint32_t d = d0 + 16 * VW * (n / VW) + VW * (4 * grp + e) + n % VW;
                        acc[n][e] = acc[n][e] * alpha + pk * (FULL || d < hd ? vp[d] : 0.0f);
                    }
            }
        }
    }

    // Merge the key ways pairwise: ways [half, 2 half) hand theirs to [0, half).
    constexpr uint32_t kRec = (NT * 4 + 2) * kWave;  // floats per wavefront
#pragma clang loop unroll(disable)
    for (uint32_t half = NW / 2; half > 0; half /= 2) {
        float *rec = f32kv_lds + (size_t)(way % half) * kRec + lane;
        __syncthreads();
        if (way >= half && way < 2 * half) {
            rec[0] = m;
            rec[kWave] = l;
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) rec[(2 + n * 4 + e) * kWave] = acc[n][e];
        }
        __syncthreads();
        if (way < half) {
            const float mo = rec[0], mn = fmaxf(m, mo), mr = mn > -__builtin_inff() ? mn : 0.0f;
            const float wa = expf_glibc_nonpos(m - mr, exp_tab), wb = expf_glibc_nonpos(mo - mr, exp_tab);
            l = l * wa + rec[kWave] * wb;
            m = mn;
#pragma unroll
            for (int n = 0; n < NT; ++n)
#pragma unroll
                for (int e = 0; e < 4; ++e) acc[n][e] = acc[n][e] * wa + rec[(2 + n * 4 + e) * kWave] * wb;
        }
    }
    if (way == 0 && slot0 + col < slots) {
        // Lane (slot col, grp): per V piece h, 4 VW consecutive dims from
        // d0 + 16 VW h + 4 VW grp.
        const float inv = l > 0.0f ? 1.0f / l : 0.0f;
#pragma unroll
        for (int h = 0; h < VH; ++h)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const uint32_t d = d0 + 16 * VW * h + VW * (4 * grp + e);
                float r[VW];
#pragma unroll
                for (int x = 0; x < VW; ++x) r[x] = l > 0.0f ? acc[h * VW + x][e] * inv : 0.0f;
                // Element stores, which become one vector store of any 4-byte
                // alignment; a branch on out's alignment made two of each.
                if (FULL || d < hd) {
#pragma unroll
                    for (int x = 0; x < VW; ++x) a.out[qoff + d + x] = r[x];
                }
            }
    }
}

template <int HD, int NT, int NW>
int launch_f32kv(const F32kvArgs &a, hipStream_t st) {
    constexpr uint32_t DS = HD / 16 / NT;
    constexpr size_t kStage = (size_t)kTileKeys * HD * NW;
    constexpr size_t kMerge = (size_t)(NW / 2) * (NT * 4 + 2) * kWave;
    constexpr size_t lds = (kStage > kMerge ? kStage : kMerge) * sizeof(float);
    static_assert(lds <= 160 * 1024 - 256, "the CU's LDS less the exp table");
    const uint32_t slots = a.rows * (a.n_heads / a.n_kv);
    const dim3 grid(a.n_kv * DS * ((slots + 15) / 16)), block(NW * kWave);
    if (a.hd == (uint32_t)HD)
        FELLM_LAUNCH((attention_f32kv_kernel<HD, NT, NW, true>), grid, block, lds, st, a);
    else
        FELLM_LAUNCH((attention_f32kv_kernel<HD, NT, NW, false>), grid, block, lds, st, a);
    return launch_status();
}

// A quarter of the output dims per workgroup, and eight key ways, while one
// slot tile per workgroup leaves three CUs in four idle (the copies of Q.K
// then cost idle CUs only).  Not with out == q: the four workgroups of a slot
// tile read the same q, which the first to end would overwrite; one workgroup
// reads its q before its first barrier and writes after its last.
template <int HD>
int choose_f32kv(const F32kvArgs &a, hipStream_t st) {
    const uint64_t slots = (uint64_t)a.rows * (a.n_heads / a.n_kv);
    if (a.q != a.out && a.n_kv * ((slots + 15) / 16) * 4 <= (uint64_t)cu_count())
        return launch_f32kv<HD, HD / 64, 8>(a, st);
    return launch_f32kv<HD, HD / 16, 4>(a, st);
}

int attention_f32kv_common(const float *q, float *out, uint32_t rows, uint32_t n_heads, uint32_t n_kv_heads,
                           uint32_t head_dim, const float *k1, const float *v1, uint32_t begin1, uint32_t end1,
                           const float *k2, const float *v2, uint32_t n2, float scale, uint32_t row_mode,
                           uint32_t window, uint32_t head_major, void *stream) {
    if (!q || !out) return FELLM_ERR_ARITY;
    if (end1 > begin1 && (!k1 || !v1)) return FELLM_ERR_ARITY;
    if (n2 && (!k2 || !v2)) return FELLM_ERR_ARITY;
    if (!n_kv_heads || n_heads % n_kv_heads || head_dim == 0 || head_dim % 4 || head_dim > 256) return FELLM_ERR_SHAPE;
    const uint32_t G = n_heads / n_kv_heads;
    if (G > 16 || (uint64_t)G * head_dim > 2048) return FELLM_ERR_SHAPE;
    for (const void *p : {(const void *)q, (const void *)k1, (const void *)v1, (const void *)k2, (const void *)v2})
        if (p && !aligned_to(p, 16)) return FELLM_ERR_SHAPE;
    if (rows == 0) return FELLM_OK;
    if (!(scale > 0.0f)) scale = 1.0f / sqrtf((float)head_dim);
    F32kvArgs a{q, out, k1, v1, k2, v2, rows, n_heads, n_kv_heads, head_dim, begin1, end1, n2, scale, row_mode,
                window, head_major};
    hipStream_t st = as_stream(stream);
    if (head_dim <= 64) return choose_f32kv<64>(a, st);
    if (head_dim <= 128) return choose_f32kv<128>(a, st);
    return choose_f32kv<256>(a, st);
}

}  // namespace
}  // namespace fellm

extern "C" int fellm_rocm_attention_f32kv(const float *q, float *out, uint32_t rows, uint32_t n_heads,
                                          uint32_t n_kv_heads, uint32_t head_dim, const float *k1, const float *v1,
                                          uint32_t begin1, uint32_t end1, const float *k2, const float *v2, uint32_t n2,
                                          float scale, void *stream) {
    return fellm::attention_f32kv_common(q, out, rows, n_heads, n_kv_heads, head_dim, k1, v1, begin1, end1, k2, v2,
                                         n2, scale, 0, 0, 0, stream);
}

extern "C" int fellm_rocm_attention_f32kv_rows(const float *q, float *out, uint32_t query_len, uint32_t n_heads,
                                               uint32_t n_kv_heads, uint32_t head_dim, const float *k,
                                               const float *v, uint32_t kv_len, float scale, uint32_t causal,
                                               uint32_t window, void *stream) {
    if (query_len == 0) return FELLM_OK;
    if (causal && kv_len < query_len) return FELLM_ERR_SHAPE;  // the query rows end at the last key
    if (kv_len == 0) return FELLM_ERR_SHAPE;
    return fellm::attention_f32kv_common(q, out, query_len, n_heads, n_kv_heads, head_dim, k, v, 0, kv_len, nullptr,
                                         nullptr, 0, scale, causal ? 1 : 2, window, 1, stream);
}
