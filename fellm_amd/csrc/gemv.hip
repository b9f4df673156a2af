// K-quant GEMV (one activation vector) and the fused gate/up GEMV with the
// SwiGLU epilogue.
//
// Reference: crates/backend-cpu/src/backend.rs:944-1002 (launch_gate_up_swiglu)
//   -> kernels/matmul.rs:404-531 (matvec_quant_multi: x quantized once to
//      Q8_K, every gate row then every up row dotted against it) and
//      swiglu.rs:5-16 (out = silu(gate) * up);
//   matmul.rs:534-600 (matvec_quant) for the plain GEMV;
//   Q8_K activations: matmul.rs:213-270 (quantize_row_q8_k_avx2: amax,
//      iscale = 127/amax, round-to-nearest-even, saturate, bsums, d = amax/127);
//   block dots: Q4_K vec_dot_q4k.rs:296-333, Q5_K vec_dot_q5k.rs:189-218,
//      Q6_K matmul.rs:1597-1644 (fused_q6_k_block).
//
// Layout and schedule.  Weights are the GGUF row-major block streams
// (row r = cols/256 blocks of 144 / 176 / 210 bytes), read exactly once with
// non-temporal loads; they are the only HBM traffic that scales with the
// problem.  Each workgroup quantizes x to Q8_K in LDS (cols bytes of qs,
// cols/16 int16 bsums, cols/256 f32 scales) while its first weight loads are
// in flight; every wavefront then keeps the slice of x that it needs in
// registers.  A wavefront walks units of at most 32 blocks per matrix (a group
// of 32/cols*256 whole rows, or its share of the blocks of a longer row): the
// unit's bytes arrive by coalesced 16-byte loads (lane l, chunk 64i + l) into
// registers one unit ahead, are written to the wavefront's LDS stage, and are
// reduced from there by lane pairs, two lanes per block (lane half h covers
// elements 128h .. 128h+127).  The block values of whole rows are folded from
// LDS in parallel lanes, one per row and matrix, and the even lanes apply
// silu(gate) * up.
//
// Arithmetic.  Integer parts are exact: 4-byte dot products (v_dot4) give the
// per-group sums, combined with the 6-bit scales/mins exactly as the CPU's
// i32 arithmetic does, reduced over the lane pair of a block.  The f32 part
// follows the CPU's portable path operation by operation:
//   Q4_K/Q5_K block: ((-dmin)*xd)*f(sumi_min) + (d*xd)*f(sumi);
//   Q6_K block: 16 terms (d*sc)*f(dot) accumulated in (half, group, k)
//     order, times xd;
//   row: serial f32 sum over blocks from 0.0.
// The CPU's SIMD paths for Q4_K/Q5_K (AVX2/VNNI/AVX-512) share the integer
// parts and reorder only that f32 combine.
#include <mutex>
#include <tuple>
#include <vector>

#include "common.hpp"

// Build knob: workgroups in the grid-stride launch (each quantizes x once).
// 512 = two resident workgroups per CU for the LDS-heavy fused formats.
#ifndef FELLM_GEMV_MAX_GRID
#define FELLM_GEMV_MAX_GRID 512
#endif

// Build knob: the widest grid for launches with many units per wavefront.
#ifndef FELLM_GEMV_WIDE_GRID
#define FELLM_GEMV_WIDE_GRID 768
#endif


namespace fellm {
namespace {

constexpr int kGemvBlock = 256;
constexpr int kGemvWaves = kGemvBlock / kWave;
// Build knob: wavefronts per workgroup for rows of at most 32 blocks.  8
// measured slower at the 8B gate/up shape: 16.2 us with 384 workgroups, 18.8
// with 512, against 14.5 us for 4.
#ifndef FELLM_GEMV_ONE_WAVES
#define FELLM_GEMV_ONE_WAVES 4
#endif
constexpr uint32_t kGemvMaxCols = 49152;
// Dynamic LDS a workgroup may take: the CU's 160 KB less the kernel's static
// LDS (the exp table) with room to spare.
constexpr uint32_t kGemvLdsLimit = 160 * 1024 - 1024;
#ifndef FELLM_GEMV_MAX_GRID_PRE
#define FELLM_GEMV_MAX_GRID_PRE 1024
#endif
constexpr uint32_t kGemvMaxGridPre = FELLM_GEMV_MAX_GRID_PRE;

// Q8_K copy of x in (dynamic) LDS: qs[cols], bsums[cols/16], d[cols/256],
// then the per-wavefront row-fold buffers [waves][rows][matrices][nb rounded up to 4].
struct XLds {
    int8_t *qs;
    int16_t *bs;
    float *d;
    float *fold;
};
__host__ __device__ constexpr uint32_t gemv_fold_off(uint32_t nb) { return (nb * 292 + 15) / 16 * 16; }
// fold_per_wave: floats of row-fold buffer per wavefront.
__host__ __device__ constexpr uint32_t gemv_lds_bytes(uint32_t nb, uint32_t fold_per_wave,
                                                     uint32_t waves = kGemvWaves) {
    return gemv_fold_off(nb) + waves * fold_per_wave * 4;
}
__device__ __forceinline__ XLds carve_lds(uint8_t *base, uint32_t nb) {
    return {reinterpret_cast<int8_t *>(base), reinterpret_cast<int16_t *>(base + nb * 256),
            reinterpret_cast<float *>(base + nb * 288), reinterpret_cast<float *>(base + gemv_fold_off(nb))};
}

// quantize_row_q8_k_avx2 (matmul.rs:213-270) for the 256-element blocks of x:
// wavefront `first` takes blocks first, first + stride, ...; lane l holds
// elements 4l..4l+3.  xl may point into LDS or global memory.  The x loads of
// kXBatch blocks go out together before any of them is reduced, and the
// batch's amax reductions (DPP inside each 16-lane row, then the four rows'
// values read as scalars) run side by side: the prologue is a short chain,
// not one LDS shuffle round trip per reduction step and block.
// fmaxf ignores a NaN operand, so the reduction order does not change amax.
__device__ __forceinline__ float block_absmax(const float4 v) {
    float a = fmaxf(fmaxf(__builtin_fabsf(v.x), __builtin_fabsf(v.y)), fmaxf(__builtin_fabsf(v.z), __builtin_fabsf(v.w)));
    a = group_max_f32<16>(a);
    const int ai = __float_as_int(a);
    const float r0 = __int_as_float(__builtin_amdgcn_readlane(ai, 0)), r1 = __int_as_float(__builtin_amdgcn_readlane(ai, 16));
    const float r2 = __int_as_float(__builtin_amdgcn_readlane(ai, 32)), r3 = __int_as_float(__builtin_amdgcn_readlane(ai, 48));
    return fmaxf(fmaxf(r0, r1), fmaxf(r2, r3));
}

__device__ __forceinline__ void quantize_block(const float4 v, const float a, uint32_t b, const XLds &xl,
                                               uint32_t lane) {
    int32_t q[4] = {0, 0, 0, 0};
    if (a != 0.0f) {
        const float iscale = 127.0f / a;
        const float e[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // x86 cvtps_epi32 gives INT32_MIN for NaN and |p| >= 2^31 (iscale is
            // inf when amax < ~3.7e-37); the saturating packs make it -128.
            const float p = e[k] * iscale;
            const float r = __builtin_rintf(p);
            q[k] = !(__builtin_fabsf(p) < 0x1p31f) ? -128 : r < -128.0f ? -128 : r > 127.0f ? 127 : (int32_t)r;
        }
    }
    const uint32_t packed = (uint32_t)(q[0] & 0xff) | (uint32_t)(q[1] & 0xff) << 8 | (uint32_t)(q[2] & 0xff) << 16 |
                            (uint32_t)(q[3] & 0xff) << 24;
    *reinterpret_cast<uint32_t *>(&xl.qs[b * 256 + lane * 4]) = packed;
    int32_t s = q[0] + q[1] + q[2] + q[3];
    s += (int32_t)dpp_u32<0xB1>((uint32_t)s);  // quad xor 1
    s += (int32_t)dpp_u32<0x4E>((uint32_t)s);  // quad xor 2
    if ((lane & 3) == 0) xl.bs[b * 16 + lane / 4] = (int16_t)s;
    if (lane == 0) xl.d[b] = a / 127.0f;
}

constexpr int kXBatch = 8;

// This wavefront's number in its workgroup, as a scalar.
__device__ __forceinline__ uint32_t wave_id() { return __builtin_amdgcn_readfirstlane(threadIdx.x / kWave); }

__device__ __forceinline__ void load_x_batch(const float *__restrict__ x, uint32_t nb, uint32_t b0, uint32_t stride,
                                             float4 (&v)[kXBatch]) {
    const uint32_t lane = threadIdx.x % kWave;
#pragma unroll
    for (int j = 0; j < kXBatch; ++j) {
        const uint32_t b = b0 + j * stride;
        v[j] = b < nb ? *reinterpret_cast<const float4 *>(x + (size_t)b * 256 + lane * 4)
                      : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
    }
}

__device__ __forceinline__ void quantize_batch(const float4 (&v)[kXBatch], uint32_t nb, uint32_t b0, uint32_t stride,
                                               const XLds &xl) {
    const uint32_t lane = threadIdx.x % kWave;
    float a[kXBatch];
    // In pairs, so that two reductions run side by side and a short row's
    // absent blocks (b0 and stride are the same in every lane) cost nothing:
    // against reducing all 8 whatever the row, 2048 x 2048 Q4_K 4.25 -> 3.91
    // us, 6144 x 4096 6.63 -> 6.29, gate/up 8192 x 2048 7.85 -> 7.24.
#pragma unroll
    for (int g = 0; g < kXBatch; g += 2) {
        if (b0 + g * stride >= nb) break;
#pragma unroll
        for (int j = g; j < g + 2; ++j) a[j] = block_absmax(v[j]);
#pragma unroll
        for (int j = g; j < g + 2; ++j) {
            const uint32_t b = b0 + j * stride;
            if (b < nb) quantize_block(v[j], a[j], b, xl, lane);
        }
    }
}

__device__ void quantize_x(const float *__restrict__ x, uint32_t nb, const XLds &xl, uint32_t first,
                           uint32_t stride) {
    for (uint32_t b0 = first; b0 < nb; b0 += stride * kXBatch) {
        float4 v[kXBatch];
        load_x_batch(x, nb, b0, stride, v);
        quantize_batch(v, nb, b0, stride, xl);
    }
}

// The Q8_K activation blob: the same layout in global memory as in LDS
// (qs[nb * 256] int8, bsums[nb * 16] int16, d[nb] f32; nb * 292 bytes).
__host__ __device__ constexpr uint32_t q8k_blob_bytes(uint32_t nb) { return nb * 292; }

// x into the workgroup's LDS: quantized here (PREQ = false), or copied from a
// blob that fellm_rocm_quantize_q8k wrote once for the whole launch.  In two
// halves: x_issue requests the thread's first batch of x (or of the blob)
// into registers, x_finish quantizes (copies) it and the rest.  The kernel
// issues x before its first weight loads, so that x does not queue behind
// the weight stream (x is on every wavefront's critical path).
constexpr int kBlobBatch = 4;
template <bool PREQ>
struct XFirst {
    float4 v[kXBatch];
};
template <>
struct XFirst<true> {
    uint32_t v[kBlobBatch];
};

template <bool PREQ>
__device__ __forceinline__ void x_issue(const void *__restrict__ xsrc, uint32_t nb, XFirst<PREQ> &f) {
    if constexpr (PREQ) {
        const uint32_t words = q8k_blob_bytes(nb) / 4;
        const uint32_t *src = static_cast<const uint32_t *>(xsrc);
#pragma unroll
        for (int j = 0; j < kBlobBatch; ++j) {
            const uint32_t i = threadIdx.x + j * blockDim.x;
            f.v[j] = i < words ? src[i] : 0u;
        }
    } else {
        load_x_batch(static_cast<const float *>(xsrc), nb, wave_id(), blockDim.x / kWave, f.v);
    }
}

template <bool PREQ>
__device__ __forceinline__ void x_finish(const void *__restrict__ xsrc, uint32_t nb, const XLds &xl, uint8_t *smem,
                                         const XFirst<PREQ> &f) {
    if constexpr (PREQ) {
        const uint32_t words = q8k_blob_bytes(nb) / 4;
        const uint32_t *src = static_cast<const uint32_t *>(xsrc);
        uint32_t *dst = reinterpret_cast<uint32_t *>(smem);
#pragma unroll
        for (int j = 0; j < kBlobBatch; ++j) {
            const uint32_t i = threadIdx.x + j * blockDim.x;
            if (i < words) dst[i] = f.v[j];
        }
        for (uint32_t i0 = threadIdx.x + blockDim.x * kBlobBatch; i0 < words; i0 += blockDim.x * kBlobBatch) {
            uint32_t v[kBlobBatch];
#pragma unroll
            for (int j = 0; j < kBlobBatch; ++j) {
                const uint32_t i = i0 + j * blockDim.x;
                v[j] = i < words ? src[i] : 0u;
            }
#pragma unroll
            for (int j = 0; j < kBlobBatch; ++j) {
                const uint32_t i = i0 + j * blockDim.x;
                if (i < words) dst[i] = v[j];
            }
        }
    } else {
        const float *x = static_cast<const float *>(xsrc);
        const uint32_t first = wave_id();
        const uint32_t nw = blockDim.x / kWave;
        quantize_batch(f.v, nb, first, nw, xl);
        quantize_x(x, nb, xl, first + nw * kXBatch, nw);
    }
}

template <bool PREQ>
__device__ __forceinline__ void fill_x(const void *__restrict__ xsrc, uint32_t nb, const XLds &xl, uint8_t *smem) {
    XFirst<PREQ> f;
    x_issue<PREQ>(xsrc, nb, f);
    x_finish<PREQ>(xsrc, nb, xl, smem, f);
}

__device__ __forceinline__ uint4 lds_u4(const void *p) { return *reinterpret_cast<const uint4 *>(p); }

// Weight streams are read through a buffer resource whose range is the
// launch's rows: a load past the end returns zeros without touching memory,
// so the next row group is requested unconditionally (no branch around the
// loads, hence exact wait counts) and the last request costs nothing.
// Cache policy 2 = non-temporal (read once).
using Rsrc = __amdgpu_buffer_rsrc_t;
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
__device__ __forceinline__ Rsrc weight_rsrc(const uint8_t *w, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t *>(w), 0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ float f16_bits(uint32_t b) { return (float)__builtin_bit_cast(_Float16, (uint16_t)b); }

// Partner lane of a pair (lane ^ 1): DPP quad_perm [1,0,3,2].
__device__ __forceinline__ uint32_t pair_swap(uint32_t v) { return dpp_u32<0xB1>(v); }

// ---- lane layout ----------------------------------------------------------------
// Two lanes per 256-element block: lane half h (= lane & 1) covers elements
// 128h .. 128h+127.  The 32 lane pairs of a wavefront take 32 block slots:
// with nb <= 32 blocks per row, slot s is block s % nb of row s / nb of the
// wavefront's current row group (32 / nb rows at once); with nb > 32 it is
// block s of the wavefront's share of a row.  Bytes both lanes of a block need (the
// Q4_K/Q5_K header, the Q5_K high bits) are loaded half by each lane and
// exchanged with one DPP swap: lanes reading the same address in one load
// slow the memory pipeline measurably.

// Lane's Q8_K slice of x for its half block.
struct XHalf {
    uint4 q[8];      // x quants of elements 128h .. 128h+127
    int32_t s2[4];   // Q4_K/Q5_K: bsums of the 4 32-element groups
    int32_t s1[8];   // Q6_K: bsums of the 8 16-element groups
    float d;
};

__device__ __forceinline__ void load_x(const XLds &xl, uint32_t b, uint32_t h, XHalf &x) {
    const int8_t *q = xl.qs + b * 256 + 128 * h;
#pragma unroll
    for (int i = 0; i < 8; ++i) x.q[i] = lds_u4(q + 16 * i);
    const int16_t *bs = xl.bs + b * 16 + 8 * h;
#pragma unroll
    for (int g = 0; g < 8; ++g) x.s1[g] = bs[g];
#pragma unroll
    for (int j = 0; j < 4; ++j) x.s2[j] = x.s1[2 * j] + x.s1[2 * j + 1];
    x.d = xl.d[b];
}

// The 4 (scale, min) pairs of groups j = 4h .. 4h+3 from the 12 scale bytes
// (get_scale_min_k4, dequant.rs:295-305) as packed bytes, four at a time:
// h = 0: sc = q[j] & 63, m = q[j+4] & 63;
// h = 1: sc = (q[j+4] & 15) | (q[j-4] >> 6) << 4, m = (q[j+4] >> 4) | (q[j] >> 6) << 4.
__device__ __forceinline__ void k4_scales_half(uint32_t s0, uint32_t s1, uint32_t s2, uint32_t h, uint32_t &sc,
                                               uint32_t &m) {
    const uint32_t sc_hi = (s2 & 0x0f0f0f0fu) | ((s0 >> 2) & 0x30303030u);
    const uint32_t m_hi = ((s2 >> 4) & 0x0f0f0f0fu) | ((s1 >> 2) & 0x30303030u);
    sc = h ? sc_hi : (s0 & 0x3f3f3f3fu);
    m = h ? m_hi : (s1 & 0x3f3f3f3fu);
}

// ---- weight formats ---------------------------------------------------------------
// Raw per-lane block bytes, read from the wavefront's LDS stage (where the
// row group was streamed with coalesced 16-byte loads).  Lane half h.
struct Q4K {
    static constexpr uint32_t kBytes = 144;
    struct Raw {
        uint4 hdr;   // d, dmin, 12 scale bytes
        uint4 q[4];  // qs bytes 64h .. 64h+63
    };
    __device__ static Raw read(const uint8_t *blk, uint32_t h) {
        Raw r;
        r.hdr = lds_u4(blk);
#pragma unroll
        for (int i = 0; i < 4; ++i) r.q[i] = lds_u4(blk + 16 + 64 * h + 16 * i);
        return r;
    }
};

struct Q5K {
    static constexpr uint32_t kBytes = 176;
    struct Raw {
        uint4 hdr;
        uint4 qh[2];  // the 32 high-bit bytes
        uint4 q[4];   // qs bytes 64h .. 64h+63
    };
    __device__ static Raw read(const uint8_t *blk, uint32_t h) {
        Raw r;
        r.hdr = lds_u4(blk);
        r.qh[0] = lds_u4(blk + 16);
        r.qh[1] = lds_u4(blk + 32);
#pragma unroll
        for (int i = 0; i < 4; ++i) r.q[i] = lds_u4(blk + 48 + 64 * h + 16 * i);
        return r;
    }
};

// 210-byte Q6_K blocks sit at 2-byte aligned LDS offsets; gfx950 serves the
// unaligned 16- and 8-byte LDS reads directly.
__device__ __forceinline__ uint4 lds_u4_any(const uint8_t *p) {
    uint4 v;
    __builtin_memcpy(&v, p, 16);
    return v;
}

struct Q6K {
    static constexpr uint32_t kBytes = 210;
    struct Raw {
        uint4 ql[4];  // ql bytes 64h .. 64h+63
        uint4 qh[2];  // qh bytes 32h .. 32h+31
        uint2 sc;     // int8 scales 8h .. 8h+7
        uint32_t d;
    };
    __device__ static Raw read(const uint8_t *blk, uint32_t h) {
        Raw r;
#pragma unroll
        for (int i = 0; i < 4; ++i) r.ql[i] = lds_u4_any(blk + 64 * h + 16 * i);
        r.qh[0] = lds_u4_any(blk + 128 + 32 * h);
        r.qh[1] = lds_u4_any(blk + 144 + 32 * h);
        __builtin_memcpy(&r.sc, blk + 192 + 8 * h, 8);
        uint16_t dd;
        __builtin_memcpy(&dd, blk + 208, 2);
        r.d = dd;
        return r;
    }
};

__device__ __forceinline__ uint32_t u4_at(const uint4 &v, int i) { return i == 0 ? v.x : i == 1 ? v.y : i == 2 ? v.z : v.w; }

// Q4_K / Q5_K block value.  Lane h: chunks c = 2h, 2h+1 (qs bytes 32c .. 32c+31,
// low nibbles -> group 2c, high -> 2c+1), groups j = 4h .. 4h+3.  The exact
// integers of both halves are summed over the lane pair; both lanes then form
// ((-dmin)*xd)*f(sumi_min) + (d*xd)*f(sumi) (vec_dot_q4k.rs:296-333).
template <typename W>
__device__ __forceinline__ float k45_value(const typename W::Raw &r, uint32_t h, const XHalf &x) {
    uint32_t scp, mp;
    k4_scales_half(r.hdr.y, r.hdr.z, r.hdr.w, h, scp, mp);
    uint32_t qh[8];
    if constexpr (W::kBytes == 176) {
        qh[0] = r.qh[0].x;
        qh[1] = r.qh[0].y;
        qh[2] = r.qh[0].z;
        qh[3] = r.qh[0].w;
        qh[4] = r.qh[1].x;
        qh[5] = r.qh[1].y;
        qh[6] = r.qh[1].z;
        qh[7] = r.qh[1].w;
    }
    int32_t si = 0, sm = 0;
#pragma unroll
    for (int cc = 0; cc < 2; ++cc) {
        int32_t dlo = 0, dhi = 0;
#pragma unroll
        for (int i = 0; i < 8; ++i) {
            const uint32_t q = u4_at(r.q[2 * cc + i / 4], i % 4);
            uint32_t lo = q & 0x0f0f0f0fu, hi = (q >> 4) & 0x0f0f0f0fu;
            if constexpr (W::kBytes == 176) {
                // bit 2c (low) / 2c+1 (high) of qh byte l adds 16 (unpack_q5_k_aux8)
                const uint32_t c2 = 2 * (2 * h + cc);
                lo |= ((qh[i] >> c2) & 0x01010101u) << 4;
                hi |= ((qh[i] >> (c2 + 1)) & 0x01010101u) << 4;
            }
            dlo = __builtin_amdgcn_sdot4((int)lo, (int)u4_at(x.q[4 * cc + i / 4], i % 4), dlo, false);
            dhi = __builtin_amdgcn_sdot4((int)hi, (int)u4_at(x.q[4 * cc + 2 + i / 4], i % 4), dhi, false);
        }
        const int32_t sc_lo = (scp >> (16 * cc)) & 0xff, sc_hi = (scp >> (16 * cc + 8)) & 0xff;
        const int32_t m_lo = (mp >> (16 * cc)) & 0xff, m_hi = (mp >> (16 * cc + 8)) & 0xff;
        si += sc_lo * dlo + sc_hi * dhi;
        sm += m_lo * x.s2[2 * cc] + m_hi * x.s2[2 * cc + 1];
    }
    si += (int32_t)pair_swap((uint32_t)si);
    sm += (int32_t)pair_swap((uint32_t)sm);
    const float d = f16_bits(r.hdr.x & 0xffffu), dmin = f16_bits(r.hdr.x >> 16);
    const float t_min = (-dmin * x.d) * (float)sm;
    const float t_sc = (d * x.d) * (float)si;
    return t_min + t_sc;
}

// Q6_K block value (matmul.rs:1597-1644).  Lane h covers half h: for group
// parity is and k = 0..3 the run 128h + 16is + 32k.  The lane forms its 8
// terms (d*sc[8h+is+2k]) * dot in (is, k) order; lane 0's partial sum is
// handed to lane 1, which adds its 8 terms: the CPU's (h, is, k) order.  The
// block value acc * xd is valid in lane h = 1.
__device__ __forceinline__ float q6k_value(const Q6K::Raw &r, uint32_t h, const XHalf &x) {
    const float d = f16_bits(r.d);
    float t[8];
#pragma unroll
    for (int is = 0; is < 2; ++is) {
        int32_t dots[4] = {0, 0, 0, 0};
#pragma unroll
        for (int i = 0; i < 4; ++i) {  // dword i of the 16-byte run l = 16is + 4i ..
            const uint32_t A = u4_at(r.ql[is], i), B = u4_at(r.ql[2 + is], i), H = u4_at(r.qh[is], i);
            const uint32_t w1 = (A & 0x0f0f0f0fu) | ((H << 4) & 0x30303030u);
            const uint32_t w2 = (B & 0x0f0f0f0fu) | ((H << 2) & 0x30303030u);
            const uint32_t w3 = ((A >> 4) & 0x0f0f0f0fu) | (H & 0x30303030u);
            const uint32_t w4 = ((B >> 4) & 0x0f0f0f0fu) | ((H >> 2) & 0x30303030u);
            dots[0] = __builtin_amdgcn_sdot4((int)w1, (int)u4_at(x.q[is], i), dots[0], false);
            dots[1] = __builtin_amdgcn_sdot4((int)w2, (int)u4_at(x.q[2 + is], i), dots[1], false);
            dots[2] = __builtin_amdgcn_sdot4((int)w3, (int)u4_at(x.q[4 + is], i), dots[2], false);
            dots[3] = __builtin_amdgcn_sdot4((int)w4, (int)u4_at(x.q[6 + is], i), dots[3], false);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            // q - 32 in every weight: dot(q - 32, x) = dot(q, x) - 32 * bsum of the run
            const int32_t dk = dots[k] - 32 * x.s1[is + 2 * k];
            const uint32_t sb = is + 2 * k;  // scale byte within the half's 8
            const int32_t sc = (int8_t)((sb < 4 ? r.sc.x : r.sc.y) >> (8 * (sb & 3)));
            t[4 * is + k] = (d * (float)sc) * (float)dk;
        }
    }
    float a = 0.0f;
    if (h == 0) {
#pragma unroll
        for (int i = 0; i < 8; ++i) a += t[i];
    }
    const float from0 = __uint_as_float(dpp_u32<0x111>(__float_as_uint(a)));  // row_shr:1
    if (h == 1) {
        a = from0;
#pragma unroll
        for (int i = 0; i < 8; ++i) a += t[i];
    }
    return a * x.d;
}

template <typename W>
__device__ __forceinline__ float block_value(const typename W::Raw &r, uint32_t h, const XHalf &x) {
    if constexpr (W::kBytes == 210)
        return q6k_value(r, h, x);
    else
        return k45_value<W>(r, h, x);
}

__device__ __forceinline__ void wave_lds_sync() {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront", "local");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront", "local");
}

// Serial f32 sum of a row's n block values in LDS, in block order, onto acc
// (16-byte reads; f is 16-byte aligned).
__device__ __forceinline__ float fold_serial(const float *f, uint32_t n, float acc) {
    const float4 *f4 = reinterpret_cast<const float4 *>(f);
    uint32_t i = 0;
    for (; i + 4 <= n; i += 4) {
        const float4 t = f4[i / 4];
        acc += t.x;
        acc += t.y;
        acc += t.z;
        acc += t.w;
    }
    for (; i < n; ++i) acc += f[i];
    return acc;
}

// ---- staging: coalesced 16-byte loads of a contiguous byte range ---------------
// A wavefront's unit of work is a contiguous byte range of each matrix (a
// group of whole rows, or its share of a longer row) of at most 32 blocks.
// It is fetched as aligned 16-byte chunks, lane l taking chunk 64i + l, so
// one load instruction covers 1 KB of consecutive bytes (the pattern that
// reaches the copy-kernel bandwidth; per-block lane patterns measured
// 25-45% slower), and written to the wavefront's LDS stage.  The lanes then
// read their block's bytes from the stage.  Chunks past the unit read outside
// the buffer range: zeros, no traffic.
// 1 KB chunks per lane per unit: 32 blocks + up to 15 alignment bytes
// (Q4_K 5, Q5_K 6, Q6_K 7).
template <typename W>
constexpr uint32_t kChunks = (32 * W::kBytes + 15 + 1023) / 1024;

template <typename W>
struct Staged {
    u32x4 v[kChunks<W>];
};
template <typename W>
__device__ __forceinline__ void stage_issue(Rsrc w, uint32_t begin, uint32_t end, uint32_t lane, Staged<W> &s) {
    const uint32_t a0 = begin & ~15u;
#pragma unroll
    for (uint32_t i = 0; i < kChunks<W>; ++i) {
        const uint32_t off = a0 + 1024 * i + 16 * lane;
        s.v[i] = __builtin_amdgcn_raw_buffer_load_b128(w, off < end ? off : 0x80000000u, 0, 2);
    }
}
template <typename W>
__device__ __forceinline__ void stage_store(uint8_t *st, uint32_t lane, const Staged<W> &s) {
#pragma unroll
    for (uint32_t i = 0; i < kChunks<W>; ++i) *reinterpret_cast<u32x4 *>(st + 1024 * i + 16 * lane) = s.v[i];
}
// LDS stage bytes per wavefront.
template <typename GW, typename UW, bool FUSED>
constexpr uint32_t kStagePerWave = 1024 * (kChunks<GW> + (FUSED ? kChunks<UW> : 0));

// Rows of at most 32 blocks.  GW: gate (or the only) format; UW: up format
// (unused unless FUSED).  A unit is a group of rp = 32/nb consecutive rows;
// lane pair slot s works on block s % nb of row s / nb; the lane's x slice
// stays in registers for the whole launch.
// Each step: next unit's loads issued -> block values of the staged unit ->
// fold buffer, from which lanes 0 .. mats*rows-1 each fold one
// (row, matrix) serially over its block values from 0.0 and the even lanes
// apply silu(gate) * up; then the next unit is written to the stage.
template <typename GW, typename UW, bool FUSED, bool PREQ, int NW = kGemvWaves>
__global__ __launch_bounds__(NW * kWave) void kquant_gemv_kernel(const uint8_t *__restrict__ gw,
                                                                  const uint8_t *__restrict__ uw,
                                                                  const void *__restrict__ x, float *__restrict__ out,
                                                                  uint32_t rows, uint32_t nb, uint32_t rp) {
    constexpr uint32_t kMats = FUSED ? 2 : 1;
    extern __shared__ __align__(16) uint8_t gemv_smem[];
    __shared__ uint64_t tab_lds[32];
    const XLds xl = carve_lds(gemv_smem, nb);
    const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint32_t h = lane & 1, slot = lane >> 1;
    const uint32_t nbp = (nb + 3) & ~3u;
    const uint32_t fold_floats = kMats * rp * nbp;
    uint8_t *stage = reinterpret_cast<uint8_t *>(xl.fold + NW * fold_floats) + wave * kStagePerWave<GW, UW, FUSED>;
    uint8_t *ustage = stage + 1024 * kChunks<GW>;
    float *fold = xl.fold + wave * fold_floats;
    const uint32_t grb = nb * GW::kBytes, urb = nb * UW::kBytes;
    const uint32_t g_end = rows * grb, u_end = rows * urb;
    const Rsrc wg = weight_rsrc(gw, g_end);
    const Rsrc wu = weight_rsrc(FUSED ? uw : gw, FUSED ? u_end : g_end);
    const uint32_t wstride = gridDim.x * NW;
    const uint32_t wid = blockIdx.x * NW + wave;

    // unit n of this wavefront: its first row and its byte range per matrix
    auto unit_row = [&](uint32_t n) { return (wid + n * wstride) * rp; };
    auto range = [&](uint32_t n, uint32_t rb, uint32_t lim, uint32_t &b0, uint32_t &b1) {
        const uint32_t r = unit_row(n);
        b0 = r < rows ? r * rb : 0;
        b1 = r < rows ? b0 + rp * rb : 0;
        if (b1 > lim) b1 = lim;
    };

    // Everything the prologue waits for (x, the exp table) is requested
    // before the first unit's weights: loads complete in order, so a wait
    // for a later load would wait for the whole weight burst too.
    XFirst<PREQ> xf;
    x_issue<PREQ>(x, nb, xf);
    uint64_t tab_v = 0;
    {
        constexpr ExpfTable T = make_expf_table();
        if (threadIdx.x < 32) tab_v = T.tab[threadIdx.x];
    }
    Staged<GW> sg;
    Staged<UW> su;
    uint32_t gb0, gb1, ub0 = 0, ub1 = 0;
    range(0, grb, g_end, gb0, gb1);
    stage_issue(wg, gb0, gb1, lane, sg);
    if constexpr (FUSED) {
        range(0, urb, u_end, ub0, ub1);
        stage_issue(wu, ub0, ub1, lane, su);
    }
    if (threadIdx.x < 32) tab_lds[threadIdx.x] = tab_v;
    x_finish<PREQ>(x, nb, xl, gemv_smem, xf);
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");

    const uint32_t ro = slot / nb, b = slot - ro * nb;
    const bool on = ro < rp;
    XHalf xh;
    load_x(xl, b, h, xh);
    stage_store(stage, lane, sg);
    if constexpr (FUSED) stage_store(ustage, lane, su);

    // Block values of the staged unit n (byte ranges starting at cg0 / cu0),
    // then the row folds and the stores.
    auto work = [&](uint32_t n, uint32_t cg0, uint32_t cu0) {
        const uint32_t row0 = unit_row(n);
        wave_lds_sync();
        {
            const uint8_t *blk = stage + (cg0 & 15u) + ro * grb + b * GW::kBytes;
            const float v = block_value<GW>(GW::read(blk, h), h, xh);
            if (on && h == (GW::kBytes == 210 ? 1u : 0u)) fold[ro * kMats * nbp + b] = v;
        }
        if constexpr (FUSED) {
            const uint8_t *blk = ustage + (cu0 & 15u) + ro * urb + b * UW::kBytes;
            const float v = block_value<UW>(UW::read(blk, h), h, xh);
            if (on && h == (UW::kBytes == 210 ? 1u : 0u)) fold[(ro * kMats + 1) * nbp + b] = v;
        }
        wave_lds_sync();
        float acc = 0.0f;
        if (lane < kMats * rp) acc = fold_serial(fold + lane * nbp, nb, 0.0f);
        if constexpr (FUSED) {
            const float up = dpp_f32<0x101>(acc);  // row_shl:1, lane i reads lane i+1
            const uint32_t r = row0 + lane / 2;
            if (lane < 2 * rp && (lane & 1) == 0 && r < rows) out[r] = silu(acc, tab_lds) * up;
        } else {
            if (lane < rp && row0 + lane < rows) out[row0 + lane] = acc;
        }
        wave_lds_sync();
    };

    for (uint32_t n = 0;; ++n) {
        if (unit_row(n) >= rows) break;
        const uint32_t cg0 = gb0, cu0 = ub0;  // staged unit's byte ranges start here
        range(n + 1, grb, g_end, gb0, gb1);
        stage_issue(wg, gb0, gb1, lane, sg);
        if constexpr (FUSED) {
            range(n + 1, urb, u_end, ub0, ub1);
            stage_issue(wu, ub0, ub1, lane, su);
        }
        work(n, cg0, cu0);
        stage_store(stage, lane, sg);
        if constexpr (FUSED) stage_store(ustage, lane, su);
    }
}

// Rows of more than 32 blocks.  A row's blocks are divided over `passes`
// wavefronts (at most 32 each), so that a wavefront's x slice stays in
// registers for the launch; a workgroup of passes * groups wavefronts works on
// `groups` rows at a time.  (One wavefront walking a row's passes re-read its
// x slice from LDS for every 32 blocks, at an eight-way bank conflict, and
// folded its row in a single lane: 8192 x 28672 Q4_K 41.2 -> 28.4 us, Q6_K 58.6
// -> 43.3, 4096 x 14336 Q4_K 13.0 -> 11.3, 5120 x 13824 20.0 -> 13.2; with 8
// wavefronts per workgroup instead of 16 31.1, 46.0, 11.5 and 13.5.)  The
// workgroup has more wavefronts than the launch's passes * groups: the others
// take their part of x's quantization and end (256 x 16384 Q4_K in workgroups
// of two wavefronts 16.3 us, with 14 more for x 7.1).  The block values of kFoldRows
// rows per group collect in LDS; after a barrier one wavefront, another for
// every batch, folds all of them, a lane per (row, matrix), while the others go
// on into the second fold buffer.
constexpr uint32_t kFoldRows = 4;
constexpr uint32_t gemv_pass_lds(uint32_t nb, uint32_t passes, uint32_t groups, uint32_t mats, uint32_t stage) {
    const uint32_t nbp = (nb + 3) & ~3u;
    return gemv_fold_off(nb) + 2 * groups * kFoldRows * mats * nbp * 4 + passes * groups * stage;
}

template <typename GW, typename UW, bool FUSED, bool PREQ, int MAXW>
__global__ __launch_bounds__(MAXW * kWave) void kquant_gemv_passes(const uint8_t *__restrict__ gw,
                                                                    const uint8_t *__restrict__ uw,
                                                                    const void *__restrict__ x, float *__restrict__ out,
                                                                    uint32_t rows, uint32_t nb, uint32_t passes,
                                                                    uint32_t groups) {
    constexpr uint32_t kMats = FUSED ? 2 : 1;
    extern __shared__ __align__(16) uint8_t gemv_smem[];
    __shared__ uint64_t tab_lds[32];
    const XLds xl = carve_lds(gemv_smem, nb);
    const uint32_t wave = __builtin_amdgcn_readfirstlane(threadIdx.x / kWave), lane = threadIdx.x % kWave;
    const uint32_t h = lane & 1, slot = lane >> 1;
    const uint32_t nbp = (nb + 3) & ~3u;
    const uint32_t pass = wave % passes, group = wave / passes, waves = passes * groups;
    const uint32_t per = (nb + passes - 1) / passes, first = pass * per;
    const bool helper = wave >= waves;  // prepares x and ends
    const uint32_t mine = first < nb && !helper ? (nb - first < per ? nb - first : per) : 0;
    const uint32_t batch_floats = groups * kFoldRows * kMats * nbp;
    uint8_t *stage = reinterpret_cast<uint8_t *>(xl.fold + 2 * batch_floats) + wave * kStagePerWave<GW, UW, FUSED>;
    uint8_t *ustage = stage + 1024 * kChunks<GW>;
    const uint32_t grb = nb * GW::kBytes, urb = nb * UW::kBytes;
    const Rsrc wg = weight_rsrc(gw, rows * grb);
    const Rsrc wu = weight_rsrc(FUSED ? uw : gw, FUSED ? rows * urb : rows * grb);

    auto row_of = [&](uint32_t n, uint32_t g) { return (n * gridDim.x + blockIdx.x) * groups + g; };
    const uint32_t steps = (rows + gridDim.x * groups - 1) / (gridDim.x * groups);
    auto range = [&](uint32_t n, uint32_t rb, uint32_t kb, uint32_t &b0, uint32_t &b1) {
        const uint32_t r = row_of(n, group);
        b0 = r < rows && !helper ? r * rb + first * kb : 0;
        b1 = r < rows ? b0 + mine * kb : 0;
    };

    // x and the exp table before the first unit's weights, as in the kernel above.
    XFirst<PREQ> xf;
    x_issue<PREQ>(x, nb, xf);
    uint64_t tab_v = 0;
    {
        constexpr ExpfTable T = make_expf_table();
        if (threadIdx.x < 32) tab_v = T.tab[threadIdx.x];
    }
    Staged<GW> sg;
    Staged<UW> su;
    uint32_t gb0, gb1, ub0 = 0, ub1 = 0;
    auto issue = [&](uint32_t n) {
        range(n, grb, GW::kBytes, gb0, gb1);
        stage_issue(wg, gb0, gb1, lane, sg);
        if constexpr (FUSED) {
            range(n, urb, UW::kBytes, ub0, ub1);
            stage_issue(wu, ub0, ub1, lane, su);
        }
    };
    auto store = [&] {
        stage_store(stage, lane, sg);
        if constexpr (FUSED) stage_store(ustage, lane, su);
    };
    auto barrier = [&] {  // orders LDS only: the weight loads stay in flight
        __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
        __builtin_amdgcn_s_barrier();
        __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
    };
    issue(0);
    if (threadIdx.x < 32) tab_lds[threadIdx.x] = tab_v;
    x_finish<PREQ>(x, nb, xl, gemv_smem, xf);
    barrier();
    if (helper) return;  // an ended wavefront takes no part in the barriers below
    const bool on = slot < mine;
    XHalf xh;
    load_x(xl, on ? first + slot : 0, h, xh);
    store();

    uint32_t turn = 0;
    for (uint32_t n0 = 0; n0 < steps; n0 += kFoldRows) {
        float *fold = xl.fold + (n0 / kFoldRows % 2) * batch_floats;
        const uint32_t n1 = steps - n0 < kFoldRows ? steps - n0 : kFoldRows;
        for (uint32_t i = 0; i < n1; ++i) {
            const uint32_t cg0 = gb0, cu0 = ub0;  // the staged unit starts here
            issue(n0 + i + 1);
            wave_lds_sync();
            float *f = fold + (group * kFoldRows + i) * kMats * nbp + first + slot;
            {
                const float v = block_value<GW>(GW::read(stage + (cg0 & 15u) + slot * GW::kBytes, h), h, xh);
                if (on && h == (GW::kBytes == 210 ? 1u : 0u)) f[0] = v;
            }
            if constexpr (FUSED) {
                const float v = block_value<UW>(UW::read(ustage + (cu0 & 15u) + slot * UW::kBytes, h), h, xh);
                if (on && h == (UW::kBytes == 210 ? 1u : 0u)) f[nbp] = v;
            }
            wave_lds_sync();
            store();
        }
        barrier();
        if (wave == turn) {
            const uint32_t e = lane / kMats, g = e / kFoldRows, i = e % kFoldRows;
            const uint32_t r = row_of(n0 + i, g);
            const bool live = g < groups && i < n1 && r < rows;
            float acc = 0.0f;
            if (live) acc = fold_serial(fold + lane * nbp, nb, 0.0f);
            if constexpr (FUSED) {
                const float up = dpp_f32<0x101>(acc);  // row_shl:1, lane i reads lane i+1
                if (live && (lane & 1) == 0) out[r] = silu(acc, tab_lds) * up;
            } else {
                if (live) out[r] = acc;
            }
        }
        turn = turn + 1 < waves ? turn + 1 : 0;
    }
}

// Rows whose bytes do not end on a 16-byte boundary (Q6_K rows of nb % 8 != 0
// blocks) are finished by this direct kernel so that no staged chunk reaches
// past the matrix: one wavefront per row, blocks read straight from memory.
template <typename GW, typename UW, bool FUSED, bool PREQ>
__global__ __launch_bounds__(kGemvBlock) void kquant_gemv_direct(const uint8_t *__restrict__ gw,
                                                                  const uint8_t *__restrict__ uw,
                                                                  const void *__restrict__ x, float *__restrict__ out,
                                                                  uint32_t rows, uint32_t nb) {
    constexpr uint32_t kMats = FUSED ? 2 : 1;
    extern __shared__ __align__(16) uint8_t gemv_smem[];
    __shared__ uint64_t tab_lds[32];
    const XLds xl = carve_lds(gemv_smem, nb);
    const uint32_t wave = threadIdx.x / kWave, lane = threadIdx.x % kWave;
    const uint32_t h = lane & 1, slot = lane >> 1;
    const uint32_t nbp = (nb + 3) & ~3u;
    stage_expf_table(tab_lds);
    fill_x<PREQ>(x, nb, xl, gemv_smem);
    __syncthreads();
    float *fold = xl.fold + wave * kMats * nbp;
    for (uint32_t row = blockIdx.x * kGemvWaves + wave; row < rows; row += gridDim.x * kGemvWaves) {
        for (uint32_t b0 = 0; b0 < nb; b0 += 32) {
            const uint32_t b = b0 + slot, bb = b < nb ? b : nb - 1;
            XHalf xh;
            load_x(xl, bb, h, xh);
            const float vg = block_value<GW>(GW::read(gw + ((size_t)row * nb + bb) * GW::kBytes, h), h, xh);
            if (b < nb && h == (GW::kBytes == 210 ? 1u : 0u)) fold[b] = vg;
            if constexpr (FUSED) {
                const float vu = block_value<UW>(UW::read(uw + ((size_t)row * nb + bb) * UW::kBytes, h), h, xh);
                if (b < nb && h == (UW::kBytes == 210 ? 1u : 0u)) fold[nbp + b] = vu;
            }
        }
        wave_lds_sync();
        float acc = 0.0f;
        if (lane < kMats) acc = fold_serial(fold + lane * nbp, nb, 0.0f);
        if constexpr (FUSED) {
            const float up = dpp_f32<0x101>(acc);
            if (lane == 0) out[row] = silu(acc, tab_lds) * up;
        } else {
            if (lane == 0) out[row] = acc;
        }
        wave_lds_sync();
    }
}

// Standalone Q8_K quantization of x into a blob (one wavefront per block).
__global__ __launch_bounds__(kGemvBlock) void quantize_q8k_kernel(const float *__restrict__ x, uint32_t nb,
                                                                   uint8_t *__restrict__ blob) {
    const XLds xl = carve_lds(blob, nb);
    quantize_x(x, nb, xl, blockIdx.x * kGemvWaves + threadIdx.x / kWave, gridDim.x * kGemvWaves);
}

// Workgroups for `units` row groups of at most 32 blocks.  Each workgroup
// quantizes x once, so a launch keeps to FELLM_GEMV_MAX_GRID (512) unless
// its wavefronts would each get more than two units; then it widens to at
// most FELLM_GEMV_WIDE_GRID (768), and never past the workgroups that can be
// resident at once (the LDS stage sets that).  With x already quantized the
// prologue is a copy, so more workgroups pay off at every size.
template <bool PREQ, typename K>
uint32_t gemv_grid(K kernel, uint32_t lds, uint32_t units, uint32_t nw = kGemvWaves) {
    const uint32_t need = (units + nw - 1) / nw;
    // the caps count wavefronts in kGemvWaves-wavefront workgroups
    uint32_t grid = (PREQ ? kGemvMaxGridPre : FELLM_GEMV_MAX_GRID) * kGemvWaves / nw;
    if (!PREQ && units / (2 * nw) > grid) {
        // resident workgroups for this kernel and LDS size, looked up once each
        static std::mutex mu;
        static std::vector<std::tuple<const void *, uint32_t, uint32_t>> seen;
        uint32_t cap = 0;
        {
            std::lock_guard<std::mutex> lock(mu);
            for (const auto &[k, l, c] : seen)
                if (k == reinterpret_cast<const void *>(kernel) && l == lds) cap = c;
            if (cap == 0) {
                cap = resident_grid(kernel, (int)nw * kWave, lds, 8);
                seen.emplace_back(reinterpret_cast<const void *>(kernel), lds, cap);
            }
        }
        uint32_t wide = units / (2 * nw);
        if (wide > FELLM_GEMV_WIDE_GRID * kGemvWaves / nw) wide = FELLM_GEMV_WIDE_GRID * kGemvWaves / nw;
        if (wide > cap) wide = cap;
        if (wide > grid) grid = wide;
    }
    return need < grid ? need : grid;
}

template <typename GW, typename UW, bool FUSED, bool PREQ = false>
int launch_gemv(const void *gw, const void *uw, const void *x, float *out, uint32_t rows, uint32_t cols,
                hipStream_t s) {
    const uint32_t nb = cols / 256;
    const uint32_t mats = FUSED ? 2 : 1;
    const uint32_t nbp = (nb + 3) & ~3u;
    const uint8_t *g8 = static_cast<const uint8_t *>(gw), *u8 = static_cast<const uint8_t *>(uw);
    // Staged rows: every matrix's staged bytes end on a 16-byte boundary.
    uint32_t m = 1;
    while ((uint64_t)m * nb * GW::kBytes % 16 || (FUSED && (uint64_t)m * nb * UW::kBytes % 16)) ++m;
    const uint32_t rows_main = rows / m * m;
    // Buffer ranges are 32-bit: stage at most 2^31 - 1 bytes of a matrix per launch.
    const uint64_t rb = (uint64_t)nb * (GW::kBytes > UW::kBytes ? GW::kBytes : UW::kBytes);
    const uint32_t chunk = (uint32_t)(((1ull << 31) - 1) / rb) / m * m;
    for (uint32_t r0 = 0; r0 < rows_main; r0 += chunk) {
        const uint32_t n = rows_main - r0 < chunk ? rows_main - r0 : chunk;
        const uint8_t *g = g8 + (uint64_t)r0 * nb * GW::kBytes;
        const uint8_t *u = FUSED ? u8 + (uint64_t)r0 * nb * UW::kBytes : nullptr;
        if (nb <= 32) {
            const uint32_t rp = 32 / nb;
            constexpr int NWO = FELLM_GEMV_ONE_WAVES;
            const uint32_t lds = gemv_lds_bytes(nb, mats * rp * nbp, NWO) + NWO * kStagePerWave<GW, UW, FUSED>;
            const uint32_t units = (n + rp - 1) / rp;
            const uint32_t grid = gemv_grid<PREQ>(kquant_gemv_kernel<GW, UW, FUSED, PREQ, NWO>, lds, units, NWO);
            FELLM_LAUNCH((kquant_gemv_kernel<GW, UW, FUSED, PREQ, NWO>), dim3(grid), dim3(NWO * kWave), lds, s, g, u, x,
                               out + r0, n, nb, rp);
        } else {
            // As many groups as fit MAXW wavefronts and the LDS, and no more
            // than give every CU a workgroup (each quantizes x: 2048 x 9472
            // Q4_K 7.6 us in 256 workgroups, 9.6 in 512 half as wide); among
            // those of at least half as many, the one that leaves the fewest
            // group slots of the last step empty.  What one step of more than
            // half of the wavefronts would take goes in two steps of half as
            // many, the second's weights on their way during the first: 2048 x
            // 16384 Q4_K 10.1 -> 9.3 us, Q6_K 14.1 -> 12.3, from a blob 8.8 ->
            // 7.6 and 13.1 -> 11.0; 1024 x 28672 Q4_K 13.3 -> 12.4.
            constexpr int MAXW = FUSED ? 8 : 16;
            const uint32_t passes = (nb + 31) / 32;
            auto lds_of = [&](uint32_t g) { return gemv_pass_lds(nb, passes, g, mats, kStagePerWave<GW, UW, FUSED>); };
            uint32_t most = MAXW / passes;
            while (most > 1 && lds_of(most) > kGemvLdsLimit) --most;
            const uint32_t one_step = (n + (uint32_t)cu_count() - 1) / (uint32_t)cu_count();
            if (one_step < most) most = one_step;
            auto grid_of = [&](uint32_t g) {
                uint32_t per_cu = kGemvLdsLimit / lds_of(g);
                if (per_cu > (uint32_t)MAXW / (passes * g)) per_cu = MAXW / (passes * g);
                const uint32_t all = (uint32_t)cu_count() * (per_cu ? per_cu : 1), need = (n + g - 1) / g;
                return need < all ? need : all;
            };
            const bool two_steps = !FUSED && one_step <= most && passes * one_step > MAXW / 2;
            uint32_t groups = two_steps ? (one_step + 1) / 2 : most;
            uint64_t best = ~0ull;
            for (uint32_t g = most; !two_steps && 2 * g >= most && g > 0; --g) {
                const uint64_t per_step = (uint64_t)grid_of(g) * g, slots = (n + per_step - 1) / per_step * per_step;
                if (slots < best) best = slots, groups = g;
            }
            // A blob's copy wants fewer helpers: 700 x 25600 Q6_K 10.7 us with 8
            // wavefronts in all, 11.1 with 16; 256 x 16384 7.0 with 2, 5.7 with 16.
            const uint32_t waves = std::max(passes * groups, PREQ ? 8u : (uint32_t)MAXW);
            const uint32_t grid = two_steps ? (uint32_t)cu_count() : grid_of(groups);
            FELLM_LAUNCH((kquant_gemv_passes<GW, UW, FUSED, PREQ, MAXW>), dim3(grid), dim3(waves * kWave), lds_of(groups),
                         s, g, u, x, out + r0, n, nb, passes, groups);
        }
        const int rc = launch_status();
        if (rc != FELLM_OK) return rc;
    }
    if (rows_main < rows) {
        const uint32_t n = rows - rows_main;
        const uint8_t *g = g8 + (uint64_t)rows_main * nb * GW::kBytes;
        const uint8_t *u = FUSED ? u8 + (uint64_t)rows_main * nb * UW::kBytes : nullptr;
        FELLM_LAUNCH((kquant_gemv_direct<GW, UW, FUSED, PREQ>), dim3((n + kGemvWaves - 1) / kGemvWaves),
                           dim3(kGemvBlock), gemv_lds_bytes(nb, mats * nbp), s, g, u, x, out + rows_main, n, nb);
        const int rc = launch_status();
        if (rc != FELLM_OK) return rc;
    }
    return FELLM_OK;
}

bool kquant_ok(uint32_t dt) { return dt == FELLM_DTYPE_Q4K || dt == FELLM_DTYPE_Q5K || dt == FELLM_DTYPE_Q6K; }

// Q4_K and Q5_K blocks (144 and 176 bytes) are read with aligned 16-byte loads.
bool weight_aligned(const void *w, uint32_t dt) { return dt == FELLM_DTYPE_Q6K || aligned_to(w, 16); }

int check_gemv(const void *w, uint32_t dt, const void *x, const float *out, uint32_t cols) {
    if (!w || !x || !out) return FELLM_ERR_ARITY;
    if (!kquant_ok(dt)) return FELLM_ERR_DTYPE;
    if (cols == 0 || cols % 256 != 0 || cols > kGemvMaxCols) return FELLM_ERR_SHAPE;
    if (!aligned_to(x, 16) || !weight_aligned(w, dt)) return FELLM_ERR_SHAPE;
    return FELLM_OK;
}

}  // namespace
}  // namespace fellm

extern "C" int fellm_rocm_gate_up_swiglu(const void *gate_w, uint32_t gate_dtype, const void *up_w, uint32_t up_dtype,
                                         uint32_t rows, uint32_t cols, const float *x, float *out, void *stream) {
    using namespace fellm;
    if (rows == 0 && kquant_ok(gate_dtype) && kquant_ok(up_dtype) && cols % 256 == 0) return FELLM_OK;
    int rc = check_gemv(gate_w, gate_dtype, x, out, cols);
    if (rc == FELLM_OK) rc = check_gemv(up_w, up_dtype, x, out, cols);
    if (rc != FELLM_OK) return rc;
    hipStream_t s = as_stream(stream);
#define FELLM_GU(GT, GD, UT, UD) \
    if (gate_dtype == GD && up_dtype == UD) return launch_gemv<GT, UT, true>(gate_w, up_w, x, out, rows, cols, s);
#define FELLM_GU_ROW(GT, GD)                 \
    FELLM_GU(GT, GD, Q4K, FELLM_DTYPE_Q4K)   \
    FELLM_GU(GT, GD, Q5K, FELLM_DTYPE_Q5K)   \
    FELLM_GU(GT, GD, Q6K, FELLM_DTYPE_Q6K)
    FELLM_GU_ROW(Q4K, FELLM_DTYPE_Q4K)
    FELLM_GU_ROW(Q5K, FELLM_DTYPE_Q5K)
    FELLM_GU_ROW(Q6K, FELLM_DTYPE_Q6K)
#undef FELLM_GU_ROW
#undef FELLM_GU
    return FELLM_ERR_DTYPE;
}

extern "C" int fellm_rocm_matvec_kquant(const void *w, uint32_t w_dtype, uint32_t rows, uint32_t cols, const float *x,
                                        float *y, void *stream) {
    using namespace fellm;
    if (rows == 0 && kquant_ok(w_dtype) && cols % 256 == 0) return FELLM_OK;
    const int rc = check_gemv(w, w_dtype, x, y, cols);
    if (rc != FELLM_OK) return rc;
    hipStream_t s = as_stream(stream);
    if (w_dtype == FELLM_DTYPE_Q4K) return launch_gemv<Q4K, Q4K, false>(w, nullptr, x, y, rows, cols, s);
    if (w_dtype == FELLM_DTYPE_Q5K) return launch_gemv<Q5K, Q5K, false>(w, nullptr, x, y, rows, cols, s);
    return launch_gemv<Q6K, Q6K, false>(w, nullptr, x, y, rows, cols, s);
}

extern "C" uint64_t fellm_rocm_q8k_bytes(uint32_t cols) {
    using namespace fellm;
    return cols % 256 ? 0 : q8k_blob_bytes(cols / 256);
}

extern "C" int fellm_rocm_quantize_q8k(const float *x, uint32_t cols, void *xq, void *stream) {
    using namespace fellm;
    if (!x || !xq) return FELLM_ERR_ARITY;
    if (cols == 0 || cols % 256 != 0 || cols > kGemvMaxCols) return FELLM_ERR_SHAPE;
    if (!aligned_to(x, 16) || !aligned_to(xq, 16)) return FELLM_ERR_SHAPE;
    const uint32_t nb = cols / 256;
    FELLM_LAUNCH(quantize_q8k_kernel, dim3((nb + kGemvWaves - 1) / kGemvWaves), dim3(kGemvBlock), 0,
                       as_stream(stream), x, nb, static_cast<uint8_t *>(xq));
    return launch_status();
}

extern "C" int fellm_rocm_gate_up_swiglu_q8k(const void *gate_w, uint32_t gate_dtype, const void *up_w,
                                             uint32_t up_dtype, uint32_t rows, uint32_t cols, const void *xq,
                                             float *out, void *stream) {
    using namespace fellm;
    if (rows == 0 && kquant_ok(gate_dtype) && kquant_ok(up_dtype) && cols % 256 == 0) return FELLM_OK;
    int rc = check_gemv(gate_w, gate_dtype, xq, out, cols);
    if (rc == FELLM_OK) rc = check_gemv(up_w, up_dtype, xq, out, cols);
    if (rc != FELLM_OK) return rc;
    hipStream_t s = as_stream(stream);
#define FELLM_GU(GT, GD, UT, UD) \
    if (gate_dtype == GD && up_dtype == UD) return launch_gemv<GT, UT, true, true>(gate_w, up_w, xq, out, rows, cols, s);
#define FELLM_GU_ROW(GT, GD)                 \
    FELLM_GU(GT, GD, Q4K, FELLM_DTYPE_Q4K)   \
    FELLM_GU(GT, GD, Q5K, FELLM_DTYPE_Q5K)   \
    FELLM_GU(GT, GD, Q6K, FELLM_DTYPE_Q6K)
    FELLM_GU_ROW(Q4K, FELLM_DTYPE_Q4K)
    FELLM_GU_ROW(Q5K, FELLM_DTYPE_Q5K)
    FELLM_GU_ROW(Q6K, FELLM_DTYPE_Q6K)
#undef FELLM_GU_ROW
#undef FELLM_GU
    return FELLM_ERR_DTYPE;
}

extern "C" int fellm_rocm_matvec_kquant_q8k(const void *w, uint32_t w_dtype, uint32_t rows, uint32_t cols,
                                            const void *xq, float *y, void *stream) {
    using namespace fellm;
    if (rows == 0 && kquant_ok(w_dtype) && cols % 256 == 0) return FELLM_OK;
    const int rc = check_gemv(w, w_dtype, xq, y, cols);
    if (rc != FELLM_OK) return rc;
    hipStream_t s = as_stream(stream);
    if (w_dtype == FELLM_DTYPE_Q4K) return launch_gemv<Q4K, Q4K, false, true>(w, nullptr, xq, y, rows, cols, s);
    if (w_dtype == FELLM_DTYPE_Q5K) return launch_gemv<Q5K, Q5K, false, true>(w, nullptr, xq, y, rows, cols, s);
    return launch_gemv<Q6K, Q6K, false, true>(w, nullptr, xq, y, rows, cols, s);
}
