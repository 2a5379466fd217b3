// q4k.hip -- Q4_K weight x int8 activation GEMV for one decode token, and the
// activation quantiser it consumes (gfx950).
//
// Reference: src/kernel/q4k_gemv.cu.  Weights are ggml block_q4_K super-blocks
// (include/nova/quant/q4_k.h:19-25): 144 B per 256 weights -- fp16 d, fp16
// dmin, 12 B of packed 6-bit (scale, min) for 8 sub-blocks of 32, and 128 B of
// nibbles (bytes 32g..32g+31 hold sub-block 2g in the low nibbles and 2g+1 in
// the high nibbles).  Activations are ActQ8 (include/nova/kernel/types.h:24-28):
// int8 codes, an fp32 scale per 32 and the int sum of each 16 codes, so that
//   w . x = sum over sub-blocks of dx * (d*sc*sum(q*c) - dmin*m*sum(c)).
//
// gfx950 design (HBM-bound on the weights, 4.5 bits each):
//  * One token: a workgroup of 4 waves stages the whole activation (codes,
//    scales, sums) in LDS once and then walks rows (grid-stride), so the
//    activation is read from L2 once per workgroup, not per row.  A wave covers
//    16 super-blocks per step: lane (j, c) = (lane >> 2, lane & 3) takes the 32
//    nibble bytes at offset 32c of super-block 16s + j -- all 32 weights of
//    sub-block 2c (low nibbles) and of 2c+1 (high).  Rows of up to 4 steps
//    (cols <= 16384: the hidden widths 1536, 3584, 5120) are one wave's, with
//    the step loop unrolled at compile time and all of a row's loads issued
//    before any is consumed; wider rows (the FFN widths) are shared by the 4
//    waves of a workgroup, at most 4 steps each, reduced through LDS in a fixed
//    order.  Grids are sized to what is resident at once and grid-stride
//    beyond.  Products: v_dot4_i32_i8 on nibbles unpacked with a mask and a
//    shift; the per-sub-block float combination is the reference's; the row sum
//    is a wave reduction.  The large launches run at what HBM gives them:
//    37888 x 3584 with ActQ8 16.25 us, 152064 x 3584 57 us (5.4 TB/s); the same
//    products from registers alone, or with the weights through LDS rings filled
//    by direct loads (per workgroup or per wave), measured 16.0-16.5 and 55-57.
//  * Four tokens: int8 MFMA, see gemv4_kernel.
#include <hip/hip_runtime.h>
#include <cstdint>
#include <mutex>

#include "check.h"
#include "nova_kernel.h"

namespace nova {
namespace {

typedef uint32_t u4 __attribute__((ext_vector_type(4)));
typedef int32_t i4 __attribute__((ext_vector_type(4)));
typedef float f4 __attribute__((ext_vector_type(4)));

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

constexpr int kQK = 256;                       // weights per super-block
constexpr int kBlockBytes = 144;
constexpr int QT = 256;                        // threads per workgroup
constexpr int kMaxCols = 32768;                // the activation (and its scales, sums) fits LDS
// One-token lane geometry: 4 lanes per super-block, each with the 32 nibble
// bytes of one sub-block pair (64 weights: sub-block 2c in the low nibbles,
// 2c+1 in the high), 16 super-blocks per wave step.  (8 lanes of half that
// width: a 7B layer's projections 50.8 us against 48.7: more, smaller steps.)
constexpr int kLps = 4;
constexpr int kSbPerStep = 64 / kLps;
constexpr int kNibWords = 32 / kLps;           // nibble dwords per lane
struct Nib {
    uint32_t w[kNibWords];
};
// 16 B at any address (weights in a mapped file): one load all the same
using u4_any __attribute__((aligned(1))) = u4;

// ---------------------------------------------------------------- quant
// One 32-element block of quant_kernel, q4k_gemv.cu:9-33: d = amax / 127,
// codes rint(x * 127 / amax), the int sums of the two 16-code halves.  The
// GEMV's in-kernel staging: one thread per block (a workgroup has few, and
// spreading one over 8 lanes as quant_kernel does measured no faster there,
// the wide widths up to 5% slower).
__device__ __forceinline__ void quant_block(const float* __restrict__ xp, u4& lo, u4& hi, float& scale, int& s0,
                                            int& s1) {
    float v[32];
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 32; i += 4) {
        const float4 t = *reinterpret_cast<const float4*>(xp + i);
        v[i] = t.x; v[i + 1] = t.y; v[i + 2] = t.z; v[i + 3] = t.w;
    }
#pragma unroll
    for (int i = 0; i < 32; ++i) amax = fmaxf(amax, fabsf(v[i]));
    scale = amax * (1.f / 127.f);
    const float inv = amax > 0.f ? 127.f / amax : 0.f;
    s0 = 0;
    s1 = 0;
    uint32_t packed[8];
#pragma unroll
    for (int i = 0; i < 32; ++i) {
        const int q = (int)rintf(v[i] * inv);
        if (i < 16) s0 += q; else s1 += q;
        if ((i & 3) == 0) packed[i >> 2] = 0;
        packed[i >> 2] |= ((uint32_t)q & 0xFFu) << (8 * (i & 3));
    }
    lo = u4{packed[0], packed[1], packed[2], packed[3]};
    hi = u4{packed[4], packed[5], packed[6], packed[7]};
}

// Lane exchanges inside a row of 16 lanes (DPP: one VALU instruction, no LDS
// round trip): lanes xor 1, xor 2, and mirrored within each 8.
template <int kCtrl>
__device__ __forceinline__ int dpp_i(int v) {
    return __builtin_amdgcn_update_dpp(0, v, kCtrl, 0xF, 0xF, true);
}
template <int kCtrl>
__device__ __forceinline__ float dpp_f(float v) {
    return __builtin_bit_cast(float, dpp_i<kCtrl>(__builtin_bit_cast(int, v)));
}
constexpr int kXor1 = 0xB1, kXor2 = 0x4E, kHalfMirror = 0x141;

// quant_kernel: the same block over 8 lanes of 4 elements each (the arithmetic
// of quant_block per element; maxima and integer sums do not depend on the
// order, so the bits are the same).  Latency-bound: a decode token's activation
// is a few hundred blocks, which one thread per block left to 3 workgroups of
// long serial threads reading 128 B each; consecutive lanes now read
// consecutive 16 B.  18944 values 2.71 -> 1.78 us, 4 x 3584 2.60 -> 1.75 us (an
// empty launch: 1.6 us).
__global__ void __launch_bounds__(256) quant_kernel(int8_t* __restrict__ qs, float* __restrict__ d,
                                                    int32_t* __restrict__ sums, const float* __restrict__ x, int64_t n4) {
    const int64_t e = (int64_t)blockIdx.x * 256 + threadIdx.x;      // 4-element piece; rows are whole blocks
    const bool in = e < n4;                                         // the same for a block's 8 lanes
    const f4 v = *reinterpret_cast<const f4*>(x + 4 * (in ? e : 0));
    float amax = 0.f;
#pragma unroll
    for (int i = 0; i < 4; ++i) amax = fmaxf(amax, fabsf(v[i]));
    amax = fmaxf(amax, dpp_f<kXor1>(amax));
    amax = fmaxf(amax, dpp_f<kXor2>(amax));
    amax = fmaxf(amax, dpp_f<kHalfMirror>(amax));
    const float inv = amax > 0.f ? 127.f / amax : 0.f;
    uint32_t packed = 0;
    int sum = 0;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const int q = (int)rintf(v[i] * inv);
        sum += q;
        packed |= ((uint32_t)q & 0xFFu) << (8 * i);
    }
    sum += dpp_i<kXor1>(sum);                                       // over 16 codes: 4 lanes
    sum += dpp_i<kXor2>(sum);
    if (!in) return;
    *reinterpret_cast<uint32_t*>(qs + 4 * e) = packed;
    if ((e & 7) == 0) d[e >> 3] = amax * (1.f / 127.f);
    if ((e & 3) == 0) sums[e >> 2] = sum;
}

// ---------------------------------------------------------------- gemv
__device__ __forceinline__ float half_to_float(uint32_t h) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

// get_scale_min_k4, q4_k.h:44-52, for sub-block j of the 12 scale bytes
// held as three little-endian words
__device__ __forceinline__ void scale_min(int j, const uint32_t sw[3], uint32_t& sc, uint32_t& m) {
    const uint32_t b0 = sw[0] >> (8 * (j & 3)), b1 = sw[1] >> (8 * (j & 3)), b2 = sw[2] >> (8 * (j & 3));
    if (j < 4) {
        sc = b0 & 63;
        m = b1 & 63;
    } else {
        sc = (b2 & 0xF) | ((b0 >> 6 & 3) << 4);
        m = (b2 >> 4 & 0xF) | ((b1 >> 6 & 3) << 4);
    }
}

__device__ __forceinline__ Nib load_nib(const uint8_t* blk, int c) {
    Nib n;
    const uint8_t* p = blk + 16 + 4 * kNibWords * c;
#pragma unroll
    for (int h = 0; h < kNibWords / 4; ++h) {
        const u4 v = *reinterpret_cast<const u4_any*>(p + 16 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) n.w[4 * h + e] = v[e];
    }
    return n;
}

// Lane c's share of a super-block: its nibbles as int8 lanes of
// v_dot4_i32_i8 (sub-block 2c low, 2c+1 high) and the two (d*scale, dmin*min)
// pairs, unpacked ahead of the products with the activation staged in LDS
// (codes, scales per 32, sums per 16).  (As one function the loads of a row's
// later steps end up behind the earlier steps' arithmetic: a 5120-wide layer
// 3% slower.)  The float combination is the reference's:
// dx * (d*sc*sum(q*c) - dmin*m*sum(c)).
struct SbW {
    int lo[kNibWords], hi[kNibWords];
    float al, bl, ah, bh;
};

__device__ __forceinline__ SbW sb_prep(const u4 hd, const Nib& nb, int c) {
    SbW w;
#pragma unroll
    for (int e = 0; e < kNibWords; ++e) {
        w.lo[e] = (int)(nb.w[e] & 0x0F0F0F0Fu);
        w.hi[e] = (int)((nb.w[e] >> 4) & 0x0F0F0F0Fu);
    }
    const uint32_t sw[3] = {hd[1], hd[2], hd[3]};
    uint32_t scl, mcl, sch, mch;
    scale_min(2 * c, sw, scl, mcl);
    scale_min(2 * c + 1, sw, sch, mch);
    const float dd = half_to_float(hd[0] & 0xFFFFu);
    const float dm = half_to_float(hd[0] >> 16);
    w.al = dd * (float)scl;
    w.bl = dm * (float)mcl;
    w.ah = dd * (float)sch;
    w.bh = dm * (float)mch;
    return w;
}

// k0: the lane's first element (low nibbles) in the row; high nibbles at k0 + 32
__device__ __forceinline__ float sb_dot(const SbW& w, int k0, const int8_t* s_q, const float* s_d, const float* s_s) {
    int dlo = 0, dhi = 0;
#pragma unroll
    for (int h = 0; h < kNibWords / 4; ++h) {
        const i4 alo = *reinterpret_cast<const i4*>(s_q + k0 + 16 * h);
        const i4 ahi = *reinterpret_cast<const i4*>(s_q + k0 + 32 + 16 * h);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            dlo = __builtin_amdgcn_sdot4(w.lo[4 * h + e], alo[e], dlo, false);
            dhi = __builtin_amdgcn_sdot4(w.hi[4 * h + e], ahi[e], dhi, false);
        }
    }
    const float dxl = s_d[k0 >> 5], dxh = s_d[(k0 + 32) >> 5];
    float sml = s_s[k0 >> 4], smh = s_s[(k0 + 32) >> 4];
    sml += s_s[(k0 >> 4) + 1];
    smh += s_s[((k0 + 32) >> 4) + 1];
    return dxl * (w.al * (float)dlo - w.bl * sml) + dxh * (w.ah * (float)dhi - w.bh * smh);
}

__device__ __forceinline__ float sb_terms(const u4 hd, const Nib& nb, int sb, int c, int elo, const int8_t* s_q,
                                          const float* s_d, const float* s_s) {
    return sb_dot(sb_prep(hd, nb, c), sb * kQK + elo, s_q, s_d, s_s);
}

// Up to 4 matrices of the same width that read one activation (q/k/v,
// gate/up), walked as one row space: matrix m owns rows [end[m-1], end[m]).
constexpr int kMaxMats = 4;
struct GemvSet {
    const uint8_t* w[kMaxMats];
    float* out[kMaxMats];
    int64_t end[kMaxMats];
    int n;
    int cols;
    const int8_t* xq;          // pre-quantised activation (ActQ8) ...
    const float* xd;
    const int32_t* xs;
    const float* x;            // ... or fp32, quantised while it is staged
};

__device__ __forceinline__ int mat_of(const GemvSet& g, int64_t r) {
    int m = 0;
#pragma unroll
    for (int k = 0; k < kMaxMats - 1; ++k) m += (k + 1 < g.n && r >= g.end[k]) ? 1 : 0;
    return m;
}

// The activation (codes, scales per 32, sums per 16) into LDS, once per
// workgroup; from ActQ8 as given, or quantised here from fp32.  The sums are
// kept as floats (exact: |sum| <= 16 * 127), so no dot product converts them.
// Copies an ActQ8 activation of n columns (codes, per-32 scales, per-16
// sums, the sums converted to exact floats) into LDS; NT threads, n <= MAXC.
// The loads of a round all go out before its LDS stores: a strided copy loop
// waits out one load latency per element, which at the FFN width was 3 us of
// the down projection's 11.4.  Codes go in rounds of 8 x 16 B per thread, the
// sums and scales as 16 B loads with the first round.  No barrier.
template <int NT, int MAXC>
__device__ __forceinline__ void stage_q8(const int8_t* xq, const float* xd, const int32_t* xs, int n, int8_t* s_q,
                                         float* s_d, float* s_s) {
    constexpr int NQ = (MAXC / 16 + NT - 1) / NT < 8 ? (MAXC / 16 + NT - 1) / NT : 8;
    constexpr int NS = (MAXC / 64 + NT - 1) / NT;
    constexpr int ND = (MAXC / 128 + NT - 1) / NT;
    const int t = threadIdx.x;
    i4 vs[NS];
    f4 vd[ND];
#pragma unroll
    for (int k = 0; k < NS; ++k)
        if (t + k * NT < n / 64) vs[k] = *reinterpret_cast<const i4*>(xs + 4 * (t + k * NT));
#pragma unroll
    for (int k = 0; k < ND; ++k)
        if (t + k * NT < n / 128) vd[k] = *reinterpret_cast<const f4*>(xd + 4 * (t + k * NT));
#pragma unroll 1
    for (int b = t; b < n / 16; b += NQ * NT) {
        u4 vq[NQ];
#pragma unroll
        for (int k = 0; k < NQ; ++k)
            if (b + k * NT < n / 16) vq[k] = *reinterpret_cast<const u4*>(xq + 16 * (b + k * NT));
#pragma unroll
        for (int k = 0; k < NQ; ++k)
            if (b + k * NT < n / 16) *reinterpret_cast<u4*>(s_q + 16 * (b + k * NT)) = vq[k];
    }
#pragma unroll
    for (int k = 0; k < NS; ++k)
        if (t + k * NT < n / 64) {
            const i4 v = vs[k];
            *reinterpret_cast<f4*>(s_s + 4 * (t + k * NT)) = f4{(float)v[0], (float)v[1], (float)v[2], (float)v[3]};
        }
#pragma unroll
    for (int k = 0; k < ND; ++k)
        if (t + k * NT < n / 128) *reinterpret_cast<f4*>(s_d + 4 * (t + k * NT)) = vd[k];
}

template <bool kF32, int MAXC = kMaxCols>
__device__ __forceinline__ void stage_activation(const GemvSet& g, int8_t* s_q, float* s_d, float* s_s) {
    const int cols = g.cols;
    if constexpr (kF32) {
        for (int b = threadIdx.x; b < cols / 32; b += QT) {
            u4 lo, hi;
            float scale;
            int s0, s1;
            quant_block(g.x + 32 * b, lo, hi, scale, s0, s1);
            *reinterpret_cast<u4*>(s_q + 32 * b) = lo;
            *reinterpret_cast<u4*>(s_q + 32 * b + 16) = hi;
            s_d[b] = scale;
            s_s[2 * b] = (float)s0;
            s_s[2 * b + 1] = (float)s1;
        }
    } else {
        stage_q8<QT, MAXC>(g.xq, g.xd, g.xs, cols, s_q, s_d, s_s);
    }
    __syncthreads();
}

// Rows of at most 4 steps (16 super-blocks per step, cols <= 16384): the step
// loop is unrolled at compile time, one row per wave, all of the row's loads
// issued before any is consumed.  (Measured on gfx950: taking 2 or 4 rows per
// wave at once, or loading the next row while the current one is reduced,
// keeps more bytes in flight per wave but costs occupancy and is slower.)
template <int STEPS, bool kF32>
__global__ void __launch_bounds__(QT) gemv_fixed_kernel(GemvSet g) {
    extern __shared__ __attribute__((aligned(16))) unsigned char s_x[];
    const int cols = g.cols;
    int8_t* s_q = reinterpret_cast<int8_t*>(s_x);
    float* s_d = reinterpret_cast<float*>(s_x + cols);
    float* s_s = reinterpret_cast<float*>(s_x + cols + 4 * (cols / 32));   // 16-sums as exact floats
    stage_activation<kF32, STEPS * kSbPerStep * kQK>(g, s_q, s_d, s_s);

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform: scalar row addressing
    const int j = lane / kLps, c = lane % kLps;
    const int elo = 64 * c;
    const int nsb = cols / kQK;
    const int64_t row_bytes = (int64_t)nsb * kBlockBytes;
    const int64_t rows = kF32 ? g.end[g.n - 1] : g.end[0];   // one matrix on the ActQ8 path

    for (int64_t r = (int64_t)blockIdx.x * 4 + wave; r < rows; r += (int64_t)gridDim.x * 4) {
        const int m = kF32 ? mat_of(g, r) : 0;
        const int64_t lr = m ? r - g.end[m - 1] : r;
        const uint8_t* wr = g.w[m] + lr * row_bytes;
        u4 hdr[STEPS];
        Nib nib[STEPS];
#pragma unroll
        for (int t = 0; t < STEPS; ++t) {
            const int sb = kSbPerStep * t + j;
            if (sb < nsb) {
                const uint8_t* blk = wr + (int64_t)sb * kBlockBytes;
                hdr[t] = *reinterpret_cast<const u4_any*>(blk);
                nib[t] = load_nib(blk, c);
            }
        }
        float acc = 0.f;
#pragma unroll
        for (int t = 0; t < STEPS; ++t) {
            const int sb = kSbPerStep * t + j;
            if (sb < nsb) acc += sb_terms(hdr[t], nib[t], sb, c, elo, s_q, s_d, s_s);
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
        if (lane == 0) g.out[m][lr] = acc;
    }
}

// Rows wider than 4 steps (the FFN widths): KS waves share a row, each with
// at most STEPS steps whose loads all go out at once; the KS partial sums
// meet in LDS and are added in a fixed order.  4 / KS rows per workgroup
// iteration.
template <int STEPS, int KS, bool kF32>
__global__ void __launch_bounds__(QT) gemv_split_kernel(GemvSet g) {
    extern __shared__ __attribute__((aligned(16))) unsigned char s_x[];
    __shared__ float s_part[4];
    const int cols = g.cols;
    int8_t* s_q = reinterpret_cast<int8_t*>(s_x);
    float* s_d = reinterpret_cast<float*>(s_x + cols);
    float* s_s = reinterpret_cast<float*>(s_x + cols + 4 * (cols / 32));   // 16-sums as exact floats
    stage_activation<kF32, (STEPS * kSbPerStep * kQK * KS < kMaxCols ? STEPS * kSbPerStep * kQK * KS : kMaxCols)>(g, s_q, s_d, s_s);

    constexpr int RPI = 4 / KS;
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // wave-uniform: scalar row addressing
    const int part = wave % KS;
    const int j = lane / kLps, c = lane % kLps;
    const int elo = 64 * c;
    const int nsb = cols / kQK;
    const int sb0 = kSbPerStep * STEPS * part + j;
    const int64_t row_bytes = (int64_t)nsb * kBlockBytes;
    const int64_t rows = kF32 ? g.end[g.n - 1] : g.end[0];   // one matrix on the ActQ8 path
    const int64_t stride = (int64_t)gridDim.x * RPI;

    for (int64_t base = (int64_t)blockIdx.x * RPI; base < rows; base += stride) {   // uniform per workgroup
        const int64_t r = base + wave / KS;
        const int m = (kF32 && r < rows) ? mat_of(g, r) : 0;
        const int64_t lr = m ? r - g.end[m - 1] : r;
        float acc = 0.f;
        if (r < rows) {
            const uint8_t* wr = g.w[m] + lr * row_bytes;
            u4 hdr[STEPS];
            Nib nib[STEPS];
#pragma unroll
            for (int t = 0; t < STEPS; ++t) {
                const int sb = sb0 + kSbPerStep * t;
                if (sb < nsb) {
                    const uint8_t* blk = wr + (int64_t)sb * kBlockBytes;
                    hdr[t] = *reinterpret_cast<const u4_any*>(blk);
                    nib[t] = load_nib(blk, c);
                }
            }
#pragma unroll
            for (int t = 0; t < STEPS; ++t) {
                const int sb = sb0 + kSbPerStep * t;
                if (sb < nsb) acc += sb_terms(hdr[t], nib[t], sb, c, elo, s_q, s_d, s_s);
            }
        }
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
        if (lane == 0) s_part[wave] = acc;
        __syncthreads();
        if (part == 0 && lane == 0 && r < rows) {
            float sum = s_part[wave];
#pragma unroll
            for (int p = 1; p < KS; ++p) sum += s_part[wave + p];
            g.out[m][lr] = sum;
        }
        __syncthreads();
    }
}

// ---------------------------------------------------------------- direct loads
// Direct global -> LDS loads: the wave's 64 pieces of 16 B go to the 1 KiB at
// LDS byte address lds.  Inline asm, so that the compiler's vmcnt bookkeeping
// does not see them (it would drain them before every LDS read it cannot prove
// disjoint); gemv4_kernel waits for them.  m0 cannot be declared clobbered, so
// the statement saves and restores it.  An LDS load needs one wait state after a
// scalar write of m0, which neither the hardware nor, inside a statement, the
// compiler supplies.
__device__ __forceinline__ void stream_load(const void* base, uint32_t off, uint32_t lds) {
    // wave-uniform base: kept in scalar registers whatever the compiler made of
    // it.  A vector memory instruction needs five wait states after v_readfirstlane
    // wrote its base; a scalar copy waits for such a write by itself and may be
    // read at once, and it is m0's wait state too.
    const uint64_t b = (uint64_t)base;
    const uint64_t sb = ((uint64_t)(uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(b >> 32)) << 32) |
                        (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)b);
    uint32_t saved;
    uint64_t copy;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %4\n\ts_mov_b64 %1, %2\n\tglobal_load_lds_dwordx4 %3, %1\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved), "=&s"(copy)
        : "s"(sb), "v"(off), "s"(lds)
        : "memory");
}

// The same with an address per lane.
__device__ __forceinline__ void stream_load_at(const void* p, uint32_t lds) {
    uint32_t saved;
    asm volatile(
        "s_mov_b32 %0, m0\n\t"
        "s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %1, off\n\t"
        "s_mov_b32 m0, %0"
        : "=&s"(saved)
        : "v"(p), "s"(lds)
        : "memory");
}

__device__ __forceinline__ uint32_t lds_address(const unsigned char* p) {
    return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const unsigned char*)p;
}

// Four tokens at once (the reference's gemv4_kernel, q4k_gemv.cu:98-180, as
// Engine::decode_batch uses it for every projection, model.cpp:270-311), on the
// matrix cores: each weight is read once for the four activations.
//
// A unit is one super-block of 16 rows.  v_mfma_i32_16x16x64_i8 multiplies the
// activations' codes (A) by the rows' nibbles (B): lane (g,c) reads, for each
// half h of the super-block, row c's 16 nibble bytes at offset 16(g&1) of
// sub-block pair 2h + (g>>1); the low nibbles are the B operand of the first
// MFMA (sub-blocks 4h and 4h+2), the high nibbles that of the second (4h+1 and
// 4h+3).  A's row 4j + t is token t against sub-block 4h + j: lane (g, 4j+t)
// holds its 16 codes at 16(g&1) when j>>1 == g>>1 and zeros otherwise.  Rows
// whose sub-block is the other MFMA's hold garbage; lane (g,c) takes the C tile
// of MFMA g&1, whose rows 4g..4g+3 are the four tokens against sub-block 4h+g
// of row c.  One header read and one scale decode thus serve four values of
// the float combination dx * (d*sc*sum(q*c) - dmin*m*sum(c)); the tokens' scales
// and sums sit in one register each (lane t of a row of 16: the scale of token
// t, lane 4 + t: its sum) and reach the lanes as DPP row broadcasts.
//
// What bounds it: bytes in flight.  A unit's operands reach the wave through
// two unit buffers of LDS that belong to it alone (the next unit is on its way
// during this one's arithmetic): direct global -> LDS loads of 16 B pieces in
// address order.  Loaded into registers the MFMA's way, the 16 rows put every
// lane of a load on a line of its own: 370 cache accesses per unit (counted)
// against 90, and the cache's one access per clock set the pace (18944 x 3584:
// 13.1 us against 11.6).  The activations come the same way, per unit and from
// L2: staging all four first, as a dot4 kernel and an earlier form of this one
// did, delays every launch by a round trip and a barrier.  No barrier holds a
// wave to the others' pace.  Three or four buffers leave fewer waves per CU and
// are slower (18944 x 3584: 11.7, 13.2 us; 3584 x 18944: 12.7, 13.5 against
// 12.4); one ring per workgroup of 16 waves is faster on the largest (306 MB:
// 60 against 75 us) and slower elsewhere (3584 x 3584: 5.7 against 4.5 us).
// Measured against the dot4 kernel (below 32M weights) and the staged MFMA
// kernel (above) that it replaces, us per launch: 512 x 3584 5.6 -> 4.2,
// 3584 x 3584 6.5 -> 4.5, 18944 x 3584 14.4 -> 11.6, 3584 x 18944 16.5 -> 12.4,
// 1536 x 1536 4.4 -> 3.4, 5120 x 13824 19.3 -> 15.7, 152064 x 3584 85 -> 75.
// ks waves share a 16-row block's super-blocks; their sums meet in LDS and are
// added in a fixed order.
constexpr int kTok4 = 4;
constexpr int kMaxCols4 = 28672;
constexpr int kMaxKs4 = 16;                    // waves of a workgroup, at most
constexpr int kLdsMax = 160 * 1024;
// a unit in LDS: 144 weight pieces, 8 of scales ([token][8]), 16 of sums
// ([token][16]), 24 unused, 64 of codes ([token][256])
constexpr int kUnitLoads = 4, kUnitBytes = 4096, kUnitX = 144 * 16, kUnitA = 3072;

// lane N of each row of 16 lanes, to the whole row
template <int N>
__device__ __forceinline__ float row_lane(float v) {
    return dpp_f<0x150 + N>(v);
}

__global__ void __launch_bounds__(64 * kMaxKs4) gemv4_kernel(const uint8_t* __restrict__ w, int64_t rows, int cols,
                                                          const int8_t* __restrict__ xq,
                                                          const float* __restrict__ xd,
                                                          const int32_t* __restrict__ xs, float* __restrict__ out,
                                                          int share, int extra) {
    extern __shared__ __attribute__((aligned(16))) unsigned char s_x[];
    const int tid = threadIdx.x, lane = tid & 63, ks = blockDim.x >> 6;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int g = lane >> 4, c = lane & 15, t = c & 3, j = c >> 2;
    const int nsb = cols / kQK;
    const int sb_a = wave * nsb / ks, sb_b = (wave + 1) * nsb / ks;
    const uint32_t row_bytes = (uint32_t)nsb * kBlockBytes;
    // LDS: the waves' buffers | 16 zero bytes per wave | the waves' sums of two row blocks
    unsigned char* ring = s_x + wave * (2 * kUnitBytes);
    unsigned char* s_zero = s_x + ks * (2 * kUnitBytes) + 16 * wave;
    f4* s_part = reinterpret_cast<f4*>(s_x + ks * (2 * kUnitBytes + 16));
    const uint32_t lds0 = __builtin_amdgcn_readfirstlane(lds_address(ring));

    // this workgroup's 16-row blocks, one after the other
    const int bid = (int)blockIdx.x;
    const int my = share + (bid < extra ? 1 : 0);
    const int64_t rb0 = (int64_t)bid * share + (bid < extra ? bid : extra);
    // the next unit to fetch: row block at fw with fleft rows from it on, super-block fsb
    const uint8_t* fw = w + rb0 * 16 * row_bytes;
    int64_t fleft = rows - rb0 * 16;
    int fsb = sb_a;
    // pieces of the three weight loads: row and offset of the lane's piece; the
    // third's lanes past the weights take the scales and sums
    uint32_t voff[3];
    auto set_rows = [&](int nr) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const int e = lane + 64 * i < 144 ? lane + 64 * i : 143;
            const int r = e / 9;
            voff[i] = (uint32_t)(r < nr ? r : nr - 1) * row_bytes + 16u * (e - 9 * r);
        }
    };
    set_rows(fleft < 16 ? (int)fleft : 16);
    const int xe = lane - 16;                  // 0..7: scales, 8..23: sums (the rest as the last)
    const char* xbase = xe < 8 ? reinterpret_cast<const char*>(xd + (xe >> 1) * (cols / 32)) + 16 * (xe & 1)
                               : reinterpret_cast<const char*>(xs + (xe < 24 ? (xe - 8) >> 2 : 3) * (cols / 16)) +
                                     16 * (xe < 24 ? (xe - 8) & 3 : 3);
    const int xstep = xe < 8 ? 32 : 64;
    const uint32_t aoff = (lane >> 4) * cols + 16 * (lane & 15);
    auto fetch = [&](uint32_t buf) {
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");       // the buffer's last reads are done
        const uint8_t* base = fw + fsb * kBlockBytes;
        stream_load(base, voff[0], lds0 + buf);
        stream_load(base, voff[1], lds0 + buf + 1024);
        const char* p = lane < 16 ? reinterpret_cast<const char*>(base) + voff[2] : xbase + fsb * xstep;
        stream_load_at(p, lds0 + buf + 2048);
        stream_load(xq + fsb * kQK, aoff, lds0 + buf + kUnitA);
        if (++fsb == sb_b) {                   // on to the next row block
            fsb = sb_a;
            fw += 16 * row_bytes;
            fleft -= 16;
            if (fleft < 16 && fleft > 0) set_rows((int)fleft);
        }
    };
    const int n_units = my * (sb_b - sb_a);
    fetch(0);
    if (lane == 0) *reinterpret_cast<f4*>(s_zero) = f4{0.f, 0.f, 0.f, 0.f};

    int64_t left = rows - rb0 * 16;
    float* op = out + rb0 * 16;
    auto put = [&](int parity, float* o, int64_t n) {             // the sums of a row block of n rows (or more)
        const int r = tid & 15, tok = tid >> 4;
        if (tid >= 64 || r >= n) return;
        const float* p = reinterpret_cast<const float*>(s_part + parity * ks * 16 + r) + tok;
        float v = *p;
        for (int u = 1; u < ks; ++u) v += p[64 * u];
        o[tok * rows + r] = v;
    };
    const uint32_t woff = c * kBlockBytes;
    const uint32_t noff = woff + 16 + 32 * (g >> 1) + 16 * (g & 1);
    const bool live = (j >> 1) == (g >> 1);
    const uint32_t coff = kUnitA + t * kQK + 32 * j + 16 * (g & 1);
    const bool is_d = j == 0;
    const uint32_t xoff = kUnitX + (is_d ? t * 32 + 4 * g : 128 + t * 64 + 8 * g);
    const uint32_t xhalf = is_d ? 16 : 32;
    uint32_t buf = 0;                          // the unit being multiplied
    int to_come = n_units - 1;                 // units after it
    // tokens 0..3 of row c, sub-blocks 4h+g; one sum per h: half as many roundings in a row
    f4 acc2[2] = {{0.f, 0.f, 0.f, 0.f}, {0.f, 0.f, 0.f, 0.f}};
    for (int b = 0; b < my; ++b) {
        for (int sb = sb_a; sb < sb_b; ++sb) {
            if (to_come > 0) {
                fetch(kUnitBytes - buf);       // into the buffer of the unit before
                asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kUnitLoads) : "memory");
            } else {
                asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
            }
            --to_come;
            const unsigned char* u = ring + buf;
            const u4 hd = *reinterpret_cast<const u4*>(u + woff);
            const float dd = half_to_float(hd[0] & 0xFFFFu);
            const float dm = half_to_float(hd[0] >> 16);
            const uint32_t b0 = hd[1] >> (8 * g), b1 = hd[2] >> (8 * g), b2 = hd[3] >> (8 * g);
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const u4 raw = *reinterpret_cast<const u4*>(u + noff + 64 * h);
                const i4 a = *reinterpret_cast<const i4*>(live ? u + coff + 128 * h : s_zero);
                const int32_t* xp = reinterpret_cast<const int32_t*>(u + xoff + h * xhalf);
                const int32_t x0 = xp[0], x1 = xp[1];
                i4 lo, hi;
#pragma unroll
                for (int e = 0; e < 4; ++e) {
                    lo[e] = (int)(raw[e] & 0x0F0F0F0Fu);
                    hi[e] = (int)((raw[e] >> 4) & 0x0F0F0F0Fu);
                }
                const i4 c0 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, lo, i4{0, 0, 0, 0}, 0, 0, 0);
                const i4 c1 = __builtin_amdgcn_mfma_i32_16x16x64_i8(a, hi, i4{0, 0, 0, 0}, 0, 0, 0);
                // get_scale_min_k4 of sub-block 4h + g
                const uint32_t sc = h ? (b2 & 0xF) | ((b0 >> 6 & 3) << 4) : b0 & 63;
                const uint32_t mn = h ? (b2 >> 4 & 0xF) | ((b1 >> 6 & 3) << 4) : b1 & 63;
                const float al = dd * (float)sc, bl = dm * (float)mn;
                const float x = __builtin_bit_cast(float, x0), sm = (float)(x0 + x1);   // exact: |sum| <= 32 * 127
                const float v[4] = {row_lane<4>(sm), row_lane<5>(sm), row_lane<6>(sm), row_lane<7>(sm)};
                const float dx[4] = {row_lane<0>(x), row_lane<1>(x), row_lane<2>(x), row_lane<3>(x)};
#pragma unroll
                for (int i = 0; i < 4; ++i)
                    acc2[h][i] += dx[i] * (al * (float)(g & 1 ? c1[i] : c0[i]) - bl * v[i]);
            }
            buf = kUnitBytes - buf;
        }
        // over the four groups of lanes, then with the other waves' after the barrier
        f4 acc = acc2[0] + acc2[1];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(acc[i]), __float_as_uint(acc[i]), false, false);
            acc[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
            const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(acc[i]), __float_as_uint(acc[i]), false, false);
            acc[i] = __uint_as_float(q[0]) + __uint_as_float(q[1]);
        }
        if (g == 0) s_part[((b & 1) * ks + wave) * 16 + c] = acc;
        acc2[0] = acc2[1] = f4{0.f, 0.f, 0.f, 0.f};
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        put(b & 1, op, left);                  // the next write here comes after the next barrier
        left -= 16;
        op += 16;
    }
}

// ---------------------------------------------------------------- four tokens, weights anywhere
// Weights that do not start on 16 B (a file mapped at an odd offset) cannot take
// the direct loads.  Here they are read into registers, once for the four
// tokens, with the one-token kernels' lanes, steps and order of sums: the bits
// are those of launch_gemv_q4k for each token.
//
// Bound by LDS reads of the activations, one row against four of them.  The
// codes therefore lie in four planes per token, chunk q of every quarter
// super-block in plane q: a read's 64 lanes take 1 KiB without bank conflicts,
// where the one-token layout's 64 B between lanes cost this kernel half its time
// (18944 x 3584: 22.5 us, in planes 13.5); the scale and the sum of a 32 sit
// side by side, one read for both sub-blocks.  A row's first loads go out before
// the activations are staged.  The four sums of a row share their cross-lane
// steps (wave_sums4).  Workgroups of 512 threads; with 1024, a CU holds fewer of
// a narrow launch's waves (5120 x 5120: 11.3 us against 9.5).
// us per launch, weights at + 4 B / + 1 B, against four one-token launches:
// 512 x 3584 3.8 / 4.2 (12.2 / 12.9), 3584 x 3584 6.0 / 6.5 (16.9 / 19.2),
// 18944 x 3584 13.5 / 15.9 (34.9 / 42.5), 3584 x 18944 16.9 / 18.0 (39.0 / 43.8),
// 5120 x 13824 19.6 / 22.5 (41.0 / 48.7), 152064 x 3584 82 / 97 (226 / 338).  The
// direct loads, on 16 B: 3.7, 4.5, 11.6, 12.4, 15.7, 75.

// One token's products of a lane's share: chunk q of four (16 codes: sub-block 2c
// q = 0, 1; sub-block 2c + 1 q = 2, 3) at sq + q * plane, scale and sum of both
// sub-blocks in ds.  The combination is sb_dot's.
__device__ __forceinline__ float sb_dot_planes(const SbW& w, const int8_t* sq, int plane, const f4 ds) {
    int dlo = 0, dhi = 0;
#pragma unroll
    for (int h = 0; h < 2; ++h) {
        const i4 alo = *reinterpret_cast<const i4*>(sq + h * plane);
        const i4 ahi = *reinterpret_cast<const i4*>(sq + (2 + h) * plane);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            dlo = __builtin_amdgcn_sdot4(alo[e], w.lo[4 * h + e], dlo, false);
            dhi = __builtin_amdgcn_sdot4(ahi[e], w.hi[4 * h + e], dhi, false);
        }
    }
    return ds[0] * (w.al * (float)dlo - w.bl * ds[1]) + ds[2] * (w.ah * (float)dhi - w.bh * ds[3]);
}

// Four ActQ8 activations into LDS: codes as four planes per token (chunk q of
// every quarter super-block), scale and sum of each 32 side by side.  No barrier.
template <int NT>
__device__ __forceinline__ void stage_planes4(const int8_t* xq, const float* xd, const int32_t* xs, int cols, int8_t* s_q,
                                              float2* s_ds) {
    const int per = cols / 16, n = kTok4 * per, nd = kTok4 * (cols / 32);
    constexpr int NQ = 4;
    for (int b = threadIdx.x; b < n; b += NQ * NT) {
        u4 v[NQ];
        float d[NQ];
        int2 sm[NQ];
        const int bd = b - (int)threadIdx.x;
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
            if (b + k * NT < n) v[k] = *reinterpret_cast<const u4*>(xq + 16 * (b + k * NT));
            if (k < NQ / 2) {
                const int e = bd / 2 + (int)threadIdx.x + k * NT;
                if (e < nd) {
                    d[k] = xd[e];
                    sm[k] = *reinterpret_cast<const int2*>(xs + 2 * e);
                }
            }
        }
#pragma unroll
        for (int k = 0; k < NQ; ++k) {
            const int u = b + k * NT, t = u / per, i = u - t * per;
            if (u < n) *reinterpret_cast<u4*>(s_q + t * cols + (i & 3) * (cols / 4) + (i >> 2) * 16) = v[k];
            if (k < NQ / 2) {
                const int e = bd / 2 + (int)threadIdx.x + k * NT;
                if (e < nd) s_ds[e] = float2{d[k], (float)(sm[k].x + sm[k].y)};
            }
        }
    }
}

// Sums of four values over the 64 lanes, in __shfl_xor's order 32, 16, 8, 4, 2, 1;
// lane 16t gets the sum of a[t'], t' = (t >> 1) | (t & 1) << 1.
__device__ __forceinline__ float wave_sums4(const float* a) {
    float h[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {             // lanes < 32: a[2i], others: a[2i + 1]
        const auto p = __builtin_amdgcn_permlane32_swap(__float_as_uint(a[2 * i]), __float_as_uint(a[2 * i + 1]), false, false);
        h[i] = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    }
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(h[0]), __float_as_uint(h[1]), false, false);
    float v = __uint_as_float(p[0]) + __uint_as_float(p[1]);
    v += dpp_f<0x128>(v);                      // row_ror:8: lane ^ 8
    v += dpp_f<0x104>(v);                      // row_shl:4: lanes 0..3 of a row
    v += dpp_f<kXor2>(v);
    return v + dpp_f<kXor1>(v);
}

// STEPS and KS as in gemv_fixed_kernel (KS == 1) and gemv_split_kernel, whose
// fourth wave per row has nothing below 97 super-blocks: KS == 3 there.  Aligned
// weights of few rows, whose order of sums is free, also with STEPS == 1, KS > 1.
template <int STEPS, int KS, int NT>
__global__ void __launch_bounds__(NT) gemv4_rows_kernel(const uint8_t* __restrict__ w, int64_t rows, int cols,
                                                        const int8_t* __restrict__ xq, const float* __restrict__ xd,
                                                        const int32_t* __restrict__ xs, float* __restrict__ out) {
    static_assert(NT % (64 * KS) == 0, "whole rows per workgroup");
    constexpr int RPI = NT / 64 / KS;          // rows per workgroup iteration
    // the next row's loads behind this row's unpacking; with more steps the
    // registers cost more waves than that hides (1536 x 8960: 7.9 us, 7.6 without)
    constexpr bool kAhead = STEPS == 1 || KS > 1;
    extern __shared__ __attribute__((aligned(16))) unsigned char s_x[];
    __shared__ float s_part[2][KS > 1 ? NT / 64 : 1][kTok4];
    int8_t* s_q = reinterpret_cast<int8_t*>(s_x);                        // [4 tokens][4 planes][cols/4]
    float2* s_ds = reinterpret_cast<float2*>(s_x + kTok4 * cols);        // [4][cols/32]

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int part = wave % KS;
    const int j = lane / kLps, c = lane % kLps;
    const int nsb = cols / kQK;
    const int sb0 = kSbPerStep * STEPS * part + j;
    const int64_t row_bytes = (int64_t)nsb * kBlockBytes;
    const int64_t stride = (int64_t)gridDim.x * RPI;

    u4 hdr[STEPS];
    Nib nib[STEPS];
    auto load = [&](int64_t r, int t) {        // a wave past the end: the last row, unused
        const int sb = sb0 + kSbPerStep * t;
        if (sb >= nsb) return;
        const uint8_t* blk = w + (r < rows ? r : rows - 1) * row_bytes + (int64_t)sb * kBlockBytes;
        hdr[t] = *reinterpret_cast<const u4_any*>(blk);
        nib[t] = load_nib(blk, c);
    };
    int64_t r = (int64_t)blockIdx.x * RPI + wave / KS;
#pragma unroll
    for (int t = 0; t < STEPS; ++t) load(r, t);
    stage_planes4<NT>(xq, xd, xs, cols, s_q, s_ds);
    __syncthreads();
    int parity = 0;
    // the same number of rounds for every wave of the workgroup
    for (int64_t base = (int64_t)blockIdx.x * RPI; base < rows; base += stride, r += stride) {
        float acc[kTok4] = {0.f, 0.f, 0.f, 0.f};
        const bool more = base + stride < rows;
#pragma unroll
        for (int t = 0; t < STEPS; ++t) {
            const int sb = sb0 + kSbPerStep * t;
            const SbW wv = sb_prep(hdr[t], nib[t], c);
            if (kAhead && more) load(r + stride, t);
            if (sb < nsb)
#pragma unroll
                for (int k = 0; k < kTok4; ++k)
                    acc[k] += sb_dot_planes(wv, s_q + k * cols + 16 * (4 * sb + c), cols / 4,
                                            *reinterpret_cast<const f4*>(s_ds + k * (cols / 32) + 8 * sb + 2 * c));
        }
        if (!kAhead && more)
#pragma unroll
            for (int t = 0; t < STEPS; ++t) load(r + stride, t);
        const float v = wave_sums4(acc);
        const int tok = (lane >> 5) | (lane >> 4 & 1) << 1;
        if constexpr (KS == 1) {
            if ((lane & 15) == 0 && r < rows) out[tok * rows + r] = v;
        } else {
            if ((lane & 15) == 0) s_part[parity][wave][tok] = v;
            __syncthreads();
            if (part == 0 && lane < kTok4 && r < rows) {
                float sum = s_part[parity][wave][lane];
#pragma unroll
                for (int p = 1; p < KS; ++p) sum += s_part[parity][wave + p][lane];
                out[lane * rows + r] = sum;
            }
            parity ^= 1;                       // the next write here comes after the next barrier
        }
    }
}

// Workgroups: one per rows_per_wg rows, but no more than can be resident at
// once (this kernel's occupancy at this LDS size times the CUs); beyond that
// the kernels grid-stride, so no second partial round of workgroups forms a
// tail (measured: gate projection 9.8 -> 9.0 us against a fixed cap of 8
// workgroups per CU, of which 7 fit).
template <typename K>
int gemv_grid(K kernel, int64_t rows, int rows_per_wg, size_t lds, int block = QT) {
    int dev = 0, cus = 0, per_cu = 0;
    NOVA_HIP(hipGetDevice(&dev));
    NOVA_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    NOVA_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, block, lds));
    if (per_cu < 1) per_cu = 1;
    const int64_t want = (rows + rows_per_wg - 1) / rows_per_wg;
    const int64_t cap = (int64_t)per_cu * cus;
    return (int)(want < cap ? want : cap);
}


template <int STEPS, bool kF32>
void launch_fixed(const GemvSet& g, size_t lds, hipStream_t s) {
    auto k = gemv_fixed_kernel<STEPS, kF32>;
    hipLaunchKernelGGL(k, dim3((unsigned)gemv_grid(k, g.end[g.n - 1], 4, lds)), dim3(QT), lds, s, g);
}

template <int STEPS, bool kF32>
void launch_split(const GemvSet& g, size_t lds, hipStream_t s) {
    auto k = gemv_split_kernel<STEPS, 4, kF32>;
    hipLaunchKernelGGL(k, dim3((unsigned)gemv_grid(k, g.end[g.n - 1], 1, lds)), dim3(QT), lds, s, g);
}

int device_cus() {
    int dev = 0, cus = 0;
    NOVA_HIP(hipGetDevice(&dev));
    NOVA_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    return cus;
}

// Waves per 16-row block: the fewest rounds of resident workgroups (LDS bounds
// them) times the units that each of their waves takes, and among equals the
// fewest waves: more of them only split the sums further.  Within 4% of the best
// of 1..16 on the shapes above.
void launch_gemv4(const uint8_t* blocks, int64_t rows, int cols, const int8_t* xq, const float* xd, const int32_t* xs,
                  float* out, hipStream_t s) {
    static std::once_flag once;                // dynamic LDS beyond 64 KB must be allowed per kernel
    std::call_once(once, [&] {
        NOVA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(gemv4_kernel), hipFuncAttributeMaxDynamicSharedMemorySize, kLdsMax));
    });
    const int cus = device_cus();
    auto lds_of = [](int k) { return (size_t)k * (2 * kUnitBytes + 16 + 2 * 16 * 16); };
    const int64_t n_rb = (rows + 15) / 16;
    const int nsb = cols / kQK;
    int ks = 1;
    int64_t best = INT64_MAX;
    for (int k = 1; k <= kMaxKs4 && k <= nsb && lds_of(k) <= (size_t)kLdsMax; ++k) {
        const int64_t cap = (int64_t)cus * (kLdsMax / lds_of(k));
        const int64_t cost = (n_rb + cap - 1) / cap * ((nsb + k - 1) / k);
        if (cost < best) {
            best = cost;
            ks = k;
        }
    }
    const int64_t cap = (int64_t)cus * (kLdsMax / lds_of(ks));
    NOVA_REQUIRE(n_rb < (int64_t)1 << 31);
    const int grid = (int)(n_rb < cap ? n_rb : cap);
    hipLaunchKernelGGL(gemv4_kernel, dim3(grid), dim3(64 * ks), lds_of(ks), s, blocks, rows, cols, xq, xd, xs, out,
                       (int)(n_rb / grid), (int)(n_rb % grid));
}

template <int STEPS, int KS, int NT>
void launch_rows4(const uint8_t* blocks, int64_t rows, int cols, const int8_t* xq, const float* xd, const int32_t* xs,
                  float* out, hipStream_t s) {
    auto k = gemv4_rows_kernel<STEPS, KS, NT>;
    static std::once_flag once;                // dynamic LDS beyond 64 KB must be allowed per kernel
    std::call_once(once, [&] {
        NOVA_HIP(hipFuncSetAttribute(reinterpret_cast<const void*>(k), hipFuncAttributeMaxDynamicSharedMemorySize,
                                     kTok4 * kMaxCols4 * 5 / 4));
    });
    const size_t lds = kTok4 * ((size_t)cols + 8 * (size_t)(cols / 32));
    hipLaunchKernelGGL(k, dim3((unsigned)gemv_grid(k, rows, NT / 64 / KS, lds, NT)), dim3(NT), lds, s, blocks, rows, cols,
                       xq, xd, xs, out);
}

// rows of more than 64 super-blocks.  12 waves: one workgroup fits a CU's LDS
// (3584 x 18944: 9 waves 17.3 us, 12 16.9, 15 16.8; 9000 x 18944: 34.0, 31.4, 34.5)
void launch_rows4_wide(const uint8_t* blocks, int64_t rows, int cols, const int8_t* xq, const float* xd,
                       const int32_t* xs, float* out, hipStream_t s) {
    if (cols / kQK <= 6 * kSbPerStep) launch_rows4<2, 3, 768>(blocks, rows, cols, xq, xd, xs, out, s);
    else launch_rows4<2, 4, 768>(blocks, rows, cols, xq, xd, xs, out, s);
}

template <bool kF32>
void launch_set(const GemvSet& g, hipStream_t st) {
    const int cols = g.cols;
    const size_t lds = (size_t)cols + 4 * (size_t)(cols / 32) + 4 * (size_t)(cols / 16);
    switch ((cols / kQK + kSbPerStep - 1) / kSbPerStep) {
        case 1: launch_fixed<1, kF32>(g, lds, st); break;
        case 2: launch_fixed<2, kF32>(g, lds, st); break;
        case 3: launch_fixed<3, kF32>(g, lds, st); break;
        case 4: launch_fixed<4, kF32>(g, lds, st); break;
        // wider rows: 4 waves per row, at most 4 steps each (measured: down
        // projection 3584 x 18944, 12.7 -> 11.7 us against one wave per row)
        case 5: case 6: case 7: case 8: launch_split<2, kF32>(g, lds, st); break;
        case 9: case 10: case 11: case 12: launch_split<3, kF32>(g, lds, st); break;
        default: launch_split<4, kF32>(g, lds, st); break;
    }
    NOVA_LAUNCHED();
}

}  // namespace
}  // namespace nova

using namespace nova;

extern "C" {

void launch_quant_q8(int8_t* qs, float* d, int32_t* sums, const float* x, int rows, int cols, nova_stream_t s) {
    NOVA_REQUIRE(qs && d && sums && x && rows >= 0 && cols > 0 && cols % 32 == 0);
    const int64_t n4 = (int64_t)rows * (cols / 4);
    if (n4 == 0) return;
    // one launch takes fewer than 2^32 threads; whole blocks (8 pieces) per launch
    constexpr int64_t kMost = (int64_t)1 << 31;
    for (int64_t at = 0; at < n4; at += kMost) {
        const int64_t n = n4 - at < kMost ? n4 - at : kMost;
        hipLaunchKernelGGL(quant_kernel, dim3((unsigned)((n + 255) / 256)), dim3(256), 0,
                           reinterpret_cast<hipStream_t>(s), qs + 4 * at, d + at / 8, sums + at / 4, x + 4 * at, n);
        NOVA_LAUNCHED();
    }
}

void launch_gemv_q4k(const uint8_t* blocks, int64_t rows, int cols, const int8_t* xq, const float* xd,
                     const int32_t* xs, float* out, nova_stream_t s) {
    NOVA_REQUIRE(blocks && xq && xd && xs && out && rows >= 0);
    NOVA_REQUIRE(cols > 0 && cols % kQK == 0 && cols <= kMaxCols);
    NOVA_REQUIRE(aligned16(xq) && aligned16(xd) && aligned16(xs));   // staged with 16 B loads
    if (rows == 0) return;
    GemvSet g{};
    g.w[0] = blocks;
    g.out[0] = out;
    g.end[0] = rows;
    g.n = 1;
    g.cols = cols;
    g.xq = xq;
    g.xd = xd;
    g.xs = xs;
    launch_set<false>(g, reinterpret_cast<hipStream_t>(s));
}

void launch_gemv4_q4k(const uint8_t* blocks, int64_t rows, int cols, const int8_t* xq, const float* xd,
                      const int32_t* xs, float* out, nova_stream_t s) {
    NOVA_REQUIRE(blocks && xq && xd && xs && out && rows >= 0);
    NOVA_REQUIRE(cols > 0 && cols % kQK == 0 && cols <= kMaxCols4);
    NOVA_REQUIRE(aligned16(xq) && aligned16(xd) && aligned16(xs));   // staged with 16 B loads
    if (rows == 0) return;
    const hipStream_t st = reinterpret_cast<hipStream_t>(s);
    const int steps = (cols / kQK + kSbPerStep - 1) / kSbPerStep;
    if (!aligned16(blocks)) {
        // the direct loads to LDS move aligned 16 B; loads to registers take any address
        switch (steps) {                       // launch_set's shapes, for its order of sums
            case 1: launch_rows4<1, 1, 512>(blocks, rows, cols, xq, xd, xs, out, st); break;
            case 2: launch_rows4<2, 1, 512>(blocks, rows, cols, xq, xd, xs, out, st); break;
            case 3: launch_rows4<3, 1, 512>(blocks, rows, cols, xq, xd, xs, out, st); break;
            case 4: launch_rows4<4, 1, 512>(blocks, rows, cols, xq, xd, xs, out, st); break;
            default: launch_rows4_wide(blocks, rows, cols, xq, xd, xs, out, st); break;
        }
    } else if (steps > 2 && (rows + 15) / 16 <= device_cus() / 4) {
        // Few rows, and long ones: the 16-row blocks would leave three CUs of four
        // idle while their 16 waves take more than two units each, one after the
        // other.  By rows, every wave or three or four of them on a row of its own:
        // 1024 x 20480 8.8 us (16-row blocks 11.6), 512 x 18944 7.5 (10.6), 1024 x
        // 14336 6.5 (9.1), 512 x 10240 4.6 (5.9), 130 x 18944 6.4 (8.0).  Past that
        // line the blocks win: 1536 x 8960 6.8 us, by rows 7.3.
        switch (steps) {
            case 3: launch_rows4<1, 3, 768>(blocks, rows, cols, xq, xd, xs, out, st); break;
            case 4: launch_rows4<1, 4, 1024>(blocks, rows, cols, xq, xd, xs, out, st); break;
            default: launch_rows4_wide(blocks, rows, cols, xq, xd, xs, out, st); break;
        }
    } else {
        launch_gemv4(blocks, rows, cols, xq, xd, xs, out, st);
    }
    NOVA_LAUNCHED();
}

void launch_gemv_q4k_f32(const uint8_t* const* blocks, const int64_t* rows, float* const* outs, int n_mat,
                         int cols, const float* x, nova_stream_t s) {
    NOVA_REQUIRE(blocks && rows && outs && x && n_mat >= 1 && n_mat <= kMaxMats);
    NOVA_REQUIRE(cols > 0 && cols % kQK == 0 && cols <= kMaxCols);
    GemvSet g{};
    int64_t total = 0;
    for (int m = 0; m < n_mat; ++m) {
        NOVA_REQUIRE(blocks[m] && outs[m] && rows[m] >= 0);
        total += rows[m];
        g.w[m] = blocks[m];
        g.out[m] = outs[m];
        g.end[m] = total;
    }
    if (total == 0) return;
    g.n = n_mat;
    g.cols = cols;
    g.x = x;
    launch_set<true>(g, reinterpret_cast<hipStream_t>(s));
}

}  // extern "C"
