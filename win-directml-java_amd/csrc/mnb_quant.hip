// mnb_quant.hip -- int4 quantization of a dense matrix on the device, and the
// read-back of a resident weight into the reference's arrays.
//
// The quantizer restates Qwen2Weights.quantizeDenseRowsToUInt4 with
// calculateUInt4QuantizationBlock and quantizeDenseBlockToUInt4
// (directml-inference/src/main/java/com/aresstack/windirectml/inference/qwen/
// Qwen2Weights.java:1352-1422): per block of bs values of a row,
//   max == min: |max| < 1e-8 -> scale 1, zp 0; max > 0 -> scale max/15, zp 0;
//               otherwise scale -min/15, zp 15
//   else:       scale = (max - min)/15, zp = clamp(round(-min/scale), 0, 15)
//   q = clamp(round(v/scale + zp), 0, 15)
// with fp32 IEEE division and addition and Java's Math.round (floor(v + 1/2),
// NaN -> 0, saturating), so the bytes equal the reference's.  It writes the
// tiled HBM layout directly, one wave per 16-row x 128-k tile.
#include <algorithm>

#include "mnb_device.h"

namespace mnb {

constexpr int kQuantThreads = 256;

__device__ __forceinline__ int java_round_f(float a) {
    if (a != a) return 0;
    if (a >= 2147483647.0f) return 2147483647;
    if (a <= -2147483648.0f) return -2147483647 - 1;
    const float fl = floorf(a);
    const float diff = a - fl;  // exact
    return (int)fl + (diff >= 0.5f ? 1 : 0);
}

__device__ __forceinline__ int clamp_u4(int v) { return v < 0 ? 0 : (v > 15 ? 15 : v); }

// The EPL values of one 16-byte load, widened (exact).
template <typename InT>
__device__ __forceinline__ void widen(const u32x4_t &r, float *v) {
    InT e[16 / sizeof(InT)];
    __builtin_memcpy(e, &r, 16);
#pragma unroll
    for (int i = 0; i < 16 / (int)sizeof(InT); ++i) v[i] = (float)e[i];
}

// bit position of value i (k order) in a tiled dword
__device__ __forceinline__ constexpr int nib_pos(int i) { return (i & 1) ? 16 + 4 * (i >> 1) : 4 * (i >> 1); }

// clamp(round(v / scale + zf), 0, 15) of EPL (4 or 8) consecutive values with
// the reference's fp32 division, addition and rounding, at the positions of
// the first EPL values of a tiled dword.  An IEEE division is ten
// instructions, so the value is first estimated as u = v * (1 / scale) + zf +
// 1/2 with one fma.  Where |v / scale| < 32 (the values a quotient between -1
// and 16 can come from) u is within 2^-17 of the reference's rounded sum plus
// 1/2: 2^-19 from the reciprocal's rounding, 2^-20 each from its own rounding
// and from the reference's quotient and sum.  Beyond that both sides clamp to
// the same end.  So floor(u) decides the nibble wherever u's fraction stays
// kTieMargin away from 0 and 1; the division runs for the lane's values
// otherwise (one value in 2^15; also for NaN, and all of a block whose scale
// has no safe reciprocal, rcp = NaN).
constexpr float kTieMargin = 0x1p-16f;
template <int EPL>
__device__ __forceinline__ uint32_t quantize_piece(const float *v, float scale, float rcp, float zf) {
    const float zh = zf + 0.5f;   // exact
    uint32_t d = 0;
    bool ok = true;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        const float u = fmaf(v[i], rcp, zh);
        const float fl = floorf(u);
        ok = ok && fabsf((u - fl) - 0.5f) <= 0.5f - kTieMargin;   // false for NaN
        const uint32_t nib = (uint32_t)__builtin_amdgcn_fmed3f(fl, 0.0f, 15.0f);
        d |= nib << nib_pos(i);
    }
    if (ok) return d;
    d = 0;
#pragma unroll
    for (int i = 0; i < EPL; ++i) {
        const float tq = v[i] / scale + zf;
        const uint32_t nib = (uint32_t)clamp_u4(java_round_f(tq));
        d |= nib << nib_pos(i);
    }
    return d;
}

// A value of another lane of the group of eight: lane ^ 1, lane ^ 2, or the
// mirrored lane 7 - p (a lane of the other half).
constexpr int kDppXor1 = 0xB1, kDppXor2 = 0x4E, kDppMirror8 = 0x141;
template <int CTRL>
__device__ __forceinline__ uint32_t lane_dpp(uint32_t v) {
    return (uint32_t)__builtin_amdgcn_mov_dpp((int)v, CTRL, 0xF, 0xF, true);
}
template <int CTRL>
__device__ __forceinline__ void min_max_step(float &mn, float &mx) {
    const float o_mn = __builtin_bit_cast(float, lane_dpp<CTRL>(__builtin_bit_cast(uint32_t, mn)));
    const float o_mx = __builtin_bit_cast(float, lane_dpp<CTRL>(__builtin_bit_cast(uint32_t, mx)));
    mn = o_mn < mn ? o_mn : mn;
    mx = o_mx > mx ? o_mx : mx;
}
// min / max over L (2, 4 or 8) consecutive lanes; NaN operands are left out,
// as the reference's comparisons leave them (mn and mx start as infinities).
template <int L>
__device__ __forceinline__ void lanes_min_max(float &mn, float &mx) {
    min_max_step<kDppXor1>(mn, mx);
    if constexpr (L > 2) min_max_step<kDppXor2>(mn, mx);
    if constexpr (L > 4) min_max_step<kDppMirror8>(mn, mx);
}

// Memory-bound: a tile reads 8 KiB (fp32) and writes 1.1 KiB.  Each load
// covers whole 128-byte lines: lane 8 a + p brings 16 bytes at line offset
// 16 p of row a or 8 + a, so a lane holds 2 rows x NP pieces of EPL values and
// a block's min / max is reduced over at most eight neighbouring lanes.  The
// grid fills the chip once and each wave strides over the tiles, the next
// tile's values in flight while the current one is quantized, so the largest
// scale of the weight (its fold exponent, below) leaves each workgroup as one
// value of `part` and no pass over the scales is needed to find it.  Qwen's
// [151936, 896] table in fp32: 113-115 us (618 MB, 5.4 TB/s); a wave per tile
// with 32 bytes of each of 16 rows per lane and a division for every value
// took 135-145 us.
template <typename InT, int BS>
__global__ __launch_bounds__(kQuantThreads) void quantize_tiles_kernel(WeightGeom g, const InT *__restrict__ data,
                                                                       uint32_t *__restrict__ q_t,
                                                                       float *__restrict__ s_t,
                                                                       uint8_t *__restrict__ zp_t,
                                                                       float *__restrict__ part) {
    constexpr int SPS = kTileK / BS;  // blocks of a row inside one super-tile
    constexpr int ZB = SPS <= 2 ? 1 : SPS / 2;
    constexpr int WPB = kQuantThreads / 64;
    constexpr int EPL = 16 / (int)sizeof(InT);     // values per load: 4 or 8
    constexpr int PK = 8 * EPL, NP = kTileK / PK;  // k per piece (a 128-byte line), pieces per row
    constexpr int NB = BS >= PK ? SPS : NP;        // blocks of a row a lane has values of
    constexpr int PPB = NP / NB;                   // pieces per block
    constexpr int L = BS >= PK ? 8 : BS / EPL;     // lanes that share a block
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const int p = lane & 7, a = lane >> 3;
    const int cols = g.K;  // a multiple of BS, so a block is entirely inside or outside [0, cols)
    const int64_t tiles = (int64_t)g.NT * g.ST;
    const int64_t step = (int64_t)gridDim.x * WPB;
    float smax = 0.0f;
    // values outside the matrix load its first ones instead (straight-line
    // loads) and are replaced below
    u32x4_t raw[2][NP];
    auto inside = [&](int nt, int st, int h, int i) {
        return nt * kTileRows + 8 * h + a < g.N && st * kTileK + i * PK + EPL * p < cols;
    };
    auto issue = [&](int64_t t) {
        const int nt = (int)(t / g.ST), st = (int)(t - (int64_t)nt * g.ST);
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < NP; ++i)
                raw[h][i] = gld_nt((const u32x4_t *)(data + (inside(nt, st, h, i) ? (size_t)(nt * kTileRows + 8 * h + a) * cols +
                                                                                        st * kTileK + i * PK + EPL * p
                                                                                  : 0)));
    };
    int64_t t = (int64_t)blockIdx.x * WPB + wave;
    if (t < tiles) issue(t);
    for (; t < tiles; t += step) {
        const int nt = (int)(t / g.ST), st = (int)(t - (int64_t)nt * g.ST);
        float v[2][NP][EPL];
#pragma unroll
        for (int h = 0; h < 2; ++h)
#pragma unroll
            for (int i = 0; i < NP; ++i) widen<InT>(raw[h][i], v[h][i]);
        issue(min(t + step, tiles - 1));   // past the end: loaded, never used

        uint32_t d[2][NP];   // the lane's nibbles of each piece
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int row = 8 * h + a;
            uint32_t zp_pair = 0;
#pragma unroll
            for (int b = 0; b < NB; ++b) {
                // A block is inside or outside the matrix as a whole, so all
                // its lanes agree.
                const bool valid = inside(nt, st, h, b * PPB);
                float mn = __builtin_inff(), mx = -__builtin_inff();
#pragma unroll
                for (int i = b * PPB; i < (b + 1) * PPB; ++i)
#pragma unroll
                    for (int e = 0; e < EPL; ++e) {
                        mn = v[h][i][e] < mn ? v[h][i][e] : mn;
                        mx = v[h][i][e] > mx ? v[h][i][e] : mx;
                    }
                lanes_min_max<L>(mn, mx);
                float scale = 0.0f;
                int z = 0;
                if (valid) {
                    if (mx == mn) {
                        if (fabsf(mx) < 1.0e-8f) {
                            scale = 1.0f;
                        } else if (mx > 0.0f) {
                            scale = mx / 15.0f;
                        } else {
                            scale = -mn / 15.0f;
                            z = 15;
                        }
                    } else {
                        scale = (mx - mn) / 15.0f;
                        z = clamp_u4(java_round_f(-mn / scale));
                    }
                }
                smax = fmaxf(smax, fabsf(scale));   // a NaN scale is left out
                // a scale whose reciprocal is a normal number, else NaN (every
                // value of the block takes the division)
                const float rcp = scale >= 0x1p-120f && scale <= 0x1p120f ? 1.0f / scale : __builtin_nanf("");
#pragma unroll
                for (int i = b * PPB; i < (b + 1) * PPB; ++i)
                    d[h][i] = valid ? quantize_piece<EPL>(v[h][i], scale, rcp, (float)z) : 0u;
                // the first lane of a block writes its scale; zero points as
                // the nibbles of the row's entry, put together over its lanes
                const int blk = BS >= PK ? b : b * (PK / BS) + p / L;
                const size_t e = (size_t)t * kTileRows + row;
                if (p % L == 0) s_t[e * SPS + blk] = scale;
                uint32_t zbits = (uint32_t)z << (4 * (blk & 1));
                if constexpr (SPS > 1) {
                    // nibbles of blocks 2 i and 2 i + 1 share a byte
                    if constexpr (BS < PK) {
                        zbits |= __shfl_xor(zbits, L);
                        if (p % (2 * L) == 0) zp_t[e * ZB + blk / 2] = (uint8_t)zbits;
                    } else {
                        if (b & 1) zp_pair |= zbits;
                        else zp_pair = zbits;
                        if ((b & 1) && p == 0) zp_t[e * ZB + blk / 2] = (uint8_t)zp_pair;
                    }
                } else if (p == 0) {
                    zp_t[e] = (uint8_t)zbits;
                }
            }
        }
        // The lane's 16-byte chunk of the tile: one row, lane group gg, the dwords
        // of the four 32-k steps.  Two lanes hold it for two rows: each keeps
        // one row and receives the other lane's part of it.
        u32x4_t out;
        int row, gg;
        if constexpr (EPL == 4) {   // halves of the same dwords
            const bool odd = p & 1;
            row = odd ? 8 + a : a;
            gg = p >> 1;
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const uint32_t keep = (odd ? d[1][i] : d[0][i]) << (odd ? 8 : 0);
                const uint32_t give = (odd ? d[0][i] : d[1][i]) << (odd ? 8 : 0);
                out[i] = keep | lane_dpp<kDppXor1>(give);
            }
        } else {                    // even and odd steps
            const bool odd = p >> 2;
            row = odd ? 8 + a : a;
            gg = p & 3;
#pragma unroll
            for (int i = 0; i < NP; ++i) {
                const uint32_t keep = odd ? d[1][i] : d[0][i], got = __shfl_xor(odd ? d[0][i] : d[1][i], 4);
                out[2 * i] = odd ? got : keep;
                out[2 * i + 1] = odd ? keep : got;
            }
        }
        *(u32x4_t *)(q_t + ((size_t)t * 64 + gg * 16 + row) * 4) = out;
    }

    // the workgroup's largest |scale|
    __shared__ float wmax[WPB];
#pragma unroll
    for (int m = 1; m < 64; m <<= 1) smax = fmaxf(smax, __shfl_xor(smax, m));
    if (lane == 0) wmax[wave] = smax;
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int i = 1; i < WPB; ++i) smax = fmaxf(smax, wmax[i]);
        part[blockIdx.x] = smax;
    }
}

// Multiplies the quantized scales by 2^fold_exp, the weight's fold exponent
// from the quantizer's n_part partial maxima (every workgroup reduces them,
// at most 4 KiB, for itself), and stores the exponent in *fold.
__global__ __launch_bounds__(kQuantThreads) void fold_scales_kernel(float4_t *__restrict__ s, size_t n4,
                                                                    const float *__restrict__ part, int n_part,
                                                                    int32_t *__restrict__ fold) {
    constexpr int WPB = kQuantThreads / 64;
    const size_t i = (size_t)blockIdx.x * kQuantThreads + threadIdx.x;
    float4_t v = {0.f, 0.f, 0.f, 0.f};
    if (i < n4) v = s[i];
    float m = 0.0f;
#pragma unroll
    for (int x = 0; x < (int)kQuantMaxWgs / kQuantThreads; ++x) {
        const int at = x * kQuantThreads + (int)threadIdx.x;
        m = fmaxf(m, part[at < n_part ? at : 0]);
    }
#pragma unroll
    for (int x = 1; x < 64; x <<= 1) m = fmaxf(m, __shfl_xor(m, x));
    __shared__ float wmax[WPB];
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
#pragma unroll
    for (int x = 0; x < WPB; ++x) m = fmaxf(m, wmax[x]);
    const int e = fold_exponent((double)m);
    if (blockIdx.x == 0 && threadIdx.x == 0) *fold = e;
    if (e != 0 && i < n4) s[i] = v * pow2f(e);
}

template <typename InT>
static hipError_t quantize_dispatch(const WeightGeom &g, const InT *data, void *q_t, float *s_t, uint8_t *zp_t,
                                    float *part, unsigned wgs, hipStream_t stream) {
    const dim3 grid(wgs), block(kQuantThreads);
    uint32_t *q = (uint32_t *)q_t;
    switch (g.bs) {
    case 16: hipLaunchKernelGGL((quantize_tiles_kernel<InT, 16>), grid, block, 0, stream, g, data, q, s_t, zp_t, part); break;
    case 32: hipLaunchKernelGGL((quantize_tiles_kernel<InT, 32>), grid, block, 0, stream, g, data, q, s_t, zp_t, part); break;
    case 64: hipLaunchKernelGGL((quantize_tiles_kernel<InT, 64>), grid, block, 0, stream, g, data, q, s_t, zp_t, part); break;
    case 128: hipLaunchKernelGGL((quantize_tiles_kernel<InT, 128>), grid, block, 0, stream, g, data, q, s_t, zp_t, part); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

hipError_t launch_quantize(const WeightGeom &g, const void *data, int32_t data_type, void *q_t, float *s_t,
                           uint8_t *zp_t, void *scratch, hipStream_t stream) {
    const size_t tiles = (size_t)g.NT * g.ST;
    const unsigned wgs = (unsigned)std::min<size_t>(kQuantMaxWgs, (tiles + kQuantThreads / 64 - 1) / (kQuantThreads / 64));
    int32_t *fold = (int32_t *)scratch;
    float *part = (float *)scratch + kQuantPartAt;
    const hipError_t e = data_type == MNB_F32
                             ? quantize_dispatch(g, (const float *)data, q_t, s_t, zp_t, part, wgs, stream)
                             : quantize_dispatch(g, (const _Float16 *)data, q_t, s_t, zp_t, part, wgs, stream);
    if (e != hipSuccess) return e;
    const size_t n4 = tiles * kTileRows * g.SPS / 4;
    hipLaunchKernelGGL(fold_scales_kernel, dim3((unsigned)((n4 + kQuantThreads - 1) / kQuantThreads)), dim3(kQuantThreads), 0,
                       stream, (float4_t *)s_t, n4, part, (int)wgs, fold);
    return hipGetLastError();
}

// ---------------------------------------------------------------------------
// read-back: tiled layout -> the reference's arrays
// ---------------------------------------------------------------------------

// Tiled dword -> natural dword (k0 in the low nibble ... k7 in the high one).
__device__ __forceinline__ uint32_t zip_nibbles(uint32_t t) {
    uint32_t s = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const int pos = (i & 1) ? 16 + 4 * (i >> 1) : 4 * (i >> 1);
        s |= ((t >> pos) & 0xFu) << (4 * i);
    }
    return s;
}

__global__ void unpack_q_kernel(WeightGeom g, const uint32_t *__restrict__ q_t, uint8_t *__restrict__ q_nat) {
    const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (c >= (size_t)g.NT * g.ST * 64) return;
    const int lane = (int)(c & 63);
    const size_t tile = c >> 6;
    const int st = (int)(tile % g.ST), nt = (int)(tile / g.ST);
    const int r = lane & 15, gg = lane >> 4;
    const int n = nt * kTileRows + r;
    if (n >= g.N) return;
    const size_t row_bytes = (size_t)g.Kpad / 2;
    const u32x4_t in = *(const u32x4_t *)(q_t + c * 4);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int k0 = st * kTileK + 32 * j + 8 * gg;
        if (k0 < g.Kpad) *(uint32_t *)(q_nat + (size_t)n * row_bytes + (size_t)(k0 / 2)) = zip_nibbles(in[j]);
    }
}

// One thread per (tile, row): the row's SPS scales and zero points of this
// super-tile; a block longer than a super-tile is written once, from the
// super-tile where it starts.  Zero points come out one byte per block (8
// when the weight has the implicit zero point).
template <typename ScaleT>
__global__ void unpack_scales_zp_kernel(WeightGeom g, const ScaleT *__restrict__ s_t, const uint8_t *__restrict__ zp_t,
                                        float *__restrict__ s_nat, uint8_t *__restrict__ zp_blocks) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)g.NT * g.ST * kTileRows) return;
    const int r = (int)(e % kTileRows);
    const size_t tile = e / kTileRows;
    const int st = (int)(tile % g.ST), nt = (int)(tile / g.ST);
    const int n = nt * kTileRows + r;
    if (n >= g.N) return;
    uint32_t bits = 0;
    if (zp_t)
        for (int b = 0; b < g.ZB; ++b) bits |= (uint32_t)zp_t[e * g.ZB + b] << (8 * b);
    for (int i = 0; i < g.SPS; ++i) {
        const int blk = g.bs >= kTileK ? (st * kTileK) / g.bs : st * g.SPS + i;
        if (blk >= g.kb) continue;
        if (g.bs > kTileK && st * kTileK != blk * g.bs) continue;
        s_nat[(size_t)n * g.kb + blk] = (float)s_t[e * g.SPS + i] * pow2f(-g.fold_exp);
        zp_blocks[(size_t)n * g.kb + blk] = zp_t ? (uint8_t)((bits >> (4 * i)) & 0xFu) : (uint8_t)8;
    }
}

hipError_t launch_unpack(const mnb_weight *w, uint8_t *q_nat, float *s_nat, uint8_t *zp_blocks, hipStream_t stream) {
    const WeightGeom &g = w->g;
    const unsigned T = 256;
    const size_t nq = (size_t)g.NT * g.ST * 64;
    hipLaunchKernelGGL(unpack_q_kernel, dim3((unsigned)((nq + T - 1) / T)), dim3(T), 0, stream, g,
                       (const uint32_t *)w->q_t, q_nat);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    const size_t ns = (size_t)g.NT * g.ST * kTileRows;
    const dim3 grid((unsigned)((ns + T - 1) / T));
    if (g.scale_f32)
        hipLaunchKernelGGL(unpack_scales_zp_kernel<float>, grid, dim3(T), 0, stream, g, (const float *)w->s_t,
                           (const uint8_t *)w->zp_t, s_nat, zp_blocks);
    else
        hipLaunchKernelGGL(unpack_scales_zp_kernel<_Float16>, grid, dim3(T), 0, stream, g, (const _Float16 *)w->s_t,
                           (const uint8_t *)w->zp_t, s_nat, zp_blocks);
    return hipGetLastError();
}

}  // namespace mnb
