// mnb_layout.hip -- one-time weight repack into the tiled HBM layout, the
// activation staging kernel and the dequantize-only kernel.
//
// The dequantize-only kernel restates MatMulNBitsKernel.dequantizeInt4
// (directml-windows-bindings/src/main/java/com/aresstack/windirectml/windows/
// MatMulNBitsKernel.java:2674-2705): w = float(nibble - zp) * scale in fp32,
// low nibble first.  Its fp32 output is bit-identical to that function.
#include "mnb_device.h"

namespace mnb {

typedef u32x4_t u32x4_dq_alias_t __attribute__((may_alias));
// 16, 8 and 4 bytes of a row of fp16 or fp32
typedef u32x4_t u32x4_row_t __attribute__((may_alias, aligned(2)));
typedef u32x2_t u32x2_row_t __attribute__((may_alias, aligned(2)));
typedef uint32_t u32_row_t __attribute__((may_alias, aligned(2)));
constexpr int kDequantThreads = 256;

WeightGeom make_geom(int32_t N, int32_t K, int32_t bs) {
    WeightGeom g;
    g.N = N;
    g.K = K;
    g.bs = bs;
    g.kb = (K + bs - 1) / bs;
    g.Kpad = g.kb * bs;
    g.NT = (N + kTileRows - 1) / kTileRows;
    g.ST = (g.Kpad + kTileK - 1) / kTileK;
    g.SPS = bs >= kTileK ? 1 : kTileK / bs;
    g.ZB = g.SPS <= 2 ? 1 : g.SPS / 2;
    return g;
}

// Natural packed dword (k0 | k1<<4 | ... | k7<<28, bytes low nibble first)
// -> tiled order (k0,k2,k4,k6 in bits 0..15; k1,k3,k5,k7 in bits 16..31).
__device__ __forceinline__ uint32_t unzip_nibbles(uint32_t s) {
    uint32_t t = 0;
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        uint32_t nib = (s >> (4 * i)) & 0xFu;
        int pos = (i & 1) ? 16 + 4 * (i >> 1) : 4 * (i >> 1);
        t |= nib << pos;
    }
    return t;
}

// Tiled dword -> natural nibble i (0..7) of its 8 consecutive k.
__device__ __forceinline__ uint32_t tiled_nibble(uint32_t t, int i) {
    int pos = (i & 1) ? 16 + 4 * (i >> 1) : 4 * (i >> 1);
    return (t >> pos) & 0xFu;
}

__global__ void repack_q_kernel(WeightGeom g, const uint8_t *__restrict__ q_nat, uint32_t *__restrict__ q_t) {
    const size_t c = (size_t)blockIdx.x * blockDim.x + threadIdx.x;   // one lane chunk (16 bytes)
    const size_t total = (size_t)g.NT * g.ST * 64;
    if (c >= total) return;
    const int lane = (int)(c & 63);
    const size_t tile = c >> 6;
    const int st = (int)(tile % g.ST);
    const int nt = (int)(tile / g.ST);
    const int r = lane & 15, gg = lane >> 4;
    const int n = nt * kTileRows + r;
    const size_t row_bytes = (size_t)g.Kpad / 2;
    u32x4_t out;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const int k0 = st * kTileK + 32 * j + 8 * gg;
        uint32_t v = 0;
        if (n < g.N && k0 < g.Kpad) {
            const uint32_t s = *(const uint32_t *)(q_nat + (size_t)n * row_bytes + (size_t)(k0 / 2));
            v = unzip_nibbles(s);
        }
        out[j] = v;
    }
    *(u32x4_t *)(q_t + c * 4) = out;
}

// s * 2^e rounded to the scale type (exact: the product stays within the
// type's finite range by the choice of the exponents).  The fp32 product is
// kept in a register first: fused into one mixed-precision multiply-add with a
// +0 addend, a -0 scale would come out as +0.
template <typename ScaleT, typename SrcT>
__device__ __forceinline__ ScaleT scaled(SrcT s, float factor) {
    float f = (float)s * factor;
    asm volatile("" : "+v"(f));
    return (ScaleT)f;
}

// Scales in tile order, times 2^fold_exp.
template <typename ScaleT>
__global__ void repack_scales_kernel(WeightGeom g, const ScaleT *__restrict__ s_nat, ScaleT *__restrict__ s_t) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t total = (size_t)g.NT * g.ST * kTileRows * g.SPS;
    if (e >= total) return;
    const int i = (int)(e % g.SPS);
    const size_t rest = e / g.SPS;
    const int r = (int)(rest % kTileRows);
    const size_t tile = rest / kTileRows;
    const int st = (int)(tile % g.ST);
    const int nt = (int)(tile / g.ST);
    const int n = nt * kTileRows + r;
    const int blk = g.bs >= kTileK ? (st * kTileK) / g.bs : st * g.SPS + i;
    ScaleT v = (ScaleT)0;
    if (n < g.N && blk < g.kb) v = scaled<ScaleT>(s_nat[(size_t)n * g.kb + blk], pow2f(g.fold_exp));
    s_t[e] = v;
}

__global__ void repack_zp_kernel(WeightGeom g, const uint8_t *__restrict__ zp_flat, uint8_t *__restrict__ zp_t) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    const size_t total = (size_t)g.NT * g.ST * kTileRows;
    if (e >= total) return;
    const int r = (int)(e % kTileRows);
    const size_t tile = e / kTileRows;
    const int st = (int)(tile % g.ST);
    const int nt = (int)(tile / g.ST);
    const int n = nt * kTileRows + r;
    uint32_t bits = 0;
    for (int i = 0; i < g.SPS; ++i) {
        const int blk = g.bs >= kTileK ? (st * kTileK) / g.bs : st * g.SPS + i;
        if (n < g.N && blk < g.kb) {
            const size_t idx = (size_t)n * g.kb + blk;
            const uint32_t nib = (zp_flat[idx / 2] >> (4 * (idx & 1))) & 0xFu;
            bits |= nib << (4 * i);
        }
    }
    for (int b = 0; b < g.ZB; ++b) zp_t[e * g.ZB + b] = (uint8_t)(bits >> (8 * b));
}

static inline unsigned blocks_for(size_t n, unsigned t) { return (unsigned)((n + t - 1) / t); }

hipError_t launch_repack(const WeightGeom &g, const uint8_t *q_nat, const void *s_nat, const uint8_t *zp_flat,
                         void *q_t, void *s_t, void *zp_t, hipStream_t stream) {
    const unsigned T = 256;
    size_t nq = (size_t)g.NT * g.ST * 64;
    hipLaunchKernelGGL(repack_q_kernel, dim3(blocks_for(nq, T)), dim3(T), 0, stream, g, q_nat, (uint32_t *)q_t);
    hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    size_t ns = (size_t)g.NT * g.ST * kTileRows * g.SPS;
    if (g.scale_f32)
        hipLaunchKernelGGL(repack_scales_kernel<float>, dim3(blocks_for(ns, T)), dim3(T), 0, stream, g,
                           (const float *)s_nat, (float *)s_t);
    else
        hipLaunchKernelGGL(repack_scales_kernel<_Float16>, dim3(blocks_for(ns, T)), dim3(T), 0, stream, g,
                           (const _Float16 *)s_nat, (_Float16 *)s_t);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    if (g.has_zp) {
        size_t nz = (size_t)g.NT * g.ST * kTileRows;
        hipLaunchKernelGGL(repack_zp_kernel, dim3(blocks_for(nz, T)), dim3(T), 0, stream, g, zp_flat,
                           (uint8_t *)zp_t);
        e = hipGetLastError();
    }
    return e;
}

// Row fusion: one thread per (source row, super-tile) moves that row's four
// 16-byte lane chunks of packed nibbles, its SPS scales and its ZB zero-point
// bytes to the destination row.  Both weights share K and the block size, so
// ST, SPS and ZB agree; padding k, blocks >= kb and rows past the end stay as
// the zeroed destination holds them.
template <typename SrcS, typename DstS>
__global__ void copy_rows_kernel(WeightGeom sg, const uint32_t *__restrict__ sq, const SrcS *__restrict__ ss,
                                 const uint8_t *__restrict__ sz, WeightGeom dg, uint32_t *__restrict__ dq,
                                 DstS *__restrict__ ds, uint8_t *__restrict__ dz, int32_t row0) {
    const size_t e = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (e >= (size_t)sg.N * sg.ST) return;
    const int st = (int)(e % sg.ST);
    const int rs = (int)(e / sg.ST);
    const int rd = row0 + rs;
    const size_t ts = (size_t)(rs / kTileRows) * sg.ST + st;
    const size_t td = (size_t)(rd / kTileRows) * dg.ST + st;
    const int ls = rs % kTileRows, ld = rd % kTileRows;
#pragma unroll
    for (int gg = 0; gg < 4; ++gg)
        *(u32x4_t *)(dq + (td * 64 + gg * 16 + ld) * 4) = *(const u32x4_t *)(sq + (ts * 64 + gg * 16 + ls) * 4);
    const float factor = pow2f(dg.fold_exp - sg.fold_exp);
    for (int i = 0; i < sg.SPS; ++i)
        ds[(td * kTileRows + ld) * dg.SPS + i] = scaled<DstS>(ss[(ts * kTileRows + ls) * sg.SPS + i], factor);
    if (!dz) return;
    if (sz) {
        for (int b = 0; b < sg.ZB; ++b) dz[(td * kTileRows + ld) * dg.ZB + b] = sz[(ts * kTileRows + ls) * sg.ZB + b];
        return;
    }
    uint32_t bits = 0;  // implicit zero point 8 for the blocks the row holds
    for (int i = 0; i < sg.SPS; ++i) {
        const int blk = sg.bs >= kTileK ? (st * kTileK) / sg.bs : st * sg.SPS + i;
        if (blk < sg.kb) bits |= 8u << (4 * i);
    }
    for (int b = 0; b < dg.ZB; ++b) dz[(td * kTileRows + ld) * dg.ZB + b] = (uint8_t)(bits >> (8 * b));
}

hipError_t launch_copy_rows(const WeightGeom &sg, const void *sq, const void *ss, const void *sz, const WeightGeom &dg,
                            void *dq, void *ds, void *dz, int32_t row0, hipStream_t stream) {
    const unsigned T = 256;
    const size_t n = (size_t)sg.N * sg.ST;
    if (n == 0) return hipSuccess;
    const dim3 grid(blocks_for(n, T)), block(T);
    if (!dg.scale_f32)
        hipLaunchKernelGGL((copy_rows_kernel<_Float16, _Float16>), grid, block, 0, stream, sg, (const uint32_t *)sq,
                           (const _Float16 *)ss, (const uint8_t *)sz, dg, (uint32_t *)dq, (_Float16 *)ds,
                           (uint8_t *)dz, row0);
    else if (sg.scale_f32)
        hipLaunchKernelGGL((copy_rows_kernel<float, float>), grid, block, 0, stream, sg, (const uint32_t *)sq,
                           (const float *)ss, (const uint8_t *)sz, dg, (uint32_t *)dq, (float *)ds, (uint8_t *)dz,
                           row0);
    else
        hipLaunchKernelGGL((copy_rows_kernel<_Float16, float>), grid, block, 0, stream, sg, (const uint32_t *)sq,
                           (const _Float16 *)ss, (const uint8_t *)sz, dg, (uint32_t *)dq, (float *)ds,
                           (uint8_t *)dz, row0);
    return hipGetLastError();
}

// fp16 copy of x with rows padded to ldx (a multiple of 8).  A launch-bound
// copy: one thread per 8 values of a row, read in 16-byte pieces at whatever
// alignment x's rows have, and 32-bit index arithmetic unless x has 2^32
// pieces or more.  A row's last piece is read so that it ends at the row's
// end and shifted into place.  Whole products with their staging, same box,
// one value per thread -> this: 3072 -> 3072 at M = 200 from aligned fp32
// 17.0 -> 15.4 us, from fp32 off by one 17.0 -> 15.5; 8190 -> 512 at M = 512
// from fp32 22.0 -> 19.5; 3076 -> 1024 at M = 2048 from fp16 44.7 -> 36.4;
// 1001 -> 1024 at M = 4 4.7 -> 4.7.  (Eight element loads per thread where a
// row is unaligned took 24.9 us of the third and 5.2 of the last.)
template <typename XT, typename IdxT>
__global__ __launch_bounds__(256) void stage_x_kernel(const XT *__restrict__ x, IdxT pieces, int32_t K, int32_t ldx,
                                                      _Float16 *__restrict__ out) {
    const IdxT e = (IdxT)blockIdx.x * 256 + threadIdx.x;
    if (e >= pieces) return;
    const IdxT per_row = (IdxT)(ldx / 8);
    const IdxT m = e / per_row;
    const int k = (int)(e - m * per_row) * 8;
    const XT *row = x + (size_t)m * K;
    half8_t h;
    if (K >= 8) {
        const int kc = min(k, K - 8);
        XT v[8];
        u32x4_row_t raw[sizeof(XT) / 2];
#pragma unroll
        for (int i = 0; i < (int)sizeof(XT) / 2; ++i)
            raw[i] = ((const __attribute__((address_space(1))) u32x4_row_t *)(row + kc))[i];
        __builtin_memcpy(v, raw, sizeof v);
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = (_Float16)v[i];
        if (kc != k) h = __builtin_bit_cast(half8_t, __builtin_bit_cast(unsigned __int128, h) >> (16 * (k - kc)));
    } else {
#pragma unroll
        for (int i = 0; i < 8; ++i) h[i] = i < K ? (_Float16)row[i] : (_Float16)0.0f;
    }
    *(half8_t *)(out + (size_t)m * ldx + k) = h;
}

template <typename XT>
static hipError_t stage_x_typed(const XT *x, int32_t M, int32_t K, int32_t ldx, _Float16 *out, hipStream_t stream) {
    const uint64_t pieces = (uint64_t)M * (uint64_t)(ldx / 8);
    const dim3 grid(blocks_for(pieces, 256)), block(256);
    if (pieces <= 0xFFFFFF00u)
        hipLaunchKernelGGL((stage_x_kernel<XT, uint32_t>), grid, block, 0, stream, x, (uint32_t)pieces, K, ldx, out);
    else
        hipLaunchKernelGGL((stage_x_kernel<XT, uint64_t>), grid, block, 0, stream, x, pieces, K, ldx, out);
    return hipGetLastError();
}

hipError_t launch_stage_x(const void *x, int32_t x_type, int32_t M, int32_t K, int32_t ldx, _Float16 *out,
                          hipStream_t stream) {
    return x_type == MNB_F32 ? stage_x_typed((const float *)x, M, K, ldx, out, stream)
                             : stage_x_typed((const _Float16 *)x, M, K, ldx, out, stream);
}

// Stores the first n (fewer than there are) of the fp32 or fp16 values in v.
__device__ __forceinline__ void store_head(float *p, const u32x4_t &v, int n) {
    if (n & 2) *(u32x2_row_t *)p = (u32x2_t){v[0], v[1]};
    if (n & 1) p[n - 1] = __builtin_bit_cast(float, n & 2 ? v[2] : v[0]);
}
__device__ __forceinline__ void store_head(_Float16 *p, const u32x4_t &v, int n) {
    const uint32_t lo = n & 4 ? v[2] : v[0], hi = n & 4 ? v[3] : v[1];
    if (n & 4) *(u32x2_row_t *)p = (u32x2_t){v[0], v[1]};
    if (n & 2) *(u32_row_t *)(p + (n & 4)) = lo;
    if (n & 1) p[n - 1] = __builtin_bit_cast(_Float16, (uint16_t)(n & 2 ? hi : lo));
}

// w = float(q - zp) * scale, formed as (float(q - zp) * stored scale) *
// 2^-fold_exp: the power of two makes the two roundings one.
//
// Bound by its writes (a tile is 1 KiB of nibbles and 4 or 8 KiB of output).
// One wave per tile: its nibbles pass through LDS, so that every store
// instruction writes whole consecutive pieces of 16 bytes per lane (two rows
// of 512 bytes in fp32, four of 256 in fp16).  Qwen's [151936, 896] head with
// fp32 scales to fp32: 100-106 us (618 MB, 5.9 TB/s; 108-112 with cached
// stores); a thread per 8 k with a load of its own dword and 32-byte strided
// stores took 332-334 us.  VEC: rows of out are 16-byte aligned.  Otherwise the
// pieces are stored at the alignment they have, cached (lines at the pieces'
// ends are shared), and a row's shorter last piece in parts of 8, 4 and 2
// bytes: 3072 -> 9216 off by one element to fp32 25 us, to fp16 17 (a thread per
// 8 k 71 and 39, element stores 46 and 42, non-temporal 37 and 21); 1001 ->
// 9728 to fp16 7.3 (17.3; 19.8).  The tile index stays uniform and 32-bit:
// small matrices are bound by one wave's latency (203 -> 4096 to fp16 4.4 us;
// 4.8 with a 64-bit division per lane).
template <typename ScaleT, typename OutT, bool HAS_ZP, bool VEC>
__global__ __launch_bounds__(kDequantThreads) void dequant_kernel(WeightGeom g, const uint32_t *__restrict__ q_t,
                                                                  const ScaleT *__restrict__ s_t,
                                                                  const uint8_t *__restrict__ zp_t,
                                                                  OutT *__restrict__ out) {
    constexpr int E = 16 / (int)sizeof(OutT);   // elements per lane and store
    constexpr int LPR = kTileK / E;             // lanes per row
    constexpr int RPS = 64 / LPR;               // rows per store
    // lane group g of the tile at g * (64 + 8) dwords: the 64 lanes of a read
    // (RPS rows, 4 dwords of each of 4 lane groups) then touch distinct banks
    constexpr int GSTRIDE = 64 + 8;
    __shared__ __align__(16) uint32_t smem[kDequantThreads / 64][4 * GSTRIDE];
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const uint32_t tile = blockIdx.x * (kDequantThreads / 64) + wave;   // below 2^31: a tile is 1 KiB of nibbles
    if (tile >= (uint32_t)g.NT * (uint32_t)g.ST) return;   // whole waves; a wave uses its own LDS only
    const int nt = (int)(tile / (uint32_t)g.ST), st = (int)(tile - (uint32_t)nt * (uint32_t)g.ST);
    *(u32x4_dq_alias_t *)&smem[wave][(lane >> 4) * GSTRIDE + (lane & 15) * 4] =
        gld_nt((const u32x4_t *)q_t + (size_t)tile * 64 + lane);
    asm volatile("" ::: "memory");   // a wave's LDS accesses run in order
    const int kk = (lane % LPR) * E;            // k of the lane's elements inside the tile
    const int k0 = st * kTileK + kk;
    const int j = kk / 32, gg = (kk % 32) / 8, i0 = kk % 8;
    const int si = kk * g.SPS / kTileK;   // the block of kk; 0 where a block spans the tile
    const float unfold = pow2f(-g.fold_exp);
    float sc[kTileRows / RPS];
    int zv[kTileRows / RPS];
    u32x4_t ov[kTileRows / RPS];
#pragma unroll
    for (int i = 0; i < kTileRows / RPS; ++i) {
        const size_t e = (size_t)tile * kTileRows + i * RPS + lane / LPR;
        sc[i] = (float)s_t[e * g.SPS + si];
        zv[i] = HAS_ZP ? (zp_t[e * g.ZB + si / 2] >> (4 * (si & 1))) & 0xF : 8;
    }
#pragma unroll
    for (int i = 0; i < kTileRows / RPS; ++i) {
        const int r = i * RPS + lane / LPR, n = nt * kTileRows + r;
        const uint32_t d = smem[wave][gg * GSTRIDE + r * 4 + j] >> (2 * i0);   // E = 4: k0..3 or k4..7 of the dword
        OutT o[E];
#pragma unroll
        for (int x = 0; x < E; ++x) {
            const int w = (int)tiled_nibble(d, x) - zv[i];
            float v = (float)w * sc[i] * unfold;
            // Keep the binary32 product in a register before the fp16 rounding:
            // otherwise the multiply and the conversion are fused into
            // v_fma_mix(scale, w, +0), which turns a -0 product into +0.
            asm volatile("" : "+v"(v));
            o[x] = (OutT)v;
        }
        OutT *p = out + (size_t)n * g.K + k0;
        __builtin_memcpy(&ov[i], o, 16);
        if constexpr (VEC) {
            if (n < g.N && k0 < g.K) __builtin_nontemporal_store(ov[i], (u32x4_t *)p);
        } else {
            if (n < g.N && k0 + E <= g.K) *(__attribute__((address_space(1))) u32x4_row_t *)p = ov[i];
        }
    }
    if constexpr (!VEC) {
        // the last, shorter piece of the rows
        const int rem = g.K - k0;
        if (rem > 0 && rem < E) {
#pragma unroll
            for (int i = 0; i < kTileRows / RPS; ++i) {
                const int n = nt * kTileRows + i * RPS + lane / LPR;
                if (n < g.N) store_head(out + (size_t)n * g.K + k0, ov[i], rem);
            }
        }
    }
}

template <typename ScaleT, typename OutT>
static hipError_t dequant_typed(const mnb_weight *w, OutT *out, hipStream_t stream) {
    const WeightGeom &g = w->g;
    const uint32_t *q = (const uint32_t *)w->q_t;
    const ScaleT *s = (const ScaleT *)w->s_t;
    const uint8_t *z = (const uint8_t *)w->zp_t;
    const dim3 grid(blocks_for((size_t)g.NT * g.ST, kDequantThreads / 64)), block(kDequantThreads);
    const bool vec = (size_t)g.K * sizeof(OutT) % 16 == 0 && (uintptr_t)out % 16 == 0;
    if (g.has_zp) {
        if (vec) hipLaunchKernelGGL((dequant_kernel<ScaleT, OutT, true, true>), grid, block, 0, stream, g, q, s, z, out);
        else hipLaunchKernelGGL((dequant_kernel<ScaleT, OutT, true, false>), grid, block, 0, stream, g, q, s, z, out);
    } else {
        if (vec) hipLaunchKernelGGL((dequant_kernel<ScaleT, OutT, false, true>), grid, block, 0, stream, g, q, s, z, out);
        else hipLaunchKernelGGL((dequant_kernel<ScaleT, OutT, false, false>), grid, block, 0, stream, g, q, s, z, out);
    }
    return hipGetLastError();
}

hipError_t launch_dequant(const mnb_weight *w, void *out, int32_t out_type, hipStream_t stream) {
    if (out_type == MNB_F32)
        return w->g.scale_f32 ? dequant_typed<float, float>(w, (float *)out, stream)
                              : dequant_typed<_Float16, float>(w, (float *)out, stream);
    return w->g.scale_f32 ? dequant_typed<float, _Float16>(w, (_Float16 *)out, stream)
                          : dequant_typed<_Float16, _Float16>(w, (_Float16 *)out, stream);
}

}  // namespace mnb
