// kxw4_pack.hip — load-time weight kernels: pack natural int4 codes into the
// gfx950 tile layout, unpack it, import the reference's DPAS layout, and the
// E2M3 -> asymmetric int4 repack (kernels_dpas.cpp:229-344; K32, K16 and
// K64 groups), and the W8A8 tier's int8 pack and repack.
//
// Packed tile (16 rows x 128 K, 1024 bytes): lane l owns bytes [16l, 16l+16),
// row l%16; dword i of the lane holds k = 32i + 8(l/16) + b with b = 0..3 in
// the low nibbles of bytes 0..3 and b = 4..7 in the high nibbles, so one
// 16-byte load per lane feeds two K64 MFMAs (or four K32 MFMAs). The W8A8
// tier's int8 tiles (2048 bytes) follow the same K slots, below.
#include "kxw4_device.hpp"
#include "kxw4_internal.hpp"

#include <algorithm>

namespace kxw4 {

// Tile-local coordinates of packed dword `d` (0..255 within a tile).
struct DwordCoord {
    int row;   // row within the 16-row group
    int k0;    // first K of the dword, within the 128-K tile
};

__device__ __forceinline__ DwordCoord dword_coord(int d) {
    const int lane = d >> 2, i = d & 3;
    return {lane & 15, 32 * i + 8 * (lane >> 4)};
}

__global__ void pack_codes_kernel(const int8_t *__restrict__ codes, int M, int K,
                                  uint32_t *__restrict__ out) {
    const size_t total = (size_t)M * K / 8;
    const size_t d = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= total) return;
    const int NT = K / kTileK;
    const size_t tile = d >> 8;
    const DwordCoord c = dword_coord((int)(d & 255));
    const int rg = (int)(tile / NT), kb = (int)(tile % NT);
    const int8_t *src = codes + (size_t)(rg * 16 + c.row) * K + kb * kTileK + c.k0;
    uint32_t w = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const uint32_t lo = (uint32_t)src[b] & 0xFu, hi = (uint32_t)src[b + 4] & 0xFu;
        w |= (lo | (hi << 4)) << (8 * b);
    }
    out[d] = w;
}

__global__ void unpack_codes_kernel(const uint32_t *__restrict__ in, int M, int K,
                                    int8_t *__restrict__ codes) {
    const size_t total = (size_t)M * K / 8;
    const size_t d = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= total) return;
    const int NT = K / kTileK;
    const size_t tile = d >> 8;
    const DwordCoord c = dword_coord((int)(d & 255));
    const int rg = (int)(tile / NT), kb = (int)(tile % NT);
    int8_t *dst = codes + (size_t)(rg * 16 + c.row) * K + kb * kTileK + c.k0;
    const uint32_t w = in[d];
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        dst[b] = (int8_t)sext4(w >> (8 * b));
        dst[b + 4] = (int8_t)sext4(w >> (8 * b + 4));
    }
}

// scales [M][G] (natural) <-> [M/16][G][16] (row within row-group fastest).
__global__ void scales_to_tiled_kernel(const uint16_t *__restrict__ in, int M, int G,
                                       uint16_t *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * G) return;
    const int row = (int)(i / G), g = (int)(i % G);
    out[((size_t)(row >> 4) * G + g) * 16 + (row & 15)] = in[i];
}

__global__ void scales_to_natural_kernel(const uint16_t *__restrict__ in, int M, int G,
                                         uint16_t *__restrict__ out) {
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * G) return;
    const int row = (int)(i / G), g = (int)(i % G);
    out[i] = in[((size_t)(row >> 4) * G + g) * 16 + (row & 15)];
}

// Reference layout (kernels_dpas.cpp:327-342): tile (rg, kt32) of 256 bytes;
// row n owns bytes [16n, 16n+16); k = 32kt + 8i + 2b + h sits in dword i,
// byte b, low nibble for h = 0.
__device__ __forceinline__ uint32_t ref_nibble(const uint8_t *__restrict__ ref, int Kt, int row,
                                               int k) {
    const int rg = row >> 4, n = row & 15, kt = k >> 5, j = k & 31;
    const uint8_t v = ref[((size_t)rg * Kt + kt) * 256u + (size_t)(n * 4 + (j >> 3)) * 4u +
                          (size_t)((j & 7) >> 1)];
    return (j & 1) ? (uint32_t)(v >> 4) : (uint32_t)(v & 0xFu);
}

__global__ void import_ref_codes_kernel(const uint8_t *__restrict__ ref, int M, int K,
                                        uint32_t *__restrict__ out) {
    const size_t total = (size_t)M * K / 8;
    const size_t d = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= total) return;
    const int NT = K / kTileK, Kt = K / 32;
    const size_t tile = d >> 8;
    const DwordCoord c = dword_coord((int)(d & 255));
    const int rg = (int)(tile / NT), kb = (int)(tile % NT);
    const int row = rg * 16 + c.row, k = kb * kTileK + c.k0;
    uint32_t w = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) {
        const uint32_t lo = ref_nibble(ref, Kt, row, k + b);
        const uint32_t hi = ref_nibble(ref, Kt, row, k + b + 4);
        w |= (lo | (hi << 4)) << (8 * b);
    }
    out[d] = w;
}

// ---- E2M3 -> asymmetric int4 (kernels_dpas.cpp:49-69, 229-344) -----------
//
// One thread per (row, group), the 16 rows of a row-group fastest, then the
// groups: a wave covers 16 rows x 4 groups, whose payload, codes and scales
// are contiguous. What bounds it is the fit's arithmetic, four quotients per
// weight (three refinements and the codes), not memory: 89 M weights (K =
// 5120, M = 17408, group 32) move 117 MB, 24 us at the rate a large copy
// reaches. With a byte load or two per code and an IEEE division per quotient
// (about 12 instructions) it took 215 us; with three 16-byte loads per thread,
// quotients of five operations and coalesced stores 107 us (W8, M = 7408, K =
// 2048: 39 -> 15 us).

// Six-bit code as a float: the five magnitude bits are the exponent and
// mantissa of an E2M3 number, put where FP32's lie and scaled by 2^126 (an
// exponent field of 0 is subnormal in both formats, so the product is exact).
__device__ __forceinline__ float e2m3f(uint32_t c) {
    const float v = __uint_as_float((c & 0x1Fu) << 20) * __uint_as_float(0x7E800000u);
    return __uint_as_float(__float_as_uint(v) | ((c & 0x20u) << 26));
}

// The 32 codes of (row, K32 tile): lanes 4*(row%16/2) .. +3 of the tile's 384
// bytes, 12 bytes each holding eight columns of an even and an odd row as a
// 96-bit stream (codes 0-3 even, 4-7 odd, 8-11 even, 12-15 odd).
__device__ __forceinline__ void e2m3_unit(const uint8_t *__restrict__ payload, size_t tile, int n, float b,
                                          float *wf) {
    const uint8_t *src = payload + tile * 384u + (size_t)(n >> 1) * 48u;
    uint32_t w[12] = {};
    if ((reinterpret_cast<uintptr_t>(payload) & 15) == 0) {
#pragma unroll
        for (int i = 0; i < 3; ++i) {
            const v4u v = reinterpret_cast<const v4u *>(src)[i];
            w[4 * i] = v.x;
            w[4 * i + 1] = v.y;
            w[4 * i + 2] = v.z;
            w[4 * i + 3] = v.w;
        }
    } else {                                                 // (a payload that starts anywhere)
#pragma unroll
        for (int i = 0; i < 48; ++i) w[i >> 2] |= (uint32_t)src[i] << (8 * (i & 3));
    }
    const bool odd = n & 1;
#pragma unroll
    for (int l = 0; l < 4; ++l) {
        const uint32_t x = w[3 * l], y = w[3 * l + 1], z = w[3 * l + 2];
        const uint32_t first = odd ? (x >> 24) | (y << 8) : x;
        const uint32_t second = odd ? z >> 8 : (y >> 16) | (z << 16);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            wf[8 * l + i] = e2m3f(first >> (6 * i)) * b;
            wf[8 * l + 4 + i] = e2m3f(second >> (6 * i)) * b;
        }
    }
}

// a / s in round to nearest. SAFE: the two-step refinement of a * y with
// y = fl(1/s) (Markstein: from a faithful quotient q and a correctly rounded
// reciprocal, fl(q + fl(a - q s) y) is the correctly rounded quotient, the
// remainder being exact), for operands far from the ends of the range.
template <bool SAFE>
__device__ __forceinline__ float quot(float a, float s, float y) {
    if constexpr (!SAFE) return a / s;
    float q = a * y;
    q = __builtin_fmaf(__builtin_fmaf(-q, s, a), y, q);
    return __builtin_fmaf(__builtin_fmaf(-q, s, a), y, q);
}

// Block scales this far from the ends of the range keep every weight, fitted
// scale, quotient and remainder normal (the scales lie in [b/120, 8b], or are
// 1 where every weight is 0; the FP16 scale is checked by itself).
__device__ __forceinline__ bool safe_scale(float b) { return b > 0x1p-60f && b < 0x1p60f; }
__device__ __forceinline__ bool safe_half(float s) { return s > 0.0f && s < 65536.0f; }

// min(max(x, lo), hi) of a number that is not NaN (clampf's result then)
template <bool SAFE>
__device__ __forceinline__ float clampq(float x, float lo, float hi) {
    return SAFE ? __builtin_amdgcn_fmed3f(x, lo, hi) : clampf(x, lo, hi);
}

// fit_int4_asym with the least-squares sums evaluated as fused multiply-adds.
template <int N, bool SAFE>
__device__ __forceinline__ uint16_t fit_int4_asym(const float *wf, int *out_z) {
    float lo = 0.0f, hi = 0.0f;
#pragma unroll
    for (int j = 0; j < N; ++j) {
        lo = fminf(lo, wf[j]);
        hi = fmaxf(hi, wf[j]);
    }
    float s = (hi - lo) / 15.0f;
    if (!(s > 0.0f)) s = 1.0f;
#pragma unroll 1
    for (int iter = 0; iter < 3; ++iter) {
        const float zf = (float)(int)clampf(rintf(-lo / s) - 8.0f, -8.0f, 7.0f), y = 1.0f / s;
        float num = 0.0f, den = 0.0f;
#pragma unroll
        for (int j = 0; j < N; ++j) {
            const float q = clampq<SAFE>(rintf(quot<SAFE>(wf[j], s, y) + zf), -8.0f, 7.0f);
            const float c = q - zf;
            num = __builtin_fmaf(wf[j], c, num);
            den = __builtin_fmaf(c, c, den);
        }
        if (den > 0.0f) s = num / den;
    }
    *out_z = (int)clampf(rintf(-lo / s) - 8.0f, -8.0f, 7.0f);
    uint16_t sh = __builtin_bit_cast(uint16_t, (_Float16)s);
    sh = (uint16_t)((sh + 8u) & 0xFFF0u);
    return sh;
}

// Fit N weights and return their scale word; their 4-bit codes go to q4.
template <int N>
__device__ __forceinline__ uint16_t quant_int4(const float *wf, bool safe, uint32_t *q4) {
    int z = 0;
    const uint16_t sh = safe ? fit_int4_asym<N, true>(wf, &z) : fit_int4_asym<N, false>(wf, &z);
    const float gs = half_bits_to_float(sh), zf = (float)z;
    if (safe && safe_half(gs)) {
        const float y = 1.0f / gs;
#pragma unroll
        for (int j = 0; j < N; ++j)
            q4[j] = (uint32_t)(int)clampq<true>(rintf(quot<true>(wf[j], gs, y) + zf), -8.0f, 7.0f) & 0xFu;
    } else {
#pragma unroll
        for (int j = 0; j < N; ++j) q4[j] = (uint32_t)(int)clampf(rintf(wf[j] / gs + zf), -8.0f, 7.0f) & 0xFu;
    }
    return (uint16_t)(sh | (z & 0xF));
}

// The four packed dwords of one K32 unit of a row: dword u of lane groups
// gl = 0..3 (k = 32u + 8gl + b, b = 0..3 low nibbles, 4..7 high).
__device__ __forceinline__ void store_unit(uint32_t *__restrict__ tile, int n, int u, const uint32_t *q4) {
#pragma unroll
    for (int gl = 0; gl < 4; ++gl) {
        uint32_t w = 0;
#pragma unroll
        for (int b = 0; b < 4; ++b) w |= (q4[8 * gl + b] | (q4[8 * gl + b + 4] << 4)) << (8 * b);
        tile[(n + 16 * gl) * 4 + u] = w;
    }
}

// GROUP 32 or 64: a thread's group is one or two whole K32 units. GROUP 16
// (mode 1, the K16 tier, kernels_dpas.cpp:287-296): a thread fits the two
// halves of one K32 unit.
template <int GROUP>
__global__ __launch_bounds__(256) void repack_e2m3_kernel(const uint8_t *__restrict__ payload,
                                                          const float *__restrict__ bs, int scale_cols, int M, int K,
                                                          uint32_t *__restrict__ out_codes,
                                                          uint16_t *__restrict__ out_scales) {
    constexpr int SPAN = GROUP < 32 ? 32 : GROUP, UNITS = SPAN / 32;
    const int SG = K / SPAN, Kt = K / 32, NT = K / kTileK;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * SG) return;
    const int n = (int)(i & 15);
    const size_t rgg = i >> 4;                               // row-group * SG + span
    const int mt = (int)(rgg / SG), g = (int)(rgg - (size_t)mt * SG);
    float wf[SPAN];
    bool safe = true;
#pragma unroll
    for (int v = 0; v < UNITS; ++v) {
        const int kt = g * UNITS + v;
        const float b = bs[(size_t)(mt >> 3) * scale_cols + (scale_cols == Kt ? kt : kt >> 2)];
        safe = safe && safe_scale(b);
        e2m3_unit(payload, (size_t)mt * Kt + kt, n, b, wf + 32 * v);
    }
    uint32_t q4[SPAN];
    if constexpr (GROUP < 32) {
#pragma unroll
        for (int h = 0; h < 2; ++h)
            out_scales[((size_t)mt * 2 * Kt + 2 * g + h) * 16 + n] = quant_int4<16>(wf + 16 * h, safe, q4 + 16 * h);
    } else {
        out_scales[((size_t)mt * SG + g) * 16 + n] = quant_int4<GROUP>(wf, safe, q4);
    }
#pragma unroll
    for (int v = 0; v < UNITS; ++v) {
        const int kt = g * UNITS + v;
        store_unit(out_codes + ((size_t)mt * NT + (kt >> 2)) * 256, n, kt & 3, q4 + 32 * v);
    }
}

// ---- the W8A8 tier (kernels_dpas.cpp:346-399, 558-575) --------------------
//
// W8 tile (16 rows x 128 K, 2048 bytes): half h at byte 1024h; lane l owns
// bytes [1024h + 16l, +16), row l%16, holding K32 unit j = 2h (bytes 0..7)
// and j = 2h + 1 (bytes 8..15); byte b of a unit is k = 32j + 8(l/16) + b.
// So one 16-byte load per lane and half is the operand of two K32 MFMAs,
// with the same K slots the W4 unpack produces.
__device__ __forceinline__ DwordCoord dword_coord_s8(int d) {
    const int h = d >> 8, lane = (d >> 2) & 63, e = d & 3;
    return {lane & 15, 32 * (2 * h + (e >> 1)) + 8 * (lane >> 4) + 4 * (e & 1)};
}

__global__ void pack_s8_kernel(const int8_t *__restrict__ codes, int M, int K, uint32_t *__restrict__ out) {
    const size_t total = (size_t)M * K / 4;
    const size_t d = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= total) return;
    const int NT = K / kTileK;
    const size_t tile = d >> 9;
    const DwordCoord c = dword_coord_s8((int)(d & 511));
    const int rg = (int)(tile / NT), kb = (int)(tile % NT);
    const int8_t *src = codes + (size_t)(rg * 16 + c.row) * K + kb * kTileK + c.k0;
    uint32_t w = 0;
#pragma unroll
    for (int b = 0; b < 4; ++b) w |= ((uint32_t)(uint8_t)src[b]) << (8 * b);
    out[d] = w;
}

__global__ void unpack_s8_kernel(const uint32_t *__restrict__ in, int M, int K, int8_t *__restrict__ codes) {
    const size_t total = (size_t)M * K / 4;
    const size_t d = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (d >= total) return;
    const int NT = K / kTileK;
    const size_t tile = d >> 9;
    const DwordCoord c = dword_coord_s8((int)(d & 511));
    const int rg = (int)(tile / NT), kb = (int)(tile % NT);
    int8_t *dst = codes + (size_t)(rg * 16 + c.row) * K + kb * kTileK + c.k0;
    const uint32_t w = in[d];
#pragma unroll
    for (int b = 0; b < 4; ++b) dst[b] = (int8_t)(w >> (8 * b));
}

// w8_repack_kernel's fit with the least-squares sums as fused multiply-adds:
// s = max(hi/127, neg/128), two refinements, FP16 by round to nearest even.
template <bool SAFE>
__device__ __forceinline__ uint16_t fit_int8(const float *wf) {
    float hi = 0.0f, neg = 0.0f;
#pragma unroll
    for (int j = 0; j < 32; ++j) {
        hi = fmaxf(hi, wf[j]);
        neg = fmaxf(neg, -wf[j]);
    }
    float s = fmaxf(hi / 127.0f, neg / 128.0f);
    if (!(s > 0.0f)) s = 1.0f;
#pragma unroll 1
    for (int iter = 0; iter < 2; ++iter) {
        const float y = 1.0f / s;
        float num = 0.0f, den = 0.0f;
#pragma unroll
        for (int j = 0; j < 32; ++j) {
            const float q = clampq<SAFE>(rintf(quot<SAFE>(wf[j], s, y)), -128.0f, 127.0f);
            num = __builtin_fmaf(wf[j], q, num);
            den = __builtin_fmaf(q, q, den);
        }
        if (den > 0.0f) s = num / den;
    }
    return __builtin_bit_cast(uint16_t, (_Float16)s);
}

// One thread per (row, K32), rows of a row-group fastest (as the int4 repack
// above, which says what bounds it): decode, fit, write the unit's 8 dwords
// (two per lane group, one 8-byte store) and its tiled FP16 scale.
__global__ __launch_bounds__(256) void repack_e2m3_s8_kernel(const uint8_t *__restrict__ payload,
                                                             const float *__restrict__ bs, int scale_cols, int M, int K,
                                                             uint32_t *__restrict__ out_codes,
                                                             uint16_t *__restrict__ out_scales) {
    const int Kt = K / 32, NT = K / kTileK;
    const size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= (size_t)M * Kt) return;
    const int n = (int)(i & 15);
    const size_t unit = i >> 4;                              // row-group * Kt + K32 tile
    const int mt = (int)(unit / Kt), kt = (int)(unit - (size_t)mt * Kt);
    const float b = bs[(size_t)(mt >> 3) * scale_cols + (scale_cols == Kt ? kt : kt >> 2)];
    const bool safe = safe_scale(b);
    float wf[32];
    e2m3_unit(payload, unit, n, b, wf);
    const uint16_t sh = safe ? fit_int8<true>(wf) : fit_int8<false>(wf);
    out_scales[unit * 16 + n] = sh;
    const float st = half_bits_to_float(sh);
    uint32_t w[8] = {};
    if (safe && safe_half(st)) {
        const float y = 1.0f / st;
#pragma unroll
        for (int j = 0; j < 32; ++j)
            w[j >> 2] |= (uint32_t)(uint8_t)(int)clampq<true>(rintf(quot<true>(wf[j], st, y)), -128.0f, 127.0f) << (8 * (j & 3));
    } else {
#pragma unroll
        for (int j = 0; j < 32; ++j)
            w[j >> 2] |= (uint32_t)(uint8_t)(int)clampf(rintf(wf[j] / st), -128.0f, 127.0f) << (8 * (j & 3));
    }
    const int j = kt & 3;
    uint32_t *tile = out_codes + ((size_t)mt * NT + (kt >> 2)) * 512 + 256 * (j >> 1);
#pragma unroll
    for (int gl = 0; gl < 4; ++gl) {
        v2u o;
        o.x = w[2 * gl];
        o.y = w[2 * gl + 1];
        *reinterpret_cast<v2u *>(tile + (n + 16 * gl) * 4 + 2 * (j & 1)) = o;
    }
}

static inline unsigned blocks_for(size_t n, int bs) { return (unsigned)((n + bs - 1) / bs); }

int launch_pack_s8(const int8_t *codes, const uint16_t *scales, int M, int K, uint8_t *out_codes,
                   uint16_t *out_scales, hipStream_t st) {
    const size_t nd = (size_t)M * K / 4, ns = (size_t)M * (K / 32);
    hipLaunchKernelGGL(pack_s8_kernel, dim3(blocks_for(nd, 256)), dim3(256), 0, st, codes, M, K,
                       reinterpret_cast<uint32_t *>(out_codes));
    hipLaunchKernelGGL(scales_to_tiled_kernel, dim3(blocks_for(ns, 256)), dim3(256), 0, st, scales, M,
                       K / 32, out_scales);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

int launch_unpack_s8(const uint8_t *codes, const uint16_t *scales, int M, int K, int8_t *out_codes,
                     uint16_t *out_scales, hipStream_t st) {
    const size_t nd = (size_t)M * K / 4, ns = (size_t)M * (K / 32);
    hipLaunchKernelGGL(unpack_s8_kernel, dim3(blocks_for(nd, 256)), dim3(256), 0, st,
                       reinterpret_cast<const uint32_t *>(codes), M, K, out_codes);
    if (out_scales)
        hipLaunchKernelGGL(scales_to_natural_kernel, dim3(blocks_for(ns, 256)), dim3(256), 0, st, scales,
                           M, K / 32, out_scales);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

int launch_repack_e2m3_s8(const uint8_t *payload, const float *bs, int scale_cols, int M, int K,
                          uint8_t *out_codes, uint16_t *out_scales, hipStream_t st) {
    const size_t n = (size_t)M * (K / 32);
    hipLaunchKernelGGL(repack_e2m3_s8_kernel, dim3(blocks_for(n, 256)), dim3(256), 0, st, payload, bs,
                       scale_cols, M, K, reinterpret_cast<uint32_t *>(out_codes), out_scales);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

int launch_pack(const int8_t *codes, const uint16_t *scales, int M, int K, int group,
                uint8_t *out_codes, uint16_t *out_scales, hipStream_t st) {
    const size_t nd = (size_t)M * K / 8, ns = (size_t)M * (K / group);
    hipLaunchKernelGGL(pack_codes_kernel, dim3(blocks_for(nd, 256)), dim3(256), 0, st, codes, M,
                       K, reinterpret_cast<uint32_t *>(out_codes));
    hipLaunchKernelGGL(scales_to_tiled_kernel, dim3(blocks_for(ns, 256)), dim3(256), 0, st,
                       scales, M, K / group, out_scales);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

int launch_unpack(const uint8_t *codes, const uint16_t *scales, int M, int K, int group,
                  int8_t *out_codes, uint16_t *out_scales, hipStream_t st) {
    const size_t nd = (size_t)M * K / 8, ns = (size_t)M * (K / group);
    hipLaunchKernelGGL(unpack_codes_kernel, dim3(blocks_for(nd, 256)), dim3(256), 0, st,
                       reinterpret_cast<const uint32_t *>(codes), M, K, out_codes);
    if (out_scales)
        hipLaunchKernelGGL(scales_to_natural_kernel, dim3(blocks_for(ns, 256)), dim3(256), 0, st,
                           scales, M, K / group, out_scales);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

int launch_import_ref(const uint8_t *ref_codes, const uint16_t *ref_scales, int M, int K,
                      int group, uint8_t *out_codes, uint16_t *out_scales, hipStream_t st) {
    const size_t nd = (size_t)M * K / 8, ns = (size_t)M * (K / group);
    hipLaunchKernelGGL(import_ref_codes_kernel, dim3(blocks_for(nd, 256)), dim3(256), 0, st,
                       ref_codes, M, K, reinterpret_cast<uint32_t *>(out_codes));
    if (hipMemcpyAsync(out_scales, ref_scales, ns * sizeof(uint16_t), hipMemcpyDeviceToDevice,
                       st) != hipSuccess)
        return -6;
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

int launch_repack_e2m3(const uint8_t *payload, const float *bs, int scale_cols, int M, int K,
                       int group, uint8_t *out_codes, uint16_t *out_scales, hipStream_t st) {
    const size_t n = (size_t)M * (K / std::max(group, 32));
    auto k = group == 16 ? repack_e2m3_kernel<16> : group == 32 ? repack_e2m3_kernel<32> : repack_e2m3_kernel<64>;
    hipLaunchKernelGGL(k, dim3(blocks_for(n, 256)), dim3(256), 0, st, payload, bs, scale_cols, M, K,
                       reinterpret_cast<uint32_t *>(out_codes), out_scales);
    return hipGetLastError() == hipSuccess ? 0 : -6;
}

}  // namespace kxw4
