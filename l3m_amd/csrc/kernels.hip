// HIP kernels for the batch-1 decode hot path on CDNA4 (gfx950), and their launchers.
//
// Matrix-vector products read weights in the lane-tile layout (host.h): a workgroup of 4 wavefronts
// owns up to 4 tiles of 16 output rows; inside a wavefront lane = 16*sub + row, and the 4 subs walk
// consecutive 32-input blocks, so each step of a wavefront is one contiguous 1-4 KiB run of 128-bit
// loads. The activation vector is prepared once per workgroup into LDS (l3m's per-32-block int8
// quantization, or bf16, or f32) and broadcast from there. Per-block integer dots use v_dot4_i32_i8;
// q4_0 nibbles go to v_dot8 as they are stored; mxfp4 e2m1 codes convert to f16 for v_dot2 in the decode
// step, and go as they are stored to the matrix cores (fp4 operand) in the large standalone matvecs.
// Reductions are fixed-order (wavefront shuffles, then LDS), so results are run-to-run identical.
#include <hip/hip_runtime.h>
#include <hip/hip_ext.h>
#include <math.h>
#include <pthread.h>
#include <stdint.h>
#include <stdio.h>
#include <stdlib.h>
#include <string.h>
#include <type_traits>
#include "dev.h"
#include "format.h"

namespace {

constexpr int RT = 16;    // rows per tile
constexpr int NT = 256;   // threads per workgroup

__host__ __device__ constexpr int qbytes(int dt) { return dt == L3M_F32 ? 128 : dt == L3M_BF16 ? 64 : dt == L3M_Q8_0 ? 32 : 16; }
__host__ __device__ constexpr int sbytes(int dt) { return dt == L3M_Q8_0 || dt == L3M_Q4_0 ? 2 : dt == L3M_MXFP4 ? 1 : 0; }
__host__ __device__ constexpr bool quantized(int dt) { return dt >= L3M_Q8_0; }
__host__ __device__ inline int kpad(int k) { return (k + 31) & ~31; }
// The prepared input of the wide matrices (q/k/v, gate/up, head) is padded to whole slots of 4 blocks with
// zero values, scales and sums, so the tile form reads the 4 blocks of every slot unconditionally.
__host__ __device__ inline int kwide(int k) { return (k + 127) & ~127; }
// A prepared activation (l3m_vec_prepare's values, pack.c:101-123) in the form the matvec of a dtype reads:
//   q8_0   per 32-block the 32 int8 values q
//   q4_0   per 32-block 16 bytes of high nibbles h = q >> 4 and 16 of low nibbles l = q & 15, dword k of each
//          pairing values 4k + i (nibble 2i) and 4k + i + 16 (nibble 2i + 1), as a q4_0 weight dword pairs its
//          inputs (its byte j holds inputs j and j + 16)
//   mxfp4  per 32-block 16 f16 pairs (q[j], q[j + 16]), as a code byte's two e2m1 values convert
// then the nb block scales (f32) and the nb block sums (int32: the sum of q, for q4_0 the sum of l); bf16
// and f32 activations are plain vectors.
__host__ __device__ constexpr int act_qbytes(int dt) { return dt == L3M_MXFP4 ? 64 : 32; }
__host__ __device__ inline size_t act_size(int dt, int k) {
    const int kp = kpad(k);
    return quantized(dt) ? (size_t)act_qbytes(dt) * (kp / 32) + 8 * (size_t)(kp / 32) : dt == L3M_BF16 ? 2 * (size_t)kp : 4 * (size_t)kp;
}
// The standalone prepared activation (l3m_k_prep, l3m_k_gemv): the same, and for mxfp4 then per 32-block the
// values' exact fp8 (e4m3) parts h = floor(q / 16) and l = q - 16 h, 32 bytes each in the f16 pairs' element
// order (the form the matrix-core matvec reads, k_gemv_mx).
__host__ __device__ inline size_t act_bytes(int dt, int k) { return act_size(dt, k) + (dt == L3M_MXFP4 ? (size_t)64 * (kpad(k) / 32) : 0); }
__host__ __device__ inline size_t align16(size_t n) { return (n + 15) & ~(size_t)15; }

// Reads through explicit global (address space 1) pointers: pointers taken from descriptors in device
// memory would otherwise be flat, and flat loads also count against the LDS wait counter, so every LDS
// barrier would wait for the weight stream in flight.
#define GLOBAL __attribute__((address_space(1)))
template <class T> __device__ __forceinline__ const GLOBAL T *gp(const void *p) { return (const GLOBAL T *)p; }
// Stores through explicit global pointers too: a flat store also counts against the LDS counter, so the
// next barrier would wait for it to reach memory.
template <class T> __device__ __forceinline__ GLOBAL T *gw(T *p) { return (GLOBAL T *)p; }
typedef unsigned u32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned u32x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint4 ldg16(const void *p, size_t i) {
    const u32x4 v = gp<u32x4>(p)[i];
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ float4 ldg16f(const void *p, size_t i) {
    const f32x4 v = gp<f32x4>(p)[i];
    return make_float4(v.x, v.y, v.z, v.w);
}
// Device-scope cache policy (sc1) of a buffer access: a load sees the newest data in this XCD's L2 or
// in memory, never a stale clean copy; a store writes through to memory.
constexpr int SC1 = 16;
// A raw buffer over p (a workgroup-uniform base): 16-byte accesses at a per-lane byte offset, with the
// cache policy the global instructions cannot take from C++.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf(const void *p) {
    return __builtin_amdgcn_make_buffer_rsrc((void *)p, 0, 0x7FFFFFFF, 0x00020000);
}
// 16 bytes that another workgroup wrote during this kernel, element i of a uniform base p: one
// device-coherent load (it reads past any stale copy in this XCD's L2, so no cache-wide invalidation is
// needed to see the data).
__device__ __forceinline__ uint4 ldcoh16(const void *p, size_t i) {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(buf(p), (uint32_t)(16 * i), 0, SC1));
    return make_uint4(v.x, v.y, v.z, v.w);
}
// 16 bytes stored through to memory (for readers on another XCD), element i of a uniform base p.
__device__ __forceinline__ void stcoh16(void *p, size_t i, float4 x) {
    const u32x4 v = {__float_as_uint(x.x), __float_as_uint(x.y), __float_as_uint(x.z), __float_as_uint(x.w)};
    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(__attribute__((ext_vector_type(4))) unsigned, v), buf(p), (uint32_t)(16 * i), 0, SC1);
}
__device__ __forceinline__ void stcoh4(void *p, size_t i, float x) {
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(x), buf(p), (uint32_t)(4 * i), 0, SC1);
}
// Element i of a weight plane p (a uniform base, under 2 GiB), or zeros with no memory access when ok is
// false: the offset of a load that is not wanted lies past the buffer's range, which the hardware answers
// with zeros and no request. A wavefront's loads for tiles or pairs past a matrix's end then cost no cache or
// memory bandwidth, and no branch ties a load to its use (a branch around loads would make the compiler
// merge the loaded registers where the branches join, and wait for the loads there).
constexpr uint32_t OOB = 0x80000000u;
__device__ __forceinline__ uint4 ldg16_if(const void *p, size_t i, bool ok) {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(buf(p), ok ? (uint32_t)(16 * i) : OOB, 0, 0));
    return make_uint4(v.x, v.y, v.z, v.w);
}
__device__ __forceinline__ uint32_t ldg2_if(const void *p, size_t i, bool ok) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(buf(p), ok ? (uint32_t)(2 * i) : OOB, 0, 0);
}
__device__ __forceinline__ uint32_t ldg1_if(const void *p, size_t i, bool ok) {
    return (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(buf(p), ok ? (uint32_t)i : OOB, 0, 0);
}
template <bool COH> __device__ __forceinline__ uint4 ld16(const void *p, size_t i) { return COH ? ldcoh16(p, i) : ldg16(p, i); }
// Element i of a uniform base p, or zeros with no memory access when ok is false (the offset past the
// buffer's range): a load that needs no branch around it.
template <bool COH> __device__ __forceinline__ uint4 ld16_if(const void *p, uint32_t byte, bool ok) {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(buf(p), ok ? byte : OOB, 0, COH ? SC1 : 0));
    return make_uint4(v.x, v.y, v.z, v.w);
}
template <bool COH> __device__ __forceinline__ float4 ld16f_if(const void *p, size_t i, bool ok) {
    const u32x4 v = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(buf(p), ok ? (uint32_t)(16 * i) : OOB, 0, COH ? SC1 : 0));
    return make_float4(__uint_as_float(v.x), __uint_as_float(v.y), __uint_as_float(v.z), __uint_as_float(v.w));
}
template <bool COH> __device__ __forceinline__ float4 ld16f(const void *p, size_t i) {
    if constexpr (COH) {
        const uint4 u = ldcoh16(p, i);
        return make_float4(__uint_as_float(u.x), __uint_as_float(u.y), __uint_as_float(u.z), __uint_as_float(u.w));
    }
    return ldg16f(p, i);
}

// ------------------------------------------------------------------------------------------ scalars

__device__ __forceinline__ float f16_f32(uint32_t h) { return (float)__builtin_bit_cast(_Float16, (uint16_t)h); }
__device__ __forceinline__ float bf16_f32(uint32_t h) { return __uint_as_float(h << 16); }
__device__ __forceinline__ uint16_t f32_bf16(float f) {       // nearest even, as the reference (ops.h:6)
    const uint32_t u = __float_as_uint(f);
    return (uint16_t)((u + 0x7FFFu + ((u >> 16) & 1u)) >> 16);
}
// 2^(e-128): the mxfp4 block scale 2^(e-127)/2, exact; e < 2 gives an f32 subnormal.
__device__ __forceinline__ float e8m0_half(uint32_t e) {
    const int x = (int)e - 128;
    return x >= -126 ? __uint_as_float((uint32_t)(x + 127) << 23) : __uint_as_float(1u << (x + 149));
}
__device__ __forceinline__ int dot4(uint32_t a, int b, int c) { return __builtin_amdgcn_sdot4((int)a, b, c, false); }

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float dot2bf(uint32_t a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));
__device__ __forceinline__ float fdot2h(f16x2 a, uint32_t b, float c) {
    return __builtin_amdgcn_fdot2(a, __builtin_bit_cast(f16x2, b), c, false);
}

// Elements i..i+3 (i a multiple of 4) of row r of a lane-tile matrix, exactly dequantized (the
// reference's dequant_row, pack.c:55-62): one block, loaded together.
__device__ float4 lt_elem4(const l3m_dmat &m, int r, int i) {
    const size_t slot = ((size_t)(r >> 4) * m.nb + (i >> 5)) * RT + (r & 15);
    const int j = i & 31;
    switch (m.dtype) {
    case L3M_F32: return ldg16f(m.q, slot * 8 + (j >> 2));
    case L3M_BF16: {
        const u32x2 v = gp<u32x2>(m.q)[slot * 8 + (j >> 2)];      // 32 bf16 = 8 x 8 bytes per slot
        return make_float4(bf16_f32(v.x & 0xFFFF), bf16_f32(v.x >> 16), bf16_f32(v.y & 0xFFFF), bf16_f32(v.y >> 16));
    }
    case L3M_Q8_0: {
        const float d = f16_f32(gp<uint16_t>(m.s)[slot]);
        const uint32_t v = gp<uint32_t>(m.q)[slot * 8 + (j >> 2)];
        return make_float4(d * (float)(int8_t)v, d * (float)(int8_t)(v >> 8), d * (float)(int8_t)(v >> 16), d * (float)(int8_t)(v >> 24));
    }
    default: {
        const uint32_t b = gp<uint32_t>(m.q)[slot * 4 + ((j & 15) >> 2)], n = j < 16 ? b & 0x0F0F0F0Fu : (b >> 4) & 0x0F0F0F0Fu;
        if (m.dtype == L3M_Q4_0) {
            const float d = f16_f32(gp<uint16_t>(m.s)[slot]);
            return make_float4(d * (float)((int)(n & 15) - 8), d * (float)((int)(n >> 8 & 15) - 8), d * (float)((int)(n >> 16 & 15) - 8),
                               d * (float)((int)(n >> 24) - 8));
        }
        const float d = e8m0_half(gp<uint8_t>(m.s)[slot]);
        const int8_t e2m1x2[16] = {0, 1, 2, 3, 4, 6, 8, 12, 0, -1, -2, -3, -4, -6, -8, -12};
        return make_float4(d * (float)e2m1x2[n & 15], d * (float)e2m1x2[n >> 8 & 15], d * (float)e2m1x2[n >> 16 & 15], d * (float)e2m1x2[n >> 24]);
    }
    }
}

// ------------------------------------------------------------------------------- workgroup helpers

template <int N> __device__ __forceinline__ float lanes_sum(float v);   // cross-lane sums, below
template <int N> __device__ __forceinline__ float lanes_max(float v);
template <int N> __device__ __forceinline__ int lanes_sumi(int v);
template <int N> __device__ __forceinline__ int lanes_mini(int v);

// (value, index) maximum; ties and NaN go to the lower index, as the reference's strict '>' scan
// (engine.c:294, 300).
__device__ __forceinline__ void better(float &v, int &i, float v2, int i2) {
    if (v2 > v || (v2 == v && i2 < i) || (v != v && v2 == v2)) { v = v2; i = i2; }
}

typedef int i32x8 __attribute__((ext_vector_type(8)));
// Two fp8 (e4m3) bytes of a and b in the low (HI false) or high half of old.
template <bool HI> __device__ __forceinline__ uint32_t pk_fp8(float a, float b, uint32_t old) {
    return (uint32_t)__builtin_amdgcn_cvt_pk_fp8_f32(a, b, (int)old, HI);
}
// The integer activation q = 16 h + l of four f16 pairs (one 16-byte word of the mxfp4 form): h = floor(q / 16)
// in [-8, 7] and l in [0, 15] as fp8 bytes, both exact (e4m3 holds every integer up to 16), in the word's
// element order.
__device__ __forceinline__ void split_hl(uint4 w, u32x2 &h, u32x2 &l) {
    const uint32_t d[4] = {w.x, w.y, w.z, w.w};
    float hv[8], lv[8];
#pragma unroll
    for (int i = 0; i < 8; i++) {
        const float q = f16_f32(d[i >> 1] >> (16 * (i & 1)));
        hv[i] = floorf(q * 0.0625f);
        lv[i] = fmaf(-16.f, hv[i], q);
    }
    h.x = pk_fp8<true>(hv[2], hv[3], pk_fp8<false>(hv[0], hv[1], 0));
    h.y = pk_fp8<true>(hv[6], hv[7], pk_fp8<false>(hv[4], hv[5], 0));
    l.x = pk_fp8<true>(lv[2], lv[3], pk_fp8<false>(lv[0], lv[1], 0));
    l.y = pk_fp8<true>(lv[6], lv[7], pk_fp8<false>(lv[4], lv[5], 0));
}
// The lane holding values 4m..4m+3 of a 32-block (m = lane & 7) writes its share of the block's prepared
// form at blk (the block's bytes): P = its four int8 values packed, Pp = those of lane m + 4 (values
// 4m + 16 ..), used by lanes m < 4 only. Returns the lane's part of the block sum.
template <int DT>
__device__ __forceinline__ int put_block(uint8_t *blk, int m, uint32_t P, uint32_t Pp, int q0, int q1, int q2, int q3) {
    if constexpr (DT == L3M_Q4_0) {
        if (m < 4) {
            // byte i: nibble 0 this lane's value i, nibble 1 the partner's value i
            ((uint32_t *)blk)[m] = ((P >> 4) & 0x0F0F0F0Fu) | (Pp & 0xF0F0F0F0u);
            ((uint32_t *)blk)[4 + m] = (P & 0x0F0F0F0Fu) | ((Pp & 0x0F0F0F0Fu) << 4);
        }
        return (q0 & 15) + (q1 & 15) + (q2 & 15) + (q3 & 15);
    } else if constexpr (DT == L3M_MXFP4) {
        if (m < 4) {
            uint32_t d[4];
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const _Float16 lo = (_Float16)(float)(int8_t)(P >> (8 * i)), hi = (_Float16)(float)(int8_t)(Pp >> (8 * i));
                d[i] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | (uint32_t)__builtin_bit_cast(uint16_t, hi) << 16;
            }
            *(uint4 *)(blk + 16 * m) = make_uint4(d[0], d[1], d[2], d[3]);
        }
        return q0 + q1 + q2 + q3;
    } else {
        ((uint32_t *)blk)[m] = P;
        return q0 + q1 + q2 + q3;
    }
}

// ------------------------------------------------------------------------------------- matvec core

// One row-block: acc += (x.scale[b] * d) * (integer dot - offset * x.sum[b]) for the quantized dtypes
// (kernels_scalar.c:30-75), or the bf16 / f32 dot (kernels_scalar.c:9-28).
// The quantized dtypes from the block's own pointers: xq its values, xsp its scale, xsum its sum.
template <int DT>
__device__ __forceinline__ float block_fma_at(float acc, const uint4 *w, uint32_t sc, const uint8_t *xq, const float *xsp, const int *xsum);
template <int DT>
__device__ __forceinline__ float block_fma(float acc, const uint4 *w, uint32_t sc, const uint8_t *act, int kp, int b) {
    if constexpr (quantized(DT)) {
        const int nb = kp >> 5;
        return block_fma_at<DT>(acc, w, sc, act + (size_t)act_qbytes(DT) * b, (const float *)(act + act_qbytes(DT) * nb) + b,
                                (const int *)(act + act_qbytes(DT) * nb + 4 * nb) + b);
    } else if constexpr (DT == L3M_BF16) {
        const uint4 *xv = (const uint4 *)(act + b * 64);
#pragma unroll
        for (int v = 0; v < 4; v++) {
            const uint4 x = xv[v];
            acc = dot2bf(w[v].x, x.x, acc); acc = dot2bf(w[v].y, x.y, acc);
            acc = dot2bf(w[v].z, x.z, acc); acc = dot2bf(w[v].w, x.w, acc);
        }
        return acc;
    } else {
        const float4 *xv = (const float4 *)(act + b * 128);
#pragma unroll
        for (int v = 0; v < 8; v++) {
            const float4 x = xv[v];
            acc = fmaf(__uint_as_float(w[v].x), x.x, acc); acc = fmaf(__uint_as_float(w[v].y), x.y, acc);
            acc = fmaf(__uint_as_float(w[v].z), x.z, acc); acc = fmaf(__uint_as_float(w[v].w), x.w, acc);
        }
        return acc;
    }
}
template <int DT>
__device__ __forceinline__ float block_fma_at(float acc, const uint4 *w, uint32_t sc, const uint8_t *xq, const float *xsp, const int *xsum) {
    static_assert(quantized(DT), "block_fma_at: quantized dtypes");
    {
        const float xs = *xsp;
        if constexpr (DT == L3M_Q8_0) {
            const int4 *xv = (const int4 *)xq;
            const int4 x0 = xv[0], x1 = xv[1];
            int dot = 0;
            dot = dot4(w[0].x, x0.x, dot); dot = dot4(w[0].y, x0.y, dot);
            dot = dot4(w[0].z, x0.z, dot); dot = dot4(w[0].w, x0.w, dot);
            dot = dot4(w[1].x, x1.x, dot); dot = dot4(w[1].y, x1.y, dot);
            dot = dot4(w[1].z, x1.z, dot); dot = dot4(w[1].w, x1.w, dot);
            return fmaf(xs * f16_f32(sc), (float)dot, acc);
        } else if constexpr (DT == L3M_Q4_0) {
            // sum (n - 8) q over the block with q = 16 h + l: 16 * sum (n - 8) h (signed 4-bit dots, the
            // codes' top bits flipped make n - 8) + sum n l (unsigned 4-bit dots) - 8 * sum l
            // the unsigned dots start from -8 sum l (two's complement: the sums wrap exactly), so the block's
            // integer is one shift-and-add of the two chains; the block scale multiplies the f16 scale in
            // one mixed-precision fma (the same single rounding as the product of its f32 value)
            const uint4 *xv = (const uint4 *)xq;
            const uint4 h = xv[0], l = xv[1];
            const int lsum = *xsum;
            int dh = 0;
            unsigned dl = (unsigned)(-8 * lsum);
            dh = __builtin_amdgcn_sdot8((int)(w[0].x ^ 0x88888888u), (int)h.x, dh, false);
            dh = __builtin_amdgcn_sdot8((int)(w[0].y ^ 0x88888888u), (int)h.y, dh, false);
            dh = __builtin_amdgcn_sdot8((int)(w[0].z ^ 0x88888888u), (int)h.z, dh, false);
            dh = __builtin_amdgcn_sdot8((int)(w[0].w ^ 0x88888888u), (int)h.w, dh, false);
            dl = __builtin_amdgcn_udot8(w[0].x, l.x, dl, false);
            dl = __builtin_amdgcn_udot8(w[0].y, l.y, dl, false);
            dl = __builtin_amdgcn_udot8(w[0].z, l.z, dl, false);
            dl = __builtin_amdgcn_udot8(w[0].w, l.w, dl, false);
            const float sd = __builtin_fmaf(f16_f32(sc), xs, 0.0f);
            return fmaf(sd, (float)(int)(((unsigned)dh << 4) + dl), acc);
        } else {
            // each code byte's two e2m1 values, doubled, as f16 (exact), dotted with the (q[j], q[j + 16])
            // pairs in f32: every partial sum is an integer below 2^24, so the dot is exact
            const uint4 *xv = (const uint4 *)xq;
            float dot = 0.f;
            const uint32_t v[4] = {w[0].x, w[0].y, w[0].z, w[0].w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint4 x = xv[j];
                dot = fdot2h(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v[j], 2.0f, 0), x.x, dot);
                dot = fdot2h(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v[j], 2.0f, 1), x.y, dot);
                dot = fdot2h(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v[j], 2.0f, 2), x.z, dot);
                dot = fdot2h(__builtin_amdgcn_cvt_scalef32_pk_f16_fp4(v[j], 2.0f, 3), x.w, dot);
            }
            return fmaf(xs * e8m0_half(sc), dot, acc);
        }
    }
}

// One batch of a lane's blocks: U blocks of its row, 4 blocks apart (the quarter-wavefronts interleave).
template <int DT> constexpr int lane_batch() { return DT == L3M_F32 ? 1 : DT == L3M_BF16 ? 2 : DT == L3M_Q8_0 ? 4 : 8; }
template <int DT, int UB = lane_batch<DT>()> struct LaneBatch {
    static constexpr int QBY = qbytes(DT), SBY = sbytes(DT), NV = QBY / 16;
    static constexpr int U = UB;
    uint4 w[U][NV];
    uint32_t sc[U];
};
template <int DT, int UB>
__device__ __forceinline__ void lane_load(const l3m_dmat &m, int tile, int b, int b1, int lane, LaneBatch<DT, UB> &x) {
    using L = LaneBatch<DT, UB>;
    const size_t base = (size_t)tile * m.nb * RT + (lane & 15);
    const uint8_t *__restrict__ qp = m.q + base * L::QBY;
    const uint8_t *__restrict__ sp = L::SBY ? m.s + base * L::SBY : nullptr;
    // every load is issued (past b1 the index stays on block b1 - 1, b0 < b1): loads under a branch
    // would make the compiler wait for all of them where the branches join
#pragma unroll
    for (int u = 0; u < L::U; u++) {
        const int bb = min(b + 4 * u, b1 - 1);
        const uint4 *src = (const uint4 *)(qp + (size_t)bb * RT * L::QBY);
#pragma unroll
        for (int v = 0; v < L::NV; v++) x.w[u][v] = src[v];
        x.sc[u] = 0;
        if constexpr (L::SBY == 2) x.sc[u] = *(const uint16_t *)(sp + (size_t)bb * RT * 2);
        if constexpr (L::SBY == 1) x.sc[u] = sp[(size_t)bb * RT];
    }
}
// This lane's partial dot for row (lane & 15) of `tile`, over blocks b0 + sub, b0 + sub + 4, ... < b1.
// x: its first batch, already requested by the caller.
template <int DT, int UB>
__device__ __forceinline__ float lane_dot(const l3m_dmat &m, int tile, int b0, int b1, const uint8_t *act, int kp, int lane,
                                          LaneBatch<DT, UB> x) {
    constexpr int U = UB;
    float acc = 0.f;
    int b = b0 + (lane >> 4);
    for (;;) {
#pragma unroll
        for (int u = 0; u < U; u++)
            if (b + 4 * u < b1) acc = block_fma<DT>(acc, x.w[u], x.sc[u], act, kp, b + 4 * u);
        b += 4 * U;
        if (b >= b1) break;
        lane_load<DT>(m, tile, b, b1, lane, x);
    }
    return acc;
}

// 16-byte words of the activation each k_gemv thread holds in registers while its first weights load
constexpr int GEMV_ACT_REGS = 4;
// k_gemv's LDS: the prepared activation, then the wavefronts' sums (16 rows each).
__host__ __device__ inline size_t gemv_lds(int dt, int k) { return align16(act_size(dt, k)) + 4 * 64; }
constexpr size_t LDS_MAX = 65536;   // dynamic LDS per workgroup without opting in to more
// The inputs l3m_k_prep and l3m_k_gemv take: rows whose prepared form and f32 values fit LDS_MAX together (what one
// workgroup staging both holds; callers size by it, and k_gemv's own LDS is always less).
inline bool act_fits(int dt, int k) { return align16(act_size(dt, k)) + 4 * (size_t)kpad(k) + 576 <= LDS_MAX; }

int pick_split(int nb) { return nb >= 16 ? 4 : nb >= 8 ? 2 : 1; }

// ------------------------------------------------------------------------------------------ kernels

extern "C" __global__ void __launch_bounds__(NT) k_dummy() {}

// A plain streaming copy of n16 16-byte words: the known-size kernel that calibrates the HBM counters
// (FETCH_SIZE, WRITE_SIZE) against which the step kernels' traffic is read.
__global__ void __launch_bounds__(NT) k_copy(u32x4 *__restrict__ dst, const u32x4 *__restrict__ src, size_t n16) {
    for (size_t i = (size_t)blockIdx.x * NT + threadIdx.x; i < n16; i += (size_t)gridDim.x * NT) dst[i] = src[i];
}

// One streaming read of n16 16-byte words: the --cold eviction (engine.c:330-338). Read through L2 and the
// Infinity Cache, a buffer larger than the Infinity Cache leaves none of the weights in either. sink keeps
// the loads.
__global__ void __launch_bounds__(NT) k_evict(const u32x4 *__restrict__ buf, size_t n16, unsigned *sink) {
    u32x4 acc = {0u, 0u, 0u, 0u};
    for (size_t i = (size_t)blockIdx.x * NT + threadIdx.x; i < n16; i += (size_t)gridDim.x * NT) acc ^= gp<u32x4>(buf)[i];
    const unsigned v = acc.x ^ acc.y ^ acc.z ^ acc.w;
    if (v == 0x9E3779B9u) gw(sink)[0] = v;            // practically never: keeps the loads
}

// The read of the measured matvec roofline: every thread issues its four words (a grid's width apart;
// indices past the end clamped, their words not used) before using any, so a buffer of up to four words per
// thread is in flight at once. sink keeps the loads.
__global__ void __launch_bounds__(NT) k_read(const u32x4 *__restrict__ buf, size_t n16, unsigned *sink) {
    const size_t width = (size_t)gridDim.x * NT;
    u32x4 acc = {0u, 0u, 0u, 0u};
    for (size_t i0 = (size_t)blockIdx.x * NT + threadIdx.x; i0 < n16; i0 += 4 * width) {
        u32x4 v[4];
#pragma unroll
        for (int u = 0; u < 4; u++) v[u] = gp<u32x4>(buf)[min(i0 + u * width, n16 - 1)];
#pragma unroll
        for (int u = 0; u < 4; u++) acc ^= i0 + u * width < n16 ? v[u] : u32x4{0u, 0u, 0u, 0u};
    }
    const unsigned x = acc.x ^ acc.y ^ acc.z ^ acc.w;
    if (x == 0x9E3779B9u) gw(sink)[0] = x;            // practically never: keeps the loads
}

// Vectors at addresses aligned to their elements alone (callers' pointers) or not at all (a prepared activation):
// the hardware takes global accesses of any alignment.
typedef f32x4 f32x4_a4 __attribute__((aligned(4)));
typedef u32x4 u32x4_a1 __attribute__((aligned(1)));
typedef u32x2 u32x2_a1 __attribute__((aligned(1)));
typedef uint32_t u32_a1 __attribute__((aligned(1)));
// Elements i .. i + 3 of x, zeros from k on.
__device__ __forceinline__ float4 load4(const float *__restrict__ x, int i, int k) {
    if (i + 3 < k) {
        const f32x4 v = *(const f32x4_a4 *)(x + i);
        return make_float4(v.x, v.y, v.z, v.w);
    }
    return make_float4(i < k ? x[i] : 0.f, i + 1 < k ? x[i + 1] : 0.f, i + 2 < k ? x[i + 2] : 0.f, 0.f);
}

// The standalone activation prep (pack.c:101-123: per 32-block amax, inv = 127 / amax, q = rint(x * inv), scale =
// amax / 127, sum = sum(q), stored in the form the dtype's matvec reads (act_size); bf16 nearest even): a thread 4
// values, 8 threads a block, one load each and straight to memory at any alignment (put_block's forms, which the decode
// step keeps for aligned LDS: with one definition for both it compiled to 0.6% slower tokens), over as many workgroups
// as the vector fills. Bound by one kernel's latency: q4_0 4096 values 2.1 us; 7.0 in one workgroup through LDS, copied out byte by byte.
template <int DT>
__global__ void __launch_bounds__(NT) k_prep(const float *__restrict__ x, int k, uint8_t *__restrict__ out) {
    const int kp = kpad(k), i = 4 * (blockIdx.x * NT + threadIdx.x);
    const float4 v = load4(x, i, k);
    if constexpr (quantized(DT)) {
        const int nb = kp / 32, b = i >> 5, m = threadIdx.x & 7;
        const float am = lanes_max<8>(fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w))));
        const float inv = am > 0.f ? 127.0f / am : 0.f;
        const int q0 = (int)rintf(v.x * inv), q1 = (int)rintf(v.y * inv), q2 = (int)rintf(v.z * inv), q3 = (int)rintf(v.w * inv);
        const uint32_t P = (uint32_t)(q0 & 255) | (uint32_t)(q1 & 255) << 8 | (uint32_t)(q2 & 255) << 16 | (uint32_t)(q3 & 255) << 24;
        const uint32_t Pp = (uint32_t)__shfl_xor((int)P, 4);
        const int s = lanes_sumi<8>(DT == L3M_Q4_0 ? (q0 & 15) + (q1 & 15) + (q2 & 15) + (q3 & 15) : q0 + q1 + q2 + q3);
        if (i >= kp) return;                          // whole blocks of lanes
        uint8_t *blk = out + (size_t)b * act_qbytes(DT);
        if constexpr (DT == L3M_Q8_0) ((u32_a1 *)blk)[m] = P;
        if constexpr (DT == L3M_Q4_0) {
            if (m < 4) {                              // put_block's nibble planes
                ((u32_a1 *)blk)[m] = ((P >> 4) & 0x0F0F0F0Fu) | (Pp & 0xF0F0F0F0u);
                ((u32_a1 *)blk)[4 + m] = (P & 0x0F0F0F0Fu) | ((Pp & 0x0F0F0F0Fu) << 4);
            }
        }
        if constexpr (DT == L3M_MXFP4) {
            if (m < 4) {                              // a 16-byte word of f16 pairs, and its fp8 parts
                uint32_t d[4];
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    const _Float16 lo = (_Float16)(float)(int8_t)(P >> (8 * j)), hi = (_Float16)(float)(int8_t)(Pp >> (8 * j));
                    d[j] = (uint32_t)__builtin_bit_cast(uint16_t, lo) | (uint32_t)__builtin_bit_cast(uint16_t, hi) << 16;
                }
                u32x2 h, l;
                split_hl(make_uint4(d[0], d[1], d[2], d[3]), h, l);
                *(u32x4_a1 *)(blk + 16 * m) = u32x4{d[0], d[1], d[2], d[3]};
                uint8_t *o = out + act_size(DT, k) + 64 * (size_t)b + 8 * m;
                *(u32x2_a1 *)o = h;
                *(u32x2_a1 *)(o + 32) = l;
            }
        }
        if (m == 0) {
            *(u32_a1 *)(out + (size_t)act_qbytes(DT) * nb + 4 * (size_t)b) = __float_as_uint(am / 127.0f);
            *(u32_a1 *)(out + (size_t)(act_qbytes(DT) + 4) * nb + 4 * (size_t)b) = (uint32_t)s;
        }
    } else if (i < kp) {
        if constexpr (DT == L3M_BF16)
            *(u32x2_a1 *)(out + 2 * (size_t)i) = u32x2{(uint32_t)f32_bf16(v.x) | (uint32_t)f32_bf16(v.y) << 16, (uint32_t)f32_bf16(v.z) | (uint32_t)f32_bf16(v.w) << 16};
        else
            *(u32x4_a1 *)(out + 4 * (size_t)i) = u32x4{__float_as_uint(v.x), __float_as_uint(v.y), __float_as_uint(v.z), __float_as_uint(v.w)};
    }
}

// The reference's host tiles (kernels.h:1-11) as lane-tile planes, a thread per row of a block: per tile of 16 rows
// f32 [k][16]; bf16 [k/2][16][2]; quantized per 32 inputs the 16 scales, then bytes: q8 value + 128 at
// (i / 4 * 16 + row) * 4 + i % 4, q4 and mxfp4 inputs 8g + j (low nibble) and 8g + 4 + j (high) at
// (g * 16 + row) * 4 + j. The same bytes l3m_lt_pack_ltiles writes (2048 x 768 q8_0: 4.4 us, about 0.7 ms there).
template <int DT>
__global__ void __launch_bounds__(NT) k_ltiles(const uint8_t *__restrict__ src, int ntiles, int k, uint8_t *__restrict__ q, uint8_t *__restrict__ s) {
    const int nb = kpad(k) / 32, id = blockIdx.x * NT + threadIdx.x, c = id & 15, b = (id >> 4) % nb, t = (id >> 4) / nb;
    if (t >= ntiles) return;
    const size_t slot = (size_t)id;                   // (tile * nb + block) * 16 + row
    if constexpr (quantized(DT)) {
        constexpr int SB = DT == L3M_MXFP4 ? 16 : 32;
        const uint8_t *blk = src + ((size_t)t * nb + b) * (SB + 16 * qbytes(DT));
        const uint32_t *w = (const uint32_t *)(blk + SB) + c;
        if constexpr (DT == L3M_MXFP4) s[slot] = blk[c];
        else ((uint16_t *)s)[slot] = ((const uint16_t *)blk)[c];
        uint4 *o = (uint4 *)(q + slot * qbytes(DT));
        if constexpr (DT == L3M_Q8_0) {
            uint32_t d[8];
#pragma unroll
            for (int i = 0; i < 8; i++) d[i] = w[16 * i] ^ 0x80808080u;
            o[0] = make_uint4(d[0], d[1], d[2], d[3]);
            o[1] = make_uint4(d[4], d[5], d[6], d[7]);
        } else {
            const uint32_t d0 = w[0], d1 = w[16], d2 = w[32], d3 = w[48], L = 0x0F0F0F0Fu, H = 0xF0F0F0F0u;
            o[0] = make_uint4((d0 & L) | (d2 & L) << 4, (d0 >> 4 & L) | (d2 & H), (d1 & L) | (d3 & L) << 4, (d1 >> 4 & L) | (d3 & H));
        }
    } else if constexpr (DT == L3M_BF16) {
        const uint16_t *e = (const uint16_t *)(src + (size_t)t * k * 32);
        uint32_t *o = (uint32_t *)(q + slot * 64);
#pragma unroll
        for (int p = 0; p < 16; p++) {
            const int i = 32 * b + 2 * p;
            const size_t at = ((size_t)(i >> 1) * 16 + c) * 2;
            o[p] = (i < k ? (uint32_t)e[at] : 0u) | (i + 1 < k ? (uint32_t)e[at + 1] << 16 : 0u);
        }
    } else {
        const uint32_t *e = (const uint32_t *)(src + (size_t)t * k * 64);
        uint32_t *o = (uint32_t *)(q + slot * 128);
#pragma unroll
        for (int p = 0; p < 32; p++) {
            const int i = 32 * b + p;
            o[p] = i < k ? e[(size_t)i * 16 + c] : 0u;
        }
    }
}

// STAGED: the activation is 16-byte aligned and at most GEMV_ACT_REGS * NT 16-byte words (gemv_staged).
template <int DT, bool STAGED>
__global__ void __launch_bounds__(NT) k_gemv(l3m_dmat m, const uint8_t *__restrict__ act_g, int k, float *__restrict__ y, int S) {
    extern __shared__ __align__(16) uint8_t smem[];
    uint8_t *act = smem;
    float *red = (float *)(smem + align16(act_size(DT, k)));
    const int kp = kpad(k), tid = threadIdx.x, wave = tid >> 6, lane = tid & 63;
    // the workgroup's 4/S tiles from tile0, each split over S wavefronts along the inputs
    const int tpw = 4 / S, tile0 = blockIdx.x * tpw, tile = tile0 + wave / S, split = wave % S;
    const int b0 = split * m.nb / S, b1 = (split + 1) * m.nb / S;
    const bool live = tile < m.tiles;
    const int ltile = min(tile, m.tiles - 1);   // a wavefront past the last tile loads the last one and discards it
    const size_t bytes = act_size(DT, k);   // 40 bytes per 32 inputs when quantized: whole words, not whole uint4
    const int n16 = (int)(bytes / 16), ntail = (int)(bytes % 16) / 4;
    LaneBatch<DT> x;
    // b0 < b1 holds: pick_split gives every split at least one block. Every load below is issued
    // unconditionally: a load under a branch makes the compiler wait for all loads where the branches join.
    if constexpr (STAGED) {
        // The activation's loads go out first and the wavefront's first batch of weights right behind
        // them. Loads complete in order, so the activation reaches LDS while the weights are on the way.
        u32x4 a[GEMV_ACT_REGS];
        uint32_t at;
#pragma unroll
        for (int r = 0; r < GEMV_ACT_REGS; r++) a[r] = ((const u32x4 *)act_g)[min(tid + r * NT, n16 - 1)];   // clamped
        at = ((const uint32_t *)act_g)[4 * n16 - 1 + min(tid + 1, ntail)];   // tail word tid, or a word in range
        lane_load<DT>(m, ltile, b0 + (lane >> 4), b1, lane, x);
        // clamped slots are written by several threads, with the same value
#pragma unroll
        for (int r = 0; r < GEMV_ACT_REGS; r++) ((u32x4 *)act)[min(tid + r * NT, n16 - 1)] = a[r];
        ((uint32_t *)act)[4 * n16 - 1 + min(tid + 1, ntail)] = at;
    } else {
        for (size_t i = tid; i < bytes / 4; i += NT) ((uint32_t *)act)[i] = ((const uint32_t *)act_g)[i];
        lane_load<DT>(m, ltile, b0 + (lane >> 4), b1, lane, x);
    }
    __syncthreads();
    float acc = lane_dot<DT>(m, ltile, b0, b1, act, kp, lane, x);
    if (!live) acc = 0.f;
    acc += __shfl_xor(acc, 16);
    acc += __shfl_xor(acc, 32);
    if (lane < 16) red[wave * 16 + lane] = acc;
    __syncthreads();
    if (tid < tpw * 16) {
        const int tt = tid >> 4, r = tid & 15, row = (tile0 + tt) * RT + r;
        float v = red[(tt * S) * 16 + r];
        for (int sp = 1; sp < S; sp++) v += red[(tt * S + sp) * 16 + r];
        if (row < m.rows) y[row] = v;
    }
}

// One query head over positions 0..n-1 (ops.c:58-73): scores q.K[t] / sqrt(hd), softmax, sum of p[t] V[t]. K, V
// rows are `stride` elements apart.
//
// Groups of L lanes (the power of two from hd / 8 on) take a row each, 16 bytes a lane, ATT_U rows a batch with
// every K and V load of the batch issued before the scores, and keep a running maximum, sum and output of their
// own; nothing crosses a group before the end. The groups meet by shuffles and LDS, and the workgroups' parts (`per` rows each)
// in ws: the last workgroup to finish (a device-scope count) adds them in order, so the result does not depend on
// which one that is. One launch, whatever n. Bound by latency: two loads deep, then the hand-over between the
// workgroups. 4001 rows of 128 (2 MB): 12.9 us in
// 63 workgroups, 60.9 in one; 229 in one workgroup of a thread per row (dependent 16-byte and 2-byte loads).
constexpr int ATT_U = 4, ATT_SPLITS = 64, ATT_PART = 256 + 8;   // rows a group loads at once; workgroups; floats of a part
constexpr size_t ATT_WS = 256 + (size_t)4 * ATT_SPLITS * ATT_PART;   // the count, then the parts [max, sum, .., hd outputs]
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));             // V rows need no alignment beyond an element's
template <int L>
__global__ void __launch_bounds__(NT) k_attend(float *__restrict__ out, const float *__restrict__ q, const uint16_t *__restrict__ kc,
                                               const uint16_t *__restrict__ vc, int n, int hd, int stride, int per, uint8_t *ws) {
    constexpr int ROWS = NT / L * ATT_U, W = NT / 64;             // rows of a workgroup's batch; wavefronts
    __shared__ __align__(16) float o_s[W][ATT_PART];              // [8 + d]: a wavefront's outputs; [0], [1]: its maximum and sum
    __shared__ __align__(16) float sum_s[NT][4];
    __shared__ float f_s[ATT_SPLITS];
    __shared__ unsigned last;
    const int tid = threadIdx.x, grp = tid / L, d8 = tid % L, d0 = 8 * d8 < hd ? 8 * d8 : 0;
    const bool dl = 8 * d8 < hd;                                  // lanes past the head hold zeros
    const float scale = 1.0f / sqrtf((float)hd);
    float qv[8], o[8], m = -INFINITY, l = 0.f;
#pragma unroll
    for (int j = 0; j < 8; j++) { qv[j] = dl ? q[d0 + j] : 0.f; o[j] = 0.f; }
    const int t0 = blockIdx.x * per, t1 = min(t0 + per, n);
    for (int tb = t0; tb < t1; tb += ROWS) {
        uint4 kk[ATT_U];
        u32x4 vv[ATT_U];
#pragma unroll
        for (int u = 0; u < ATT_U; u++) {
            const size_t row = (size_t)min(tb + u * (NT / L) + grp, n - 1) * stride + d0;   // rows past the end: not used
            kk[u] = *(const uint4 *)(kc + row);
            vv[u] = *(const u32x4_a2 *)(vc + row);
        }
        float s[ATT_U], nm = m;
#pragma unroll
        for (int u = 0; u < ATT_U; u++) {
            float dot = 0.f;
            const uint32_t w[4] = {kk[u].x, kk[u].y, kk[u].z, kk[u].w};
#pragma unroll
            for (int j = 0; j < 4; j++) {
                dot = fmaf(qv[2 * j], dl ? bf16_f32(w[j] & 0xFFFF) : 0.f, dot);
                dot = fmaf(qv[2 * j + 1], dl ? bf16_f32(w[j] >> 16) : 0.f, dot);
            }
            for (int x = 1; x < L; x <<= 1) dot += __shfl_xor(dot, x);
            s[u] = tb + u * (NT / L) + grp < t1 ? dot * scale : -INFINITY;
            nm = fmaxf(nm, s[u]);
        }
        const float base = nm == -INFINITY ? 0.f : nm, r = expf(m - base);   // no row yet: every p is 0
        l *= r;
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] *= r;
#pragma unroll
        for (int u = 0; u < ATT_U; u++) {
            const float p = expf(s[u] - base);
            const bool ok = tb + u * (NT / L) + grp < t1;
            l += p;
#pragma unroll
            for (int j = 0; j < 4; j++) {
                const uint32_t w = ok ? vv[u][j] : 0u;
                o[2 * j] = fmaf(p, bf16_f32(w & 0xFFFF), o[2 * j]);
                o[2 * j + 1] = fmaf(p, bf16_f32(w >> 16), o[2 * j + 1]);
            }
        }
        m = nm;
    }
    // a part's factor at the common maximum: one without a row (or with no score above -infinity, sum 0) counts nothing
    auto meet = [](float mw, float mm) { return mw == -INFINITY ? 0.f : expf(mw - mm); };
    // the wavefront's groups, pairwise
#pragma unroll
    for (int x = L; x < 64; x <<= 1) {
        const float m2 = __shfl_xor(m, x), l2 = __shfl_xor(l, x), nm = fmaxf(m, m2), f = meet(m, nm), f2 = meet(m2, nm);
        l = l * f + l2 * f2;
#pragma unroll
        for (int j = 0; j < 8; j++) o[j] = o[j] * f + __shfl_xor(o[j], x) * f2;
        m = nm;
    }
    const int w = tid >> 6;
    if ((tid & 63) == 0) { o_s[w][0] = m; o_s[w][1] = l; }
    if ((tid & 63) < L && dl)
#pragma unroll
        for (int j = 0; j < 8; j++) o_s[w][8 + d0 + j] = o[j];
    __syncthreads();
    // the wavefronts in order, one thread a dim
    float mm = o_s[0][0], sum = 0.f, y = 0.f;
#pragma unroll
    for (int g = 1; g < W; g++) mm = fmaxf(mm, o_s[g][0]);
    if (tid < hd) {
#pragma unroll
        for (int g = 0; g < W; g++) {
            const float f = meet(o_s[g][0], mm);
            sum += o_s[g][1] * f;
            y += o_s[g][8 + tid] * f;
        }
    }
    if (gridDim.x == 1) {
        if (tid < hd) out[tid] = y / sum;
        return;
    }
    float *parts = (float *)(ws + 256), *part = parts + (size_t)blockIdx.x * ATT_PART;
    if (tid < hd) part[8 + tid] = y;
    if (tid == 0) { part[0] = mm; part[1] = sum; }
    __threadfence();
    __syncthreads();
    if (tid == 0) last = __hip_atomic_fetch_add((unsigned *)ws, 1u, __ATOMIC_ACQ_REL, __HIP_MEMORY_SCOPE_AGENT) == gridDim.x - 1;
    __syncthreads();
    if (!last) return;
    __threadfence();
    // thread (g, c): dims 4 c .. of parts g, g + ng, ..., the first 8 of them requested before the factors are known
    const int S = gridDim.x, h4 = hd >> 2, ng = NT / h4, g = tid / h4, c = tid - g * h4;
    float4 v[8];
#pragma unroll
    for (int i = 0; i < 8; i++) v[i] = *(const float4 *)(parts + (size_t)min(g + i * ng, S - 1) * ATT_PART + 8 + 4 * c);
    if (tid < 64) {                                               // S <= 64: a lane a part
        const float pm = parts[(size_t)min(tid, S - 1) * ATT_PART], pl = parts[(size_t)min(tid, S - 1) * ATT_PART + 1];
        float am = pm;
        for (int x = 32; x; x >>= 1) am = fmaxf(am, __shfl_xor(am, x));
        const float f = tid < S ? meet(pm, am) : 0.f;
        float al = tid < S ? pl * f : 0.f;
        for (int x = 32; x; x >>= 1) al += __shfl_xor(al, x);
        f_s[tid] = f;
        if (tid == 0) o_s[0][1] = al;
    }
    __syncthreads();
    float4 a = make_float4(0.f, 0.f, 0.f, 0.f);
    if (g < ng) {
        for (int p0 = g; p0 < S; p0 += 8 * ng) {
#pragma unroll
            for (int i = 0; i < 8; i++) {
                if (p0 + i * ng < S) {
                    const float f = f_s[p0 + i * ng];
                    a.x = fmaf(v[i].x, f, a.x); a.y = fmaf(v[i].y, f, a.y); a.z = fmaf(v[i].z, f, a.z); a.w = fmaf(v[i].w, f, a.w);
                }
                v[i] = *(const float4 *)(parts + (size_t)min(p0 + (8 + i) * ng, S - 1) * ATT_PART + 8 + 4 * c);
            }
        }
        *(float4 *)sum_s[tid] = a;
    }
    __syncthreads();
    if (tid < h4) {
        for (int i = 1; i < ng; i++) {
            const float4 b = *(const float4 *)sum_s[i * h4 + tid];
            a.x += b.x; a.y += b.y; a.z += b.z; a.w += b.w;
        }
        const float den = o_s[0][1];
        out[4 * tid] = a.x / den; out[4 * tid + 1] = a.y / den; out[4 * tid + 2] = a.z / den; out[4 * tid + 3] = a.w / den;
    }
    if (tid == 0) *(unsigned *)ws = 0;                            // for the stream's next call
}

// y = x * s * w with s = 1 / sqrt(sum x^2 / n + eps) (ops.c:13-18), one workgroup of a thread per 4 values (C of them
// each when n is past 4096), every load first. y may be x. 768 values 1.6 us; 4.1 with 256 threads staging x in
// LDS.
template <int C>
__global__ void __launch_bounds__(1024) k_rmsnorm(float *y, const float *x, const float *w, int n, float eps) {
    __shared__ float red[16];
    const int t = threadIdx.x, nt = blockDim.x, wave = t >> 6;
    float4 v[C], g[C];
    float ss = 0.f;
#pragma unroll
    for (int c = 0; c < C; c++) {
        v[c] = load4(x, 4 * (t + c * nt), n);
        g[c] = load4(w, 4 * (t + c * nt), n);
    }
#pragma unroll
    for (int c = 0; c < C; c++) ss += fmaf(v[c].x, v[c].x, v[c].y * v[c].y) + fmaf(v[c].z, v[c].z, v[c].w * v[c].w);
    ss = lanes_sum<64>(ss);
    if ((t & 63) == 0) red[wave] = ss;
    __syncthreads();
    float tot = 0.f;
    for (int i = 0; i < nt >> 6; i++) tot += red[i];
    const float s = 1.0f / sqrtf(tot / (float)n + eps);
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int i = 4 * (t + c * nt);
        const f32x4 o = {v[c].x * s * g[c].x, v[c].y * s * g[c].y, v[c].z * s * g[c].z, v[c].w * s * g[c].w};
        if (i + 3 < n) *(f32x4_a4 *)(y + i) = o;
        else
            for (int j = 0; j < 3; j++)
                if (i + j < n) y[i + j] = o[j];
    }
}

// Pairs (2i, 2i+1) of each head rotate by the table angle i (ops.c:29-40).
__device__ __forceinline__ float rope_one(float val, float partner, float c, float s, bool odd) {
    return odd ? partner * s + val * c : val * c - partner * s;
}

__global__ void __launch_bounds__(NT) k_rope(float *v, int n, int hd, const float *table) {
    const int r = blockIdx.x * NT + threadIdx.x;
    const float val = r < n ? v[r] : 0.f, partner = __shfl_xor(val, 1);
    if (r < n) {
        const int i = (r % hd) >> 1;
        v[r] = rope_one(val, partner, table[2 * i], table[2 * i + 1], r & 1);
    }
}

__device__ __forceinline__ float silu_mul(float up, float g) { return up * (g / (1.0f + expf(-g))); }

__global__ void __launch_bounds__(NT) k_silu_mul(float *h, const float *g, int n) {
    const int i = blockIdx.x * NT + threadIdx.x;
    if (i < n) h[i] = silu_mul(h[i], g[i]);
}

// The first maximum of x (engine.c:290-301): one workgroup of nt threads, each U x 4 values a round with every load
// first (16 bytes from the first aligned address on). Bound by latency: U = 1 holds one quad a thread, up to 4096
// values; past that 1024 threads and U = 12, and the quad with the largest value is read again for its place. Queued
// back to back, 1000 values 3.5 us (4.7 with 1024 threads of U = 12, 3.5 with 256 threads of 4-byte loads), 4096
// 3.5 (4.9, 5.0), 49152 3.8 (5.1, 35.2).
template <int U>
__global__ void __launch_bounds__(1024) k_argmax(const float *x, int n, int nt, int32_t *out) {
    __shared__ float sv[16];
    __shared__ int si[16];
    const int t = threadIdx.x, head = min((int)((16 - ((uintptr_t)x & 15)) & 15) >> 2, n), nq = (n - head) >> 2, tail = head + 4 * nq;
    float v = -INFINITY;
    int idx = 0x7FFFFFFF;
    // a value wins over an equal one by its lower index (and over the start, which no value is below); NaN never wins
    auto take = [&](float a, int i) {
        if (a > v || (a == v && i < idx)) { v = a; idx = i; }
    };
    auto take4 = [&](float4 a, int i) {
        take(a.x, i); take(a.y, i + 1); take(a.z, i + 2); take(a.w, i + 3);
    };
    if (t < head) take(x[t], t);
    const float4 *xq = (const float4 *)(x + head);
    if constexpr (U == 1) {
        if (t < nq) take4(xq[t], head + 4 * t);
    } else {
        // the thread's first quad with the largest value, then that value's place in it
        float vq = -INFINITY;
        int best = -1;
        for (int q0 = 0; q0 < nq; q0 += U * 1024) {
            float4 a[U];
#pragma unroll
            for (int u = 0; u < U; u++) a[u] = xq[min(q0 + u * 1024 + t, nq - 1)];   // past the end: the last again
#pragma unroll
            for (int u = 0; u < U; u++) {
                const float m = fmaxf(fmaxf(a[u].x, a[u].y), fmaxf(a[u].z, a[u].w));
                if (m > vq) { vq = m; best = min(q0 + u * 1024 + t, nq - 1); }
            }
        }
        if (best >= 0) {
            const float4 a = xq[best];
            take(vq, head + 4 * best + (a.x == vq ? 0 : a.y == vq ? 1 : a.z == vq ? 2 : 3));
        } else {                                      // nothing above -infinity: the first of those
            for (int q = t; q < nq; q += 1024) take4(xq[q], head + 4 * q);
        }
    }
    if (t < n - tail) take(x[tail + t], tail + t);
    // a wavefront's largest, then the lowest index that holds it; then the wavefronts' by the first of them
    float m = lanes_max<64>(v);
    int i = lanes_mini<64>(v == m ? idx : 0x7FFFFFFF);
    const int waves = nt >> 6;
    if (waves > 1) {
        if ((t & 63) == 0) { sv[t >> 6] = m; si[t >> 6] = i; }
        __syncthreads();
        if (t >= 64) return;
        v = t < waves ? sv[t] : -INFINITY;
        m = lanes_max<64>(v);
        i = lanes_mini<64>(t < waves && v == m ? si[t] : 0x7FFFFFFF);
    }
    if (t == 0) *out = i == 0x7FFFFFFF ? 0 : i;
}

// ------------------------------------------------------------------------------ decode step kernels
//
// Per layer: kernel A (one workgroup per head group) = norm + prep + qkv rows + RoPE + KV write +
// attention + the group's Wo column slice; kernel B (one workgroup per FFN chunk) = norm + prep + gate/up
// rows + SiLU + prep + the chunk's Wdown column slice. Each writes a partial residual (po, pd); the next
// kernel adds the partials in a fixed order, so results are run-to-run identical.
//
// Every one of the 16 wavefronts of a workgroup runs the same sequence: issue its share of the loads of
// the incoming partial residuals, then issue its share of the weights (nothing depends on them), then
// wait for the partials only (loads complete in order), build the normalized activation in LDS, and
// only then consume the weights. So the weight stream overlaps the prologue instead of following it.

constexpr int NTE = 1024, NWE = NTE / 64;

// The thread's index, read through an opaque move: values derived from it are then computed where they
// are used. Otherwise the compiler hoists every lane-dependent address out of the persistent kernel's
// layer and step loops and keeps them all live across it, which spills.
__device__ __forceinline__ int tidx() {
    int t;
    asm volatile("v_mov_b32 %0, %1" : "=v"(t) : "v"((int)threadIdx.x));
    return t;
}


// Weight slots per lane: a step kernel streams matrix A (qkv, gate/up, head rows) and matrix B (Wo,
// Wdown columns), each through its own register array; 64 (tile, block) pairs per slot and workgroup.
template <int DT> constexpr int nslot_a() { return DT == L3M_F32 ? 1 : DT == L3M_BF16 ? 2 : DT == L3M_Q8_0 ? 5 : 6; }
template <int DT> constexpr int nslot_b() { return DT == L3M_F32 ? 1 : DT == L3M_BF16 ? 1 : 3; }
// The attention block keeps its Wo slots live through the attention; q8_0 gives one up to stay in registers.
template <int DT> constexpr int nslot_wo() { return DT == L3M_Q8_0 || DT == L3M_Q4_0 ? 2 : nslot_b<DT>(); }
// The wide matrices (q/k/v rows, gate/up rows, the head) take the tile form (tile_rows) in the quantized
// dtypes, whose slot batch holds a whole row of the benchmark shapes (up to 24 blocks); bf16 takes the
// matrix cores (tile_rows_mfma: the v_dot2 tile form, with a third slot, measured 3% slower on stories15M
// than mv and rows_sum4), f32 mv and rows_sum4. The head's slots: one row's in the tile form.
template <int DT> constexpr bool tiled() { return quantized(DT); }
template <int DT> constexpr int nslot_h() { return tiled<DT>() ? nslot_a<DT>() : nslot_a<DT>() + nslot_b<DT>(); }

template <int DT, int NS>
struct Pref {
    uint4 w[NS][qbytes(DT) / 16];
    uint32_t sc[NS];
};

// Slot s of this lane holds pair p = (wave + (s0 + s) * NWE) * 4 + sub of m, a pair being (tile, block)
// = (p / nb, p % nb) and the lane reading row (lane & 15) of it: 4 consecutive pairs = one contiguous
// 64 * QBYTES run per wavefront. Loads are unconditional: past the end they return zeros with no memory
// access (ldg16_if). m has at least one pair.
// The wavefront index as a scalar (uniform) value, so index arithmetic on it runs on the scalar unit.
__device__ __forceinline__ int wave_id() { return __builtin_amdgcn_readfirstlane(tidx() >> 6); }

template <int DT, int NS>
__device__ __forceinline__ void pref_load(Pref<DT, NS> &pf, const l3m_dmat &m, int s0) {
    constexpr int QBY = qbytes(DT), SBY = sbytes(DT), NV = QBY / 16;
    const int wave = wave_id(), sub = (tidx() >> 4) & 3, row = tidx() & 15, n = m.tiles * m.nb;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int p = (wave + (s0 + s) * NWE) * 4 + sub;
        const bool ok = p < n;                        // pairs past the end: zeros, no memory access
        const size_t slot = (size_t)p * 16 + row;
#pragma unroll
        for (int v = 0; v < NV; v++) pf.w[s][v] = ldg16_if(m.q, slot * NV + v, ok);
        if constexpr (SBY == 2) pf.sc[s] = ldg2_if(m.s, slot, ok);
        if constexpr (SBY == 1) pf.sc[s] = ldg1_if(m.s, slot, ok);
        if constexpr (SBY == 0) pf.sc[s] = 0;
    }
}

// The tile form of a matrix: wavefront w takes tiles w, w + NWE, ... in turn, each in slots of 4 blocks
// of its 16 rows (lane quarter sub = lane / 16 takes blocks sub, sub + 4, ...), NS slots per batch.
// pref_load_tile loads slots j0 .. j0 + NS - 1 of tile t: 4 consecutive pairs per slot, as pref_load;
// blocks past nb and tiles past the end are zeros, with no memory access (not used).
template <int DT, int NS>
__device__ __forceinline__ void pref_load_tile(Pref<DT, NS> &pf, const l3m_dmat &m, int t, int j0) {
    constexpr int QBY = qbytes(DT), SBY = sbytes(DT), NV = QBY / 16;
    const int sub = (tidx() >> 4) & 3, row = tidx() & 15, nb = m.nb;
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int b = 4 * (j0 + s) + sub;
        const bool ok = t < m.tiles && b < nb;
        const size_t slot = ((size_t)t * nb + b) * 16 + row;
#pragma unroll
        for (int v = 0; v < NV; v++) pf.w[s][v] = ldg16_if(m.q, slot * NV + v, ok);
        if constexpr (SBY == 2) pf.sc[s] = ldg2_if(m.s, slot, ok);
        if constexpr (SBY == 1) pf.sc[s] = ldg1_if(m.s, slot, ok);
        if constexpr (SBY == 0) pf.sc[s] = 0;
    }
}

// res[pair * 16 + row] for this lane's slots. The lane's pair advances by 4 * NWE from slot to slot, so
// its block (pair % nb) advances by (4 * NWE) % nb, with one wrap.
template <int DT, int NS>
__device__ __forceinline__ void pref_compute(Pref<DT, NS> &pf, const l3m_dmat &m, int s0, const uint8_t *act, int kp, float *res) {
    const int wave = wave_id(), lane = tidx() & 63, nb = m.nb, n = m.tiles * nb;
    // x % nb = x - nb * floor((x + 0.5) / nb) with a reciprocal good to 1 ulp: exact for x < 2^20
    const float inb = __builtin_amdgcn_rcpf((float)nb);
    const int x0 = (tidx() >> 4) + 4 * NWE * s0;      // the lane's pair in slot 0
    int b = x0 - (int)(((float)x0 + 0.5f) * inb) * nb;
    const int step = __builtin_amdgcn_readfirstlane(4 * NWE - (int)(((float)(4 * NWE) + 0.5f) * inb) * nb);
    const unsigned stepm = (unsigned)__builtin_amdgcn_readfirstlane(step - nb);
    // Pin the loaded registers here: otherwise the compiler hoists their first use (the f16 scale
    // conversion) up to the loads, and every wavefront stalls on its first load at entry.
#pragma unroll
    for (int s = 0; s < NS; s++) {
        asm volatile("" : "+v"(pf.sc[s]));
#pragma unroll
        for (int v = 0; v < qbytes(DT) / 16; v++) asm volatile("" : "+v"(pf.w[s][v].x), "+v"(pf.w[s][v].y), "+v"(pf.w[s][v].z), "+v"(pf.w[s][v].w));
    }
    // a wavefront stops at its first slot past the end (a scalar branch); in its last slot the up to 3
    // pairs past the end (loads repeat the last pair) write into the padding of res (res_bytes)
    float *rp = res + wave * 64 + lane;              // res[p0 * 16 + lane] = rp[slot * NWE * 64]
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int p0 = (wave + (s0 + s) * NWE) * 4;
        if (p0 >= n) break;
        rp[(s0 + s) * NWE * 64] = block_fma<DT>(0.f, pf.w[s], pf.sc[s], act, kp, b);
        // b + step - nb when that is not negative, else b + step (step < nb): one unsigned minimum
        b = (int)__builtin_elementwise_min((unsigned)b + (unsigned)step, (unsigned)b + stepm);
    }
}

// All pairs of m: the prefetched batch, then any further batches (loaded here).
template <int DT, int NS>
__device__ __forceinline__ void mv(Pref<DT, NS> &pf, const l3m_dmat &m, const uint8_t *act, int kp, float *res) {
    pref_compute<DT, NS>(pf, m, 0, act, kp, res);
    for (int s0 = NS; s0 * NWE * 4 < m.tiles * m.nb; s0 += NS) {
        pref_load<DT, NS>(pf, m, s0);
        pref_compute<DT, NS>(pf, m, s0, act, kp, res);
    }
}

// ------------------------------------------------------------------------------ cross-lane sums
// DPP and gfx950 permlane swaps: every lane of an aligned group of N lanes gets the group's sum (max),
// added in one fixed order, so the value is identical in every lane and every run. All 64 lanes of the
// wavefront must be active.
template <int C> __device__ __forceinline__ float dppf(float v) {
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), C, 0xF, 0xF, false));
}
template <int C> __device__ __forceinline__ int dppi(int v) { return __builtin_amdgcn_update_dpp(0, v, C, 0xF, 0xF, false); }
// (lanes with bit 4 clear, lanes with bit 4 set) of each 32, and (lanes 0-31, lanes 32-63)
__device__ __forceinline__ void swap16(float v, float &lo, float &hi) {
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    lo = __uint_as_float(r[0]); hi = __uint_as_float(r[1]);
}
__device__ __forceinline__ void swap32(float v, float &lo, float &hi) {
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    lo = __uint_as_float(r[0]); hi = __uint_as_float(r[1]);
}
constexpr int QP_X1 = 0xB1, QP_X2 = 0x4E, ROW_HALF_MIRROR = 0x141, ROW_MIRROR = 0x140, ROW_ROR4 = 0x124, ROW_ROR8 = 0x128;

template <int N> __device__ __forceinline__ float lanes_sum(float v) {
    if constexpr (N >= 2) v += dppf<QP_X1>(v);
    if constexpr (N >= 4) v += dppf<QP_X2>(v);
    if constexpr (N >= 8) v += dppf<ROW_HALF_MIRROR>(v);
    if constexpr (N >= 16) v += dppf<ROW_MIRROR>(v);
    if constexpr (N >= 32) { float lo, hi; swap16(v, lo, hi); v = lo + hi; }
    if constexpr (N >= 64) { float lo, hi; swap32(v, lo, hi); v = lo + hi; }
    return v;
}
template <int N> __device__ __forceinline__ float lanes_max(float v) {
    if constexpr (N >= 2) v = fmaxf(v, dppf<QP_X1>(v));
    if constexpr (N >= 4) v = fmaxf(v, dppf<QP_X2>(v));
    if constexpr (N >= 8) v = fmaxf(v, dppf<ROW_HALF_MIRROR>(v));
    if constexpr (N >= 16) v = fmaxf(v, dppf<ROW_MIRROR>(v));
    if constexpr (N >= 32) { float lo, hi; swap16(v, lo, hi); v = fmaxf(lo, hi); }
    if constexpr (N >= 64) { float lo, hi; swap32(v, lo, hi); v = fmaxf(lo, hi); }
    return v;
}
template <int N> __device__ __forceinline__ int lanes_sumi(int v) {
    if constexpr (N >= 2) v += dppi<QP_X1>(v);
    if constexpr (N >= 4) v += dppi<QP_X2>(v);
    if constexpr (N >= 8) v += dppi<ROW_HALF_MIRROR>(v);
    return v;
}
// Sum over groups of n (4, 8, 16 or 32; uniform) aligned lanes.
__device__ __forceinline__ float lanes_sum_n(float v, int n) {
    v = lanes_sum<4>(v);
    if (n >= 8) v += dppf<ROW_HALF_MIRROR>(v);
    if (n >= 16) v += dppf<ROW_MIRROR>(v);
    if (n >= 32) { float lo, hi; swap16(v, lo, hi); v = lo + hi; }
    return v;
}
// Sum over the lanes of a wavefront that share (lane % n), n = 4, 8, 16 or 32 (uniform); lanes
// with lane < n hold the results.
__device__ __forceinline__ float strided_sum(float v, int n) {
    float lo, hi;
    if (n <= 4) v += dppf<ROW_ROR4>(v);
    if (n <= 8) v += dppf<ROW_ROR8>(v);
    if (n <= 16) { swap16(v, lo, hi); v = lo + hi; }
    swap32(v, lo, hi);
    return lo + hi;
}

// The matvec of m in the tile form (the first batch of the wavefront's first tile loaded by
// pref_load_tile beforehand): lane (sub, row) accumulates its blocks sub, sub + 4, ... in block order as
// they come out of its slots (block_fma's fma into the running sum), the four quarter sums meet by
// permlane swaps ((q0 + q1) + (q2 + q3)), and f(i, y, partner, lead) runs for the tile's 16 rows, with
// no LDS round trip or barrier. The block offsets are constants per slot (no index arithmetic).
template <int DT, int NS, class F>
__device__ __forceinline__ void tile_rows(Pref<DT, NS> &pf, const l3m_dmat &m, const uint8_t *act, int kp, int rows, F f) {
    const int wave = wave_id(), lane = tidx() & 63, sub = lane >> 4, row = lane & 15, nb = m.nb, spt = (nb + 3) >> 2;
    constexpr int QB = act_qbytes(DT);
    // the lane's block sub (values, scale, sum) of act's na blocks (kp = kwide(k): whole slots, the blocks
    // past nb zero with scale 0); slot s adds 4 s blocks, a constant offset
    const int na = kp >> 5;
    const uint8_t *xq = act + QB * sub;
    const float *xsp = (const float *)(act + QB * na) + sub;
    const int *xsum = (const int *)(act + QB * na + 4 * na) + sub;
    float y = 0.f;
    auto batch = [&](int j0) {
        // pin the loaded registers here, as pref_compute does
#pragma unroll
        for (int s = 0; s < NS; s++) {
            asm volatile("" : "+v"(pf.sc[s]));
#pragma unroll
            for (int v = 0; v < qbytes(DT) / 16; v++)
                asm volatile("" : "+v"(pf.w[s][v].x), "+v"(pf.w[s][v].y), "+v"(pf.w[s][v].z), "+v"(pf.w[s][v].w));
        }
#pragma unroll
        for (int s = 0; s < NS; s++) {
            if (j0 + s >= spt) break;
            // blocks past nb: weights of block nb - 1 (pref_load_tile) times zero values with scale 0
            const int o = 4 * (j0 + s);
            y = block_fma_at<DT>(y, pf.w[s], pf.sc[s], xq + QB * o, xsp + o, xsum + o);
        }
    };
    auto finish = [&](int t) {
        float lo, hi;
        swap16(y, lo, hi);                            // q0 + q1, q2 + q3
        y = lo + hi;
        swap32(y, lo, hi);                            // (q0 + q1) + (q2 + q3), in all four lanes
        y = lo + hi;
        const float partner = dppf<QP_X1>(y);        // row i ^ 1 is the neighbouring lane
        const int i = t * 16 + row;
        if (i < rows) f(i, y, partner, sub == 0);
        y = 0.f;
    };
    if (wave < m.tiles) {
        batch(0);
        for (int j0 = NS; j0 < spt; j0 += NS) {
            pref_load_tile<DT, NS>(pf, m, wave, j0);
            batch(j0);
        }
        finish(wave);
        for (int t = wave + NWE; t < m.tiles; t += NWE) {
            for (int j0 = 0; j0 < spt; j0 += NS) {
                pref_load_tile<DT, NS>(pf, m, t, j0);
                batch(j0);
            }
            finish(t);
        }
    }
}

// A matrix of nb = 1, 2 or 4 blocks per row, its rows summed where the slots computed them: a slot's 4
// pairs are then whole rows of 16 (nb 4: the 4 blocks of one tile; nb 2: two tiles; nb 1: four), so the
// quarter sums of rows_sum4 meet in registers (permlane swaps, the same values added in the same order)
// and f(i, y, lead) takes each row from the slot that computed it, with no LDS round trip or barrier.
template <int DT, int NS, class F>
__device__ __forceinline__ void slots_rows(Pref<DT, NS> &pf, const l3m_dmat &m, int s0, const uint8_t *act, int kp, int rows, F f) {
    const int wave = wave_id(), lane = tidx() & 63, nb = m.nb, n = m.tiles * nb, sub = lane >> 4, row = lane & 15;
    const int b = sub & (nb - 1), sh = nb >> 1 == 2 ? 2 : nb >> 1;   // the lane's block, log2(nb)
#pragma unroll
    for (int s = 0; s < NS; s++) {
        asm volatile("" : "+v"(pf.sc[s]));
#pragma unroll
        for (int v = 0; v < qbytes(DT) / 16; v++) asm volatile("" : "+v"(pf.w[s][v].x), "+v"(pf.w[s][v].y), "+v"(pf.w[s][v].z), "+v"(pf.w[s][v].w));
    }
#pragma unroll
    for (int s = 0; s < NS; s++) {
        const int p0 = (wave + (s0 + s) * NWE) * 4;
        if (p0 >= n) break;
        // rows_sum4 for nb <= 4: quarter q = 0.f + block q (when q < nb), then (q0 + q1) + (q2 + q3)
        const float v = 0.f + block_fma<DT>(0.f, pf.w[s], pf.sc[s], act, kp, b);
        float lo, hi, y;
        if (nb == 4) {
            swap16(v, lo, hi);
            y = lo + hi;
            swap32(y, lo, hi);
            y = lo + hi;
        } else if (nb == 2) {
            swap16(v, lo, hi);
            y = (lo + hi) + (0.f + 0.f);
        } else {
            y = (v + 0.f) + (0.f + 0.f);
        }
        const int i = ((p0 + sub) >> sh) * 16 + row;   // pairs past the end give i >= rows
        if (i < rows) f(i, y, b == 0);
    }
}
template <int DT, int NS, class F>
__device__ __forceinline__ void mv_rows(Pref<DT, NS> &pf, const l3m_dmat &m, const uint8_t *act, int kp, float *res, int rows, F f) {
    if (m.nb == 1 || m.nb == 2 || m.nb == 4) {
        slots_rows<DT, NS>(pf, m, 0, act, kp, rows, f);
        for (int s0 = NS; s0 * NWE * 4 < m.tiles * m.nb; s0 += NS) {
            pref_load<DT, NS>(pf, m, s0);
            slots_rows<DT, NS>(pf, m, s0, act, kp, rows, f);
        }
        return;
    }
    mv<DT, NS>(pf, m, act, kp, res);
    __syncthreads();
    rows_sum4(m, res, rows, [&](int i, float y, float, bool lead) { f(i, y, lead); });
}

// Scratch for workgroup reductions (norm_prep): the wavefront results go to one of two 16-float slots of
// scr, used alternately, so a slot is only rewritten after every thread has passed the barrier of the
// reduction in between. All threads take part, in the same order.
struct Red {
    float *scr;    // 32 floats of LDS
    int k;
};
template <int N> __device__ __forceinline__ int lanes_mini(int v) {
    if constexpr (N >= 2) v = min(v, dppi<QP_X1>(v));
    if constexpr (N >= 4) v = min(v, dppi<QP_X2>(v));
    if constexpr (N >= 8) v = min(v, dppi<ROW_HALF_MIRROR>(v));
    if constexpr (N >= 16) v = min(v, dppi<ROW_MIRROR>(v));
    if constexpr (N >= 32) { float lo, hi; swap16(__int_as_float(v), lo, hi); v = min(__float_as_int(lo), __float_as_int(hi)); }
    if constexpr (N >= 64) { float lo, hi; swap32(__int_as_float(v), lo, hi); v = min(__float_as_int(lo), __float_as_int(hi)); }
    return v;
}
// (value, index) maximum with the reference's tie rule (the larger value, then the lower index;
// a NaN never wins) into every thread: a wavefront's largest value (fmaxf passes NaN over), then the
// lowest index that holds it; then the same over the wavefronts' results, which every wavefront reads
// after one barrier. sv, si: NWE words each, not read again before a later barrier.
// The same into wavefront 0 only (the head's key comes from thread 0): the wavefronts at and past
// `busy` hold no rows, and store their empty result without reducing it; only wavefront 0 takes the
// second stage, so the others leave at the barrier.
__device__ void block_argmax0(float &v, int &i, float *sv, int *si, int busy) {
    const int w = wave_id();
    float m = -INFINITY;
    int ci = 0x7FFFFFFF;
    if (w < busy) {
        m = lanes_max<64>(v);
        ci = lanes_mini<64>(v == m ? i : 0x7FFFFFFF);
    }
    if ((tidx() & 63) == 0) { sv[w] = m; si[w] = ci; }
    __syncthreads();
    if (w == 0) {
        const int k = tidx() & (NWE - 1);
        const float vk = sv[k];
        const int ik = si[k];
        m = lanes_max<NWE>(vk);
        ci = lanes_mini<NWE>(vk == m ? ik : 0x7FFFFFFF);
    }
    v = m;
    i = ci;
}
__device__ void block_argmax(float &v, int &i, float *sv, int *si) {
    float m = lanes_max<64>(v);
    int ci = lanes_mini<64>(v == m ? i : 0x7FFFFFFF);
    if ((tidx() & 63) == 0) { sv[wave_id()] = m; si[wave_id()] = ci; }
    __syncthreads();
    const int k = tidx() & (NWE - 1);                 // each aligned group of NWE lanes holds every result
    const float vk = sv[k];
    const int ik = si[k];
    m = lanes_max<NWE>(vk);
    ci = lanes_mini<NWE>(vk == m ? ik : 0x7FFFFFFF);
    v = m;
    i = ci;
}

// Matvec results res[pair * 16 + row] summed per row: four quarter sums of the blocks, each in block
// order, added pairwise ((q0 + q1) + (q2 + q3)). Rows of more than 4 blocks take 4 lanes, one per quarter:
// a wavefront takes the 16 rows of one tile, row r in lanes r, r + 16, r + 32, r + 48, and quarter q
// holds blocks q, q + 4, q + 8, ..., so the 32 lanes the LDS serves at once (quarters q and q + 1) read
// 32 different banks (block b lies 16 b floats into the tile). Rows of at most 4 blocks take one lane
// (all four quarters: block q, if any), which gives the same sums in a quarter of the passes.
// f(i, y, partner, lead) runs in every lane for rows i < rows, partner being row i ^ 1's value and lead
// true in one lane per row.
template <class F>
__device__ __forceinline__ void rows_sum4(const l3m_dmat &m, const float *res, int rows, F f) {
    const int nb = m.nb;
    // Reads are unconditional (row and block clamped into range) and issued together; the sums then take
    // only the values in range, in block order.
    if (nb <= 4) {
        // each quarter holds at most one block: quarter q has block q when q < nb
        for (int base = 0; base < rows; base += NTE) {
            const int i = base + tidx(), ic = i < rows ? i : rows - 1;
            const float *p = res + (size_t)(ic >> 4) * nb * 16 + (ic & 15);
            float v[4];
#pragma unroll
            for (int b = 0; b < 4; b++) v[b] = p[(b < nb ? b : nb - 1) * 16];
            float s[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int q = 0; q < 4; q++)
                if (i < rows && q < nb) s[q] += v[q];
            const float y = (s[0] + s[1]) + (s[2] + s[3]);
            const float partner = dppf<QP_X1>(y);     // row i ^ 1 is the neighbouring lane
            if (i < rows) f(i, y, partner, true);
        }
        return;
    }
    const int lane = tidx() & 63, q = lane >> 4;
    for (int base = 0; base < rows; base += NTE / 4) {
        const int i = base + 16 * wave_id() + (lane & 15);
        float y = 0.f;
        if (i < rows) {
            const float *p = res + (size_t)(i >> 4) * nb * 16 + (i & 15);
#pragma unroll 4
            for (int b = q; b < nb; b += 4) y += p[b * 16];
        }
        float lo, hi;
        swap16(y, lo, hi);                            // q0 + q1, q2 + q3
        y = lo + hi;
        swap32(y, lo, hi);                            // (q0 + q1) + (q2 + q3), in all four lanes
        y = lo + hi;
        const float partner = dppf<QP_X1>(y);        // row i ^ 1 is the neighbouring lane
        if (i < rows) f(i, y, partner, q == 0);
    }
}

// ------------------------------------------------------------------------------- phase stamps
// Per-phase timing of the decode step, in a build of its own (L3M_PHASE_STAMPS: make -C l3m_amd/csrc
// phases, l3m_amd/libl3m_hip_phases.so; bench.py --phases): thread 0 of each attention group (role g),
// FFN chunk (64 + c) and head workgroup (128 + h) records the 100 MHz clock at each phase boundary of two
// consecutive layers at one position, armed by l3m_phase_stamps: (layer, layer + 1), or for the last
// layer (its layer and the head, then layer 0 of the next position). The product build compiles every
// stamp away.
#ifdef L3M_PHASE_STAMPS
__device__ unsigned long long g_phase[2][3 * 64][16];
__device__ unsigned long long g_phase_clk[2][3 * 64][16];   // the shader clock (s_memtime) at the same points
__device__ int g_phase_at[2];
__shared__ int s_phase_row;      // thread 0's: which of the two recorded layers this one is, or -1
// At the top of a layer (before its wait): whether this (position, layer) is recorded. One global read per
// layer, off the measured phases; the stamps then read only thread 0's LDS word.
__device__ __forceinline__ void phase_arm(int pos, int layer, int nl) {
    if (tidx() != 0) return;
    const int at_pos = __hip_atomic_load(&g_phase_at[0], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int at_layer = __hip_atomic_load(&g_phase_at[1], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const int d = layer - at_layer;
    if (pos == at_pos && (d == 0 || d == 1)) s_phase_row = d;
    else if (at_layer == nl - 1 && pos == at_pos + 1 && layer == 0) s_phase_row = 1;   // after the last layer
    else s_phase_row = -1;
}
__device__ __forceinline__ void phase(int role, int ev, int, int) {
    if (tidx() != 0 || role >= 3 * 64) return;
    const int d = s_phase_row;                        // the graph path never arms it: only 0 or 1 records
    if (d == 0 || d == 1) {
        g_phase[d][role][ev] = __builtin_amdgcn_s_memrealtime();
        g_phase_clk[d][role][ev] = __builtin_amdgcn_s_memtime();
    }
}
#else
__device__ __forceinline__ void phase_arm(int, int, int) {}
__device__ __forceinline__ void phase(int, int, int, int) {}
#endif

// ----------------------------------------------------------------------------------- prologue
// The incoming residual x = base + parts[0] + ... + parts[n-1] (or, for layer 0, the embedding row of
// tok), with thread f < dim/4 owning x[4f, 4f+4). The parts are split over G = NTE / (dim/4) thread
// groups; pro_load only issues the loads (the norm weights and RoPE angles come from pro_static),
// pro_finish adds them: each group's sum goes through LDS and the owners add the groups in order.
constexpr int FILL_PER = 4;
struct Pro {
    float4 p[FILL_PER];
    float4 base;
    float4 emb;       // layer 0: the embedding row's owned elements
};
// The inputs of a block that no other workgroup writes during the step: the owners' norm weights and, for
// attention, the RoPE (cos, sin) of angle index tid (tid < hd / 2) at the step's position. The persistent
// path loads them before it waits for the block's exchanged inputs, so their memory latency (the weight
// stream keeps them out of L2) stays off the step's critical path.
struct ProStatic {
    float4 nw;
    float2 cs;
};
struct ProGeom {
    int n4, groups, per, nparts;
};
// groups = NTE / n4 (at least 1), per = ceil(nparts / groups) (at least 1): computed on the host
// (l3m_model_layout) so that no workgroup divides by them at run time.
// As many groups of dim / 4 threads as the workgroup holds, each summing per parts, and no group more than
// the parts need (a group past the last part would only load copies of it).
__host__ __device__ inline void pro_shape(int dim, int nparts, int &groups, int &per) {
    groups = NTE / (dim >> 2) < 1 ? 1 : NTE / (dim >> 2);
    per = (nparts + groups - 1) / groups;
    if (per < 1) per = 1;
    groups = nparts > 0 ? (nparts + per - 1) / per : 1;
}
// which 0: over the n_chunks FFN partials (attention and head prologues), 1: over the n_groups ones.
__device__ __forceinline__ ProGeom pro_geom(const l3m_dmodel &M, int which) {
    ProGeom g;
    g.n4 = M.dim >> 2;
    g.groups = M.pro_groups[which];
    g.per = M.pro_per[which];
    g.nparts = which ? M.n_groups : M.n_chunks;
    return g;
}
// tid / n4 and tid % n4 (tid < NTE <= 2^10, n4 <= 2^10) without an integer division per thread:
// (tid + 0.5) / n4 is at least 0.5 / n4 >= 2^-11 away from an integer, far more than the float
// product's error, so its floor is exact.
__device__ __forceinline__ void split_tid(int tid, int n4, int &grp, int &f) {
    const float inv = __builtin_amdgcn_rcpf((float)n4);   // within 1 ulp: the margin above is far larger
    grp = (int)(((float)tid + 0.5f) * inv);
    f = tid - grp * n4;
}
// Loads are unconditional (indices clamped into range) wherever possible: a load under a branch that
// later merges makes the compiler wait for it there, before the weight stream is issued.
// embed is passed by value: a pointer into the kernel's argument struct would move that struct to scratch.
// Owners load their norm weights and, given rope_row, the angles (hd / 2 <= n4: the angles' threads are
// owners too).
__device__ __forceinline__ void pro_static(ProStatic &S, int n4, const float *nw, const float *rope_row, int hd) {
    const int tid = tidx(), own = tid < n4 ? tid : n4 - 1;
    if (wave_id() * 64 < n4) {
        S.nw = ldg16f(nw, own);
        if (rope_row) {
            const int i = tid < (hd >> 1) ? tid : (hd >> 1) - 1;
            const u32x2 c = gp<u32x2>(rope_row)[i];
            S.cs = make_float2(__uint_as_float(c.x), __uint_as_float(c.y));
        }
    }
}
template <bool COH>
__device__ __forceinline__ void pro_load(Pro &P, const float *base, const float *parts, const ProGeom &G,
                                         l3m_dmat embed, bool use_embed, int tok) {
    const int tid = tidx(), nparts = G.nparts, dim = 4 * G.n4;
    int f, grp;
    split_tid(tid, G.n4, grp, f);
    const int j0 = grp * G.per, own = tid < G.n4 ? tid : G.n4 - 1, wave = wave_id();
    // Each wavefront issues only the loads its threads use (wave-uniform branches: a memory instruction
    // costs address-unit time whether or not its lanes are needed). Owners (group 0) take the base and,
    // at layer 0, the embedding row; grouped threads their parts.
    if (wave * 64 < G.n4) P.base = ld16f<COH>(base, f);
    if (wave * 64 < G.groups * G.n4) {
#pragma unroll
        for (int j = 0; j < FILL_PER; j++)
            P.p[j] = ld16f_if<COH>(parts, (size_t)(j0 + j) * (dim >> 2) + f, j < G.per && j0 + j < nparts);
    }
    if (use_embed) P.emb = lt_elem4(embed, tok, 4 * own);   // layer 0: x = dequant(embed[tok]) (engine.c:236)
    asm volatile("" ::: "memory");                            // these loads are issued before the weights
}
// Returns x[4f, 4f+4) to owner f (zeros to the other threads); stores it to keep when given; writes the
// RoPE angles to cs_lds when given. pbuf: NTE float4 of LDS. All threads call it.
template <bool COH>
__device__ __forceinline__ float4 pro_finish(Pro &P, const float *parts, const ProGeom &G, bool use_embed, float4 *pbuf, float *keep,
                             float *cs_lds, float2 cs, int hd) {
    const int tid = tidx(), nparts = G.nparts, dim = 4 * G.n4;
    int f, grp;
    split_tid(tid, G.n4, grp, f);
    const int j0 = grp * G.per;
    if (cs_lds && tid < (hd >> 1)) ((float2 *)cs_lds)[tid] = cs;
    float4 x = make_float4(0.f, 0.f, 0.f, 0.f);
    if (use_embed) {
        if (tid < G.n4) x = P.emb;
    } else {
        if (grp < G.groups) {
            float4 v = grp == 0 ? P.base : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
            for (int j = 0; j < FILL_PER; j++) { v.x += P.p[j].x; v.y += P.p[j].y; v.z += P.p[j].z; v.w += P.p[j].w; }
            for (int j = FILL_PER; j < G.per && j0 + j < nparts; j++) {   // beyond one batch: in order
                const float4 p = ld16f<COH>(parts, (size_t)(j0 + j) * (dim >> 2) + f);
                v.x += p.x; v.y += p.y; v.z += p.z; v.w += p.w;
            }
            if (G.groups > 1) pbuf[grp * G.n4 + f] = v;
            else x = v;
        }
        if (G.groups > 1) {
            __syncthreads();
            if (tid < G.n4) {
                x = pbuf[tid];
                for (int g0 = 1; g0 < G.groups; g0 += 4) {   // 4 reads in flight, then their sums in order
                    float4 p[4];
#pragma unroll
                    for (int u = 0; u < 4; u++) p[u] = pbuf[(g0 + u < G.groups ? g0 + u : G.groups - 1) * G.n4 + tid];
#pragma unroll
                    for (int u = 0; u < 4; u++) {
                        const bool in = g0 + u < G.groups;
                        x.x += in ? p[u].x : 0.f; x.y += in ? p[u].y : 0.f; x.z += in ? p[u].z : 0.f; x.w += in ? p[u].w : 0.f;
                    }
                }
            }
        }
    }
    if (keep && tid < G.n4) {
        const f32x4 v = {x.x, x.y, x.z, x.w};
        gw((f32x4 *)keep)[tid] = v;
    }
    return x;
}

__device__ __forceinline__ float4 add4(float4 a, float4 b) { return make_float4(a.x + b.x, a.y + b.y, a.z + b.z, a.w + b.w); }

// act = the prepared activation (pack.c:101-123) of the values v[4f, 4f+4) held by thread f, f < kp/4
// (zero beyond k): the reference's per-32-block int8 quantization (8 lanes per block), bf16 or f32.
// Ends with a barrier.
template <int DT>
__device__ __forceinline__ void prep_body(float4 y, uint8_t *act, int kp) {
    const int f = tidx();
    if constexpr (quantized(DT)) {
        float am = fmaxf(fmaxf(fabsf(y.x), fabsf(y.y)), fmaxf(fabsf(y.z), fabsf(y.w)));
        am = lanes_max<8>(am);
        const float inv = am > 0.f ? 127.0f / am : 0.f;
        const int q0 = (int)rintf(y.x * inv), q1 = (int)rintf(y.y * inv), q2 = (int)rintf(y.z * inv), q3 = (int)rintf(y.w * inv);
        const uint32_t P = (uint32_t)(q0 & 255) | (uint32_t)(q1 & 255) << 8 | (uint32_t)(q2 & 255) << 16 | (uint32_t)(q3 & 255) << 24;
        // the partner lane m + 4 of the block's 8 (DPP row shift left by 4: lanes 0-3 and 8-11 of each row
        // of 16 read lanes 4-7 and 12-15)
        const uint32_t Pp = DT == L3M_Q8_0 ? 0u : (uint32_t)dppi<0x104>((int)P);
        const int nb = kp >> 5;
        int s = 0;
        if (4 * f < kp) s = put_block<DT>(act + (f >> 3) * act_qbytes(DT), f & 7, P, Pp, q0, q1, q2, q3);
        s = lanes_sumi<8>(s);
        if (4 * f < kp && (f & 7) == 0) {
            ((float *)(act + act_qbytes(DT) * nb))[f >> 3] = am / 127.0f;
            ((int *)(act + act_qbytes(DT) * nb + 4 * nb))[f >> 3] = s;
        }
    } else if constexpr (DT == L3M_BF16) {
        if (4 * f < kp)
            *(uint2 *)(act + 8 * f) = make_uint2((uint32_t)f32_bf16(y.x) | (uint32_t)f32_bf16(y.y) << 16,
                                                 (uint32_t)f32_bf16(y.z) | (uint32_t)f32_bf16(y.w) << 16);
    } else {
        if (4 * f < kp) *(float4 *)(act + 16 * f) = y;
    }
}
// Only the wavefronts that hold prepared elements (4 per thread) do the work; the others go straight to
// the barrier, so they take no issue slots from the SIMDs they share.
template <int DT>
__device__ __forceinline__ void prep_owned(float4 y, uint8_t *act, int kp) {
    if (wave_id() * 256 < kp) prep_body<DT>(y, act, kp);
    __syncthreads();
}

// RMSNorm (ops.c:13-18: s = 1/sqrt(sum x^2 / n + eps), y = x * s * w) of the owned x, then its prep.
// The sum of squares is red_sum's (same slots, same order of additions); wavefronts past the owned
// elements write their zero without the reduction work and skip the rest.
template <int DT>
__device__ __forceinline__ void norm_prep(float4 x, float4 nw, int k, int kp, float eps, uint8_t *act, Red &red) {
    const int wave = wave_id();
    const bool owner = wave * 256 < kp;               // kp >= k: these waves also write the padding
    float *slot = red.scr + 16 * (red.k++ & 1);
    const float part = owner ? lanes_sum<64>(x.x * x.x + x.y * x.y + x.z * x.z + x.w * x.w) : 0.f;
    if ((tidx() & 63) == 0) slot[wave] = part;
    __syncthreads();
    if (owner) {
        const float4 *sv = (const float4 *)slot;
        const float4 a = sv[0], b = sv[1], c = sv[2], d = sv[3];
        const float tot = (((a.x + a.y) + (a.z + a.w)) + ((b.x + b.y) + (b.z + b.w))) + (((c.x + c.y) + (c.z + c.w)) + ((d.x + d.y) + (d.z + d.w)));
        const float s = 1.0f / sqrtf(tot / (float)k + eps);
        float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
        if (4 * (int)tidx() < k) y = make_float4(x.x * s * nw.x, x.y * s * nw.y, x.z * s * nw.z, x.w * s * nw.w);
        prep_body<DT>(y, act, kp);
    }
    __syncthreads();
}

// LayerNorm (ops.c:20-27: the mean, then the mean square deviation, s = 1/sqrt(var / n + eps),
// y = (x - mean) * s * w + b) of the owned x, then its prep: the GPT-2 variant's norm. Two workgroup sums
// (same slots and order of additions as norm_prep's), only past the first does x's mean exist.
template <int DT>
__device__ __forceinline__ void ln_prep(float4 x, const float *w, const float *b, int k, int kp, float eps, uint8_t *act, Red &red) {
    const int wave = wave_id(), f = tidx();
    const bool owner = wave * 256 < kp;
    auto block_total = [&](float v) {
        float *slot = red.scr + 16 * (red.k++ & 1);
        const float part = owner ? lanes_sum<64>(v) : 0.f;
        if ((f & 63) == 0) slot[wave] = part;
        __syncthreads();
        const float4 *sv = (const float4 *)slot;
        const float4 a = sv[0], c = sv[1], d = sv[2], e = sv[3];
        return (((a.x + a.y) + (a.z + a.w)) + ((c.x + c.y) + (c.z + c.w))) + (((d.x + d.y) + (d.z + d.w)) + ((e.x + e.y) + (e.z + e.w)));
    };
    const float mean = block_total(x.x + x.y + x.z + x.w) / (float)k;
    const bool in = 4 * f < k;
    const float4 dv = in ? make_float4(x.x - mean, x.y - mean, x.z - mean, x.w - mean) : make_float4(0.f, 0.f, 0.f, 0.f);
    const float var = block_total(dv.x * dv.x + dv.y * dv.y + dv.z * dv.z + dv.w * dv.w);
    if (owner) {
        const float s = 1.0f / sqrtf(var / (float)k + eps);
        float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
        if (in) {
            const float4 wv = ((const float4 *)w)[f], bv = ((const float4 *)b)[f];
            y = make_float4(dv.x * s * wv.x + bv.x, dv.y * s * wv.y + bv.y, dv.z * s * wv.z + bv.z, dv.w * s * wv.w + bv.w);
        }
        prep_body<DT>(y, act, kp);
    }
    __syncthreads();
}
// GELU, tanh form (ops.c:53-56).
__device__ __forceinline__ float gelu_tanh(float x) { return 0.5f * x * (1.0f + tanhf(0.7978845608f * (x + 0.044715f * x * x * x))); }

// LDS regions of the step kernels (byte offsets, 16-aligned) from the layer geometry. `work` holds the
// prologue's group sums, then the per-pair matvec results.
// Matvec results take 64 bytes per (tile, block) pair; a wavefront writes whole groups of 4 pairs
// (those past the end into padding).
__host__ __device__ inline size_t res_bytes(size_t pairs) { return 64 * ((pairs + 3) / 4 * 4); }
__host__ __device__ inline size_t work_bytes(size_t a, size_t b) {
    const size_t w = a > b ? a : b;
    return align16(w > 16 * (size_t)NTE ? w : 16 * (size_t)NTE);
}

// Row stride (bf16 elements) of the LDS K/V window: hd + 8 keeps rows 16-byte aligned and puts 16
// consecutive rows' same 16 bytes on 16 different 4-bank groups, so reads down a column (the MFMA
// operand layout) are free of bank conflicts.
__host__ __device__ inline int kv_row(int hd) { return hd + 8; }
// The matrix-core attention keeps V transposed in the window, V^T [nkv][hd][vt_row(ctx)]: a P.V operand (8
// consecutive positions of one dimension) is then one 16-byte read. Rows hold every position a 32-position
// step reads, plus 8 to spread consecutive rows over the banks.
__host__ __device__ inline int vt_row(int ctx) { return ((ctx + 31) & ~31) + 8; }
// Bytes of the LDS K/V window: K [nkv][ctx][kv_row(hd)], then V in the same layout or transposed (vt).
__host__ __device__ inline size_t kv_window_bytes(int nkv, int ctx, int hd, bool vt) {
    const size_t k = (size_t)nkv * ctx * kv_row(hd), v = vt ? (size_t)nkv * hd * vt_row(ctx) : k;
    return align16(2 * (k + v));
}
// Whether attend_mfma takes the shape (hd a multiple of 16, the q parts beside the wavefront sums in vred,
// the scores and p parts within the 16 KiB minimum of the work region).
__host__ __device__ inline bool mfma_fits(int hd, int nq, int ctx) {
    return hd % 16 == 0 && 6 * nq * hd <= 4 * NWE * hd && 10 * ((ctx + 31) & ~31) <= 16 * NTE;
}
// Which attention the decode step runs for a head group of nq query heads: 2 on the matrix cores
// (attend_mfma, over the K/V window in LDS) when the shape fits it, 1 the VALU split softmax over the LDS
// window, 0 the VALU split softmax reading K and V from the cache (the window does not fit in LDS).
__host__ __device__ inline int att_mode(int kv_lds, int hd, int nq, int ctx) {
    if (!kv_lds) return 0;
    return mfma_fits(hd, nq, ctx) ? 2 : 1;
}
struct LdsA { size_t act, work, q, cur, cs, vred, att, act2, scr, kvb, total; };
__host__ __device__ inline LdsA lds_a(int dt, int dim, int ctx, int hd, const l3m_dgroup &g, int kv_lds) {
    LdsA L;
    size_t o = 0;
    const size_t pq = (size_t)g.qkv.tiles * g.qkv.nb, pw = (size_t)g.wo.tiles * g.wo.nb;
    L.act = o;  o += align16(act_size(dt, kwide(dim)));
    L.work = o; o += work_bytes(res_bytes(pq), res_bytes(pw));
    L.q = o;    o += align16(4 * (size_t)g.nq * hd);
    L.cur = o;  o += align16(4 * (size_t)g.nkv * hd);              // this step's k, v rows: bf16 [2][nkv][hd]
    L.cs = o;   o += align16(4 * (size_t)hd);
    L.vred = o; o += align16(4 * (size_t)NWE * (hd + 2));
    L.att = o;  o += align16(4 * (size_t)kpad(g.nq * hd));
    L.act2 = o; o += align16(act_size(dt, g.nq * hd));
    L.scr = o;  o += 4 * 64;
    L.kvb = o;  o += kv_lds ? kv_window_bytes(g.nkv, ctx, hd, mfma_fits(hd, g.nq, ctx)) : 0;   // K, V (or V^T) bf16
    L.total = o;
    return L;
}
// The offsets as the host stored them in the group descriptor (l3m_group_layout).
__device__ __forceinline__ LdsA lds_of(const l3m_dgroup &G) {
    LdsA L;
    L.act = G.lds[0]; L.work = G.lds[1]; L.q = G.lds[2]; L.cur = G.lds[3]; L.cs = G.lds[4];
    L.vred = G.lds[5]; L.att = G.lds[6]; L.act2 = G.lds[7]; L.scr = G.lds[8]; L.kvb = G.lds[9]; L.total = 0;
    return L;
}
struct LdsB { size_t act, work, gu, act2, scr, total; };
__host__ __device__ inline LdsB lds_b(int dt, int dim, const l3m_dchunk &c) {
    LdsB L;
    size_t o = 0;
    const size_t pg = (size_t)c.gate_up.tiles * c.gate_up.nb, pw = (size_t)c.down.tiles * c.down.nb;
    L.act = o;  o += align16(act_size(dt, kwide(dim)));
    L.work = o; o += work_bytes(res_bytes(pg), res_bytes(pw));
    L.gu = o;   o += align16(64 * (size_t)c.gate_up.tiles);
    L.act2 = o; o += align16(act_size(dt, c.nf));
    L.scr = o;  o += 4 * 64;
    L.total = o;
    return L;
}
__device__ __forceinline__ LdsB lds_of(const l3m_dchunk &C) {
    LdsB L;
    L.act = C.lds[0]; L.work = C.lds[1]; L.gu = C.lds[2]; L.act2 = C.lds[3]; L.scr = C.lds[4]; L.total = 0;
    return L;
}
struct LdsH { size_t act, work, scr, lgv, total; };
__host__ __device__ inline LdsH lds_h(int dt, int dim, int nb, int tiles_per_wg) {
    LdsH L;
    size_t o = 0;
    L.act = o;  o += align16(act_size(dt, kwide(dim)));
    L.work = o; o += work_bytes(res_bytes((size_t)tiles_per_wg * nb), 0);
    L.scr = o;  o += 4 * 64;
    L.lgv = o;  o += align16(4 * 16 * (size_t)tiles_per_wg);   // the slice's logits, kept for sampling
    L.total = o;
    return L;
}

// K and V rows 0..pos-1 of the group's kv heads, copied from the cache into the LDS window (K [nkv][ctx]
// [kv_row(hd)], then V the same or, vt, transposed). Rows up to pos - 1 were written by earlier steps, so
// the copy can start at the top of the kernel. Row-major rows go by the memory unit (global_load_lds_dwordx4:
// 64 lanes x 16 bytes into 1 KiB of LDS, no registers); V^T through registers, each lane taking one
// position's 8 dimensions and storing them down 8 rows of V^T, with zeros at the positions past pos up to
// the end of the 32-position step (P.V reads them with p = 0; zeros keep the products finite). Position
// pos is the block's own (written with this step's rows).
template <bool COH>
__device__ void kv_window_dma(uint16_t *kvb, const l3m_dmodel &M, int layer, int kv0, int nkv, int pos, bool vt) {
    const int wave = wave_id(), lane = tidx() & 63, hd = M.hd, rs = kv_row(hd);
    const size_t cwin = (size_t)M.ctx * hd, lwin = (size_t)M.kv_win * rs;   // per head: cache, LDS window
    // one row per instruction (the window's rows are padded apart, so a copy cannot span rows): hd / 8
    // lanes of 16 bytes each
    for (int head = 0; head < (vt ? nkv : 2 * nkv); head++) {
        const int which = head >= nkv ? 1 : 0, j = head - which * nkv;
        const uint16_t *src = (which ? M.vc : M.kc) + ((size_t)layer * M.n_kv + kv0 + j) * cwin;
        uint16_t *dst = kvb + (size_t)head * lwin;
        for (int t = wave; t < pos; t += NWE)
            if (lane < (hd >> 3))
                __builtin_amdgcn_global_load_lds((const GLOBAL void *)(src + (size_t)t * hd + 8 * lane),
                                                 (__attribute__((address_space(3))) void *)(dst + (size_t)t * rs), 16, 0,
                                                 COH ? 16 : 0);   // 16: sc1
    }
    if (!vt) return;
    const int vr = vt_row(M.kv_win), tend = (pos + 32) & ~31;   // the step of position pos ends at tend (<= kv_win)
    for (int j = 0; j < nkv; j++) {
        const uint16_t *src = M.vc + ((size_t)layer * M.n_kv + kv0 + j) * cwin;
        uint16_t *dst = kvb + (size_t)nkv * lwin + (size_t)j * hd * vr;
        for (int c = wave; c < (hd >> 3); c += NWE)
            for (int t = lane; t < tend; t += 64) {
                if (t == pos) continue;
                uint4 v = make_uint4(0u, 0u, 0u, 0u);
                if (t < pos) v = ld16<COH>(src, (size_t)t * (hd >> 3) + c);   // uniform base, 16-byte index
                uint16_t *d = dst + (size_t)(8 * c) * vr + t;
                d[0] = (uint16_t)v.x; d[vr] = (uint16_t)(v.x >> 16); d[2 * vr] = (uint16_t)v.y; d[3 * vr] = (uint16_t)(v.y >> 16);
                d[4 * vr] = (uint16_t)v.z; d[5 * vr] = (uint16_t)(v.z >> 16); d[6 * vr] = (uint16_t)v.w; d[7 * vr] = (uint16_t)(v.w >> 16);
            }
    }
}

__device__ __forceinline__ float dot8_bf16(const float *q, uint4 k, float acc) {
    acc = fmaf(q[0], bf16_f32(k.x & 0xFFFF), acc); acc = fmaf(q[1], bf16_f32(k.x >> 16), acc);
    acc = fmaf(q[2], bf16_f32(k.y & 0xFFFF), acc); acc = fmaf(q[3], bf16_f32(k.y >> 16), acc);
    acc = fmaf(q[4], bf16_f32(k.z & 0xFFFF), acc); acc = fmaf(q[5], bf16_f32(k.z >> 16), acc);
    acc = fmaf(q[6], bf16_f32(k.w & 0xFFFF), acc); acc = fmaf(q[7], bf16_f32(k.w >> 16), acc);
    return acc;
}

// Attention of the group's query heads over positions 0..pos (ops.c:58-73), split-softmax form: each
// head takes W wavefronts, W from the context length (at most ATT_IT position rounds per wavefront, and
// no more wavefronts than the workgroup has per head). In a wavefront, lane j of each aligned group of
// LP lanes holds dims [8j, 8j+8) of one position (LP = hd/8 rounded up to a power of two); a round scores
// 64/LP positions (lane-group sums), and the wavefront keeps a running max m, a running sum l of
// exp(s - m) and the running exp-weighted V sum o, rescaled when m grows. With W > 1 the wavefronts'
// (m, l, o) meet in LDS after one barrier and combine as exp(m_w - M) weights. K, V rows before pos come
// from the LDS window (WIN) or the cache, row pos from cur (this step's rows, bf16 as the cache holds
// them). BATCH (from the cache): a chunk's K and V rows are all requested first, by buffer loads that answer a row
// past the end with zeros and no access; loads under a branch a round are waited for one after the other. Taken by
// the bodies with int8 step matrices, which have the 32 registers (8 heads of 64, 8 layers, positions 600-664: 4.5
// us a pass less); a bf16 body's step spills with it (stories15M, which never reads the cache: 2% slower).
// vred: NWE * (hd + 2) floats of LDS. Ends with a barrier.
#ifndef L3M_ATT_LOG_IT
#define L3M_ATT_LOG_IT 2
#endif
constexpr int ATT_LOG_IT = L3M_ATT_LOG_IT, ATT_IT = 1 << ATT_LOG_IT;
template <bool WIN, bool COH, bool BATCH>
__device__ void attend_group(const l3m_dmodel &M, const l3m_dgroup &G, int layer, int pos, const float *qh, const uint16_t *cur,
                             const uint16_t *kvb, float *vred, float *att) {
    const int hd = M.hd, nv = hd >> 3, lg = nv <= 4 ? 2 : nv <= 8 ? 3 : nv <= 16 ? 4 : 5, LP = 1 << lg, PPW = 64 >> lg;
    const int lane = tidx() & 63, wave = wave_id(), j = lane & (LP - 1), gl = lane >> lg, n = pos + 1;
    const float scale = M.att_scale, ihpk = __builtin_amdgcn_rcpf((float)M.hpk);
    const int rs = WIN ? kv_row(hd) : hd;             // row stride: LDS window or cache
    const size_t win = (size_t)(WIN ? M.kv_win : M.ctx) * rs;
    // W = 2^wl wavefronts per head: the fewest that keep each at ATT_IT rounds or less, at most 2^att_wl
    const int sh = ATT_LOG_IT + 6 - lg;               // ATT_IT * PPW = 2^sh positions per wavefront
    const int need = (n + (1 << sh) - 1) >> sh;
    int wl = need <= 1 ? 0 : 32 - __builtin_clz((unsigned)(need - 1));
    wl = wl < G.att_wl ? wl : G.att_wl;
    const int W = 1 << wl, HB = NWE >> wl;            // heads per batch
    float *ml = vred + NWE * hd;                      // (m, l) per wavefront
    for (int h0 = 0; h0 < G.nq; h0 += HB) {
        const int h = h0 + (wave >> wl), wi = wave & (W - 1);
        const bool active = h < G.nq;
        if (active) {
            // (q0 + h) / hpk by an exact float reciprocal (both far below 2^20)
            const int kvl = (int)(((float)(G.q0 + h) + 0.5f) * ihpk) - G.kv0;
            const uint16_t *kw = WIN ? kvb + kvl * win : M.kc + ((size_t)layer * M.n_kv + G.kv0 + kvl) * win;
            const uint16_t *vw = WIN ? kvb + (G.nkv + kvl) * win : M.vc + ((size_t)layer * M.n_kv + G.kv0 + kvl) * win;
            const uint4 *kcur = (const uint4 *)(cur + kvl * hd), *vcur = (const uint4 *)(cur + (G.nkv + kvl) * hd);
            float q[8];
            {
                const float4 a = j < nv ? ((const float4 *)(qh + h * hd))[2 * j] : make_float4(0.f, 0.f, 0.f, 0.f);
                const float4 b = j < nv ? ((const float4 *)(qh + h * hd))[2 * j + 1] : make_float4(0.f, 0.f, 0.f, 0.f);
                q[0] = a.x; q[1] = a.y; q[2] = a.z; q[3] = a.w; q[4] = b.x; q[5] = b.y; q[6] = b.z; q[7] = b.w;
            }
            float m = -INFINITY, l = 0.f, o[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
            // rounds r = 0, 1, ... cover positions (r * W + wi) * PPW + gl; ATT_IT rounds per chunk
            for (int r0 = 0; (r0 * W + wi) * PPW < n; r0 += ATT_IT) {
                if constexpr (BATCH) {
                    // buffers over the layer's rows (a uniform base), the head's from row0 on; own: the position whose row is
                    // cur's. Lanes past the head keep zeros (their zero q times an infinity is NaN)
                    const uint16_t *kl = M.kc + (size_t)layer * M.n_kv * win, *vl = M.vc + (size_t)layer * M.n_kv * win;
                    const uint32_t row0 = (uint32_t)((G.kv0 + kvl) * M.ctx);
                    const int own = j < nv ? pos : -1;
                    float s[ATT_IT];
                    float cm = -INFINITY;
                    uint4 kb[ATT_IT], vb[ATT_IT];
#pragma unroll
                    for (int k = 0; k < ATT_IT; k++) {
                        const int t = ((r0 + k) * W + wi) * PPW + gl;
                        kb[k] = ld16_if<COH>(kl, 16 * ((row0 + (uint32_t)t) * (uint32_t)nv + (uint32_t)j), t < pos && j < nv);
                    }
#pragma unroll
                    for (int k = 0; k < ATT_IT; k++) {
                        const int t = ((r0 + k) * W + wi) * PPW + gl;
                        vb[k] = ld16_if<COH>(vl, 16 * ((row0 + (uint32_t)t) * (uint32_t)nv + (uint32_t)j), t < pos && j < nv);
                    }
                    asm volatile("" ::: "memory");
                    const uint4 kc = kcur[j < nv ? j : 0], vc = vcur[j < nv ? j : 0];
#pragma unroll
                    for (int k = 0; k < ATT_IT; k++)
                        if (((r0 + k) * W + wi) * PPW + gl == own) { kb[k] = kc; vb[k] = vc; }
#pragma unroll
                    for (int k = 0; k < ATT_IT; k++) {
                        const int t = ((r0 + k) * W + wi) * PPW + gl;
                        const float part = dot8_bf16(q, kb[k], 0.f);
                        s[k] = t < n ? lanes_sum_n(part, LP) * scale : -INFINITY;
                        cm = fmaxf(cm, s[k]);
                    }
                    const float mn = fmaxf(m, lanes_max<64>(cm));
                    const float alpha = expf(m - mn);
                    l *= alpha;
#pragma unroll
                    for (int e = 0; e < 8; e++) o[e] *= alpha;
#pragma unroll
                    for (int k = 0; k < ATT_IT; k++) {  // past the end p is 0 and the row zeros
                        const float p = expf(s[k] - mn);
                        l += p;
                        const uint4 vv = vb[k];
                        o[0] = fmaf(p, bf16_f32(vv.x & 0xFFFF), o[0]); o[1] = fmaf(p, bf16_f32(vv.x >> 16), o[1]);
                        o[2] = fmaf(p, bf16_f32(vv.y & 0xFFFF), o[2]); o[3] = fmaf(p, bf16_f32(vv.y >> 16), o[3]);
                        o[4] = fmaf(p, bf16_f32(vv.z & 0xFFFF), o[4]); o[5] = fmaf(p, bf16_f32(vv.z >> 16), o[5]);
                        o[6] = fmaf(p, bf16_f32(vv.w & 0xFFFF), o[6]); o[7] = fmaf(p, bf16_f32(vv.w >> 16), o[7]);
                    }
                    m = mn;
                    continue;
                }
                float s[ATT_IT];
                float cm = -INFINITY;
#pragma unroll
                for (int k = 0; k < ATT_IT; k++) {
                    const int t = ((r0 + k) * W + wi) * PPW + gl;
                    float part = 0.f;
                    if (t < n && j < nv) {
                        uint4 kk;
                        if (t == pos) kk = kcur[j];
                        else if (WIN) kk = ((const uint4 *)(kw + (size_t)t * rs))[j];
                        else kk = ld16<COH>(kw, (size_t)t * (hd >> 3) + j);
                        part = dot8_bf16(q, kk, 0.f);
                    }
                    s[k] = t < n ? lanes_sum_n(part, LP) * scale : -INFINITY;
                    cm = fmaxf(cm, s[k]);
                }
                const float mn = fmaxf(m, lanes_max<64>(cm));
                const float alpha = expf(m - mn);     // m = -inf at the start: alpha = 0
                l *= alpha;
#pragma unroll
                for (int e = 0; e < 8; e++) o[e] *= alpha;
#pragma unroll
                for (int k = 0; k < ATT_IT; k++) {
                    const int t = ((r0 + k) * W + wi) * PPW + gl;
                    if (t < n) {
                        const float p = expf(s[k] - mn);
                        l += p;
                        if (j < nv) {
                            uint4 vv;
                            if (t == pos) vv = vcur[j];
                            else if (WIN) vv = ((const uint4 *)(vw + (size_t)t * rs))[j];
                            else vv = ld16<COH>(vw, (size_t)t * (hd >> 3) + j);
                            o[0] = fmaf(p, bf16_f32(vv.x & 0xFFFF), o[0]); o[1] = fmaf(p, bf16_f32(vv.x >> 16), o[1]);
                            o[2] = fmaf(p, bf16_f32(vv.y & 0xFFFF), o[2]); o[3] = fmaf(p, bf16_f32(vv.y >> 16), o[3]);
                            o[4] = fmaf(p, bf16_f32(vv.z & 0xFFFF), o[4]); o[5] = fmaf(p, bf16_f32(vv.z >> 16), o[5]);
                            o[6] = fmaf(p, bf16_f32(vv.w & 0xFFFF), o[6]); o[7] = fmaf(p, bf16_f32(vv.w >> 16), o[7]);
                        }
                    }
                }
                m = mn;
            }
            // over the wavefront's position groups: lanes j < LP end up with the sums
#pragma unroll
            for (int e = 0; e < 8; e++) o[e] = strided_sum(o[e], LP);
            l = strided_sum(l, LP);
            if (W == 1) {
                if (lane < LP && j < nv) {
                    const float inv = 1.0f / l;
                    float4 *d = (float4 *)(att + h * hd + 8 * j);
                    d[0] = make_float4(o[0] * inv, o[1] * inv, o[2] * inv, o[3] * inv);
                    d[1] = make_float4(o[4] * inv, o[5] * inv, o[6] * inv, o[7] * inv);
                }
            } else {
                if (lane < LP && j < nv) {
                    float4 *d = (float4 *)(vred + wave * hd + 8 * j);
                    d[0] = make_float4(o[0], o[1], o[2], o[3]);
                    d[1] = make_float4(o[4], o[5], o[6], o[7]);
                }
                if (lane == 0) { ml[2 * wave] = m; ml[2 * wave + 1] = l; }
            }
        }
        if (W > 1) {
            __syncthreads();
            // head h's W wavefronts combine: dims d = wi * 64 + lane, + 64 * W, ... of the head
            if (active) {
                const int w0 = wave - wi;
                float mx = ml[2 * w0];
                for (int k = 1; k < W; k++) mx = fmaxf(mx, ml[2 * (w0 + k)]);
                for (int d = wi * 64 + lane; d < hd; d += 64 * W) {
                    float num = 0.f, den = 0.f;
                    for (int k = 0; k < W; k++) {
                        const float a = expf(ml[2 * (w0 + k)] - mx);
                        den = fmaf(a, ml[2 * (w0 + k) + 1], den);
                        num = fmaf(a, vred[(w0 + k) * hd + d], num);
                    }
                    att[h * hd + d] = num / den;
                }
            }
        }
        __syncthreads();
    }
}

// bf16 vectors for the gfx950 MFMA v_mfma_f32_16x16x32_bf16: A is 16 x 32, B 32 x 16, C 16 x 16 f32.
// Lane l supplies A[l % 16][8 (l / 16) + e] and B[8 (l / 16) + e][l % 16] (e = 0..7) and holds
// C[4 (l / 16) + r][l % 16] (r = 0..3).
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
__device__ __forceinline__ f32x4 mfma_bf16(bf16x8 a, bf16x8 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
// The bf16 wide matrices (q/k/v rows, gate/up rows, the head) on the matrix cores: wavefront w takes tiles
// w, w + NWE, ... in turn, and a tile's blocks go through v_mfma_f32_16x16x32_bf16 one after the other, the
// block's 16 x 32 weights as A, the activation's 32 values in every column of B, each product accumulating
// onto the last (C). Every column of the result then holds the tile's 16 row sums, already in lanes: no
// cross-lane sum, no LDS round trip, no barrier, and a quarter of the instructions of the v_dot2 form (one
// per block where each lane of that form spends 16 v_dot2 on its block). Lane l holds A's row l % 16,
// inputs 8 (l / 16) .. + 7 of each block: the 16-byte piece l / 16 of its row, so a block's 64 pieces are
// its 1 KiB of the lane-tile plane, one load per lane, as the other forms read it. The products of bf16
// values are exact in f32; the sums are f32 (the order differs from the v_dot2 form's, within its bounds).
// PrefM holds MK blocks of one tile: the most that fit the bf16 roles' registers (36 VGPRs, where the
// v_dot2 form's two slots take 32), which is every block of a 288-input row; longer rows take further
// batches of MK, loaded in turn.
constexpr int MK = 9;
struct PrefM { uint4 a[MK]; };
template <int DT, int NS> struct WideSel { using T = Pref<DT, NS>; };
template <int NS> struct WideSel<L3M_BF16, NS> { using T = PrefM; };
// The register batch of a wide matrix of dtype DT (NS slots in the v_dot2 and integer forms).
template <int DT, int NS> using Wide = typename WideSel<DT, NS>::T;

// Blocks b0 .. b0 + MK - 1 of tile t (past nb: zeros, no memory access, not used). A wavefront with no tile
// issues nothing: the bf16 roles have the registers to spare for the branch (no spills), and the loads it
// saves cost more than loads past the range (measured: stories15M 16,018 -> 16,380 tok/s). The integer
// roles, at their register limit, spill with it and keep loads past the range (ldg16_if) instead.
__device__ __forceinline__ void prefm_load(PrefM &pf, const l3m_dmat &m, int t, int b0) {
    const int lane = tidx() & 63, nb = m.nb;
    const size_t piece = (size_t)(lane & 15) * 4 + (lane >> 4);   // uint4 of the block: row l % 16, piece l / 16
    if (t >= m.tiles) return;                         // no tile for this wavefront (uniform)
#pragma unroll
    for (int k = 0; k < MK; k++) {
        const int b = b0 + k;
        pf.a[k] = ldg16_if(m.q, ((size_t)t * nb + b) * 64 + piece, b < nb);
    }
}
// The matvec of a bf16 matrix in this form (the wavefront's first batch loaded by prefm_load beforehand),
// act the bf16 activation in LDS. f(i, y, partner, lead) runs for each of the tile's 16 rows in the lanes
// l with 4 (l / 16) + l % 4 = the row's place in the tile (lead: (l / 4) % 4 == 0), partner being row
// i ^ 1's value (the neighbouring lane), as the other forms call it.
template <class F>
__device__ __forceinline__ void tile_rows_mfma(PrefM &pf, const l3m_dmat &m, const uint8_t *act, int rows, F f) {
    const int wave = wave_id(), lane = tidx() & 63, nb = m.nb, q = lane & 3;
    const uint4 *xb = (const uint4 *)act + (lane >> 4);   // block b's piece: xb[4 b]
    auto batch = [&](f32x4 c, int b0) {
        // pin the loaded registers here, as pref_compute does
#pragma unroll
        for (int k = 0; k < MK; k++) asm volatile("" : "+v"(pf.a[k].x), "+v"(pf.a[k].y), "+v"(pf.a[k].z), "+v"(pf.a[k].w));
#pragma unroll
        for (int k = 0; k < MK; k++) {
            if (b0 + k >= nb) break;
            c = mfma_bf16(__builtin_bit_cast(bf16x8, pf.a[k]), __builtin_bit_cast(bf16x8, xb[4 * (b0 + k)]), c);
        }
        return c;
    };
    auto finish = [&](f32x4 c, int t) {
        const float y = q == 0 ? c[0] : q == 1 ? c[1] : q == 2 ? c[2] : c[3];
        const float partner = dppf<QP_X1>(y);        // row i ^ 1 is the neighbouring lane
        const int i = t * 16 + 4 * (lane >> 4) + q;
        if (i < rows) f(i, y, partner, ((lane >> 2) & 3) == 0);
    };
    if (wave < m.tiles) {
        f32x4 c = {0.f, 0.f, 0.f, 0.f};
        c = batch(c, 0);
        for (int b0 = MK; b0 < nb; b0 += MK) {
            prefm_load(pf, m, wave, b0);
            c = batch(c, b0);
        }
        finish(c, wave);
        for (int t = wave + NWE; t < m.tiles; t += NWE) {
            c = f32x4{0.f, 0.f, 0.f, 0.f};
            for (int b0 = 0; b0 < nb; b0 += MK) {
                prefm_load(pf, m, t, b0);
                c = batch(c, b0);
            }
            finish(c, t);
        }
    }
}

// x as the sum of three bf16 (each rounded to nearest even from what is left): exact to 2^-24 of x, so
// three bf16 products with an exact bf16 operand give x * y to f32 accuracy.
__device__ __forceinline__ void split3(float x, __bf16 &h, __bf16 &m, __bf16 &l) {
    h = (__bf16)x;
    const float r = x - (float)h;
    m = (__bf16)r;
    l = (__bf16)(r - (float)m);
}

// Attention of the group's query heads over positions 0..pos (ops.c:58-73) on the matrix cores, for a
// head dimension that is a multiple of 16, with every K, V row in the LDS window (row stride kv_row(hd),
// row pos included: the block stores this step's rows there first). q and p are split into three bf16
// parts (split3), so each product with an exact bf16 operand is f32 exact; the three parts ride in rows
// 0-2 of the A operand of one product, the other 13 rows zero, and their sums, which land in one lane,
// are added (h + m) + l. One head at a time, three passes with a barrier after each:
//  1. scores: wavefront w takes 16-position tiles w, w + NWE, ...: S = A (row j < 3 = q's part j) times
//     K_tile^T (hd x 16, B taken from the window as it lies: lane l supplies row l % 16); lane t < 16 holds
//     rows 0-3 of column t, so s_t = ((S[0][t] + S[1][t]) + S[2][t]) / sqrt(hd) in one lane, into sc, and
//     each wavefront's maximum into smax;
//  2. p_t = exp(s_t - m) over the head's maximum m, stored as three bf16 parts (zero past pos, up to a
//     multiple of 32), and each wavefront's sum of p into lpart;
//  3. o = P V: wavefront w takes dims [16w, 16w + 16): 32 positions per step, A row j < 3 = p's part j,
//     B = V^T rows, 32 positions at a time; lanes 0-15 hold rows 0-3 of their dim's column, and
//     att = ((row 0 + row 1) + row 2) / sum(lpart).
// sc: 10 * ceil32(ctx) bytes of LDS; vred: 2 * NWE floats; qp: [3][nq * hd] bf16. Ends with a barrier.
__device__ void attend_mfma(const l3m_dmodel &M, const l3m_dgroup &G, int pos, const __bf16 *qp, const uint16_t *kvb, float *sc,
                            float *vred, float *att) {
    const int hd = M.hd, rs = kv_row(hd), vr = vt_row(M.kv_win), ctx = M.kv_win, n = pos + 1;   // ctx: the window's
    const int lane = tidx() & 63, wave = wave_id(), li = lane & 15, lg = lane >> 4;
    const float scale = M.att_scale, ihpk = __builtin_amdgcn_rcpf((float)M.hpk);
    const size_t win = (size_t)ctx * rs;
    const int tiles = (n + 15) >> 4, steps = (n + 31) >> 5, cap = (ctx + 31) & ~31, nqd = G.nq * hd;
    const int part = li < 3 ? li : 0;                 // the q (p) part this lane supplies, when li < 3
    const bf16x8 z = {};
    float *s_arr = sc, *smax = vred, *lpart = vred + NWE;
    __bf16 *pp = (__bf16 *)(sc + cap);                // [3][cap]
    for (int h = 0; h < G.nq; h++) {
        // (q0 + h) / hpk by an exact float reciprocal (both far below 2^20)
        const int kvl = (int)(((float)(G.q0 + h) + 0.5f) * ihpk) - G.kv0;
        const uint16_t *kw = kvb + (size_t)kvl * win, *vw = kvb + (size_t)G.nkv * win + (size_t)kvl * hd * vr;   // V^T
        float mx = -INFINITY;
        for (int T = wave; T < tiles; T += NWE) {
            const int row = T * 16 + li < n ? T * 16 + li : n - 1;
            f32x4 c = {0.f, 0.f, 0.f, 0.f};
            for (int kk = 0; kk < hd; kk += 32) {
                bf16x8 a = *(const bf16x8 *)(qp + part * nqd + h * hd + kk + 8 * lg),
                       b = *(const bf16x8 *)(kw + (size_t)row * rs + kk + 8 * lg);
                asm volatile("" : "+v"(a), "+v"(b));   // both read before the product
                // rows 3-15 of A are zero; so is the upper half of the last step when hd = 32 j + 16
                // (what was read there, the row's padding or the next head's q, is never multiplied)
                const bool live = kk + 8 * lg < hd;
                a = live && li < 3 ? a : z;
                b = live ? b : z;
                c = mfma_bf16(a, b, c);
            }
            // lanes 0-15: rows 0-2 (the parts) of column li, position T * 16 + li
            const int t = T * 16 + li;
            const float sv = ((c[0] + c[1]) + c[2]) * scale;
            const bool mine = lg == 0 && t < n;
            if (lg == 0) s_arr[t] = mine ? sv : -INFINITY;
            mx = fmaxf(mx, mine ? sv : -INFINITY);
        }
        if (wave < tiles) {                           // lane 0: the maximum over lanes 0-15
            mx = lanes_max<16>(mx);
        }
        if (lane == 0) smax[wave] = mx;
        __syncthreads();
        const float m = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(lanes_max<16>(smax[li]))));
        float lw = 0.f;
        for (int t = tidx(); t < 32 * steps; t += NTE) {
            const float p = t < n ? expf(s_arr[t] - m) : 0.f;
            split3(p, pp[t], pp[cap + t], pp[2 * cap + t]);
            lw += p;
        }
        if (wave * 64 < 32 * steps) lw = lanes_sum<64>(lw);   // wavefronts past the positions hold 0
        if (lane == 0) lpart[wave] = lw;
        __syncthreads();
        for (int dt = wave; dt < (hd >> 4); dt += NWE) {
            f32x4 c = {0.f, 0.f, 0.f, 0.f};
            // two 32-position steps per round, every operand read before the first product; a second
            // step past the end reads step k's operands again and is not multiplied. A: row li < 3 = p's
            // part li at positions t0..t0+7 (zero rows past 3); B: V^T row 16 dt + li, the same positions
            // (past pos the window holds zeros, p is zero there)
            for (int k = 0; k < steps; k += 2) {
                bf16x8 a[2], b[2];
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    const int t0 = 32 * (k + u < steps ? k + u : k) + 8 * lg;
                    a[u] = *(const bf16x8 *)(pp + part * cap + t0);
                    b[u] = *(const bf16x8 *)(vw + (size_t)(16 * dt + li) * vr + t0);
                }
#pragma unroll
                for (int u = 0; u < 2; u++) {
                    asm volatile("" : "+v"(a[u]), "+v"(b[u]));
                    a[u] = li < 3 ? a[u] : z;
                }
                c = mfma_bf16(a[0], b[0], c);
                if (k + 1 < steps) c = mfma_bf16(a[1], b[1], c);
            }
            // the wavefronts' sums of p: lane k < NWE reads wavefront k's (lanes 16 and up repeat them)
            const float l = __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(lanes_sum<16>(lpart[li]))));
            if (lg == 0) att[h * hd + 16 * dt + li] = ((c[0] + c[1]) + c[2]) / l;
        }
        __syncthreads();
    }
}

// ------------------------------------------------------------------ step blocks (device functions)
// One block each for the attention of a head group, the FFN of a chunk and a slice of the head. The
// graph path launches each as its own kernel (k_attn_block, k_ffn_block, k_head_block); the persistent
// path (k_decode) calls them from resident workgroups. PRE: the block's weights were issued into w
// already (the persistent path issues them while it waits for the block's inputs); otherwise they are
// issued right after the prologue's loads.

// The storage dtype of the step blocks' matrices (q/k/v rows, Wo columns, gate/up rows, Wdown columns)
// for a body of dtype DT. A q4_0 body holds them as q8_0: the same blocks with each nibble q widened to
// the byte q - 8 and the same scale, so every integer dot and every float operation is the one q4_0 would
// do, while the slot loop skips the nibble unpacking. The head stays q4_0.
#ifdef L3M_Q4_STEPS_NATIVE
// Measurement build only (make -C l3m_amd/csrc q4native): q4_0 step matrices kept as q4_0 blocks.
template <int DT> constexpr int a_dtype() { return DT; }
#else
template <int DT> constexpr int a_dtype() { return DT == L3M_Q4_0 ? L3M_Q8_0 : DT; }
#endif
template <int DT> struct AttnW { Wide<a_dtype<DT>(), nslot_a<DT>()> a; Pref<a_dtype<DT>(), nslot_wo<DT>()> b; ProStatic st; };
template <int DT> struct FfnW { Wide<a_dtype<DT>(), nslot_a<DT>()> a; Pref<a_dtype<DT>(), nslot_b<DT>()> b; ProStatic st; };
template <int DT> struct HeadW { Wide<DT, nslot_h<DT>()> a; ProStatic st; };

// A block's static prologue inputs (ProStatic), issued ahead of its weights.
__device__ __forceinline__ void attn_static(ProStatic &st, const l3m_dmodel &M, const l3m_dlayer &Lw, int pos) {
    pro_static(st, M.dim >> 2, Lw.attn_norm, M.rope + (size_t)pos * M.hd, M.hd);
}
__device__ __forceinline__ void ffn_static(ProStatic &st, const l3m_dmodel &M, const l3m_dlayer &Lw) {
    pro_static(st, M.dim >> 2, Lw.ffn_norm, nullptr, 0);
}

template <int DT, int NS> __device__ __forceinline__ void wide_issue(Pref<DT, NS> &pf, const l3m_dmat &m) {
    if constexpr (tiled<DT>()) pref_load_tile<DT, NS>(pf, m, wave_id(), 0);
    else pref_load<DT, NS>(pf, m, 0);
}
__device__ __forceinline__ void wide_issue(PrefM &pf, const l3m_dmat &m) { prefm_load(pf, m, wave_id(), 0); }
template <int DT, int NS, class F>
__device__ __forceinline__ void wide_rows(Pref<DT, NS> &pf, const l3m_dmat &m, const uint8_t *act, int kp, float *res, int rows, F f) {
    if constexpr (tiled<DT>()) {
        tile_rows<DT, NS>(pf, m, act, kp, rows, f);
    } else {
        mv<DT, NS>(pf, m, act, kp, res);
        __syncthreads();
        rows_sum4(m, res, rows, f);
    }
}
template <class F>
__device__ __forceinline__ void wide_rows(PrefM &pf, const l3m_dmat &m, const uint8_t *act, int, float *, int rows, F f) {
    tile_rows_mfma(pf, m, act, rows, f);
}
template <int DT> __device__ __forceinline__ void attn_issue(AttnW<DT> &w, const l3m_dgroup &G) {
    wide_issue(w.a, G.qkv);
    pref_load<a_dtype<DT>(), nslot_wo<DT>()>(w.b, G.wo, 0);
}
template <int DT> __device__ __forceinline__ void ffn_issue(FfnW<DT> &w, const l3m_dchunk &C) {
    wide_issue(w.a, C.gate_up);
    pref_load<a_dtype<DT>(), nslot_b<DT>()>(w.b, C.down, 0);
}
template <int DT> __device__ __forceinline__ void head_issue(HeadW<DT> &w, const l3m_dmat &V) {
    wide_issue(w.a, V);
}

// The persistent path's K/V window copy for the attention block of group G at (layer, pos): rows
// 0..pos-1 were written in earlier steps, so it can run while the block waits for its inputs.
template <int DT>
__device__ __forceinline__ void attn_kv_window(const l3m_dmodel &M, const l3m_dgroup &G, int layer, int pos, uint8_t *smem) {
    if (!M.kv_lds || pos >= M.kv_win) return;
    const LdsA L = lds_of(G);
    kv_window_dma<true>((uint16_t *)(smem + L.kvb), M, layer, G.kv0, G.nkv, pos, mfma_fits(M.hd, G.nq, M.kv_win));
}

// The attention block of head group gi (engine.c:236-258) at `layer`, position pos: x = xb + the FFN
// partials (layer 0: the embedding row of tokens[pos]), RMSNorm, prep, the group's q/k/v rows, RoPE,
// bf16 K/V into the cache, attention, prep, the group's Wo columns -> po[gi]. Group 0 keeps x in xa.
// This step's k and v rows (bf16, engine.c:247-248, in cur) into the cache, for the kv heads group G
// writes: element i0, i0 + step, ... of the 2 nkv hd.
__device__ __forceinline__ void kv_rows_store(const l3m_dmodel &M, const l3m_dgroup &G, int layer, int pos, const uint16_t *cur, int i0,
                                              int step) {
    const int hd = M.hd, nkd = G.nkv * hd;
    const float inv_hd = 1.0f / (float)hd;            // i / hd by an exact float reciprocal (i, hd < 2^12)
    for (int i = i0; i < 2 * nkd; i += step) {
        const int kv = i < nkd ? 0 : 1, jj = i - kv * nkd, kvl = (int)(((float)jj + 0.5f) * inv_hd);
        if (G.write_kv >> kvl & 1u)
            gw(kv ? M.vc : M.kc)[(((size_t)layer * M.n_kv + G.kv0 + kvl) * M.ctx + pos) * hd + (jj - kvl * hd)] = cur[i];
    }
}

template <int DT, bool PRE, bool G2 = false>
__device__ __forceinline__ void attn_block(const l3m_dmodel &M, const l3m_dlayer &Lw, const l3m_dgroup &G, int layer, int pos,
                                           int tok, int gi, AttnW<DT> &w, uint8_t *smem) {
    const int tid = tidx(), dim = M.dim, hd = M.hd, kp = kwide(dim);
    const LdsA L = lds_of(G);
    float *work = (float *)(smem + L.work), *qh = (float *)(smem + L.q), *cs = (float *)(smem + L.cs);
    float *vred = (float *)(smem + L.vred), *att = (float *)(smem + L.att);
    uint16_t *cur = (uint16_t *)(smem + L.cur), *kvb = (uint16_t *)(smem + L.kvb);
    uint8_t *act = smem + L.act, *act2 = smem + L.act2;
    Red red{(float *)(smem + L.scr), 0};

    Pro P;
    const ProGeom PG = pro_geom(M, 0);
    if constexpr (!PRE) attn_static(w.st, M, Lw, pos);
    pro_load<PRE>(P, M.xb, M.pd, PG, M.embed, layer == 0, tok);
    if constexpr (!PRE) attn_issue<DT>(w, G);
    float4 x = pro_finish<PRE>(P, M.pd, PG, layer == 0, (float4 *)work, G2 && layer == 0 ? nullptr : gi == 0 ? M.xa : nullptr, cs, w.st.cs, hd);
    phase(gi, 2, pos, layer);
    if constexpr (G2) {
        if (layer == 0) {                             // the learned position row (engine.c:237), then kept
            if (tid < (dim >> 2)) x = add4(x, ((const float4 *)(M.pos_embed + (size_t)pos * dim))[tid]);
            if (gi == 0 && tid < (dim >> 2)) ((float4 *)M.xa)[tid] = x;
        }
    }
    // K, V rows 0..pos-1 (no dependence on this step). Issued after the prologue is consumed: a copy of
    // data-dependent length ahead of it would make the compiler wait for every load in flight there.
    // The persistent path issues it before it waits for the block's inputs (attn_kv_window).
    const bool kwin = M.kv_lds && pos < M.kv_win;    // rows 0..pos fit the LDS window at this step
    if (!PRE && kwin) kv_window_dma<false>(kvb, M, layer, G.kv0, G.nkv, pos, mfma_fits(hd, G.nq, M.kv_win));
    constexpr int AT = a_dtype<DT>();                // the activations take the form the step matrices read
    if constexpr (G2) ln_prep<AT>(x, Lw.attn_norm, Lw.attn_norm_b, dim, kp, M.eps, act, red);
    else norm_prep<AT>(x, w.st.nw, dim, kp, M.eps, act, red);
    phase(gi, 3, pos, layer);

    // q, k rows: RoPE on pairs (2i, 2i+1) of each head by the angle i (ops.c:29-40); k, v rows rounded
    // to bf16 as the cache holds them (engine.c:247-248), into cur, row pos of the LDS window and, for the
    // heads this group writes, the cache
    const int nqd = G.nq * hd, nkd = G.nkv * hd;
    const float inv_hd = 1.0f / (float)hd;            // i / hd by an exact float reciprocal (i, hd < 2^12)
    // the matrix-core attention (LDS window, hd a multiple of 16, q parts fit beside vred's 2 NWE sums)
    const bool mfma_att = kwin && mfma_fits(hd, G.nq, M.kv_win);
    __bf16 *qp = (__bf16 *)(vred + 2 * NWE);
    auto qkv_row = [&](int i, float y, float partner, bool lead) {
        if constexpr (G2) y += G.bqkv[i];            // the GPT-2 variant's q, k, v biases; no RoPE
        if (!G2 && i < nqd + nkd) {
            const int local = i < nqd ? i : i - nqd, head = (int)(((float)local + 0.5f) * inv_hd);
            const float2 c = ((const float2 *)cs)[(local - head * hd) >> 1];
            y = (i & 1) ? partner * c.y + y * c.x : y * c.x - partner * c.y;
        }
        if (lead) {
            if (i < nqd) {
                qh[i] = y;
                if (mfma_att) split3(y, qp[i], qp[nqd + i], qp[2 * nqd + i]);
            } else {
                const int r = i - nqd, kv = r < nkd ? 0 : 1, jj = r - kv * nkd, kvl = (int)(((float)jj + 0.5f) * inv_hd);
                const uint16_t hb = f32_bf16(y);
                cur[kv * nkd + jj] = hb;
                if (mfma_att && kv)                   // V^T
                    kvb[(size_t)G.nkv * M.kv_win * kv_row(hd) + (size_t)jj * vt_row(M.kv_win) + pos] = hb;
                else if (kwin)
                    kvb[((size_t)(kv * G.nkv + kvl) * M.kv_win + pos) * kv_row(hd) + (jj - kvl * hd)] = hb;
            }
        }
    };
    wide_rows(w.a, G.qkv, act, kp, work, nqd + 2 * nkd, qkv_row);
    phase(gi, 4, pos, layer);
    // the window's copy (issued long before) is complete; this step's rows go to the cache after the
    // attention, so their store acknowledgements stay off the path to it
    if (kwin) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    phase(gi, 5, pos, layer);
    if (mfma_att) attend_mfma(M, G, pos, qp, kvb, work, vred, att);
    else if (kwin) attend_group<true, PRE, false>(M, G, layer, pos, qh, cur, kvb, vred, att);
    else attend_group<false, PRE, AT == L3M_Q8_0>(M, G, layer, pos, qh, cur, kvb, vred, att);
    phase(gi, 6, pos, layer);
    // this step's k and v rows (bf16, engine.c:247-248) into the cache, for the kv heads this group writes,
    // by the wavefronts past those that prepare the attention output next (they go straight to the prep);
    // the flag after the block waits for the stores
    // (the persistent path stores them after the block's flag instead, kv_rows_store)
    const int kq = kpad(nqd), skip = (kq + 255) >> 8 < NWE ? 64 * ((kq + 255) >> 8) : 0;
    if (!PRE && tid >= skip) kv_rows_store(M, G, layer, pos, cur, tid - skip, NTE - skip);

    // the group's attention output, prepared, through its Wo columns -> the partial residual po[group]
    prep_owned<AT>(4 * tid < nqd ? ((const float4 *)att)[tid] : make_float4(0.f, 0.f, 0.f, 0.f), act2, kq);
    phase(gi, 7, pos, layer);
    float *po = M.po + (size_t)gi * dim;
    if constexpr (G2) {
        mv<a_dtype<DT>(), nslot_wo<DT>()>(w.b, G.wo, act2, kq, work);
        __syncthreads();
        phase(gi, 8, pos, layer);
        rows_sum4(G.wo, work, dim, [&](int i, float y, float, bool lead) {
            y += gi == 0 ? Lw.bo[i] : 0.f;            // bo once, with group 0's partial
            if (lead) gw(po)[i] = y;
        });
    } else {
        mv_rows<a_dtype<DT>(), nslot_wo<DT>()>(w.b, G.wo, act2, kq, work, dim, [&](int i, float y, bool lead) {
            if (lead) gw(po)[i] = y;
        });
        phase(gi, 8, pos, layer);
    }
    phase(gi, 9, pos, layer);
}

// The FFN block of chunk ci (engine.c:259-275): x = xa + the attention partials, RMSNorm, prep, the
// chunk's gate and up rows, SiLU(gate) * up, prep, its Wdown columns -> pd[ci]. Chunk 0 keeps x in xb.
template <int DT, bool PRE, bool G2 = false>
__device__ __forceinline__ void ffn_block(const l3m_dmodel &M, const l3m_dlayer &Lw, const l3m_dchunk &C, int ci, FfnW<DT> &w,
                                          uint8_t *smem, int layer = 0, int pos = 0, bool through = false) {
    // through: the last layer of a persistent step with logits, whose x (chunk 0) and partials the head
    // workgroups on other XCDs read, stored through to memory
    const int tid = tidx(), dim = M.dim, kp = kwide(dim);
    const LdsB L = lds_of(C);
    float *work = (float *)(smem + L.work), *gu = (float *)(smem + L.gu);
    uint8_t *act = smem + L.act, *act2 = smem + L.act2;
    Red red{(float *)(smem + L.scr), 0};

    Pro P;
    const ProGeom PG = pro_geom(M, 1);
    if constexpr (!PRE) ffn_static(w.st, M, Lw);
    pro_load<PRE>(P, M.xa, M.po, PG, M.embed, false, 0);     // x += proj (engine.c:259)
    if constexpr (!PRE) ffn_issue<DT>(w, C);
    const float4 x = pro_finish<PRE>(P, M.po, PG, false, (float4 *)work, ci == 0 ? M.xb : nullptr, nullptr, w.st.cs, 0);
    if (through && ci == 0 && tid < (dim >> 2)) stcoh16(M.xb, tid, x);
    phase(64 + ci, 2, pos, layer);
    constexpr int AT = a_dtype<DT>();                // the activations take the form the step matrices read
    if constexpr (G2) ln_prep<AT>(x, Lw.ffn_norm, Lw.ffn_norm_b, dim, kp, M.eps, act, red);
    else norm_prep<AT>(x, w.st.nw, dim, kp, M.eps, act, red);
    phase(64 + ci, 3, pos, layer);
    // gate row k and up row k are rows 2k and 2k + 1 (row i ^ 1 is the partner rows_sum4 hands over):
    // the lane of gate row k forms h_k = up * silu(gate) (ops.c:49-51) there, into gu[k]
    auto gu_row = [&](int i, float y, float partner, bool lead) {
        if constexpr (G2) {
            y += i < C.nf ? C.bup[i] : 0.f;           // the up rows only, with b_up
            if (lead) gu[i] = y;
        } else {
            if (lead && !(i & 1)) gu[i >> 1] = silu_mul(partner, y);
        }
    };
    wide_rows(w.a, C.gate_up, act, kp, work, C.gate_up.rows, gu_row);
    phase(64 + ci, 4, pos, layer);
    __syncthreads();
    phase(64 + ci, 5, pos, layer);
    // h of the owned 4 rows, prepared
    const int kf = kpad(C.nf);
    float4 hv = make_float4(0.f, 0.f, 0.f, 0.f);
    if (4 * tid < C.nf) {
        if constexpr (G2) {
            float hh[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int i = 4 * tid + e;
                hh[e] = i < C.nf ? gelu_tanh(gu[i]) : 0.f;   // GELU(up) (engine.c:263-264)
            }
            hv = make_float4(hh[0], hh[1], hh[2], hh[3]);
        } else {
            hv = ((const float4 *)gu)[tid];
        }
    }
    prep_owned<AT>(hv, act2, kf);
    phase(64 + ci, 6, pos, layer);
    float *pd = M.pd + (size_t)ci * dim;
    if constexpr (G2) {
        mv<a_dtype<DT>(), nslot_b<DT>()>(w.b, C.down, act2, kf, work);
        __syncthreads();
        phase(64 + ci, 7, pos, layer);
        rows_sum4(C.down, work, dim, [&](int i, float y, float, bool lead) {
            y += ci == 0 ? Lw.bdown[i] : 0.f;         // b_down once, with chunk 0's partial
            if (lead) {
                if (through) stcoh4(pd, i, y);
                else gw(pd)[i] = y;
            }
        });
    } else {
        mv_rows<a_dtype<DT>(), nslot_b<DT>()>(w.b, C.down, act2, kf, work, dim, [&](int i, float y, bool lead) {
            if (lead) {
                if (through) stcoh4(pd, i, y);
                else gw(pd)[i] = y;
            }
        });
        phase(64 + ci, 7, pos, layer);
    }
    phase(64 + ci, 8, pos, layer);
}

// Tiles [t0, t0 + tpw) of the head as a matrix of their own (the last slice may be short).
__device__ __forceinline__ l3m_dmat head_slice(const l3m_dmodel &M, int t0, int tpw) {
    l3m_dmat V = M.head;
    const int nt = t0 + tpw <= V.tiles ? tpw : V.tiles - t0;
    V.q += (size_t)t0 * V.nb * 16 * qbytes(V.dtype);
    if (sbytes(V.dtype)) V.s += (size_t)t0 * V.nb * 16 * sbytes(V.dtype);
    V.tiles = nt;
    V.rows = nt * 16 < M.vocab - t0 * 16 ? nt * 16 : M.vocab - t0 * 16;
    return V;
}

// Final norm and the head rows of slice V (tiles from t0) at position pos (engine.c:277-301): logits
// into slot pos % nslots, and this slice's (max, lowest index) in v, idx for every thread.
template <int DT, bool PRE, bool G2 = false>
__device__ __forceinline__ void head_block(const l3m_dmodel &M, const l3m_dmat &V, int t0, int tpw, int pos, HeadW<DT> &w,
                                           uint8_t *smem, float &v, int &idx, float *keep = nullptr, int role = -1) {
    const int dim = M.dim, kp = kwide(dim);
    const LdsH L = lds_h(DT, dim, M.head.nb, tpw);
    float *work = (float *)(smem + L.work), *scr = (float *)(smem + L.scr);
    uint8_t *act = smem + L.act;
    Red red{scr, 0};

    float4 x;
    if constexpr (PRE) {
        // the persistent path: x and the last layer's FFN partials, stored through by the chunks, read
        // from memory (coherent loads); the norm weights came with the head's weights (head_issue)
        Pro P;
        const ProGeom PG = pro_geom(M, 0);
        pro_load<true>(P, M.xb, M.pd, PG, M.embed, false, 0);   // x += down (engine.c:275), last layer
        x = pro_finish<true>(P, M.pd, PG, false, (float4 *)work, nullptr, nullptr, w.st.cs, 0);
    } else {
        Pro P;
        const ProGeom PG = pro_geom(M, 0);
        pro_static(w.st, dim >> 2, M.norm, nullptr, 0);
        pro_load<false>(P, M.xb, M.pd, PG, M.embed, false, 0);   // x += down (engine.c:275), last layer
        head_issue<DT>(w, V);
        x = pro_finish<false>(P, M.pd, PG, false, (float4 *)work, nullptr, nullptr, w.st.cs, 0);
    }
    if (role >= 0) phase(role, 4, pos, 0);
    if constexpr (G2) ln_prep<DT>(x, M.norm, M.norm_b, dim, kp, M.eps, act, red);
    else norm_prep<DT>(x, w.st.nw, dim, kp, M.eps, act, red);
    if (role >= 0) phase(role, 5, pos, 0);
    // each row's logit from the lane that sums it: stored, and kept if it beats the lane's earlier rows
    float *lg = M.logits + (size_t)(pos % M.nslots) * M.vocab + (size_t)t0 * 16;
    v = -INFINITY;
    idx = 0x7FFFFFFF;
    auto logit_row = [&](int i, float yy, float, bool lead) {
        if (lead) {
            gw(lg)[i] = yy;
            if (keep) keep[i] = yy;                   // kept in LDS for sampling
            better(v, idx, yy, t0 * 16 + i);
        }
    };
    wide_rows(w.a, V, act, kp, work, V.rows, logit_row);
    if (role >= 0) phase(role, 6, pos, 0);
    // the tile forms (quantized and bf16 heads) leave tile t's rows in wavefront t; f32 heads sum rows in
    // every wavefront
    constexpr bool by_tile = tiled<DT>() || DT == L3M_BF16;
    block_argmax0(v, idx, scr, (int *)scr + 16, by_tile && V.tiles < NWE ? V.tiles : NWE);
}

// The argmax over n (value, index) partials, in index order (engine.c:294-300), into every thread.
__device__ void reduce_partials(const float *val, const int *idx_in, int n, float *scr, float &v, int &idx) {
    v = -INFINITY;
    idx = 0x7FFFFFFF;
    for (int w = tidx(); w < n; w += NTE) {
        const float pv = __hip_atomic_load(gp<float>(val + w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const int pi = __hip_atomic_load(gp<int>(idx_in + w), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        better(v, idx, pv, pi);
    }
    block_argmax(v, idx, scr, (int *)scr + 16);
}

// ------------------------------------------------------------------ temperature sampling

// xorshift64* (engine.c:98-101): three shifts of the state, then the top 53 bits of its product with the
// generator's multiplier. The reference's draw u is this integer times 2^-53.
__device__ __forceinline__ unsigned long long draw53(unsigned long long &st) {
    st ^= st >> 12;
    st ^= st << 25;
    st ^= st >> 27;
    return (st * 0x2545F4914F6CDD1DULL) >> 11;
}
// The unnormalized probability of a logit (engine.c:284-287): expf((logit - gmax) / temp), and 0 when the
// exponent is below -16.
__device__ __forceinline__ float sample_weight(float logit, float gmax, float temp) {
    const float d = (logit - gmax) / temp;
    return d < -16.0f ? 0.0f : expf(d);
}
// A weight as the integer p * 2^47, exactly: a weight is 0 or a float in [e^-16, 1], and e^-16 > 2^-24, so
// its last mantissa bit is worth at least 2^-47. Totals of up to 2^16 weights stay below 2^64, so the
// running sums and totals below are exact integers: the sampler adds in any order and still picks the
// token the exact running sums pick. (The reference's double sums round; they can pick differently only
// where u * z falls within their rounding of a boundary.) Anything else (NaN) counts as 0.
__device__ __forceinline__ unsigned long long fixp(float p) {
    if (!(p > 0.0f)) return 0;
    const uint32_t b = __float_as_uint(p), e = b >> 23;
    return (unsigned long long)((b & 0x7FFFFFu) | 0x800000u) << (e - 103);
}
// Whether a running sum c has passed the target u * z, u = k * 2^-53: c * 2^53 > k * z, in 128 bits.
__device__ __forceinline__ bool crosses(unsigned long long c, unsigned long long k, unsigned long long z) {
    return (unsigned __int128)c << 53 > (unsigned __int128)k * z;
}
// Inclusive prefix sums over the wavefront's lanes in lane order; excl gets the lanes before.
__device__ __forceinline__ unsigned long long lanes_scan_u64(unsigned long long v, unsigned long long &excl) {
    const int lane = tidx() & 63;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
        const unsigned long long t = __shfl_up(v, o, 64);
        if (lane >= o) v += t;
    }
    excl = __shfl_up(v, 1, 64);
    if (lane == 0) excl = 0;
    return v;
}
// Block prefix sums in thread order: this thread's exclusive prefix, and the total into every thread.
// uscr: NWE words of LDS, free again when it returns.
__device__ __forceinline__ unsigned long long block_scan_u64(unsigned long long v, unsigned long long &total, unsigned long long *uscr) {
    const int wave = wave_id();
    unsigned long long excl;
    const unsigned long long incl = lanes_scan_u64(v, excl);
    if ((tidx() & 63) == 63) uscr[wave] = incl;
    __syncthreads();
    unsigned long long before = 0, z = 0;
    for (int w = 0; w < NWE; w++) {
        if (w == wave) before = z;
        z += uscr[w];
    }
    __syncthreads();
    total = z;
    return before + excl;
}
// The lowest of the threads' candidates (0x7FFFFFFF: none) into every thread. iscr: NWE ints of LDS.
__device__ __forceinline__ int block_min_int(int v, int *iscr) {
    v = lanes_mini<64>(v);
    if ((tidx() & 63) == 0) iscr[wave_id()] = v;
    __syncthreads();
    v = lanes_mini<NWE>(iscr[tidx() & (NWE - 1)]);
    __syncthreads();
    return v;
}

// One workgroup samples a token from the V logits at lg, given their maximum gmax and the draw k
// (engine.c:364-379): the first i whose running sum of weights passes k * 2^-53 times their total, or V - 1
// when none does. Thread t owns logits [t per, (t + 1) per), per = ceil(V / NTE): it sums its weights, a
// block scan gives each range the sum of those before it, and every thread walks its own range again
// (the same weights, recomputed); the lowest crossing wins. Any V. lg is read with device-coherent
// loads (other workgroups wrote it). uscr: NWE words, iscr: NWE ints of LDS. Every thread gets the token.
__device__ int sample_block(const float *lg, int V, float gmax, float temp, unsigned long long k, unsigned long long *uscr, int *iscr) {
    const int tid = tidx(), per = (V + NTE - 1) / NTE, i0 = tid * per, i1 = i0 + per < V ? i0 + per : V;
    auto weight = [&](int i) {
        return fixp(sample_weight(__hip_atomic_load(gp<float>(lg + i), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT), gmax, temp));
    };
    unsigned long long sum = 0;
    for (int i = i0; i < i1; i++) sum += weight(i);
    unsigned long long z;
    unsigned long long c = block_scan_u64(sum, z, uscr);
    int cand = 0x7FFFFFFF;
    for (int i = i0; i < i1; i++) {
        c += weight(i);
        if (crosses(c, k, z)) { cand = i; break; }
    }
    const int tok = block_min_int(cand, iscr);
    return tok == 0x7FFFFFFF ? V - 1 : tok;
}

// The first batch of a deep-kernel lane (k_gemv_deep, k_gemv_mx): blocks b0 + sub + 4u (u < UB) of row
// lane & 15 of a tile, all inside the matrix. Buffer loads over a wavefront-uniform base (the tile's block b0)
// at the lane's offset plus a constant per u: no per-load address arithmetic.
template <int DT, int UB>
__device__ __forceinline__ void lane_load_deep(const l3m_dmat &m, int tile, int b0, int lane, LaneBatch<DT, UB> &x) {
    using L = LaneBatch<DT, UB>;
    const size_t first = ((size_t)tile * m.nb + b0) * RT;          // (tile, block b0, row 0)
    const __amdgpu_buffer_rsrc_t rq = buf(m.q + first * L::QBY);
    const uint32_t oq = (uint32_t)lane * L::QBY;
#pragma unroll
    for (int u = 0; u < L::U; u++) {
#pragma unroll
        for (int v = 0; v < L::NV; v++) {
            const u32x4 w = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(rq, oq + 16 * v, 64 * u * L::QBY, 0));
            x.w[u][v] = make_uint4(w.x, w.y, w.z, w.w);
        }
        x.sc[u] = 0;
    }
    if constexpr (L::SBY) {
        const __amdgpu_buffer_rsrc_t rs = buf(m.s + first * L::SBY);
        const uint32_t os = (uint32_t)lane * L::SBY;
#pragma unroll
        for (int u = 0; u < L::U; u++) {
            if constexpr (L::SBY == 2) x.sc[u] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b16(rs, os, 64 * u * 2, 0);
            else x.sc[u] = (uint32_t)__builtin_amdgcn_raw_buffer_load_b8(rs, os, 64 * u, 0);
        }
    }
}

// The matvec of a matrix of many tiles and long rows: one tile per workgroup of S wavefronts, wavefront s
// taking the s-th of S equal ranges of blocks (UB blocks per lane, one batch), so each wavefront has few
// loads to wait for and a CU holds many wavefronts to hide their latency. The S partial sums of a row are
// added in order through LDS.
template <int DT, int S, int UB> constexpr int gemv_deep_words() { return DT == L3M_MXFP4 || UB == 8 ? 2 : 1; }
template <int DT, int S, int UB>
__global__ void __launch_bounds__(64 * S) k_gemv_deep(l3m_dmat m, const uint8_t *__restrict__ act_g, int k, float *__restrict__ y) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int NTD = 64 * S;
    const int kp = kpad(k), tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, tile = blockIdx.x;
    const int b0 = wave * m.nb / S, b1 = (wave + 1) * m.nb / S;
    float *red = (float *)(smem + align16(act_size(DT, k)));
    const size_t bytes = act_size(DT, k);
    const int n16 = (int)(bytes / 16), ntail = (int)(bytes % 16) / 4;
    LaneBatch<DT, UB> x;
    // 16-byte words of the activation per thread (the launcher checks the activation fits): a load per
    // thread covers up to 8 KiB at 8 wavefronts, two the larger mxfp4 form and the 256-block rows
    constexpr int AR = gemv_deep_words<DT, S, UB>();
    u32x4 a[AR];
#pragma unroll
    for (int r = 0; r < AR; r++) a[r] = ((const u32x4 *)act_g)[min(tid + r * NTD, n16 - 1)];
    const uint32_t at = ((const uint32_t *)act_g)[4 * n16 - 1 + min(tid + 1, ntail)];
    lane_load_deep<DT, UB>(m, tile, b0, lane, x);
#pragma unroll
    for (int r = 0; r < AR; r++) ((u32x4 *)smem)[min(tid + r * NTD, n16 - 1)] = a[r];
    ((uint32_t *)smem)[4 * n16 - 1 + min(tid + 1, ntail)] = at;
    __syncthreads();
    // the wavefront's range is exactly UB batches of 4 blocks: one straight run of block dots
    float acc = 0.f;
#pragma unroll
    for (int u = 0; u < UB; u++) acc = block_fma<DT>(acc, x.w[u], x.sc[u], smem, kp, b0 + 4 * u + (lane >> 4));
    (void)b1;
    float lo, hi;
    swap16(acc, lo, hi);                              // q0 + q1, q2 + q3
    acc = lo + hi;
    swap32(acc, lo, hi);                              // (q0 + q1) + (q2 + q3)
    acc = lo + hi;
    if (lane < 16) red[wave * 16 + lane] = acc;
    __syncthreads();
    if (tid < 16) {
        float v = red[tid];
#pragma unroll
        for (int w = 1; w < S; w++) v += red[w * 16 + tid];
        const int r = tile * RT + tid;
        if (r < m.rows) y[r] = v;
    }
}

// The mxfp4 matvec of k_gemv_deep's shapes on the matrix cores. One v_mfma_scale_f32_16x16x128_f8f6f4
// takes 4 blocks of a tile's 16 rows: B is the e2m1 codes as they lie in the lane-tile plane (lane l: row
// l % 16, block l / 16 of the 4, its 16 bytes; the code bytes need no decode), A is the activation's exact
// fp8 parts h and l (q = 16 h + l, the prepared activation's last part), row 4g + p of A holding part p of
// block g and zeros outside block g's 32 inputs, so that row 4g of the result is block g's dot with h and
// row 4g + 1 its dot with l, per weight row. Both block scales of the product are 1 (e8m0 127); the products
// of e2m1 values (half the doubled codes the reference dots) with these integers, and their sums, are
// multiples of 1/2 below 2^13, exact in f32. Lane l then holds block g = l / 16 of row l % 16: the
// reference's integer dot 2 (16 D[4g] + D[4g + 1]), scaled by the reference's formula
// (kernels_scalar.c:62-75). A wavefront's lanes add their blocks in order, the 4 block lanes of a row meet by
// permlane swaps, the wavefronts through LDS.
// Memory instructions are what bounds this kernel warm (each one of 64 lanes costs the load unit its cycles
// whatever share of its lanes carry data), so every load is full width: a wavefront's 4 batches of weights,
// each 16 blocks' fp8 parts (1 KiB) in one load that it stores to its own LDS span and reads back in the
// product's layout (its own bytes only: no workgroup barrier), the block scales as 4 byte loads and the
// activation scales as 4 word loads.
template <int S, int R>
__global__ void __launch_bounds__(64 * S) k_gemv_mx(l3m_dmat m, const uint8_t *__restrict__ act_g, int k, float *__restrict__ y) {
    constexpr int UB = 4 * R;                             // R rounds of 16 blocks per wavefront
    __shared__ float red[S * 16];
    __shared__ __align__(16) uint8_t stage[S][1024 * R + 16];
    const int nb = m.nb, tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, tile = blockIdx.x;
    const int b0 = wave * nb / S;
    const uint8_t *hl = act_g + act_size(L3M_MXFP4, k);   // [nb][h, l][32] fp8
    const float *xs = (const float *)(act_g + 64 * (size_t)nb);
    // the fp8 parts first (cache hits, stored to LDS while the weights are in flight), then the weights
    const __amdgpu_buffer_rsrc_t ra = buf(hl + 64 * (size_t)b0);
    u32x4 aw[R];
#pragma unroll
    for (int r = 0; r < R; r++) aw[r] = __builtin_bit_cast(u32x4, __builtin_amdgcn_raw_buffer_load_b128(ra, 16 * lane, 1024 * r, 0));
    LaneBatch<L3M_MXFP4, UB> x;
    lane_load_deep<L3M_MXFP4, UB>(m, tile, b0, lane, x);
    const __amdgpu_buffer_rsrc_t rx = buf(xs + b0);
    const int g = lane >> 4, row = lane & 15, bb = row >> 2, part = row & 3;
    float sx[UB];
#pragma unroll
    for (int u = 0; u < UB; u++) sx[u] = __uint_as_float((uint32_t)__builtin_amdgcn_raw_buffer_load_b32(rx, 4 * g, 16 * u, 0));
    uint8_t *my = stage[wave];
#pragma unroll
    for (int r = 0; r < R; r++) *(u32x4 *)(my + 1024 * r + 16 * lane) = aw[r];
    if (lane == 0) *(u32x4 *)(my + 1024 * R) = u32x4{0u, 0u, 0u, 0u};
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    // Inputs of the product: lane group g of B holds block g's 32 codes (inputs 32 g .. 32 g + 31 of the 128),
    // lane group g of A holds inputs 16 g .. 16 g + 15 in its first 16 bytes and 64 + 16 g .. + 15 in its last
    // 16. So block bb's part p (row 4 bb + p of A) lies in the first 16 bytes of lane groups 2 bb and 2 bb + 1
    // for bb < 2, in the last 16 of lane groups 2 (bb - 2) and 2 (bb - 2) + 1 for bb >= 2; lane group g holds
    // its inputs 16 (g & 1) .. + 15 there. Every other half reads the span's 16 zero bytes.
    const bool has = part < 2 && (bb & 1) == (g >> 1), second = bb >= 2;
    const int oa = 64 * bb + 32 * part + 16 * (g & 1);
    const uint8_t *plo = has && !second ? my + oa : my + 1024 * R, *phi = has && second ? my + oa : my + 1024 * R;
    const int step = has ? 256 : 0;                       // the next 4 blocks, or the zero bytes again
    float acc = 0.f;
#pragma unroll
    for (int u = 0; u < UB; u++) {
        const u32x4 lo = *(const u32x4 *)(plo + (!second ? u * step : 0)), hi = *(const u32x4 *)(phi + (second ? u * step : 0));
        const i32x8 A = {(int)lo.x, (int)lo.y, (int)lo.z, (int)lo.w, (int)hi.x, (int)hi.y, (int)hi.z, (int)hi.w};
        const i32x8 B = {(int)x.w[u][0].x, (int)x.w[u][0].y, (int)x.w[u][0].z, (int)x.w[u][0].w, 0, 0, 0, 0};
        const f32x4 d = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(A, B, f32x4{0.f, 0.f, 0.f, 0.f}, 0, 4, 0, 127, 0, 127);
        const float dot = 2.f * fmaf(16.f, d[0], d[1]);
        // xs 2^(e - 128) as one exact scaling (the product the reference forms, rounded once either way)
        acc = fmaf(__builtin_amdgcn_ldexpf(sx[u], (int)x.sc[u] - 128), dot, acc);
    }
    float lo, hi;
    swap16(acc, lo, hi);                              // blocks g = 0 + 1, 2 + 3
    acc = lo + hi;
    swap32(acc, lo, hi);
    acc = lo + hi;
    if (lane < 16) red[wave * 16 + lane] = acc;
    __syncthreads();
    if (tid < 16) {
        float v = red[tid];
#pragma unroll
        for (int w = 1; w < S; w++) v += red[w * 16 + tid];
        const int r = tile * RT + tid;
        if (r < m.rows) y[r] = v;
    }
}

// ------------------------------------------------------------------ pieces of the decode step, alone
// For parity tests: the decode step's own device code on inputs the caller gives.

// Rows [row0, row0 + n) of a lane-tile matrix exactly dequantized by lt_elem4, the step's embedding lookup
// (engine.c:236, pack.c:55-62): out[r][0, 32 nb), one thread per 4 elements.
__global__ void __launch_bounds__(NT) k_dequant(l3m_dmat m, int row0, int n, float *out) {
    const int k4 = m.nb * 8;
    const size_t i = (size_t)blockIdx.x * NT + threadIdx.x;
    if (i >= (size_t)n * k4) return;
    const int r = (int)(i / (size_t)k4), c = (int)(i - (size_t)r * k4);
    const float4 v = lt_elem4(m, row0 + r, 4 * c);
    ((float4 *)out)[i] = v;
}

// LDS regions of k_attend_decode (byte offsets), in the order the attention block keeps them.
struct LdsAtt { size_t qh, att, cur, vred, sc, kvb, total; };
__host__ __device__ inline LdsAtt lds_att(int mode, int nq, int nkv, int hd, int ctx) {
    LdsAtt L;
    size_t o = 0;
    const size_t nqd = (size_t)nq * hd, vr = 4 * (size_t)NWE * (hd + 2), vq = 8 * (size_t)NWE + 6 * nqd;
    L.qh = o;   o += align16(4 * nqd);
    L.att = o;  o += align16(4 * nqd);
    L.cur = o;  o += align16(4 * (size_t)nkv * hd);
    L.vred = o; o += align16(vr > vq ? vr : vq);
    L.sc = o;   o += mode == 2 ? align16(10 * (size_t)((ctx + 31) & ~31)) : 0;
    L.kvb = o;  o += mode ? kv_window_bytes(nkv, ctx, hd, mode == 2) : 0;
    L.total = o;
    return L;
}

// One head group's attention exactly as the decode step runs it (attn_block): MODE 2 attend_mfma, 1
// attend_group over the LDS window, 0 attend_group reading the cache (batched or not). q: [nq][hd] f32 (after RoPE);
// kc, vc: [nkv][ctx][hd] bf16 holding rows 0..pos (row pos is this step's, which the block takes from its
// own registers into cur and the window); out: [nq][hd]. Query head h reads kv head h / (nq / nkv).
template <int MODE, bool BATCH>
__global__ void __launch_bounds__(NTE) k_attend_decode(float *out, const float *q, const uint16_t *kc, const uint16_t *vc, int nq,
                                                       int nkv, int hd, int ctx, int pos, int att_wl) {
    extern __shared__ __align__(16) uint8_t smem[];
    const LdsAtt L = lds_att(MODE, nq, nkv, hd, ctx);
    float *qh = (float *)(smem + L.qh), *att = (float *)(smem + L.att), *vred = (float *)(smem + L.vred), *sc = (float *)(smem + L.sc);
    uint16_t *cur = (uint16_t *)(smem + L.cur), *kvb = (uint16_t *)(smem + L.kvb);
    __bf16 *qp = (__bf16 *)(vred + 2 * NWE);
    l3m_dmodel M{};
    M.hd = hd; M.ctx = ctx; M.n_kv = nkv; M.hpk = nq / nkv; M.att_scale = 1.0f / sqrtf((float)hd); M.kv_lds = MODE != 0; M.kv_win = MODE != 0 ? ctx : 0;
    M.kc = (uint16_t *)kc; M.vc = (uint16_t *)vc;
    l3m_dgroup G{};
    G.q0 = 0; G.nq = nq; G.kv0 = 0; G.nkv = nkv; G.att_wl = att_wl;
    const int nqd = nq * hd, nkd = nkv * hd;
    if (MODE) kv_window_dma<false>(kvb, M, 0, 0, nkv, pos, MODE == 2);
    for (int i = tidx(); i < nqd; i += NTE) {
        const float y = q[i];
        qh[i] = y;
        if (MODE == 2) split3(y, qp[i], qp[nqd + i], qp[2 * nqd + i]);
    }
    for (int i = tidx(); i < 2 * nkd; i += NTE) {     // this step's k, v rows, as the block stores them
        const int kv = i < nkd ? 0 : 1, jj = i - kv * nkd, kvl = jj / hd, d = jj - kvl * hd;
        const uint16_t hb = (kv ? vc : kc)[((size_t)kvl * ctx + pos) * hd + d];
        cur[i] = hb;
        if (MODE == 2 && kv) kvb[(size_t)nkv * ctx * kv_row(hd) + (size_t)jj * vt_row(ctx) + pos] = hb;   // V^T
        else if (MODE) kvb[((size_t)(kv * nkv + kvl) * ctx + pos) * kv_row(hd) + d] = hb;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (MODE == 2) attend_mfma(M, G, pos, qp, kvb, sc, vred, att);
    else if (MODE == 1) attend_group<true, false, false>(M, G, 0, pos, qh, cur, kvb, vred, att);
    else attend_group<false, false, BATCH>(M, G, 0, pos, qh, cur, kvb, vred, att);
    for (int i = tidx(); i < nqd; i += NTE) out[i] = att[i];
}

// One of the decode step's matvecs alone, exactly as the step runs it: FORM 0 the wide form of the q/k/v
// rows and the gate/up rows (attn_block, ffn_block: tile_rows in the quantized dtypes, mv and rows_sum4 in
// bf16 and f32, over an input padded to whole slots), 1 the Wo columns (attn_block: mv_rows with the Wo
// slots), 2 the Wdown columns (ffn_block: mv_rows with its slots), 3 the head rows of tiles
// [blockIdx * tpw, + tpw) per workgroup (head_block's slice). m is stored as the step stores it (a_dtype
// for a body of dtype DT; the head in its own dtype DT). The weights are issued first and the int8 prep of
// x (k f32 values, the step's normalized input) follows, as in the step; y[i] for every row i of m.
template <int DT, int FORM>
__global__ void __launch_bounds__(NTE) k_step_mv(l3m_dmat m, const float *x, int k, float *y, int tpw) {
    extern __shared__ __align__(16) uint8_t smem[];
    constexpr int AT = FORM == 3 ? DT : a_dtype<DT>();
    constexpr int NS = FORM == 0 ? nslot_a<DT>() : FORM == 1 ? nslot_wo<DT>() : FORM == 2 ? nslot_b<DT>() : nslot_h<DT>();
    constexpr bool WIDE = FORM == 0 || FORM == 3;
    const int tid = tidx(), kp = WIDE ? kwide(k) : kpad(k);
    uint8_t *act = smem;
    float *work = (float *)(smem + align16(act_size(AT, kp)));
    int t0 = 0;
    if constexpr (FORM == 3) {                        // the workgroup's slice, as head_slice cuts it
        t0 = blockIdx.x * tpw;
        const int nt = t0 + tpw <= m.tiles ? tpw : m.tiles - t0;
        m.q += (size_t)t0 * m.nb * 16 * qbytes(AT);
        if (sbytes(AT)) m.s += (size_t)t0 * m.nb * 16 * sbytes(AT);
        m.rows = nt * 16 < m.rows - t0 * 16 ? nt * 16 : m.rows - t0 * 16;
        m.tiles = nt;
    }
    std::conditional_t<WIDE, Wide<AT, NS>, Pref<AT, NS>> pf;
    if constexpr (WIDE) wide_issue(pf, m);
    else pref_load<AT, NS>(pf, m, 0);
    float e[4];
#pragma unroll
    for (int j = 0; j < 4; j++) e[j] = 4 * tid + j < k ? x[4 * tid + j] : 0.f;
    prep_owned<AT>(make_float4(e[0], e[1], e[2], e[3]), act, kp);
    float *out = y + (size_t)t0 * 16;
    if constexpr (WIDE) {
        wide_rows(pf, m, act, kp, work, m.rows, [&](int i, float v, float, bool lead) {
            if (lead) out[i] = v;
        });
    } else {
        mv_rows<AT, NS>(pf, m, act, kp, work, m.rows, [&](int i, float v, bool lead) {
            if (lead) out[i] = v;
        });
    }
}
// Dynamic LDS of k_step_mv: the prepared input, then the per-pair results of the general form.
inline size_t step_mv_lds(int at, int form, int k, int tiles, int nb) {
    const int kp = form == 0 || form == 3 ? kwide(k) : kpad(k);
    return align16(act_size(at, kp)) + work_bytes(res_bytes((size_t)tiles * nb), 0);
}

// ------------------------------------------------------------------ the graph path: one kernel per block

template <int DT, bool G2 = false>
__global__ void __launch_bounds__(NTE) k_attn_block(l3m_dmodel M, l3m_dlayer Lw, int layer) {
    extern __shared__ __align__(16) uint8_t smem[];
    const l3m_dgroup G = Lw.groups[blockIdx.x];
    AttnW<DT> w;
    const int pos = *M.pos;
    attn_block<DT, false, G2>(M, Lw, G, layer, pos, layer ? 0 : M.tokens[pos], blockIdx.x, w, smem);
}

// The last layer of a step without the head advances the position (nothing in this kernel reads it).
template <int DT, bool G2 = false>
__global__ void __launch_bounds__(NTE) k_ffn_block(l3m_dmodel M, l3m_dlayer Lw, int advance) {
    extern __shared__ __align__(16) uint8_t smem[];
    const l3m_dchunk C = Lw.chunks[blockIdx.x];
    FfnW<DT> w;
    ffn_block<DT, false, G2>(M, Lw, C, blockIdx.x, w, smem);
    if (advance && blockIdx.x == 0 && tidx() == 0) *M.pos += 1;
}

// Each workgroup reduces its slice; the last one to finish reduces the partials, writes tokens[pos + 1],
// resets the counter and (advance) moves pos on.
template <int DT, bool G2 = false>
__global__ void __launch_bounds__(NTE) k_head_block(l3m_dmodel M, int advance) {
    extern __shared__ __align__(16) uint8_t smem[];
    const int tpw = M.head_tiles_per_wg, t0 = blockIdx.x * tpw, pos = *M.pos;
    const l3m_dmat V = head_slice(M, t0, tpw);
    HeadW<DT> w;
    float v;
    int idx;
    head_block<DT, false, G2>(M, V, t0, tpw, pos, w, smem, v, idx);
    float *scr = (float *)(smem + lds_h(DT, M.dim, M.head.nb, tpw).scr);
    __shared__ int last;
    if (tidx() == 0) {
        M.part_val[blockIdx.x] = v;
        M.part_idx[blockIdx.x] = idx;
        __threadfence();
        last = atomicAdd(M.done, 1u) == gridDim.x - 1;
    }
    __syncthreads();
    if (!last) return;
    __threadfence();
    reduce_partials(M.part_val, M.part_idx, gridDim.x, scr, v, idx);
    const float temp = M.samp->temp;
    if (temp > 0 && idx != 0x7FFFFFFF) {             // temperature sampling over this step's logits
        unsigned long long st = M.samp->rng[0];
        const unsigned long long k = draw53(st);
        idx = sample_block(M.logits + (size_t)(pos % M.nslots) * M.vocab, M.vocab, v, temp, k, (unsigned long long *)scr,
                           (int *)scr + 2 * NWE);
        if (tidx() == 0) M.samp->rng[0] = st;
    }
    if (tidx() == 0) {
        if (advance) {
            M.tokens[pos + 1] = idx == 0x7FFFFFFF ? 0 : idx;
            *M.pos = pos + 1;
        }
        *M.done = 0;
    }
}

// ------------------------------------------------------------------ the persistent path
// k_decode runs R.nsteps decode steps in one cooperative launch, one workgroup per CU. The body (the
// attention blocks of the n_groups head groups and the FFN blocks of the n_chunks chunks) runs on the
// workgroups of one XCD (R.body_xcc): their hand-overs then meet in that XCD's L2. Every other workgroup
// takes head tiles. Roles are dealt at launch from per-XCD tickets, so they follow where the hardware
// placed each workgroup.
//
// Hand-over, inside the body: each producer owns a flag word that it sets to its epoch once its stores
// have reached L2 (s_waitcnt, barrier, then the flag); consumers poll the producers' flags with
// device-scope loads (one lane per producer) and read the data the same way. Epochs only grow during a
// launch (the host zeroes R.sync first): attention group g sets attn[g] = s*L + l + 1 after layer l of
// step s, FFN chunk c sets ffn[c] likewise. A layer's blocks wait for all flags of the block before them.
//
// Hand-over to and from the head (other XCDs, so through memory): in the last layer of a step with
// logits, the FFN chunks store x (chunk 0) and their partials through to memory and set their flags
// device-wide; head workgroups wait for those flags, sum the final residual themselves (the prologue's
// order of additions, coherent loads), compute their tiles' logits and argmax, and store one 64-bit key
// per workgroup (the step's tag, the value in an order-preserving code, the index); the attention groups
// of the next step wait for every key with that tag and take the maximum. The attention groups are free
// after their last block: they issue the next step's first weights while the head runs, and those loads
// are complete by the time they poll for the token (a wavefront's loads return in order).
//
// Every wait is bounded: past R.spin_limit ticks of the 100 MHz clock the waiter raises the abort flag
// and every workgroup leaves at its next wait, so the grid always drains.
enum { SY_ATTN = 0, SY_FFN = 64, SY_ABORT = L3M_SYNC_ABORT, SY_TOKEN = 208, SY_TICKET = 224, SY_HEAD_TICKET = 240,
       SY_SLOTS = 256 };
constexpr int SY_SUMS = SY_SLOTS + 2 * L3M_MAX_HEAD_WGS;   // slice totals (sampling) follow the keys
static_assert(L3M_SYNC_OUT == SY_SUMS + 2 * L3M_MAX_HEAD_WGS && L3M_MAX_HEAD_WGS == 256, "keys and totals follow the flag words");
static_assert(L3M_SYNC_TOK + 128 <= L3M_SYNC_WORDS, "a run's tokens fit its output span");
// The run's token at position p + 1 (p >= head_from), into the output span the host copies back.
__device__ __forceinline__ void out_token(const l3m_run &R, int p, int tok) {
    const int f = R.pos0 > R.head_from ? R.pos0 : R.head_from;
    gw((int *)(R.sync + L3M_SYNC_TOK))[p - f] = tok;
}

__device__ __forceinline__ unsigned xcc_id() {
    unsigned x;
    asm volatile("s_getreg_b32 %0, hwreg(HW_REG_XCC_ID)" : "=s"(x));
    return x & 15;
}
__device__ __forceinline__ unsigned ld_flag(const unsigned *p) {
    return __hip_atomic_load(gp<unsigned>(p), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waits, bounded: the shared tail of every poll loop. Returns 0 to stop waiting (abort seen or raised).
__device__ __forceinline__ int keep_waiting(unsigned spin, unsigned long long t0, unsigned *abort_flag, unsigned long long limit) {
    if ((spin & 31) != 31) return 1;
    if (ld_flag(abort_flag)) return 0;
    if (__builtin_amdgcn_s_memrealtime() - t0 > limit) {
        __hip_atomic_store(gw(abort_flag), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return 0;
    }
    return 1;
}

// Wavefront 0 polls flags[0..n) (n <= 64, one lane each) until every one is >= target; the result
// reaches every thread through ok_lds. SLEEP: s_sleep between polls (64 clocks each). ALL: every wavefront
// polls for itself and goes on as soon as it sees the flags, with no barrier (the hand-overs inside the
// body XCD: measured 2.4% faster decode on stories110M); a wavefront that gives up leaves, and the others
// see the abort word at their next poll.
template <int SLEEP, bool ALL = false>
__device__ bool wait_flags(const unsigned *flags, int n, unsigned target, unsigned *abort_flag, unsigned long long limit, int *ok_lds) {
    if constexpr (ALL) {
        const int lane = tidx() & 63;
        const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
        for (unsigned spin = 0;; spin++) {
            const unsigned v = lane < n ? ld_flag(flags + lane) : target;
            if (__all(v >= target)) return true;
            if (!keep_waiting(spin, t0, abort_flag, limit)) return false;
            if constexpr (SLEEP > 0) __builtin_amdgcn_s_sleep(SLEEP);
        }
    }
    const int tid = tidx();
    if (tid < 64) {
        int ok = 1;
        const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
        for (unsigned spin = 0;; spin++) {
            const unsigned v = tid < n ? ld_flag(flags + tid) : target;
            if (__all(v >= target)) break;
            if (!keep_waiting(spin, t0, abort_flag, limit)) { ok = 0; break; }
            __builtin_amdgcn_s_sleep(SLEEP);
        }
        if (tid == 0) *ok_lds = ok;
    }
    __syncthreads();
    const int ok = *ok_lds;
    __syncthreads();                                  // ok_lds is free again
    return ok != 0;
}

// Every thread's stores have reached L2 (vmcnt), then thread 0 sets the flag: a plain store for readers
// on this XCD, a write-through one (device) for readers on others.
template <bool DEVICE>
__device__ __forceinline__ void set_flag(unsigned *flag, unsigned value) {
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    __syncthreads();
    if (tidx() == 0) {
        if constexpr (DEVICE) __hip_atomic_store(gw(flag), value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        else *gw(flag) = value;                       // write-through from L1, so it is in this XCD's L2
    }
}

// A head workgroup's argmax as a 64-bit key whose unsigned order is the reference's (larger value, then
// lower index): bits 17..48 the value in an order-preserving code, bits 0..16 0x1FFFF - index, bits 49..63
// the step's tag. No row (idx past 0x1FFFF) or NaN gives key 0, which never wins.
constexpr uint64_t KEY_BITS = (1ull << 49) - 1;
__device__ __forceinline__ uint64_t argmax_key(float v, int idx, unsigned tag) {
    uint64_t key = 0;
    if (v == v && idx >= 0 && idx <= 0x1FFFF) {
        uint32_t u = __float_as_uint(v + 0.0f);       // -0 as +0: they compare equal
        u = (u & 0x80000000u) ? ~u : (u | 0x80000000u);
        key = (uint64_t)u << 17 | (uint64_t)(0x1FFFF - idx);
    }
    return (uint64_t)tag << 49 | key;
}
__device__ __forceinline__ unsigned step_tag(int s) { return (unsigned)(s % 32767) + 1; }
__device__ __forceinline__ uint64_t max_u64(uint64_t a, uint64_t b) { return a > b ? a : b; }
// The maximum over the wavefront's 64 lanes, into every lane (DPP and permlane moves of both halves).
__device__ __forceinline__ uint64_t lanes_max_u64(uint64_t v) {
    auto hi = [](uint64_t x) { return (int)(uint32_t)(x >> 32); };
    auto lo = [](uint64_t x) { return (int)(uint32_t)x; };
    auto join = [](int h, int l) { return (uint64_t)(uint32_t)h << 32 | (uint32_t)l; };
    v = max_u64(v, join(dppi<QP_X1>(hi(v)), dppi<QP_X1>(lo(v))));
    v = max_u64(v, join(dppi<QP_X2>(hi(v)), dppi<QP_X2>(lo(v))));
    v = max_u64(v, join(dppi<ROW_HALF_MIRROR>(hi(v)), dppi<ROW_HALF_MIRROR>(lo(v))));
    v = max_u64(v, join(dppi<ROW_MIRROR>(hi(v)), dppi<ROW_MIRROR>(lo(v))));
    float h0, h1, l0, l1;
    swap16(__int_as_float(hi(v)), h0, h1); swap16(__int_as_float(lo(v)), l0, l1);
    v = max_u64(join(__float_as_int(h0), __float_as_int(l0)), join(__float_as_int(h1), __float_as_int(l1)));
    swap32(__int_as_float(hi(v)), h0, h1); swap32(__int_as_float(lo(v)), l0, l1);
    return max_u64(join(__float_as_int(h0), __float_as_int(l0)), join(__float_as_int(h1), __float_as_int(l1)));
}

// Wavefront 0 polls the n_head keys of step s until all carry the step's tag; returns their maximum (the
// winning key) in wavefront 0, or ~0 when the run is being abandoned. Each lane loads keys lane + 64 r,
// r < 4, of the 256-key area every time, and keys from n_head on are masked by selects: a load under a
// lane condition is followed by a wait for every load in flight, which would put the four loads one
// cross-XCD round trip apart instead of overlapping them.
__device__ __forceinline__ uint64_t poll_keys(const uint64_t *slots, int n_head, int s, unsigned *abort_flag, unsigned long long limit) {
    const int tid = tidx();
    const unsigned tag = step_tag(s);
    uint64_t best = 0;
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    for (unsigned spin = 0;; spin++) {
        bool all = true;
        best = 0;
        uint64_t v[4];
#pragma unroll
        for (int r = 0; r < 4; r++)
            v[r] = __hip_atomic_load(gp<uint64_t>(slots + tid + 64 * r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const bool in = tid + 64 * r < n_head;
            all = all && (!in || (unsigned)(v[r] >> 49) == tag);
            best = max_u64(best, in ? v[r] & KEY_BITS : 0ull);
        }
        if (__all(all)) break;
        if (!keep_waiting(spin, t0, abort_flag, limit)) return ~0ull;
        __builtin_amdgcn_s_sleep(1);
    }
    return lanes_max_u64(best);
}
__device__ __forceinline__ int key_token(uint64_t key) { return (key >> 17) == 0 ? 0 : 0x1FFFF - (int)(key & 0x1FFFF); }
// The value a key holds (argmax_key's order-preserving code, undone; a -0 maximum comes back as +0).
__device__ __forceinline__ float key_value(uint64_t key) {
    const uint32_t u = (uint32_t)(key >> 17);
    return __uint_as_float((u & 0x80000000u) ? (u & 0x7FFFFFFFu) : ~u);
}

// The token chosen by step s's head (the winning key's index), into every thread; -1 when the run is
// being abandoned.
__device__ int wait_token(const uint64_t *slots, int n_head, int s, unsigned *abort_flag, unsigned long long limit, int *lds) {
    const int tid = tidx();
    if (tid < 64) {
        const uint64_t best = poll_keys(slots, n_head, s, abort_flag, limit);
        if (tid == 0) *lds = best == ~0ull ? -1 : key_token(best);
    }
    __syncthreads();
    const int tok = *lds;
    __syncthreads();
    return tok;
}

// The token word: step_tag(s) << 17 | token, written by the workgroup that sampled step s.
__device__ __forceinline__ unsigned token_word(int s, int tok) { return step_tag(s) << 17 | (unsigned)tok; }
// The token sampled at step s, from the token word, into every thread; -1 when the run is being abandoned.
__device__ int wait_token_word(const unsigned *word, int s, unsigned *abort_flag, unsigned long long limit, int *lds) {
    if (tidx() == 0) {
        const unsigned tag = step_tag(s);
        int tok = -1;
        const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
        for (unsigned spin = 0;; spin++) {
            const unsigned w = ld_flag(word);
            if (w >> 17 == tag) { tok = (int)(w & 0x1FFFF); break; }
            if (!keep_waiting(spin, t0, abort_flag, limit)) break;
            __builtin_amdgcn_s_sleep(1);
        }
        *lds = tok;
    }
    __syncthreads();
    const int tok = *lds;
    __syncthreads();
    return tok;
}

// A 64-bit value through readfirstlane, one 32-bit half at a time. The builtin returns a signed int, so
// each half is taken back as uint32_t before it is widened (a sign-extended low half would set every
// high bit of the address).
__device__ __forceinline__ uint64_t first_lane64(uint64_t u) {
    const uint32_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)(u >> 32));
    const uint32_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((int)(uint32_t)u);
    return (uint64_t)hi << 32 | (uint64_t)lo;
}
// Arguments of a function that is not inlined arrive in vector registers; these are uniform, so say so
// (scalar registers, scalar loads, uniform branches).
template <class T> __device__ __forceinline__ T *uniform(T *p) { return (T *)first_lane64((uint64_t)p); }
// Parameters that stay fixed during a launch (the model, the run, the layer descriptors), read through the
// constant address space: scalar loads into scalar registers.
#define CONSTANT __attribute__((address_space(4)))
template <class T> __device__ __forceinline__ T fixed(const T *p, int i = 0) {
    static_assert(sizeof(T) % 4 == 0, "copied as 32-bit words");
    const CONSTANT uint32_t *src = (const CONSTANT uint32_t *)uniform(p) + (size_t)i * (sizeof(T) / 4);
    T v;
    uint32_t *dst = (uint32_t *)&v;
#pragma unroll
    for (size_t k = 0; k < sizeof(T) / 4; k++) dst[k] = src[k];
    return v;
}
// The same pointer, hidden from the optimizer, so loads through it are redone inside a loop (where
// they are used) instead of being hoisted in front of it and held in registers across the whole loop.
template <class T> __device__ __forceinline__ const T *per_iteration(const T *p) {
    uint64_t u = first_lane64((uint64_t)p);
    asm volatile("" : "+s"(u));
    return (const T *)u;
}
__device__ __forceinline__ int uniform(int v) { return __builtin_amdgcn_readfirstlane(v); }

// The roles, each in a function of its own (so each gets its own register allocation and nothing of one
// role stays live in another). They return false when the run is being abandoned.
// HD > 0: the model's head dimension, as a constant (the host launches the kernel built for it): the
// compiler then fixes the attention block's loops over it and its lane masks (measured +0.9% decode on
// stories110M, +2.1% on stories42M, +2.8% on SmolLM2 against reading it from the model).
template <int DT, bool G2, int HD = 0>
__device__ __noinline__ bool attn_role(const l3m_dmodel *Mp, const l3m_dlayer *layers, const l3m_run *Rp, int g, int s) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int ok_lds;
    // group 0's time waiting for its inputs (the FFN flags, the head's token) since the launch began, in
    // ticks of the 100 MHz clock: the decode's analogue of the reference's barrier wait (l3m_perf ns_wait)
    __shared__ unsigned long long waited;
    g = uniform(g); s = uniform(s);
    if (s == 0 && tidx() == 0) waited = 0;
    const int nl = fixed(Mp).n_layers;
    for (int l = 0; l < nl; l++) {
        l3m_dmodel M = fixed(per_iteration(Mp));
        if constexpr (HD > 0) M.hd = HD;
        const l3m_run R = fixed(per_iteration(Rp));
        const int pos = R.pos0 + s;
        unsigned *sync = R.sync, *abort_flag = sync + SY_ABORT;
        const l3m_dlayer Lw = fixed(layers, l);
        const l3m_dgroup G = fixed(Lw.groups, g);
        AttnW<DT> wt;
        phase_arm(pos, l, nl);
        phase(g, 0, pos, l);
        attn_static(wt.st, M, Lw, pos);
        attn_issue<DT>(wt, G);
        attn_kv_window<DT>(M, G, l, pos, smem);
        const unsigned epoch = (unsigned)(s * nl + l);
        int tok = 0;
        const unsigned long long w0 = __builtin_amdgcn_s_memrealtime();
        if (l == 0 && s > 0 && pos - 1 >= R.head_from) {
            // this step's token is the previous step's argmax (which also orders this step after every
            // read of the previous step's FFN partials)
            tok = R.temp > 0 ? wait_token_word(sync + SY_TOKEN, s - 1, abort_flag, R.spin_limit, &ok_lds)
                                   : wait_token((const uint64_t *)(sync + SY_SLOTS), R.n_head, s - 1, abort_flag, R.spin_limit, &ok_lds);
            if (tok < 0) return false;
            if (g == 0 && tidx() == 0) {
                gw(M.tokens)[pos] = tok;
                out_token(R, pos - 1, tok);
            }
        } else {
            if (epoch > 0 && !wait_flags<0, true>(sync + SY_FFN, M.n_chunks, epoch, abort_flag, R.spin_limit, &ok_lds)) return false;
            if (l == 0) tok = __hip_atomic_load(gp<int32_t>(M.tokens + pos), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // read now, added after the block: the clock read's latency overlaps the prologue's loads
        const unsigned long long w1 = __builtin_amdgcn_s_memrealtime();
        phase(g, 1, pos, l);
        attn_block<DT, true, G2>(M, Lw, G, l, pos, tok, g, wt, smem);
        set_flag<false>(sync + SY_ATTN + g, epoch + 1);
        if (g == 0 && tidx() == 0) waited += w1 - w0;
        // the K/V rows while the FFN runs: off the block's path (the next read of them is the window copy
        // of the next position's step, behind this workgroup's later flag waits)
        kv_rows_store(M, G, l, pos, (const uint16_t *)(smem + lds_of(G).cur), tidx(), NTE);
        phase(g, 10, pos, l);
    }
    if (g == 0 && tidx() == 0) gw((unsigned long long *)(fixed(Rp).sync + L3M_SYNC_WAIT))[0] = waited;
    return true;
}

template <int DT, bool G2>
__device__ __noinline__ bool ffn_role(const l3m_dmodel *Mp, const l3m_dlayer *layers, const l3m_run *Rp, int ci, int s) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int ok_lds;
    ci = uniform(ci); s = uniform(s);
    const int nl = fixed(Mp).n_layers;
    for (int l = 0; l < nl; l++) {
        const l3m_dmodel M = fixed(per_iteration(Mp));
        const l3m_run R = fixed(per_iteration(Rp));
        unsigned *sync = R.sync;
        const l3m_dlayer Lw = fixed(layers, l);
        const l3m_dchunk C = fixed(Lw.chunks, ci);
        FfnW<DT> wt;
        const int pos = R.pos0 + s;
        phase_arm(pos, l, nl);
        phase(64 + ci, 0, pos, l);
        ffn_static(wt.st, M, Lw);
        ffn_issue<DT>(wt, C);
        const unsigned epoch = (unsigned)(s * nl + l);
        if (!wait_flags<0, true>(sync + SY_ATTN, M.n_groups, epoch + 1, sync + SY_ABORT, R.spin_limit, &ok_lds)) return false;
        phase(64 + ci, 1, pos, l);
        const bool through = l == nl - 1 && pos >= R.head_from;   // the head reads this layer's partials
        ffn_block<DT, true, G2>(M, Lw, C, ci, wt, smem, l, pos, through);
        if (through) set_flag<true>(sync + SY_FFN + ci, epoch + 1);
        else set_flag<false>(sync + SY_FFN + ci, epoch + 1);
        phase(64 + ci, 9, pos, l);
    }
    return true;
}

// Temperature sampling of step s over the head workgroups, in the reference's multi-rank form
// (engine.c:290-319; the rules of engine.c:284-287 and 364-379). Head workgroup h, whose slice holds
// rows [r0, r0 + nrow) with their logits in LDS (lgv), after it stored its key:
//  1. waits for every key and takes the step's maximum from the winning one;
//  2. stores its slice's weight total (exact, fixp) tagged with the step in its slot;
//  3. waits for every slot, draws k from its own copy of the generator, and finds the slice where the
//     running total passes k * 2^-53 times the grand total;
//  4. if that slice is its own, walks it and publishes the token in the token word.
// Every workgroup draws once per sampled step, so the copies of the generator stay equal. Returns false
// when the run is being abandoned.
__device__ __forceinline__ unsigned sum_tag(int s) { return (unsigned)(s % 63) + 1; }   // 6 bits: totals < 2^58
__device__ bool sample_step(const l3m_dmodel &M, const l3m_run &R, int h, int s, int nrow, int r0, uint8_t *smem) {
    const int tid = tidx(), lane = tid & 63;
    const LdsH LH = lds_h(M.head.dtype, M.dim, M.head.nb, R.head_tpw);
    const float *lgv = (const float *)(smem + LH.lgv);
    unsigned long long *uscr = (unsigned long long *)(smem + LH.scr);
    int *iscr = (int *)(uscr + NWE);
    const float temp = R.temp;
    // 1. the step's maximum
    if (tid < 64) {
        const uint64_t key = poll_keys((const uint64_t *)(R.sync + SY_SLOTS), R.n_head, s, R.sync + SY_ABORT, R.spin_limit);
        if (tid == 0) uscr[0] = key;
    }
    __syncthreads();
    const uint64_t key = uscr[0];
    __syncthreads();
    if (key == ~0ull) return false;
    const float gmax = key_value(key);
    // 2. this slice's total (one row per thread: nrow <= 16 * 64 <= NTE)
    const unsigned long long w = tid < nrow ? fixp(sample_weight(lgv[tid], gmax, temp)) : 0;
    unsigned long long total;
    const unsigned long long before = block_scan_u64(w, total, uscr);
    unsigned long long *sums = (unsigned long long *)(R.sync + SY_SUMS);
    if (tid == 0) __hip_atomic_store(gw(sums + h), (unsigned long long)sum_tag(s) << 58 | total, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    // 3. every slice's total, the draw, the owner slice
    if (tid < 64) {
        const unsigned tag = sum_tag(s);
        unsigned long long v[4];
        const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
        bool ok = true;
        for (unsigned spin = 0;; spin++) {
            bool all = true;
#pragma unroll
            for (int r = 0; r < 4; r++)
                v[r] = __hip_atomic_load(gp<unsigned long long>(sums + lane + 64 * r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
            for (int r = 0; r < 4; r++) all = all && (lane + 64 * r >= R.n_head || (unsigned)(v[r] >> 58) == tag);
            if (__all(all)) break;
            if (!keep_waiting(spin, t0, R.sync + SY_ABORT, R.spin_limit)) { ok = false; break; }
            __builtin_amdgcn_s_sleep(1);
        }
        // slice j = lane + 64 r, in order: its running total through it, and the grand total
        unsigned long long incl[4], carry = 0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const unsigned long long sj = lane + 64 * r < R.n_head ? v[r] & ((1ull << 58) - 1) : 0;
            unsigned long long ex;
            incl[r] = carry + lanes_scan_u64(sj, ex);
            carry += __shfl(incl[r] - carry, 63, 64);
        }
        const unsigned long long z = carry;
        unsigned long long st = __hip_atomic_load(gp<unsigned long long>(&M.samp->rng[h]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const unsigned long long k = draw53(st);
        int owner = 0x7FFFFFFF;
#pragma unroll
        for (int r = 0; r < 4; r++)
            if (lane + 64 * r < R.n_head && owner == 0x7FFFFFFF && crosses(incl[r], k, z)) owner = lane + 64 * r;
        owner = lanes_mini<64>(owner);
        if (lane == 0) {
            __hip_atomic_store(gw(&M.samp->rng[h]), st, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            iscr[0] = ok ? owner : -1;
            uscr[1] = k;
            uscr[2] = z;
        }
        // the running total before the owner slice, for the owner
        unsigned long long base = 0;
#pragma unroll
        for (int r = 0; r < 4; r++) {
            const unsigned long long sj = lane + 64 * r < R.n_head ? v[r] & ((1ull << 58) - 1) : 0;
            if (lane + 64 * r == owner) base = incl[r] - sj;
        }
        if (lane + 64 * 0 == owner || lane + 64 * 1 == owner || lane + 64 * 2 == owner || lane + 64 * 3 == owner) uscr[3] = base;
    }
    __syncthreads();
    const int owner = iscr[0];
    const unsigned long long k = uscr[1], z = uscr[2], base = uscr[3];
    __syncthreads();
    if (owner < 0) return false;
    // 4. the owner walks its slice; with no owner (a zero grand total) head 0 answers the last index
    if (owner == h || (owner == 0x7FFFFFFF && h == 0)) {
        const int cand = owner == h && tid < nrow && crosses(base + before + w, k, z) ? tid : 0x7FFFFFFF;
        const int first = block_min_int(cand, iscr);
        const int tok = first == 0x7FFFFFFF ? (owner == h ? r0 + nrow - 1 : M.vocab - 1) : r0 + first;
        if (tid == 0) __hip_atomic_store(gw(R.sync + SY_TOKEN), token_word(s, tok), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    }
    return true;
}

// Head workgroup h: tiles [h * head_tpw, (h + 1) * head_tpw) of step s, once the final residual is out.
template <int DT, bool G2>
__device__ __noinline__ bool head_role(const l3m_dmodel *Mp, const l3m_run *Rp, int h, int s) {
    extern __shared__ __align__(16) uint8_t smem[];
    __shared__ int ok_lds;
    h = uniform(h); s = uniform(s);
    const l3m_dmodel M = fixed(Mp);
    const l3m_run R = fixed(Rp);
    const int pos = R.pos0 + s, t0 = h * R.head_tpw;
    const bool has_tiles = t0 < M.head.tiles;
    float v = -INFINITY;
    int idx = 0x7FFFFFFF;
    const l3m_dmat V = head_slice(M, has_tiles ? t0 : 0, R.head_tpw);
    HeadW<DT> wt;
    phase_arm(pos, M.n_layers - 1, M.n_layers);
    phase(128 + h, 0, pos, M.n_layers - 1);
    if (has_tiles) {
        pro_static(wt.st, M.dim >> 2, M.norm, nullptr, 0);
        head_issue<DT>(wt, V);
    }
    // the last layer's FFN flags, set once its partials are stored through (epoch (s + 1) L)
    if (!wait_flags<4>(R.sync + SY_FFN, M.n_chunks, (unsigned)((s + 1) * M.n_layers), R.sync + SY_ABORT, R.spin_limit, &ok_lds))
        return false;
    phase(128 + h, 1, pos, M.n_layers - 1);
    const float temp = R.temp;
    float *keep = temp > 0 ? (float *)(smem + lds_h(DT, M.dim, M.head.nb, R.head_tpw).lgv) : nullptr;
    if (has_tiles) head_block<DT, true, G2>(M, V, t0, R.head_tpw, pos, wt, smem, v, idx, keep, 128 + h);
    phase(128 + h, 2, pos, M.n_layers - 1);
    if (tidx() == 0)
        __hip_atomic_store(gw((uint64_t *)(R.sync + SY_SLOTS) + h), argmax_key(v, idx, step_tag(s)), __ATOMIC_RELAXED,
                           __HIP_MEMORY_SCOPE_AGENT);
    phase(128 + h, 3, pos, M.n_layers - 1);
    if (temp > 0 && !sample_step(M, R, h, s, has_tiles ? V.rows : 0, t0 * 16, smem)) return false;
    return true;
}

// Roles from where the workgroup runs: the first n_body workgroups to arrive on the body XCD take the
// attention groups then the FFN chunks; every other workgroup takes the next head index.
__device__ int deal_role(const l3m_run &R, int n_body, int *lds) {
    if (tidx() == 0) {
        const unsigned x = xcc_id();
        int role = -1;
        if ((int)x == R.body_xcc) {
            const unsigned t = __hip_atomic_fetch_add(gw(R.sync + SY_TICKET + x), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((int)t < n_body) role = (int)t;
        }
        if (role < 0)
            role = n_body + (int)__hip_atomic_fetch_add(gw(R.sync + SY_HEAD_TICKET), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        *lds = role;
    }
    __syncthreads();
    const int role = *lds;
    __syncthreads();
    return role;
}

// DT: the body's dtype, HDT: the head's (a file may quantize its head differently, as the reference's
// exporter allows: test_engine.py:187-191); G2: the GPT-2 variant (model.h:19-26); HD: the head dimension
// as a constant, or 0 to read it from the model (attn_role).
template <int DT, int HDT, bool G2, int HD = 0>
__global__ void __launch_bounds__(NTE) k_decode(const l3m_dmodel *__restrict__ Mp, const l3m_dlayer *__restrict__ layers,
                                                const l3m_run *__restrict__ Rp) {
    __shared__ int role_lds;
    const l3m_run R = fixed(Rp);
    const int n_groups = Mp->n_groups, n_chunks = Mp->n_chunks, n_body = n_groups + n_chunks;
    const int role = deal_role(R, n_body, &role_lds);
    for (int s = 0; s < R.nsteps; s++) {
        if (role < n_groups) {
            if (!attn_role<DT, G2, HD>(Mp, layers, Rp, role, s)) return;
        } else if (role < n_body) {
            if (!ffn_role<DT, G2>(Mp, layers, Rp, role - n_groups, s)) return;
        } else if (R.pos0 + s >= R.head_from && role - n_body < R.n_head) {
            if (!head_role<HDT, G2>(Mp, Rp, role - n_body, s)) return;
        }
    }
    // the last step's token has no next step in this launch to take it: group 0 writes it
    const int last = R.pos0 + R.nsteps - 1;
    if (role == 0 && R.nsteps > 0 && last >= R.head_from) {
        const int tok = R.temp > 0
                            ? wait_token_word(R.sync + SY_TOKEN, R.nsteps - 1, R.sync + SY_ABORT, R.spin_limit, &role_lds)
                            : wait_token((const uint64_t *)(R.sync + SY_SLOTS), R.n_head, R.nsteps - 1, R.sync + SY_ABORT, R.spin_limit, &role_lds);
        if (tok >= 0 && tidx() == 0) {
            gw(Mp->tokens)[last + 1] = tok;
            out_token(R, last, tok);
        }
    }
}

// Where the workgroups of a grid land: out[b] = the XCD of block b (the decode kernel's launch shape).
__global__ void __launch_bounds__(NTE) k_where(int *out) {
    if (tidx() == 0) out[blockIdx.x] = (int)xcc_id();
}

// ------------------------------------------------------------------ batched prompt prefill
// The prompt positions before the last one, all at once: per layer, the same
// operations as the decode step (engine.c:230-275) on P tokens, with the matrices as GEMMs on the matrix
// cores. The decode path then runs from the last prompt position on, over the K/V rows these kernels wrote.
// Weights are lane-tile planes of the full matrices, q8_0 (DT; q4_0 and mxfp4 widened exactly) or bf16; each
// token's activation is prepared as the decode step prepares it.

// x[t] = the embedding row of tokens[t] (engine.c:236), t < P; one workgroup per token.
__global__ void __launch_bounds__(NTE) k_pf_embed(l3m_dmat embed, const int32_t *tokens, int dim, float *x) {
    const int t = blockIdx.x, f = tidx();
    if (4 * f < dim) ((float4 *)(x + (size_t)t * dim))[f] = lt_elem4(embed, tokens[t], 4 * f);
}

// A prefill activation: per 16 tokens and 32-input block the tokens' blocks, [token / 16][block][16][32] int8
// with its scale beside it in [token / 16][block][16] (the prep of pack.c:101-123; the block sums are not
// needed), or [token / 16][block][16][32] bf16, so that a product's operand is one contiguous run, as a weight
// tile's is. Rows of tokens past the
// prompt's end hold whatever was there: a product's column depends on its own token alone, and theirs are not
// stored.
__device__ __forceinline__ size_t pf_slot(int t, int b, int nb) { return ((size_t)(t >> 4) * nb + b) * 16 + (t & 15); }

__device__ __forceinline__ uint2 pack_bf16(float4 y) {
    return make_uint2((uint32_t)f32_bf16(y.x) | (uint32_t)f32_bf16(y.y) << 16, (uint32_t)f32_bf16(y.z) | (uint32_t)f32_bf16(y.w) << 16);
}
// Values e .. e + 3 (e a multiple of 4) of token t's activation, 8 consecutive lanes a block: prep_body's
// formulas. All lanes of a block take part; store: whether they write.
template <int DT>
__device__ __forceinline__ void pf_put4(const l3m_pfact &a, int t, int nb, int e, float4 y, bool store) {
    if constexpr (DT == L3M_BF16) {
        if (store) *(uint2 *)(a.q + pf_slot(t, e >> 5, nb) * 64 + 2 * (e & 31)) = pack_bf16(y);
        return;
    }
    const float am = lanes_max<8>(fmaxf(fmaxf(fabsf(y.x), fabsf(y.y)), fmaxf(fabsf(y.z), fabsf(y.w))));
    const float inv = am > 0.f ? 127.0f / am : 0.f;
    const int q0 = (int)rintf(y.x * inv), q1 = (int)rintf(y.y * inv), q2 = (int)rintf(y.z * inv), q3 = (int)rintf(y.w * inv);
    if (!store) return;
    const size_t slot = pf_slot(t, e >> 5, nb);
    *(uint32_t *)(a.q + slot * 32 + (e & 31)) = (uint32_t)(q0 & 255) | (uint32_t)(q1 & 255) << 8 | (uint32_t)(q2 & 255) << 16 | (uint32_t)(q3 & 255) << 24;
    if ((e & 31) == 0) a.s[slot] = am / 127.0f;
}

// act[t] = the prep of y[t][0..k), or (NORM) of RMSNorm(y[t]) * w (engine.c:241, 261): a wavefront per token, 4
// values a lane for every 256, the sum of squares added as norm_prep adds it (per 256, then the 16 slots'
// tree). One wavefront per token instead of a 1024-thread workgroup, no LDS or barrier: 479 tokens of 576
// values 4.7 us, as before (4.8): what is left is one kernel's fixed cost, loads and launch.
template <int DT, bool NORM, int C>                  // C: 256-value pieces of a row
__global__ void __launch_bounds__(256) k_pf_rows(const float *y, int k, const float *w, float eps, l3m_pfact act, int P) {
    const int t = 4 * blockIdx.x + wave_id(), lane = tidx() & 63, nb = k >> 5;
    if (t >= P) return;
    const float *row = y + (size_t)t * k;
    // every load first (past k: buffer loads past the range, no branch and no access), the weights' among them
    float4 v[C], nw[C];
#pragma unroll
    for (int c = 0; c < C; c++) v[c] = ld16f_if<false>(row, 64 * c + lane, 256 * c + 4 * lane < k);
    if constexpr (NORM) {
#pragma unroll
        for (int c = 0; c < C; c++) nw[c] = ld16f_if<false>(w, 64 * c + lane, 256 * c + 4 * lane < k);
    }
    float s = 1.f;
    if constexpr (NORM) {
        float part[16], q[4];
#pragma unroll
        for (int c = 0; c < 16; c++) part[c] = 0.f;
#pragma unroll
        for (int c = 0; c < C; c++) part[c] = lanes_sum<64>(v[c].x * v[c].x + v[c].y * v[c].y + v[c].z * v[c].z + v[c].w * v[c].w);
#pragma unroll
        for (int i = 0; i < 4; i++) q[i] = (part[4 * i] + part[4 * i + 1]) + (part[4 * i + 2] + part[4 * i + 3]);
        s = 1.0f / sqrtf(((q[0] + q[1]) + (q[2] + q[3])) / (float)k + eps);
    }
#pragma unroll
    for (int c = 0; c < C; c++) {
        const int e = 256 * c + 4 * lane;
        float4 x = v[c];
        if constexpr (NORM) x = make_float4(x.x * s * nw[c].x, x.y * s * nw[c].y, x.z * s * nw[c].z, x.w * s * nw[c].w);
        pf_put4<DT>(act, t, nb, e, x, e < k);
    }
}

// The matrices of a prompt (the gemv of every token at once, kernels_scalar.c:16-45): per 16 rows x 16 tokens and
// 32-input block one product. q8_0: v_mfma_i32_16x16x32_i8, its i32 result scaled by the row's and the token's
// block scales into the f32 sum; bf16: v_mfma_f32_16x16x32_bf16 onto the f32 sum. Blocks in order. Lane l holds
// row (token) l % 16, the 8 values at 8 (l / 16) of the block, and gets rows 4 (l / 16) + i of token l % 16.
//
// A row's blocks fall into ranges of PF_RANGE blocks or so (pf_ranges). int8: each range is summed by itself and the sums
// added in order; bf16: every product goes onto one sum. A wavefront takes RT x TT tiles over its share of the ranges:
// KS = blockDim / (64 WR) wavefronts split them, and their sums are added in order through LDS; WR wavefronts of each share lie side by side. Operands come straight from L2 in the layouts they lie in (a contiguous run a tile and
// block), PB blocks ahead; nothing is staged. Per q8_0 product a lane spends 12 VALU instructions on the scales
// (48 clocks of its SIMD against 8 for the product), which bounds the largest shapes; RT = TT = 2 loads each
// operand once for two products. The others are bound by latency, a chain of loads over few wavefronts: they
// split the blocks (pf_gemm's rule). 479 tokens, 30 layers of dim 576 and ffn 1536 (kernel trace), against one
// 16 x 16 tile a workgroup with each token's input in a row of its own: q/k/v 14.8 -> 7.7 us, Wo 10.8 -> 7.2,
// gate/up 36.7 -> 12.0 with the SiLU and prep kernel (4.9) gone into it, Wdown 24.4 -> 9.3. bf16, 199 tokens, 6
// layers of dim 288 and ffn 768: 6.2 / 4.8 / 6.1 / 5.8 us, where the prompt had gone token by token.
//
// EPI 0: y += the product (the residual adds, engine.c:259, 275).
// EPI 1: the q/k/v rows: RoPE on q and k (pairs (2i, 2i + 1) of each head rotated by angle i of position t from
//        the host table, ops.c:29-40), q into y, the k and v rows rounded to bf16 into the cache
//        (engine.c:247-248). A lane's four rows are two whole pairs.
// EPI 2: gate and up rows (RT = 2: the same rows' gate tile and up tile), up * silu(gate) (ops.c:49-51) and its
//        prep into out: the workgroup's 2 x 16 rows are one 32-block of the next matrix's input.
typedef int v4i32 __attribute__((ext_vector_type(4)));
constexpr int PF_RANGE = 4;
__host__ __device__ inline int pf_ranges(int nb) { return min(max((nb + PF_RANGE - 1) / PF_RANGE, 1), 16); }
struct PfGemm {
    l3m_dmat W;
    l3m_pfact x, out;
    int P, ystride;
    float *y;
    const float *rope;                                // EPI 1
    uint16_t *kc, *vc;
    int layer, ctx, nq, nk, hd, n_kv;
};
template <int DT, int RT_, int TT_> struct PfFrag {
    std::conditional_t<DT == L3M_BF16, bf16x8, long> a[RT_], x[TT_];
    u32x2 sw[RT_];                                    // q8_0: the scales
    float sx[TT_];
};
template <int DT, int EPI, int RT_, int TT_, int WR, int KMAX>
__global__ void __launch_bounds__(64 * WR * KMAX) k_pf_gemm(PfGemm G) {
    constexpr int PB = 4, QB = qbytes(DT);
    using Frag = PfFrag<DT, RT_, TT_>;
    __shared__ f32x4 part[KMAX > 1 ? (KMAX - 1) * WR * RT_ * TT_ : 1][64];
    __shared__ float amx[EPI == 2 ? WR * TT_ : 1][16];
    const int lane = tidx() & 63, wave = wave_id(), c16 = lane & 15, quarter = lane >> 4;
    const int kw = wave / WR, wr = wave % WR, nb = G.W.nb;
    const int KS = KMAX > 1 ? (int)blockDim.x / (64 * WR) : 1, R = pf_ranges(nb), per = (nb + R - 1) / R;
    const int k0 = min(kw * R / KS * per, nb), k1 = min((kw + 1) * R / KS * per, nb);
    int rt[RT_], tt[TT_];                             // 16-row tiles, 16-token tiles
#pragma unroll
    for (int r = 0; r < RT_; r++)
        rt[r] = EPI == 2 ? (int)blockIdx.x * WR + wr + r * (G.W.tiles >> 1) : ((int)blockIdx.x * WR + wr) * RT_ + r;
#pragma unroll
    for (int t = 0; t < TT_; t++) tt[t] = (int)blockIdx.y * TT_ + t;
    const uint8_t *wq[RT_], *xq[TT_];
    const uint16_t *ws[RT_];
    const float *xs[TT_];
#pragma unroll
    for (int r = 0; r < RT_; r++) {
        const size_t at = (size_t)min(rt[r], G.W.tiles - 1) * nb * 16;   // tiles past the last: it again, not stored
        wq[r] = G.W.q + (at + c16) * QB + quarter * (QB / 4);
        ws[r] = (const uint16_t *)G.W.s + at + quarter * 4;
    }
#pragma unroll
    for (int t = 0; t < TT_; t++) {
        const size_t at = (size_t)tt[t] * nb * 16 + c16;
        xq[t] = G.x.q + at * QB + quarter * (QB / 4);
        xs[t] = G.x.s + at;
    }
    Frag f[PB];
    auto load = [&](Frag &g, int b) {
        b = min(b, nb - 1);                           // past the range: a block in bounds, not used
#pragma unroll
        for (int r = 0; r < RT_; r++) {
            if constexpr (DT == L3M_BF16) g.a[r] = __builtin_bit_cast(bf16x8, *gp<u32x4>(wq[r] + (size_t)b * 16 * QB));
            else {
                g.a[r] = *gp<long>(wq[r] + (size_t)b * 16 * QB);
                g.sw[r] = *gp<u32x2>(ws[r] + (size_t)b * 16);
            }
        }
#pragma unroll
        for (int t = 0; t < TT_; t++) {
            if constexpr (DT == L3M_BF16) g.x[t] = __builtin_bit_cast(bf16x8, *gp<u32x4>(xq[t] + (size_t)b * 16 * QB));
            else {
                g.x[t] = *gp<long>(xq[t] + (size_t)b * 16 * QB);
                g.sx[t] = *gp<float>(xs[t] + (size_t)b * 16);
            }
        }
    };
    f32x4 acc[RT_][TT_], cur[RT_][TT_];               // the sum of the ranges done, the current range's
#pragma unroll
    for (int r = 0; r < RT_; r++)
#pragma unroll
        for (int t = 0; t < TT_; t++) acc[r][t] = cur[r][t] = f32x4{0.f, 0.f, 0.f, 0.f};
    int next = k0 + per;
#pragma unroll
    for (int i = 0; i < PB; i++) load(f[i], k0 + i);
    for (int b0 = k0; b0 < k1; b0 += PB) {
#pragma unroll
        for (int i = 0; i < PB; i++) {
            if (b0 + i < k1) {                        // uniform
                if constexpr (DT == L3M_BF16) {
#pragma unroll
                    for (int r = 0; r < RT_; r++)
#pragma unroll
                        for (int t = 0; t < TT_; t++) acc[r][t] = mfma_bf16(f[i].a[r], f[i].x[t], acc[r][t]);
                } else {
#pragma unroll
                    for (int r = 0; r < RT_; r++) {
                        const float d[4] = {f16_f32(f[i].sw[r].x & 0xFFFF), f16_f32(f[i].sw[r].x >> 16), f16_f32(f[i].sw[r].y & 0xFFFF),
                                            f16_f32(f[i].sw[r].y >> 16)};
#pragma unroll
                        for (int t = 0; t < TT_; t++) {
                            const v4i32 c = __builtin_amdgcn_mfma_i32_16x16x32_i8(f[i].a[r], f[i].x[t], v4i32{0, 0, 0, 0}, 0, 0, 0);
#pragma unroll
                            for (int j = 0; j < 4; j++) cur[r][t][j] += (float)c[j] * (d[j] * f[i].sx[t]);
                        }
                    }
                    if (b0 + i + 1 == next || b0 + i + 1 == k1) {   // uniform: the range is done
                        next += per;
#pragma unroll
                        for (int r = 0; r < RT_; r++)
#pragma unroll
                            for (int t = 0; t < TT_; t++) { acc[r][t] += cur[r][t]; cur[r][t] = f32x4{0.f, 0.f, 0.f, 0.f}; }
                    }
                }
            }
            load(f[i], b0 + PB + i);
        }
    }
    if constexpr (KMAX > 1) {
        if (kw) {
#pragma unroll
            for (int r = 0; r < RT_; r++)
#pragma unroll
                for (int t = 0; t < TT_; t++) part[((kw - 1) * WR + wr) * RT_ * TT_ + r * TT_ + t][lane] = acc[r][t];
        }
        __syncthreads();
        if (kw == 0) {
#pragma unroll
            for (int k = 1; k < KMAX; k++) {
                if (k >= KS) break;
#pragma unroll
                for (int r = 0; r < RT_; r++)
#pragma unroll
                    for (int t = 0; t < TT_; t++) {
                        const f32x4 p = part[((k - 1) * WR + wr) * RT_ * TT_ + r * TT_ + t][lane];
                        acc[r][t][0] += p[0]; acc[r][t][1] += p[1]; acc[r][t][2] += p[2]; acc[r][t][3] += p[3];
                    }
            }
        }
    }
    if constexpr (EPI == 2) {
        float4 h[TT_];
        float am[TT_];
        if (kw == 0) {
#pragma unroll
            for (int t = 0; t < TT_; t++) {
                const f32x4 g = acc[0][t], u = acc[RT_ - 1][t];
                h[t] = make_float4(silu_mul(u[0], g[0]), silu_mul(u[1], g[1]), silu_mul(u[2], g[2]), silu_mul(u[3], g[3]));
                if constexpr (DT == L3M_BF16) {
                    const int tok = 16 * tt[t] + c16;
                    if (tok < G.P) *(uint2 *)(G.out.q + pf_slot(tok, blockIdx.x, G.W.tiles >> 2) * 64 + 32 * wr + 8 * quarter) = pack_bf16(h[t]);
                    continue;
                }
                float m = fmaxf(fmaxf(fabsf(h[t].x), fabsf(h[t].y)), fmaxf(fabsf(h[t].z), fabsf(h[t].w))), lo, hi;
                swap16(m, lo, hi); m = fmaxf(lo, hi);
                swap32(m, lo, hi); am[t] = fmaxf(lo, hi);
                if (quarter == 0) amx[wr * TT_ + t][c16] = am[t];
            }
        }
        if constexpr (DT == L3M_BF16) return;
        __syncthreads();
        if (kw == 0) {
#pragma unroll
            for (int t = 0; t < TT_; t++) {
                const int tok = 16 * tt[t] + c16;
                const float m = fmaxf(am[t], amx[(wr ^ 1) * TT_ + t][c16]);   // WR = 2: the block's other 16 rows
                const float inv = m > 0.f ? 127.0f / m : 0.f;
                const int q0 = (int)rintf(h[t].x * inv), q1 = (int)rintf(h[t].y * inv), q2 = (int)rintf(h[t].z * inv), q3 = (int)rintf(h[t].w * inv);
                if (tok < G.P) {
                    const size_t slot = pf_slot(tok, blockIdx.x, G.W.tiles >> 2);
                    *(uint32_t *)(G.out.q + slot * 32 + 16 * wr + 4 * quarter) =
                        (uint32_t)(q0 & 255) | (uint32_t)(q1 & 255) << 8 | (uint32_t)(q2 & 255) << 16 | (uint32_t)(q3 & 255) << 24;
                    if (wr == 0 && quarter == 0) G.out.s[slot] = m / 127.0f;
                }
            }
        }
        return;
    }
    if (kw) return;
#pragma unroll
    for (int r = 0; r < RT_; r++)
#pragma unroll
        for (int t = 0; t < TT_; t++) {
            const int tok = 16 * tt[t] + c16, r0 = 16 * rt[r] + 4 * quarter;
            if (tok >= G.P || r0 >= G.W.rows) continue;
            f32x4 v = acc[r][t];
            if constexpr (EPI == 0) {                 // rows: whole 32-blocks
                float4 *o = (float4 *)(G.y + (size_t)tok * G.ystride + r0);
                const float4 x = *o;
                *o = make_float4(x.x + v[0], x.y + v[1], x.z + v[2], x.w + v[3]);
            } else {
                // q, k and v rows each begin at a multiple of 8: the four rows lie in one of them
                const bool isq = r0 < G.nq, isv = r0 >= G.nq + G.nk;
                const int e = isq ? r0 : isv ? r0 - G.nq - G.nk : r0 - G.nq, hh = e / G.hd, j = e - hh * G.hd;
                if (!isv) {
                    const float4 cs = *(const float4 *)(G.rope + (size_t)tok * G.hd + j);   // the two pairs' (cos, sin)
                    const float a = v[0], b = v[1], c = v[2], d = v[3];
                    v[0] = a * cs.x - b * cs.y; v[1] = a * cs.y + b * cs.x;
                    v[2] = c * cs.z - d * cs.w; v[3] = c * cs.w + d * cs.z;
                }
                if (isq) *(float4 *)(G.y + (size_t)tok * G.ystride + r0) = make_float4(v[0], v[1], v[2], v[3]);
                else *(uint2 *)((isv ? G.vc : G.kc) + (((size_t)G.layer * G.n_kv + hh) * G.ctx + tok) * G.hd + j) =
                    pack_bf16(make_float4(v[0], v[1], v[2], v[3]));
            }
        }
}

// The form for the other head dims (k_pf_attn takes multiples of 16 up to 128).
// Attention of token t, head h over positions 0..t (ops.c:42-73): one wavefront per (t, h), positions in
// chunks of 64 (a lane per position) with a running maximum and sum; then each lane sums its output
// dims over the chunk's weights. q from qb (after RoPE), K and V from the cache as bf16.
__global__ void __launch_bounds__(64) k_pf_attend(const float *qb, int P, int n_heads, int n_kv, int hd, int ctx, int layer,
                                                  float scale, const uint16_t *kc, const uint16_t *vc, float *att) {
    constexpr int VMAX = 32;                          // V rows a lane loads per 64-position chunk (h8 <= 32)
    __shared__ float qs[256], ps[64], part[64 * 8];
    const int t = blockIdx.x, h = blockIdx.y, lane = tidx(), hpk = n_heads / n_kv, kv = h / hpk;
    const int width = n_heads * hd, h8 = hd >> 3;
    // P.V: lane = jg * h8 + dg takes dims [8 dg, 8 dg + 8) at positions jg, jg + JG, ... of a chunk
    const int JG = 64 / h8, jg = lane / h8, dg = lane - jg * h8;
    const bool vlane = jg < JG;
    for (int d = lane; d < hd; d += 64) qs[d] = qb[(size_t)t * width + h * hd + d];
    __syncthreads();
    const uint16_t *K = kc + ((size_t)layer * n_kv + kv) * ctx * hd, *V = vc + ((size_t)layer * n_kv + kv) * ctx * hd;
    float m = -INFINITY, l = 0.f, o[4] = {0.f, 0.f, 0.f, 0.f};   // output dims lane, lane + 64, ... (hd <= 256)
    for (int p0 = 0; p0 <= t; p0 += 64) {
        const int p = p0 + lane, n = t - p0 + 1 < 64 ? t - p0 + 1 : 64;
        // the V rows this lane multiplies, requested before the scores so their latency overlaps them
        uint4 vv[VMAX];
#pragma unroll
        for (int u = 0; u < VMAX; u++) {
            const int j = jg + u * JG;
            vv[u] = (u * JG < 64) ? ((const uint4 *)(V + (size_t)(p0 + (vlane && j < n ? j : 0)) * hd))[dg] : make_uint4(0u, 0u, 0u, 0u);
        }
        float sc = -INFINITY;
        if (p <= t) {
            // the lane's K row in 16-byte words, eight loads in flight before their products
            const uint4 *kr = (const uint4 *)(K + (size_t)p * hd);
            float dot = 0.f;
            for (int v0 = 0; v0 < h8; v0 += 8) {
                uint4 kk[8];
#pragma unroll
                for (int u = 0; u < 8; u++) kk[u] = kr[v0 + u < h8 ? v0 + u : h8 - 1];
#pragma unroll
                for (int u = 0; u < 8; u++)
                    if (v0 + u < h8) dot = dot8_bf16(qs + 8 * (v0 + u), kk[u], dot);
            }
            sc = dot * scale;
        }
        const float cm = lanes_max<64>(sc), nm = fmaxf(m, cm);
        const float w = p <= t ? expf(sc - nm) : 0.f, rescale = expf(m - nm);
        l = l * rescale + lanes_sum<64>(w);
        ps[lane] = w;
        __syncthreads();
        // each lane's 8 dims over its positions, then the JG partial sums of a dim added in jg order
        float acc[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int u = 0; u < VMAX; u++) {
            const int j = jg + u * JG;
            if (u * JG < 64 && vlane && j < n) {
                const float pj = ps[j];
                const uint4 x = vv[u];
                acc[0] += pj * bf16_f32(x.x & 0xFFFF); acc[1] += pj * bf16_f32(x.x >> 16);
                acc[2] += pj * bf16_f32(x.y & 0xFFFF); acc[3] += pj * bf16_f32(x.y >> 16);
                acc[4] += pj * bf16_f32(x.z & 0xFFFF); acc[5] += pj * bf16_f32(x.z >> 16);
                acc[6] += pj * bf16_f32(x.w & 0xFFFF); acc[7] += pj * bf16_f32(x.w >> 16);
            }
        }
        if (vlane) {
#pragma unroll
            for (int e = 0; e < 8; e++) part[jg * hd + 8 * dg + e] = acc[e];
        }
        __syncthreads();
#pragma unroll
        for (int i = 0; i < 4; i++) {
            const int d = lane + 64 * i;
            if (d < hd) {
                float sum = 0.f;
                for (int g = 0; g < JG; g++) sum += part[g * hd + d];
                o[i] = o[i] * rescale + sum;
            }
        }
        m = nm;
        __syncthreads();
    }
#pragma unroll
    for (int i = 0; i < 4; i++) {
        const int d = lane + 64 * i;
        if (d < hd) att[(size_t)t * n_heads * hd + h * hd + d] = o[i] / l;
    }
}

// Causal attention of the prompt on the matrix cores (ops.c:42-73), for head dims that are multiples of 16
// up to 128: a workgroup takes 16 consecutive tokens of one head, its PFA_W wavefronts every PFA_W-th chunk
// of 32 positions, each with a running maximum, and their results meet in LDS at the end.
//  - Scores transposed: A = the chunk's K rows as they lie in the cache (lane l: row l % 16, 8 dims at
//    8 (l / 16) of each 32), B = the tokens' q as three bf16 parts (split3: every product exact in f32). A
//    lane then holds one token's (l % 16) scores of positions 4 (l / 16) + i of both 16-position tiles, so
//    the softmax is per lane: the maximum meets the token's other three lanes in two permlane swaps.
//  - Those 8 positions are also the lane's share of the contraction of P.V (the order within a product is
//    free, V's operand takes the same): p, as three bf16 parts, goes from the softmax to B in registers.
//    A = V^T, dims by positions: the wavefront transposes the chunk's V rows (4 positions x 8 dims a lane)
//    into its own LDS span, rows of 40 elements, the lane's 8 positions contiguous.
// A masked position's p is 0 and a part of q may be, but 0 times an infinity or a NaN in a V or K row is NaN: where
// any of a wavefront's sums is not finite, the tile's tokens are done one at a time instead (pf_attn_token), over
// their own positions alone. (A flag from the merged outputs and a second barrier cost a prompt of 64 tokens 1%.)
// No barrier before the end. Bound by the chunk's chain (loads, two products, expf, LDS round trip), not by
// bytes or products: 9 heads of 64, 479 tokens: 11.1 us a layer, against 55.7 for k_pf_attend (one wavefront
// per token and head, a lane per position: every token reads every K and V row again); 63 tokens: 5.0 (7.0).
constexpr int PFA_W = 4, PFA_T = 16, PFA_C = 32, PFA_VROW = 40;
// Attention of one token over positions 0..tok by one wavefront, every product in f32 and no row past tok read:
// lane l scores position l of each 64, then adds dims l and l + 64 up. buf: HD + 64 floats of the wavefront's
// own LDS; the output is left in its first HD.
template <int HD>
__device__ void pf_attn_token(const float *q, const uint16_t *K, const uint16_t *V, int tok, float scale, float *buf) {
    constexpr int ND = (HD + 63) / 64;
    const int lane = tidx() & 63;
    float *ps = buf + HD;
    auto lds_done = [] { asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory"); __builtin_amdgcn_wave_barrier(); };
    lds_done();
    for (int d = lane; d < HD; d += 64) buf[d] = q[d];
    lds_done();
    float m = -INFINITY, l = 0.f, o[ND];
#pragma unroll
    for (int i = 0; i < ND; i++) o[i] = 0.f;
    for (int p0 = 0; p0 <= tok; p0 += 64) {
        const int n = min(tok - p0 + 1, 64);
        float s = -INFINITY;
        if (lane < n) {
            float dot = 0.f;
            for (int d = 0; d < HD; d++) dot = fmaf(buf[d], bf16_f32(K[(size_t)(p0 + lane) * HD + d]), dot);
            s = dot * scale;
        }
        const float nm = fmaxf(m, lanes_max<64>(s)), base = nm == -INFINITY ? 0.f : nm, r = expf(m - base);
        const float p = lane < n ? expf(s - base) : 0.f;
        l = l * r + lanes_sum<64>(p);
        ps[lane] = p;
        lds_done();
#pragma unroll
        for (int i = 0; i < ND; i++) {
            const int d = lane + 64 * i;
            if (d < HD) {
                o[i] *= r;
                for (int j = 0; j < n; j++) o[i] = fmaf(ps[j], bf16_f32(V[(size_t)(p0 + j) * HD + d]), o[i]);
            }
        }
        lds_done();
        m = nm;
    }
#pragma unroll
    for (int i = 0; i < ND; i++)
        if (lane + 64 * i < HD) buf[lane + 64 * i] = o[i] / l;
    lds_done();
}
template <int DT, int HD>
__global__ void __launch_bounds__(64 * PFA_W) k_pf_attn(const float *qb, int P, int n_heads, int n_kv, int ctx, int layer, float scale,
                                                        const uint16_t *kc, const uint16_t *vc, float *att, l3m_pfact act) {
    constexpr int KS = (HD + 31) / 32, NT16 = HD / 16, D8 = HD / 8, UNITS = (HD + 63) / 64, OROW = HD + 4;
    constexpr size_t VT = (size_t)HD * PFA_VROW * 2;                     // one wavefront's V^T chunk; its merge span is no larger
    static_assert((size_t)PFA_T * OROW * 4 <= VT, "the merge spans fit the V^T spans");
    __shared__ __align__(16) uint8_t lds[PFA_W * VT];
    static_assert((HD + 64) * 4 <= VT, "pf_attn_token's floats too");
    __shared__ float ml[2][PFA_W][PFA_T];
    __shared__ int odd[PFA_W];                        // the wavefront has a sum that is not finite
    const int lane = tidx() & 63, wave = wave_id(), c16 = lane & 15, quarter = lane >> 4;
    // the tiles with the most positions first
    const int t0 = PFA_T * ((int)gridDim.x - 1 - (int)blockIdx.x), h = blockIdx.y, kv = h / (n_heads / n_kv);
    const int width = n_heads * HD, tmax = (t0 + PFA_T < P ? t0 + PFA_T : P) - 1, tok = min(t0 + c16, tmax);
    const uint16_t *K = kc + ((size_t)layer * n_kv + kv) * ctx * HD, *V = vc + ((size_t)layer * n_kv + kv) * ctx * HD;
    uint16_t *vt = (uint16_t *)(lds + wave * VT);
    bf16x8 q[3][KS];
#pragma unroll
    for (int s = 0; s < KS; s++) {
        const int d = 32 * s + 8 * quarter;
        const float *src = qb + (size_t)tok * width + h * HD + (d < HD ? d : 0);
        const float4 a = ldg16f(src, 0), b = ldg16f(src, 1);
        const float x[8] = {a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
#pragma unroll
        for (int j = 0; j < 8; j++) {
            __bf16 p0, p1, p2;
            split3(d < HD ? x[j] : 0.f, p0, p1, p2);
            q[0][s][j] = p0; q[1][s][j] = p1; q[2][s][j] = p2;
        }
    }
    f32x4 o[NT16];
#pragma unroll
    for (int n = 0; n < NT16; n++) o[n] = f32x4{0.f, 0.f, 0.f, 0.f};
    float m = -INFINITY, l = 0.f;
    for (int p0 = PFA_C * wave; p0 <= tmax; p0 += PFA_C * PFA_W) {
        bf16x8 kk[2][KS];
        u32x4 vv[UNITS][4];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            const uint16_t *row = K + (size_t)min(p0 + 16 * u + c16, tmax) * HD;   // positions past the last: its row, masked below
#pragma unroll
            for (int s = 0; s < KS; s++) {
                const int d = 32 * s + 8 * quarter;
                kk[u][s] = __builtin_bit_cast(bf16x8, *gp<u32x4>(row + (d < HD ? d : 0)));   // past HD: times zeros of q
            }
        }
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            const int id = lane + 64 * u, dg = id % D8, pq = id / D8 < 8 ? id / D8 : 7;
#pragma unroll
            for (int e = 0; e < 4; e++) vv[u][e] = *gp<u32x4>(V + (size_t)min(p0 + 4 * pq + e, tmax) * HD + 8 * dg);
        }
        f32x4 sc[2];
#pragma unroll
        for (int u = 0; u < 2; u++) {
            sc[u] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
            for (int part = 2; part >= 0; part--)
#pragma unroll
                for (int s = 0; s < KS; s++) sc[u] = mfma_bf16(kk[u][s], q[part][s], sc[u]);
        }
        float mx = -INFINITY;
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                sc[u][i] = p0 + 16 * u + 4 * quarter + i <= tok ? sc[u][i] * scale : -INFINITY;
                mx = fmaxf(mx, sc[u][i]);
            }
        float lo, hi;
        swap16(mx, lo, hi); mx = fmaxf(lo, hi);
        swap32(mx, lo, hi); mx = fmaxf(lo, hi);
        const float nm = fmaxf(m, mx), base = nm == -INFINITY ? 0.f : nm;   // no position yet: every p is 0
        const float r = expf(m - base);
        l *= r;
        bf16x8 p[3];
#pragma unroll
        for (int u = 0; u < 2; u++)
#pragma unroll
            for (int i = 0; i < 4; i++) {
                const float e = expf(sc[u][i] - base);
                __bf16 x0, x1, x2;
                l += e;
                split3(e, x0, x1, x2);
                p[0][4 * u + i] = x0; p[1][4 * u + i] = x1; p[2][4 * u + i] = x2;
            }
        m = nm;
        // V^T: position quad pq (positions 4 pq ..) at element 4 ((pq % 4) * 2 + pq / 4), so that a lane's 8
        // positions (4 quarter + i, 16 + 4 quarter + i) are 16 contiguous bytes
#pragma unroll
        for (int u = 0; u < UNITS; u++) {
            const int id = lane + 64 * u, dg = id % D8, pq = id / D8;
            if (pq < 8) {
                uint16_t *dst = vt + (size_t)8 * dg * PFA_VROW + 4 * ((pq & 3) * 2 + (pq >> 2));
#pragma unroll
                for (int j = 0; j < 4; j++) {
                    *(u32x2 *)(dst + (2 * j) * PFA_VROW) = u32x2{__builtin_amdgcn_perm(vv[u][1][j], vv[u][0][j], 0x05040100u),
                                                                __builtin_amdgcn_perm(vv[u][3][j], vv[u][2][j], 0x05040100u)};
                    *(u32x2 *)(dst + (2 * j + 1) * PFA_VROW) = u32x2{__builtin_amdgcn_perm(vv[u][1][j], vv[u][0][j], 0x07060302u),
                                                                    __builtin_amdgcn_perm(vv[u][3][j], vv[u][2][j], 0x07060302u)};
                }
            }
        }
        // the span is the wavefront's own and its LDS accesses complete in order: only the compiler has to
        // keep them so
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int n = 0; n < NT16; n++) {
            const bf16x8 a = *(const bf16x8 *)(vt + (size_t)(16 * n + c16) * PFA_VROW + 8 * quarter);
            o[n][0] *= r; o[n][1] *= r; o[n][2] *= r; o[n][3] *= r;
#pragma unroll
            for (int part = 2; part >= 0; part--) o[n] = mfma_bf16(a, p[part], o[n]);
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        __builtin_amdgcn_wave_barrier();
    }
    float lo, hi;
    swap16(l, lo, hi); l = lo + hi;
    swap32(l, lo, hi); l = lo + hi;
    float *om = (float *)vt + c16 * OROW;
#pragma unroll
    for (int n = 0; n < NT16; n++) *(float4 *)(om + 16 * n + 4 * quarter) = make_float4(o[n][0], o[n][1], o[n][2], o[n][3]);
    if (quarter == 0) { ml[0][wave][c16] = m; ml[1][wave][c16] = l; }
    f32x4 z = {0.f, 0.f, 0.f, 0.f};                   // NaN where a sum is not finite
#pragma unroll
    for (int n = 0; n < NT16; n++) z += o[n] * 0.f;
    const int any = __any(!(z[0] + z[1] + z[2] + z[3] == 0.f));
    if (lane == 0) odd[wave] = any;
    __syncthreads();
    // the output's dims d .. d + 3 of token t
    auto put = [&](int t, int d, float4 y, bool store) {
        if constexpr (HD % 32 == 0 || DT == L3M_BF16) {   // whole blocks of the head: prepared here, 8 lanes a block
            pf_put4<DT>(act, t, (n_heads * HD) >> 5, h * HD + d, y, store);
        } else if (store) {
            *(float4 *)(att + (size_t)t * n_heads * HD + h * HD + d) = y;
        }
    };
    int redo = odd[0];
#pragma unroll
    for (int w = 1; w < PFA_W; w++) redo |= odd[w];
    if (__builtin_amdgcn_readfirstlane(redo)) {       // the wavefront's span: its merge rows are not read
        for (int tt = wave; tt < PFA_T && t0 + tt < P; tt += PFA_W) {
            float *buf = (float *)vt;
            pf_attn_token<HD>(qb + (size_t)(t0 + tt) * width + h * HD, K, V, t0 + tt, scale, buf);
            const bool mine = 4 * lane < HD;
            put(t0 + tt, 4 * lane, mine ? *(const float4 *)(buf + 4 * lane) : make_float4(0.f, 0.f, 0.f, 0.f), mine);
        }
        return;
    }
    // each thread 4 dims of a token: the wavefronts' parts in order, scaled to the common maximum (wavefront 0
    // always has position 0)
    for (int u = tidx(); u < PFA_T * HD / 4; u += 64 * PFA_W) {
        const int tt = u / (HD / 4), d4 = u % (HD / 4), t = t0 + tt;
        float mm = ml[0][0][tt];
#pragma unroll
        for (int w = 1; w < PFA_W; w++) mm = fmaxf(mm, ml[0][w][tt]);
        float den = 0.f;
        float4 y = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
        for (int w = 0; w < PFA_W; w++) {
            const float f = expf(ml[0][w][tt] - mm);
            const float4 x = *(const float4 *)((const float *)(lds + w * VT) + tt * OROW + 4 * d4);
            den += ml[1][w][tt] * f;
            y.x += x.x * f; y.y += x.y * f; y.z += x.z * f; y.w += x.w * f;
        }
        y = make_float4(y.x / den, y.y / den, y.z / den, y.w / den);
        put(t, 4 * d4, y, t < P);
    }
}

// ------------------------------------------------------------------ residency and exchange probes
// The GPU analogues of the reference's bench/residency.c (every core streams its own shard, at each
// working-set size) and bench/exchange.c (ns per barrier and exchange over a set of cores), which back the
// layout and hand-over choices of the decode kernel. Launched with one workgroup per CU; the workgroups on
// the chosen XCDs take tickets per XCD and work, the others leave at once.

// Shard streaming: workgroup (x, t) of the first `xcds` XCDs (t < per_xcd tickets) reads its n16 16-byte
// words `passes` times. sink keeps the loads alive.
__global__ void __launch_bounds__(NTE) k_probe_stream(const u32x4 *buf, size_t n16, int passes, int xcds, int per_xcd,
                                                      unsigned *tickets, unsigned *sink) {
    __shared__ int shard;
    if (tidx() == 0) {
        const unsigned x = xcc_id();
        int sh = -1;
        if ((int)x < xcds) {
            const unsigned t = __hip_atomic_fetch_add(gw(tickets + x), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((int)t < per_xcd) sh = (int)x * per_xcd + (int)t;
        }
        shard = sh;
    }
    __syncthreads();
    if (shard < 0) return;
    const u32x4 *p = buf + (size_t)shard * n16;
    u32x4 acc = {0u, 0u, 0u, 0u};
    for (int pass = 0; pass < passes; pass++)
        for (size_t i = tidx(); i < n16; i += NTE) acc ^= gp<u32x4>(p)[i];
    const unsigned v = acc.x ^ acc.y ^ acc.z ^ acc.w;
    if (v == 0x9E3779B9u) gw(sink)[0] = v;            // practically never: keeps the loads
}

// Exchange rounds among n workgroups (on XCD 0 when same_xcd, else dealt round-robin over the XCDs):
// round i, each writes its slice of a dim-float vector (two copies by parity), stores flag = i + 1 after its
// stores are in L2 (device-scope stores when the group spans XCDs), waits for every flag, then reads the
// whole vector. Workgroup 0 times `rounds` rounds with the 100 MHz clock. Every wait is bounded:
// past `limit` ticks the abort word is raised and all leave.
__global__ void __launch_bounds__(NTE) k_probe_exchange(float *vec, int dim, int n, int same_xcd, int rounds, unsigned *flags,
                                                        unsigned *tickets, unsigned long long *out, unsigned long long limit) {
    __shared__ int role, ok;
    if (tidx() == 0) {
        const unsigned x = xcc_id();
        int r = -1;
        if (same_xcd) {
            if (x == 0) {
                const unsigned t = __hip_atomic_fetch_add(gw(tickets), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if ((int)t < n) r = (int)t;
            }
        } else {
            const unsigned t = __hip_atomic_fetch_add(gw(tickets + 1 + x), 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            if ((int)(t * 8 + x) < n) r = (int)(t * 8 + x);   // member t*8 + x: round-robin over the 8 XCDs
        }
        role = r;
        ok = 1;
    }
    __syncthreads();
    const int me = role;
    if (me < 0) return;
    unsigned *abort_flag = flags + 64;
    const int lo = dim * me / n, hi = dim * (me + 1) / n;
    float acc = 0.f;
    unsigned long long t0 = 0;
    for (int i = 0; i < rounds; i++) {
        if (i == 1 && me == 0 && tidx() == 0) t0 = __builtin_amdgcn_s_memrealtime();   // round 0 warms up
        float *v = vec + (size_t)(i & 1) * dim;
        for (int j = lo + tidx(); j < hi; j += NTE) {
            if (same_xcd) gw(v)[j] = (float)(i + j);
            else __hip_atomic_store(gw((unsigned *)v + j), __float_as_uint((float)(i + j)), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        __syncthreads();
        if (tidx() == 0) __hip_atomic_store(gw(flags + me), (unsigned)i + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (tidx() < 64) {
            const unsigned long long w0 = __builtin_amdgcn_s_memrealtime();
            for (unsigned spin = 0;; spin++) {
                const unsigned f = (int)tidx() < n ? ld_flag(flags + tidx()) : (unsigned)i + 1;
                if (__all(f >= (unsigned)i + 1)) break;
                if (!keep_waiting(spin, w0, abort_flag, limit)) { ok = 0; break; }
            }
        }
        __syncthreads();
        if (!ok) return;
        for (int j = tidx(); j < dim; j += NTE) acc += __uint_as_float(__hip_atomic_load(gp<unsigned>((unsigned *)v + j), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
    }
    if (me == 0 && tidx() == 0) { out[0] = __builtin_amdgcn_s_memrealtime() - t0; out[1] = (unsigned long long)__float_as_uint(acc); }
}

__global__ void k_probe_empty() {}

// Latencies inside one workgroup, the steps every phase of the decode kernel is built from: thread 0
// reads the shader clock (s_memtime) around `iters` repetitions of one dependent step, each taking the
// previous one's result:
//   0 every thread writes an LDS word, barrier, reads another wavefront's word, barrier (a hand-over
//     through LDS); 1 a dependent LDS read; 2 a 64-lane sum (DPP and permlane swaps, lanes_sum);
//   3 a bf16 matrix-core product into its own accumulator (16x16x32); 4 a barrier; 5 an LDS write, a wait,
//   the same word read back; 6 expf.
// The step's latency is the difference of two launches (iters and 2 iters) over iters. blockDim.x is a power
// of two from 64 to NTE (with 64 threads, mode 0's word comes from the same wavefront).
template <int MODE>
__global__ void __launch_bounds__(NTE) k_probe_latency(unsigned long long *out, float *sink, int iters) {
    __shared__ float buf[2 * NTE];
    const int t = tidx(), n = blockDim.x;
    buf[t] = (float)t;
    buf[t + NTE] = 0.f;
    __syncthreads();
    float v = (float)(t & 7);
    int idx = t;
    f32x4 c = {0.f, 0.f, 0.f, 0.f};
    const bf16x8 a = {}, b = {};
    const unsigned long long t0 = __builtin_amdgcn_s_memtime();
#pragma unroll 8
    for (int i = 0; i < iters; i++) {
        if constexpr (MODE == 0) {
            buf[t] = v;
            __syncthreads();
            v += buf[(t + 65) & (n - 1)];
            __syncthreads();
        } else if constexpr (MODE == 1) {
            idx = ((int)buf[idx] + 1) & (n - 1);
        } else if constexpr (MODE == 2) {
            v = lanes_sum<64>(v) * 0.001f;
        } else if constexpr (MODE == 3) {
            c = mfma_bf16(a, b, c);
        } else if constexpr (MODE == 4) {
            __syncthreads();
        } else if constexpr (MODE == 5) {
            buf[t + NTE] = v;
            asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
            v = buf[t + NTE] + 1.0f;
        } else {
            v = expf(v * 0.5f - 1.0f);
        }
    }
    const unsigned long long t1 = __builtin_amdgcn_s_memtime();
    if (t == 0) gw(out)[0] = t1 - t0;
    if (v == 12345.f || idx < 0 || c[0] == 12345.f) gw(sink)[t] = v + (float)idx + c[0];   // keeps the work
}

// ----------------------------------------------------------------------------------------- runtime

char g_err[512];
int g_has_err;
hipStream_t g_stream;
// The device address of `scratch` (below) on each device the library set up, from hipGetSymbolAddress: the
// array's name in host code is a host-side stand-in, not a device address.
void *g_scratch_dev[16];
// k_attend's workspaces (attend_ws below), under g_attend_lock. Workspace 0 is the library stream's, 1 the null
// stream's (the library's stream before l3m_dev_init); the others go to callers' streams, each with the stream that
// used it last and that launch's own completion event. busy: a call has it and has not launched yet.
constexpr int ATT_STREAMS = 18, ATT_OWN = 2;
struct AttWs {
    hipStream_t stream;
    hipEvent_t done;
    bool busy;
};
AttWs g_attend[ATT_STREAMS];
uint8_t *g_attend_ws;
pthread_mutex_t g_attend_lock = PTHREAD_MUTEX_INITIALIZER;
int g_ready = -1;
char g_name[128];
unsigned g_lds_max = 65536;

int fail(const char *what, hipError_t e) {
    if (!g_has_err) {
        snprintf(g_err, sizeof g_err, "%s: %s", what, hipGetErrorString(e));
        g_has_err = 1;
        fprintf(stderr, "l3m: hip: %s\n", g_err);
    }
    return -1;
}
int fail_msg(const char *msg) {
    if (!g_has_err) {
        snprintf(g_err, sizeof g_err, "%s", msg);
        g_has_err = 1;
        fprintf(stderr, "l3m: hip: %s\n", g_err);
    }
    return -1;
}
#define CK(call) do { hipError_t e_ = (call); if (e_ != hipSuccess) return fail(#call, e_); } while (0)
#define CKL(what) do { hipError_t e_ = hipGetLastError(); if (e_ != hipSuccess) return fail(what, e_); } while (0)

hipStream_t as_stream(void *s) { return s ? (hipStream_t)s : g_stream; }

#define DISPATCH(dt, F, ...) \
    switch (dt) { \
    case L3M_F32: F<L3M_F32>(__VA_ARGS__); break; \
    case L3M_BF16: F<L3M_BF16>(__VA_ARGS__); break; \
    case L3M_Q8_0: F<L3M_Q8_0>(__VA_ARGS__); break; \
    case L3M_Q4_0: F<L3M_Q4_0>(__VA_ARGS__); break; \
    case L3M_MXFP4: F<L3M_MXFP4>(__VA_ARGS__); break; \
    default: return fail_msg("bad dtype"); }

template <int DT> void launch_prep(const float *x, int k, void *act, hipStream_t st) {
    hipLaunchKernelGGL(k_prep<DT>, dim3((kpad(k) / 4 + NT - 1) / NT), dim3(NT), 0, st, x, k, (uint8_t *)act);
}
template <int DT> void launch_ltiles(const uint8_t *src, int ntiles, int k, uint8_t *q, uint8_t *s, unsigned n, hipStream_t st) {
    hipLaunchKernelGGL(k_ltiles<DT>, dim3((n + NT - 1) / NT), dim3(NT), 0, st, src, ntiles, k, q, s);
}
// Nibble-block matrices (q4_0, mxfp4) of at least 128 tiles whose rows are 64, 128 or 256 blocks take
// k_gemv_deep: 8 wavefronts per tile, nb / 32 blocks per lane (measured at 14336 x 4096, warm / cold against
// the 4-wavefront k_gemv: q4_0 +10% / +7%, mxfp4 +6% / +4%; 16 wavefronts per tile was slower).
int g_gemv_deep = -1;   // L3M_GEMV_DEEP=0 keeps every matrix on k_gemv (for comparison)
int g_gemv_mx = -1;     // L3M_GEMV_MX=0 keeps mxfp4 on k_gemv_deep's VALU dots (for comparison)
template <int DT> bool gemv_deep(const l3m_dmat &m, const void *act, int k, hipStream_t st, float *y) {
    if (g_gemv_deep < 0) {
        const char *e = getenv("L3M_GEMV_DEEP");
        g_gemv_deep = !(e && !strcmp(e, "0"));
    }
    if (!g_gemv_deep || m.tiles < 128 || (m.nb != 64 && m.nb != 128 && m.nb != 256) || ((uintptr_t)act & 15)) return false;
    const uint8_t *a = (const uint8_t *)act;
    if constexpr (DT == L3M_MXFP4) {
        if (g_gemv_mx < 0) {
            const char *e = getenv("L3M_GEMV_MX");
            g_gemv_mx = !(e && !strcmp(e, "0"));
        }
        if (g_gemv_mx) {
            if (m.nb == 64) hipLaunchKernelGGL((k_gemv_mx<4, 1>), dim3(m.tiles), dim3(256), 0, st, m, a, k, y);
            else if (m.nb == 128) hipLaunchKernelGGL((k_gemv_mx<8, 1>), dim3(m.tiles), dim3(512), 0, st, m, a, k, y);
            else hipLaunchKernelGGL((k_gemv_mx<8, 2>), dim3(m.tiles), dim3(512), 0, st, m, a, k, y);
            return true;
        }
    }
    const int ub = m.nb / 32, words = ub == 2 ? gemv_deep_words<DT, 8, 2>() : ub == 4 ? gemv_deep_words<DT, 8, 4>() : gemv_deep_words<DT, 8, 8>();
    if (act_size(DT, k) / 16 > (size_t)words * 512) return false;
    const size_t lds = align16(act_size(DT, k)) + 8 * 16 * 4;
    if (m.nb == 64) hipLaunchKernelGGL((k_gemv_deep<DT, 8, 2>), dim3(m.tiles), dim3(512), lds, st, m, a, k, y);
    else if (m.nb == 128) hipLaunchKernelGGL((k_gemv_deep<DT, 8, 4>), dim3(m.tiles), dim3(512), lds, st, m, a, k, y);
    else hipLaunchKernelGGL((k_gemv_deep<DT, 8, 8>), dim3(m.tiles), dim3(512), lds, st, m, a, k, y);
    return true;
}
template <int DT> void launch_gemv(const l3m_dmat &m, const void *act, int k, float *y, int S, hipStream_t st) {
    if constexpr (DT != L3M_F32)
        if (gemv_deep<DT>(m, act, k, st, y)) return;
    const int grid = (m.tiles + 4 / S - 1) / (4 / S);
    const size_t n16 = act_size(DT, k) / 16;
    const bool staged = n16 > 0 && n16 <= (size_t)GEMV_ACT_REGS * NT && ((uintptr_t)act & 15) == 0;
    if (staged) hipLaunchKernelGGL((k_gemv<DT, true>), dim3(grid), dim3(NT), gemv_lds(DT, k), st, m, (const uint8_t *)act, k, y, S);
    else hipLaunchKernelGGL((k_gemv<DT, false>), dim3(grid), dim3(NT), gemv_lds(DT, k), st, m, (const uint8_t *)act, k, y, S);
}
// Kernels that take more than 64 KiB of dynamic LDS declare it once.
template <class K> void lds_opt_in(K kernel, unsigned bytes) {
    if (bytes > 65536) (void)hipFuncSetAttribute((const void *)kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)bytes);
}
// The GPT-2 variant (M.gpt2) runs its own instantiations of the step kernels.
template <int DT> void launch_attn(const l3m_dmodel &M, const l3m_dlayer &L, int layer, hipStream_t st) {
    auto k = M.gpt2 ? k_attn_block<DT, true> : k_attn_block<DT, false>;
    lds_opt_in(k, M.lds_a);
    hipLaunchKernelGGL(k, dim3(M.n_groups), dim3(NTE), M.lds_a, st, M, L, layer);
}
template <int DT> void launch_ffn(const l3m_dmodel &M, const l3m_dlayer &L, int advance, hipStream_t st) {
    auto k = M.gpt2 ? k_ffn_block<DT, true> : k_ffn_block<DT, false>;
    lds_opt_in(k, M.lds_b);
    hipLaunchKernelGGL(k, dim3(M.n_chunks), dim3(NTE), M.lds_b, st, M, L, advance);
}
template <int DT> void launch_head(const l3m_dmodel &M, int advance, hipStream_t st) {
    auto k = M.gpt2 ? k_head_block<DT, true> : k_head_block<DT, false>;
    lds_opt_in(k, M.lds_h);
    hipLaunchKernelGGL(k, dim3(M.head_grid), dim3(NTE), M.lds_h, st, M, advance);
}
// The persistent kernel needs every workgroup resident at once: a cooperative launch, which the runtime
// refuses (instead of starting it) when the grid does not fit. L3M_COOP=0 (read once, at l3m_dev_init)
// launches the same grid as an ordinary dispatch instead, for profiling runs: with one workgroup per CU
// (its LDS keeps a second one off each CU) on an otherwise idle GPU every workgroup is resident, and if
// one were not, the bounded waits would end the launch with the abort flag (an error), not a hang.
int g_coop = 1;
// Optional timing of the decode launches: hipEvents around each launch on its stream, collected after
// the host has waited for it (l3m_decode_timer).
// Each of the (at most two) launches in flight has its own pair of events (slot).
hipEvent_t g_dec_ev[2][2];
int g_dec_timing, g_dec_launches, g_dec_pending[2];
double g_dec_us;
// The head dimensions the Llama decode kernels of a body and head of one dtype are also built for (HD).
template <int DT, int HDT, bool G2> constexpr bool hd_consts() { return !G2 && DT == HDT && DT != L3M_F32; }
template <int DT, int HDT, bool G2, int HD> int launch_decode_hd(const l3m_dmodel *M_dev, const l3m_dlayer *layers, const l3m_run *R_dev,
                                                                 int grid, unsigned lds, hipStream_t st, int slot) {
    static unsigned opted;                            // per instantiation: set once, again only for more
    if (lds > opted) {
        lds_opt_in(k_decode<DT, HDT, G2, HD>, lds);
        opted = lds;
    }
    const l3m_dmodel *m = M_dev;
    const l3m_dlayer *ly = layers;
    const l3m_run *r = R_dev;
    void *args[] = {&m, &ly, &r};
    if (g_dec_timing) CK(hipEventRecord(g_dec_ev[slot][0], st));
    hipError_t e;
    if (g_coop) {
        e = hipLaunchCooperativeKernel((const void *)k_decode<DT, HDT, G2, HD>, dim3(grid), dim3(NTE), args, lds, st);
    } else {
        hipLaunchKernelGGL((k_decode<DT, HDT, G2, HD>), dim3(grid), dim3(NTE), lds, st, m, ly, r);
        e = hipGetLastError();
    }
    if (e != hipSuccess) return fail("decode launch", e);
    if (g_dec_timing) {
        CK(hipEventRecord(g_dec_ev[slot][1], st));
        g_dec_pending[slot] = 1;
    }
    return 0;
}
template <int DT, int HDT, bool G2> int launch_decode(const l3m_dmodel *M_dev, const l3m_dlayer *layers, const l3m_run *R_dev, int hd,
                                                      int grid, unsigned lds, hipStream_t st, int slot) {
    if constexpr (hd_consts<DT, HDT, G2>()) {
        if (hd == 64) return launch_decode_hd<DT, HDT, G2, 64>(M_dev, layers, R_dev, grid, lds, st, slot);
        if (hd == 48) return launch_decode_hd<DT, HDT, G2, 48>(M_dev, layers, R_dev, grid, lds, st, slot);
    }
    return launch_decode_hd<DT, HDT, G2, 0>(M_dev, layers, R_dev, grid, lds, st, slot);
}
template <int DT, int HDT, bool G2, int HD> int decode_fits_hd(int grid, unsigned lds) {
    lds_opt_in(k_decode<DT, HDT, G2, HD>, lds);
    int per_cu = 0, cus = 0, coop = 0;
    if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void *)k_decode<DT, HDT, G2, HD>, NTE, lds) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, 0) != hipSuccess) return 0;
    if (hipDeviceGetAttribute(&coop, hipDeviceAttributeCooperativeLaunch, 0) != hipSuccess || !coop) return 0;
    return per_cu >= 1 && grid <= per_cu * cus;
}
template <int DT, int HDT, bool G2> int decode_fits(int hd, int grid, unsigned lds) {
    if constexpr (hd_consts<DT, HDT, G2>()) {
        if (hd == 64) return decode_fits_hd<DT, HDT, G2, 64>(grid, lds);
        if (hd == 48) return decode_fits_hd<DT, HDT, G2, 48>(grid, lds);
    }
    return decode_fits_hd<DT, HDT, G2, 0>(grid, lds);
}

// k_pf_rows for rows of k <= 4096 values.
template <int DT, bool NORM> void pf_rows(const float *y, int k, const float *w, float eps, const l3m_pfact &act, int P, hipStream_t st) {
    const dim3 grid((P + 3) / 4), block(256);
    if (k <= 512) hipLaunchKernelGGL((k_pf_rows<DT, NORM, 2>), grid, block, 0, st, y, k, w, eps, act, P);
    else if (k <= 1024) hipLaunchKernelGGL((k_pf_rows<DT, NORM, 4>), grid, block, 0, st, y, k, w, eps, act, P);
    else hipLaunchKernelGGL((k_pf_rows<DT, NORM, 16>), grid, block, 0, st, y, k, w, eps, act, P);
}

// The prompt's attention in layer l: on the matrix cores for head dims of 16, 32, ... 128 (k_pf_attn), else
// k_pf_attend; its output prepared into B->act.
template <int DT> void pf_attention(const l3m_dmodel *M, const l3m_pfbuf *B, int P, int l, hipStream_t st) {
    const float *q = B->q;
    const uint16_t *kc = M->kc, *vc = M->vc;
    const int hd = M->hd, nq = M->n_heads * hd;
    const dim3 grid((P + PFA_T - 1) / PFA_T, M->n_heads), block(64 * PFA_W);
    bool rows = DT != L3M_BF16 && hd % 32;            // blocks across heads
#define PF_ATTN(HD) \
    case HD: hipLaunchKernelGGL((k_pf_attn<DT, HD>), grid, block, 0, st, q, P, M->n_heads, M->n_kv, M->ctx, l, M->att_scale, kc, vc, B->att, B->act); break;
    switch (hd) {
        PF_ATTN(16) PF_ATTN(32) PF_ATTN(48) PF_ATTN(64) PF_ATTN(80) PF_ATTN(96) PF_ATTN(112) PF_ATTN(128)
    default:
        hipLaunchKernelGGL(k_pf_attend, dim3(P, M->n_heads), dim3(64), 0, st, q, P, M->n_heads, M->n_kv, hd, M->ctx, l, M->att_scale, kc, vc, B->att);
        rows = true;
    }
#undef PF_ATTN
    if (rows) pf_rows<DT, false>(B->att, nq, nullptr, 0.f, B->act, P, st);
}

// One matrix of the prompt. Three splits, by how many 32-row x 32-token tiles there are (for EPI 2 16 gate and 16
// up rows): many, a wavefront a tile over all blocks, two side by side; fewer, a tile's ranges split over 4
// wavefronts; fewest, 32 x 16 tiles with the ranges split over up to 8. Measured (30 layers of dim 576, ffn 1536;
// us to the first logits, each split for every matrix): 64 tokens 2065 / 1685 / 1509, 200 tokens 2282 / 1918 /
// 1941, 480 tokens 2549 / 2394 / 2846; gate and up alone at 480 tokens 12.0 / 15.1 / 25.9 us, at 64 - / 7.6 / 7.0.
// bf16 has no scales to multiply and crosses at the same sizes: 64 tokens 2070 / 1838 / 1715, 200 tokens 2196 / 2008 /
// 2001, 480 tokens 2543 / 2557 / 2945, by this rule 1727 / 1944 / 2460 (runs of one side differ by 1%).
constexpr int PF_WIDE = 1024;
template <int DT, int EPI> void pf_gemm(const PfGemm &G, hipStream_t st) {
    constexpr int WR = EPI == 2 ? 2 : 1, MID = EPI == 2 ? 256 : 160;
    const int rows = EPI == 2 ? G.W.tiles * 8 : G.W.rows;   // EPI 2: the ffn rows
    const int r32 = (rows + 31) / 32, t32 = (G.P + 31) / 32, R = pf_ranges(G.W.nb), n = WR * r32 * t32;
    if (n >= PF_WIDE) hipLaunchKernelGGL((k_pf_gemm<DT, EPI, 2, 2, 2, 1>), dim3(EPI == 2 ? r32 : (r32 + 1) / 2, t32), dim3(128), 0, st, G);
    else if (n >= MID) hipLaunchKernelGGL((k_pf_gemm<DT, EPI, 2, 2, WR, 4>), dim3(r32, t32), dim3(64 * WR * min(R, 4)), 0, st, G);
    else hipLaunchKernelGGL((k_pf_gemm<DT, EPI, 2, 1, WR, 8>), dim3(r32, (G.P + 15) / 16), dim3(64 * WR * min(R, 8)), 0, st, G);
}

template <int DT> void pf_layers(const l3m_dmodel *M, const l3m_pflayer *L, const l3m_pfbuf *B, int P, hipStream_t st) {
    const int dim = M->dim, hd = M->hd, nq = M->n_heads * hd;
    for (int l = 0; l < M->n_layers; l++) {
        const l3m_pflayer &W = L[l];
        PfGemm G{};
        G.P = P;
        pf_rows<DT, true>(B->x, dim, W.attn_norm, M->eps, B->act, P, st);
        // q (after RoPE) into B->q, k and v into the cache
        G.W = W.qkv; G.x = B->act; G.y = B->q; G.ystride = nq;
        G.rope = M->rope; G.kc = M->kc; G.vc = M->vc; G.layer = l; G.ctx = M->ctx; G.nq = nq; G.nk = M->n_kv * hd; G.hd = hd; G.n_kv = M->n_kv;
        pf_gemm<DT, 1>(G, st);
        if (l == M->n_layers - 1) break;              // the last layer's K/V rows are all its prompt positions leave
        pf_attention<DT>(M, B, P, l, st);
        G.W = W.wo; G.y = B->x; G.ystride = dim;
        pf_gemm<DT, 0>(G, st);
        pf_rows<DT, true>(B->x, dim, W.ffn_norm, M->eps, B->act, P, st);
        G.W = W.gu; G.out = B->hact;
        pf_gemm<DT, 2>(G, st);
        G.W = W.down; G.x = B->hact;
        pf_gemm<DT, 0>(G, st);
    }
}

template <int DT> int launch_step_mv(int form, const l3m_dmat &m, const float *x, int k, float *y, int tpw, hipStream_t st) {
    const int at = form == 3 ? DT : a_dtype<DT>();
    if (m.dtype != at) return fail_msg("step_mv: the matrix is not stored in the dtype this form reads");
    const int tpb = form == 3 ? tpw : m.tiles;
    const size_t lds = step_mv_lds(at, form, k, tpb, m.nb);
    if (lds > g_lds_max) return fail_msg("step_mv: the matrix's per-pair results do not fit in LDS");
    const int grid = form == 3 ? (m.tiles + tpw - 1) / tpw : 1;
    auto kern = form == 0 ? k_step_mv<DT, 0> : form == 1 ? k_step_mv<DT, 1> : form == 2 ? k_step_mv<DT, 2> : k_step_mv<DT, 3>;
    lds_opt_in(kern, (unsigned)lds);
    hipLaunchKernelGGL(kern, dim3(grid), dim3(NTE), lds, st, m, x, k, y, tpw);
    CKL("k_step_mv");
    return 0;
}
}  // namespace

// The only device memory l3m_hip_attend_noalloc uses: the staged q, K rows, V rows and the output of one
// call (the staging the kernel table's attend allocates and grows on demand). One copy per GPU, held until
// the process ends; every call on a GPU shares it and it keeps the last call's contents.
constexpr size_t ATTEND_STATIC_BYTES = 4u << 20;
static __device__ __align__(256) uint8_t scratch[ATTEND_STATIC_BYTES];
// k_attend's workspaces on device 0 (g_attend).
static __device__ __align__(256) uint8_t attend_ws[ATT_STREAMS][ATT_WS];
static_assert(ATT_WS % 256 == 0, "every workspace 256-byte aligned");

// The workspace a call on st takes, or -1: none, one workgroup does it. Two calls may share one only if the
// second cannot begin before the first has ended:
//  - the library's stream and the null stream have their own, and neither is destroyed with work in flight;
//  - any other stream takes the one its handle used last, behind that call's event (a handle may name a new
//    stream whose predecessor was destroyed with the call still running), else one whose last call has ended.
//    Never one that is in use: a stream does not wait for another's work.
// None for a stream under capture (its graph may be replayed on another), the special handles (one name for several
// streams) and streams of another device (the workspaces are device 0's).
static int attend_take(hipStream_t st) {
    int dev = -1, got = -1;
    if ((uintptr_t)st == 1 || (uintptr_t)st == 2 || hipGetDevice(&dev) != hipSuccess || dev != 0) return -1;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (st && (hipStreamIsCapturing(st, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone)) return -1;
    if (st && st == g_stream) return 0;
    pthread_mutex_lock(&g_attend_lock);
    if (!st) {                                        // before l3m_dev_init: nothing resolved the array yet
        if (g_attend_ws || hipGetSymbolAddress((void **)&g_attend_ws, HIP_SYMBOL(attend_ws)) == hipSuccess) got = 1;
    } else if (g_attend_ws && hipStreamGetDevice(st, &dev) == hipSuccess && dev == 0) {
        // an event may be asked for its state while another thread captures
        hipStreamCaptureMode mode = hipStreamCaptureModeRelaxed;
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        for (int i = ATT_OWN; i < ATT_STREAMS && got < 0; i++) {
            const AttWs &w = g_attend[i];
            if (!w.busy && w.done && w.stream == st && hipStreamWaitEvent(st, w.done, 0) == hipSuccess) got = i;
        }
        if (got < 0) {
            for (int i = ATT_OWN; i < ATT_STREAMS && got < 0; i++) {
                AttWs &w = g_attend[i];
                if (!w.busy && (w.done ? hipEventQuery(w.done) : hipEventCreate(&w.done)) == hipSuccess) got = i;
            }
            (void)hipGetLastError();                  // an event not ready is no error of the call's
        }
        (void)hipThreadExchangeStreamCaptureMode(&mode);
        if (got >= 0) g_attend[got].busy = true;
    }
    pthread_mutex_unlock(&g_attend_lock);
    return got;
}

// k_attend over n rows. Up to ATT_ALONE batches of rows go to one workgroup: a second costs the hand-over (about
// 3.5 us), a batch about 0.9 us (hd 128, 256 rows: 6.8 us in one; 512 rows: 8.3 us spread, 10.4 in one). More are spread over up to ATT_SPLITS workgroups.
constexpr int ATT_ALONE = 4;
// On a caller's stream the launch carries its workspace's event (hipExtLaunchKernel; hd 128, 4001 rows queued back
// to back: 12.6-12.7 us, 12.5-12.6 without one, 15.5 with an event recorded behind the launch; waited for alone 26.5-28.9,
// 24.2-25.1, 24.8-26.1).
template <int L> static void attend_l(float *out, const float *q, const uint16_t *k, const uint16_t *v, int n, int hd, int stride, hipStream_t st) {
    const int rows = NT / L * ATT_U, batches = (n + rows - 1) / rows, own = batches > ATT_ALONE ? attend_take(st) : -1;
    uint8_t *ws = own < 0 ? nullptr : g_attend_ws + (size_t)own * ATT_WS;
    const int per = rows * (ws ? (batches + ATT_SPLITS - 1) / ATT_SPLITS : batches), grid = (n + per - 1) / per;
    if (own < ATT_OWN) {
        hipLaunchKernelGGL(k_attend<L>, dim3(grid), dim3(NT), 0, st, out, q, k, v, n, hd, stride, per, ws);
        return;
    }
    hipExtLaunchKernelGGL(k_attend<L>, dim3(grid), dim3(NT), 0, st, nullptr, g_attend[own].done, 0, out, q, k, v, n, hd, stride, per, ws);
    pthread_mutex_lock(&g_attend_lock);
    g_attend[own].stream = st;
    g_attend[own].busy = false;
    pthread_mutex_unlock(&g_attend_lock);
}
static void launch_attend(float *out, const float *q, const uint16_t *k, const uint16_t *v, int n, int hd, int stride, hipStream_t st) {
    if (hd <= 8) attend_l<1>(out, q, k, v, n, hd, stride, st);
    else if (hd <= 16) attend_l<2>(out, q, k, v, n, hd, stride, st);
    else if (hd <= 32) attend_l<4>(out, q, k, v, n, hd, stride, st);
    else if (hd <= 64) attend_l<8>(out, q, k, v, n, hd, stride, st);
    else if (hd <= 128) attend_l<16>(out, q, k, v, n, hd, stride, st);
    else attend_l<32>(out, q, k, v, n, hd, stride, st);
}

// =============================================================================================== C ABI

struct l3m_graphs {
    hipGraph_t g[2];
    hipGraphExec_t e[2];
};

extern "C" {

// Everything the library created on the device that no model owns (the stream, the decode timer's
// events), destroyed by the host before it exits (the Python package registers it with its interpreter's
// atexit; a C host may call it last or leave it to process exit). Not an atexit handler of the library's
// own: those run after a profiler's finalization, when HIP calls no longer may be made. Calls after it fail
// cleanly.
void l3m_dev_shutdown(void) {
    if (g_ready != 1) return;
    (void)hipStreamSynchronize(g_stream);
    for (int i = 0; i < 2; i++)
        for (int j = 0; j < 2; j++)
            if (g_dec_ev[i][j]) { (void)hipEventDestroy(g_dec_ev[i][j]); g_dec_ev[i][j] = nullptr; }
    for (AttWs &w : g_attend)                         // a call still running keeps its event
        if (w.done && !w.busy && hipEventQuery(w.done) == hipSuccess) { (void)hipEventDestroy(w.done); w = AttWs{}; }
    (void)hipGetLastError();
    (void)hipStreamDestroy(g_stream);
    g_stream = nullptr;
    g_ready = 0;
}

int l3m_dev_init(void) {
    if (g_ready >= 0) return g_ready ? 0 : -1;
    g_ready = 0;
    int n = 0;
    hipError_t e = hipGetDeviceCount(&n);
    if (e != hipSuccess || n < 1) { fail_msg("no HIP device"); return -1; }
    hipDeviceProp_t p;
    CK(hipGetDeviceProperties(&p, 0));
    snprintf(g_name, sizeof g_name, "%s (%s, %d CUs)", p.name, p.gcnArchName, p.multiProcessorCount);
    if (strncmp(p.gcnArchName, "gfx950", 6)) {
        char msg[256];
        snprintf(msg, sizeof msg, "device 0 is %s; this build targets gfx950", p.gcnArchName);
        return fail_msg(msg);
    }
    CK(hipSetDevice(0));
    const char *coop = getenv("L3M_COOP");
    g_coop = !(coop && !strcmp(coop, "0"));
    CK(hipGetSymbolAddress(&g_scratch_dev[0], HIP_SYMBOL(scratch)));
    CK(hipGetSymbolAddress((void **)&g_attend_ws, HIP_SYMBOL(attend_ws)));
    int lds = 0;
    if (hipDeviceGetAttribute(&lds, hipDeviceAttributeMaxSharedMemoryPerBlock, 0) == hipSuccess && lds > 0) g_lds_max = (unsigned)lds;
    CK(hipStreamCreateWithFlags(&g_stream, hipStreamNonBlocking));
    hipLaunchKernelGGL(k_dummy, dim3(1), dim3(NT), 0, g_stream);
    CKL("first launch");
    CK(hipStreamSynchronize(g_stream));
    g_ready = 1;
    return 0;
}

const char *l3m_dev_error(void) { return g_has_err ? g_err : NULL; }
// Also HIP's own last error: a refused launch (a cooperative launch while another process on the GPU holds
// the device's cooperative dispatch) would otherwise fail the next launch check of the fallback path.
void l3m_dev_clear_error(void) { (void)hipGetLastError(); g_has_err = 0; g_err[0] = 0; }
const char *l3m_dev_name(void) { return g_name; }
unsigned l3m_dev_lds_max(void) { return l3m_dev_init() ? 65536u : g_lds_max; }
void *l3m_dev_stream(void) { return (void *)g_stream; }

void *l3m_dev_alloc(size_t bytes) {
    void *p = NULL;
    if (l3m_dev_init()) return NULL;
    if (hipMalloc(&p, bytes ? bytes : 16) != hipSuccess) { fail_msg("hipMalloc failed"); return NULL; }
    if (hipMemsetAsync(p, 0, bytes ? bytes : 16, g_stream) != hipSuccess || hipStreamSynchronize(g_stream) != hipSuccess) {
        (void)hipFree(p);
        fail_msg("hipMemset failed");
        return NULL;
    }
    return p;
}
void l3m_dev_free(void *p) { if (p) (void)hipFree(p); }
// Copies run on the library's stream, after the work already queued there, and complete before returning.
int l3m_dev_upload(void *dst, const void *src, size_t bytes) {
    if (l3m_dev_init()) return -1;
    CK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_stream));
    CK(hipStreamSynchronize(g_stream));
    return 0;
}
// Queued on the library's stream without waiting: a copy from host memory that stays unchanged until the stream has
// run it (pinned, l3m_dev_host_alloc, to return at once; the kernel table's pageable tiles are staged first) and a
// fill with zero bytes.
int l3m_dev_upload_async(void *dst, const void *src, size_t bytes) {
    if (l3m_dev_init()) return -1;
    CK(hipMemcpyAsync(dst, src, bytes, hipMemcpyHostToDevice, g_stream));
    return 0;
}
int l3m_dev_zero_async(void *dst, size_t bytes) {
    if (l3m_dev_init()) return -1;
    CK(hipMemsetAsync(dst, 0, bytes, g_stream));
    return 0;
}
void *l3m_dev_host_alloc(size_t bytes) {
    void *p = NULL;
    if (l3m_dev_init()) return NULL;
    if (hipHostMalloc(&p, bytes ? bytes : 16, hipHostMallocDefault) != hipSuccess) { fail_msg("hipHostMalloc failed"); return NULL; }
    return p;
}
void l3m_dev_host_free(void *p) { if (p) (void)hipHostFree(p); }
int l3m_dev_download(void *dst, const void *src, size_t bytes) {
    if (l3m_dev_init()) return -1;
    CK(hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, g_stream));
    CK(hipStreamSynchronize(g_stream));
    return 0;
}
int l3m_dev_sync(void) {
    if (l3m_dev_init()) return -1;
    CK(hipStreamSynchronize(g_stream));
    return 0;
}
int l3m_dev_download_async(void *dst_pinned, const void *src, size_t bytes) {
    if (l3m_dev_init()) return -1;
    CK(hipMemcpyAsync(dst_pinned, src, bytes, hipMemcpyDeviceToHost, g_stream));
    return 0;
}
void *l3m_dev_event_new(void) {
    hipEvent_t e = nullptr;
    if (l3m_dev_init()) return nullptr;
    if (hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) { fail_msg("hipEventCreate failed"); return nullptr; }
    return (void *)e;
}
void l3m_dev_event_free(void *e) { if (e) (void)hipEventDestroy((hipEvent_t)e); }
int l3m_dev_event_record(void *e) {
    if (l3m_dev_init()) return -1;
    CK(hipEventRecord((hipEvent_t)e, g_stream));
    return 0;
}
int l3m_dev_event_wait(void *e) {
    if (l3m_dev_init()) return -1;
    CK(hipEventSynchronize((hipEvent_t)e));
    return 0;
}

size_t l3m_act_bytes(int dtype, int k) { return act_bytes(dtype, k); }

int l3m_gemv_matrix_cores(int on) {
    if (g_gemv_mx < 0) {
        const char *e = getenv("L3M_GEMV_MX");
        g_gemv_mx = !(e && !strcmp(e, "0"));
    }
    const int was = g_gemv_mx;
    if (on >= 0) g_gemv_mx = on != 0;
    return was;
}

int l3m_k_prep(int dtype, const float *x, int k, void *act, void *stream) {
    if (k < 1 || dtype < 0 || dtype >= L3M_NDTYPES || !act_fits(dtype, k)) return fail_msg("prep: k out of range for this dtype");
    hipStream_t st = as_stream(stream);
    DISPATCH(dtype, launch_prep, x, k, act, st);
    CKL("k_prep");
    return 0;
}

size_t l3m_ltile_bytes(int dtype, int ntiles, int k) {
    const size_t per = dtype == L3M_F32 ? (size_t)k * 64 : dtype == L3M_BF16 ? (size_t)k * 32
                                                                             : (size_t)(k / 32) * (16 * (qbytes(dtype) + sbytes(dtype)));
    return per * (size_t)ntiles;
}
int l3m_k_ltiles(int dtype, int ntiles, int k, const void *tiles, void *quant, void *scale, void *stream) {
    if (k < 1 || ntiles < 1 || dtype < 0 || dtype >= L3M_NDTYPES || (quantized(dtype) && k % 32)) return fail_msg("ltiles: bad shape");
    hipStream_t st = as_stream(stream);
    const size_t n = (size_t)ntiles * (kpad(k) / 32) * 16;
    if (n > 0x7FFFFFFF - NT) return fail_msg("ltiles: matrix too large");
    DISPATCH(dtype, launch_ltiles, (const uint8_t *)tiles, ntiles, k, (uint8_t *)quant, (uint8_t *)scale, (unsigned)n, st);
    CKL("k_ltiles");
    return 0;
}

int l3m_k_gemv(const l3m_dmat *m, const void *act, int k, float *y, void *stream) {
    if (k < 1 || m->dtype < 0 || m->dtype >= L3M_NDTYPES || kpad(k) / 32 != m->nb || m->tiles != (m->rows + 15) / 16 || m->rows < 1)
        return fail_msg("gemv: shape does not match the matrix");
    if (!act_fits(m->dtype, k)) return fail_msg("gemv: k too large for this dtype");
    hipStream_t st = as_stream(stream);
    const int S = pick_split(m->nb);
    DISPATCH(m->dtype, launch_gemv, *m, act, k, y, S, st);
    CKL("k_gemv");
    return 0;
}

// The most positions a call takes, unchanged since one workgroup held q, every score and its threads' sums in LDS
// (16,128 - hd or so; k_attend itself has no such bound): 4 (hd + ceil4(pos + 1) + NT + 8) bytes within LDS_MAX.
static bool attend_fits(int pos, int hd) { return 4 * ((size_t)hd + ((pos + 4) & ~3) + NT + 8) <= LDS_MAX; }

int l3m_k_attend(float *out, const float *q, const uint16_t *k, const uint16_t *v, int pos, int hd, int stride, void *stream) {
    if (pos < 0 || hd < 8 || hd % 8 || hd > NT || stride < hd || stride % 8) return fail_msg("attend: bad shape");
    if (!attend_fits(pos, hd)) return fail_msg("attend: pos too large");
    launch_attend(out, q, k, v, pos + 1, hd, stride, as_stream(stream));
    CKL("k_attend");
    return 0;
}

int l3m_k_rmsnorm(float *y, const float *x, const float *w, int n, float eps, void *stream) {
    if (n < 1 || 4 * ((size_t)kpad(n) + 8) > LDS_MAX) return fail_msg("rmsnorm: n out of range");
    const int quads = (n + 3) / 4;                    // at most 4088: LDS_MAX bounds n
    if (quads <= 1024) hipLaunchKernelGGL(k_rmsnorm<1>, dim3(1), dim3((quads + 63) & ~63), 0, as_stream(stream), y, x, w, n, eps);
    else hipLaunchKernelGGL(k_rmsnorm<4>, dim3(1), dim3(1024), 0, as_stream(stream), y, x, w, n, eps);
    CKL("k_rmsnorm");
    return 0;
}

int l3m_k_rope(float *v, int n_heads, int hd, int pos, const float *table, void *stream) {
    const int n = n_heads * hd;
    if (n < 2 || hd % 2) return fail_msg("rope: bad shape");
    hipLaunchKernelGGL(k_rope, dim3((n + NT - 1) / NT), dim3(NT), 0, as_stream(stream), v, n, hd, table + (size_t)pos * hd);
    CKL("k_rope");
    return 0;
}

int l3m_k_silu_mul(float *h, const float *g, int n, void *stream) {
    hipLaunchKernelGGL(k_silu_mul, dim3((n + NT - 1) / NT), dim3(NT), 0, as_stream(stream), h, g, n);
    CKL("k_silu_mul");
    return 0;
}

int l3m_dev_copy(void *dst, const void *src, size_t bytes, void *stream) {
    if (bytes % 16 || ((uintptr_t)dst | (uintptr_t)src) % 16) return fail_msg("copy: 16-byte multiples and alignment");
    const size_t n16 = bytes / 16;
    const unsigned grid = (unsigned)(n16 / NT < 4096 ? (n16 + NT - 1) / NT : 4096);
    if (grid) hipLaunchKernelGGL(k_copy, dim3(grid), dim3(NT), 0, as_stream(stream), (u32x4 *)dst, (const u32x4 *)src, n16);
    CKL("k_copy");
    return 0;
}

// l3m_kernels_hip.attend without allocating: q, the K and V rows and the output staged through `scratch`
// (its device address from l3m_dev_init), the same kernel, the same result. Calls are serialized by a
// lock; without it, two calls overlapping on one GPU would race on the one array.
static pthread_mutex_t g_scratch_lock = PTHREAD_MUTEX_INITIALIZER;
static size_t up256(size_t n) { return (n + 255) & ~(size_t)255; }

int l3m_hip_attend_noalloc(float *out, const float *q, const uint16_t *k, const uint16_t *v, int pos, int head_dim, int stride) {
    if (l3m_dev_init()) return -1;
    if (pos < 0 || head_dim < 8 || head_dim % 8 || head_dim > NT || stride < head_dim || stride % 8)
        return fail_msg("attend_noalloc: head_dim must be a multiple of 8 up to 256, stride a multiple of 8 of at least head_dim");
    const size_t kv = ((size_t)pos * stride + head_dim) * 2, vec = up256((size_t)head_dim * 4);
    if (2 * vec + 2 * up256(kv) > ATTEND_STATIC_BYTES) {
        char msg[200];
        snprintf(msg, sizeof msg, "attend_noalloc: (pos * stride + head_dim) * 2 = %zu bytes of K (and of V) exceed the %zu-byte staging array",
                 kv, (ATTEND_STATIC_BYTES - 2 * vec) / 2);
        return fail_msg(msg);
    }
    if (!attend_fits(pos, head_dim)) return fail_msg("attend_noalloc: pos too large");
    uint8_t *base = (uint8_t *)g_scratch_dev[0];
    float *dq = (float *)base, *dout = (float *)(base + vec);
    uint16_t *dk = (uint16_t *)(base + 2 * vec), *dv = (uint16_t *)(base + 2 * vec + up256(kv));
    pthread_mutex_lock(&g_scratch_lock);
    hipError_t e = hipMemcpyAsync(dq, q, (size_t)head_dim * 4, hipMemcpyHostToDevice, g_stream);
    if (e == hipSuccess) e = hipMemcpyAsync(dk, k, kv, hipMemcpyHostToDevice, g_stream);
    if (e == hipSuccess) e = hipMemcpyAsync(dv, v, kv, hipMemcpyHostToDevice, g_stream);
    if (e == hipSuccess) {
        launch_attend(dout, dq, dk, dv, pos + 1, head_dim, stride, g_stream);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(out, dout, (size_t)head_dim * 4, hipMemcpyDeviceToHost, g_stream);
    if (e == hipSuccess) e = hipStreamSynchronize(g_stream);
    pthread_mutex_unlock(&g_scratch_lock);
    return e == hipSuccess ? 0 : fail("attend_noalloc", e);
}

int l3m_dev_evict(const void *buf, size_t bytes, void *stream) {
    if (bytes < 16 || bytes % 16 || (uintptr_t)buf % 16) return fail_msg("evict: 16-byte multiples and alignment");
    const size_t n16 = bytes / 16;
    // the last 16-byte word is the sink: it is never read past the first n16 - 1 words' xor
    hipLaunchKernelGGL(k_evict, dim3(4 * (unsigned)l3m_dev_cus()), dim3(NT), 0, as_stream(stream), (const u32x4 *)buf, n16 - 1,
                       (unsigned *)((u32x4 *)buf + n16 - 1));
    CKL("k_evict");
    return 0;
}

int l3m_k_dequant(const l3m_dmat *m, int row0, int n, float *out, void *stream) {
    if (m->dtype < 0 || m->dtype >= L3M_NDTYPES || n < 1 || row0 < 0 || row0 + n > m->tiles * RT || m->nb < 1)
        return fail_msg("dequant: rows out of range");
    const size_t k4 = (size_t)m->nb * 8, threads = (size_t)n * k4;
    hipLaunchKernelGGL(k_dequant, dim3((unsigned)((threads + NT - 1) / NT)), dim3(NT), 0, as_stream(stream), *m, row0, n, out);
    CKL("k_dequant");
    return 0;
}

int l3m_attention_mode(int kv_lds, int hd, int nq, int ctx) { return att_mode(kv_lds, hd, nq, ctx); }

int l3m_phase_stamps(int mode, int pos, int layer, unsigned long long *out) {
#ifdef L3M_PHASE_STAMPS
    if (l3m_dev_init()) return -1;
    if (mode == 0) {
        static unsigned long long zero[2][3 * 64][16];
        const int at[2] = {pos, layer};
        CK(hipMemcpyToSymbol(HIP_SYMBOL(g_phase), zero, sizeof zero, 0, hipMemcpyHostToDevice));
        CK(hipMemcpyToSymbol(HIP_SYMBOL(g_phase_at), at, sizeof at, 0, hipMemcpyHostToDevice));
        return 0;
    }
    CK(hipMemcpyFromSymbol(out, HIP_SYMBOL(mode == 2 ? g_phase_clk : g_phase), sizeof(unsigned long long) * 2 * 3 * 64 * 16, 0,
                           hipMemcpyDeviceToHost));
    return 0;
#else
    (void)mode; (void)pos; (void)layer; (void)out;
    return fail_msg("phase stamps: this library was built without L3M_PHASE_STAMPS (make -C l3m_amd/csrc phases)");
#endif
}

int l3m_k_step_mv(int dtype, int form, const l3m_dmat *m, const float *x, int k, float *y, int tpw, void *stream) {
    if (l3m_dev_init()) return -1;
    if (form < 0 || form > 3 || k < 1 || k > 4 * NTE || kpad(k) / 32 != m->nb || m->tiles < 1 || m->rows > 16 * m->tiles ||
        (form == 3 && (tpw < 1 || tpw > 64)))
        return fail_msg("step_mv: shape out of range");
    int rc = -1;
    switch (dtype) {
    case L3M_F32: rc = launch_step_mv<L3M_F32>(form, *m, x, k, y, tpw, as_stream(stream)); break;
    case L3M_BF16: rc = launch_step_mv<L3M_BF16>(form, *m, x, k, y, tpw, as_stream(stream)); break;
    case L3M_Q8_0: rc = launch_step_mv<L3M_Q8_0>(form, *m, x, k, y, tpw, as_stream(stream)); break;
    case L3M_Q4_0: rc = launch_step_mv<L3M_Q4_0>(form, *m, x, k, y, tpw, as_stream(stream)); break;
    case L3M_MXFP4: rc = launch_step_mv<L3M_MXFP4>(form, *m, x, k, y, tpw, as_stream(stream)); break;
    default: return fail_msg("step_mv: bad dtype");
    }
    return rc;
}

int l3m_k_attend_decode(int mode, float *out, const float *q, const uint16_t *kc, const uint16_t *vc, int nq, int nkv, int hd, int ctx,
                        int pos, void *stream) {
    if (l3m_dev_init()) return -1;
    if (mode < 0 || mode > 2 || hd < 8 || hd % 8 || hd > 256 || nq < 1 || nkv < 1 || nq % nkv || pos < 0 || pos >= ctx ||
        (mode == 2 && !mfma_fits(hd, nq, ctx)))
        return fail_msg("attend_decode: shape out of range for this mode");
    const size_t lds = lds_att(mode, nq, nkv, hd, ctx).total;
    if (lds > g_lds_max) return fail_msg("attend_decode: the K/V window does not fit in LDS");
    int wmax = nq < NWE ? NWE / nq : 1, wl = 0;       // as l3m_group_layout
    while ((2 << wl) <= wmax) wl++;
    // the batched form's byte offsets span every kv head's rows and must lie below OOB; a model's always do (dim up
    // to 4096, ctx up to 8192: 64 MiB)
    const bool batch = 2 * (size_t)nkv * ctx * hd < OOB;
    auto k = mode == 2 ? k_attend_decode<2, false> : mode == 1 ? k_attend_decode<1, false> : batch ? k_attend_decode<0, true> : k_attend_decode<0, false>;
    lds_opt_in(k, (unsigned)lds);
    hipLaunchKernelGGL(k, dim3(1), dim3(NTE), lds, as_stream(stream), out, q, kc, vc, nq, nkv, hd, ctx, pos, wl);
    CKL("k_attend_decode");
    return 0;
}

int l3m_k_argmax(const float *x, int n, int32_t *out, void *stream) {
    const int nt = min(max((n / 4 + 63) & ~63, 64), 1024);   // n / 4 quads at most, whatever x's alignment
    if (n <= 4096) hipLaunchKernelGGL(k_argmax<1>, dim3(1), dim3(nt), 0, as_stream(stream), x, n, nt, out);
    else hipLaunchKernelGGL(k_argmax<12>, dim3(1), dim3(1024), 0, as_stream(stream), x, n, 1024, out);
    CKL("k_argmax");
    return 0;
}

unsigned l3m_lds_attn(int dtype, int dim, int ctx, int hd, const l3m_dgroup *g, int kv_lds) { return (unsigned)lds_a(dtype, dim, ctx, hd, *g, kv_lds).total; }
void l3m_group_layout(int dtype, int dim, int ctx, int hd, l3m_dgroup *g) {
    const LdsA L = lds_a(dtype, dim, ctx, hd, *g, 1);
    const size_t off[10] = {L.act, L.work, L.q, L.cur, L.cs, L.vred, L.att, L.act2, L.scr, L.kvb};
    for (int i = 0; i < 10; i++) g->lds[i] = (unsigned)off[i];
    int wmax = g->nq < NWE ? NWE / g->nq : 1, wl = 0;
    while ((2 << wl) <= wmax) wl++;
    g->att_wl = wl;
}
void l3m_chunk_layout(int dtype, int dim, l3m_dchunk *c) {
    const LdsB L = lds_b(dtype, dim, *c);
    const size_t off[5] = {L.act, L.work, L.gu, L.act2, L.scr};
    for (int i = 0; i < 5; i++) c->lds[i] = (unsigned)off[i];
}
void l3m_model_layout(l3m_dmodel *m) {
    pro_shape(m->dim, m->n_chunks, m->pro_groups[0], m->pro_per[0]);
    pro_shape(m->dim, m->n_groups, m->pro_groups[1], m->pro_per[1]);
    m->att_scale = 1.0f / sqrtf((float)m->hd);
    m->hpk = m->n_heads / m->n_kv;
}
unsigned l3m_lds_ffn(int dtype, int dim, const l3m_dchunk *c) { return (unsigned)lds_b(dtype, dim, *c).total; }
unsigned l3m_lds_head(int dtype, int dim, int nb, int tiles_per_wg) { return (unsigned)lds_h(dtype, dim, nb, tiles_per_wg).total; }
int l3m_step_a_dtype(int dtype) {
    return dtype == L3M_Q4_0 ? a_dtype<L3M_Q4_0>() : dtype;
}
int l3m_step_slots(int dtype, int which) {
    if (which) return dtype == L3M_F32 ? nslot_b<L3M_F32>() : dtype == L3M_BF16 ? nslot_b<L3M_BF16>() : dtype == L3M_Q8_0 ? nslot_b<L3M_Q8_0>() : nslot_b<L3M_Q4_0>();
    return dtype == L3M_F32 ? nslot_a<L3M_F32>() : dtype == L3M_BF16 ? nslot_a<L3M_BF16>() : dtype == L3M_Q8_0 ? nslot_a<L3M_Q8_0>() : nslot_a<L3M_Q4_0>();
}

// The shapes the prefill takes: rows of dim and n_heads * hd values fit k_pf_rows (16 pieces of 256),
// k_pf_attend's q row and outputs cover hd; longer ffn rows go token by token.
int l3m_prefill_fits(int dim, int ffn, int nqd, int hd) {
    return dim <= 4 * NTE && ffn <= 4 * NTE && nqd <= 4 * NTE && hd <= 256 && hd % 2 == 0;
}

int l3m_prefill(const l3m_dmodel *M, const l3m_pflayer *L, const l3m_pfbuf *B, int P, void *stream) {
    if (P < 1) return 0;
    if (P > M->ctx || !l3m_prefill_fits(M->dim, M->ffn, M->n_heads * M->hd, M->hd)) return fail_msg("prefill: shape out of range");
    hipStream_t st = as_stream(stream);
    hipLaunchKernelGGL(k_pf_embed, dim3(P), dim3(NTE), 0, st, M->embed, (const int32_t *)M->tokens, M->dim, B->x);
    if (L->qkv.dtype == L3M_BF16) pf_layers<L3M_BF16>(M, L, B, P, st);
    else pf_layers<L3M_Q8_0>(M, L, B, P, st);
    CKL("prefill");
    return 0;
}

int l3m_step_enqueue(const l3m_dmodel *M, const l3m_dlayer *layers, int with_head, void *stream) {
    hipStream_t st = as_stream(stream);
    for (int l = 0; l < M->n_layers; l++) {
        DISPATCH(M->body_dtype, launch_attn, *M, layers[l], l, st);
        DISPATCH(M->body_dtype, launch_ffn, *M, layers[l], !with_head && l == M->n_layers - 1, st);
    }
    if (with_head) DISPATCH(M->head.dtype, launch_head, *M, 1, st);
    CKL("decode step");
    return 0;
}

int l3m_dev_cus(void) {
    int cus = 0;
    if (l3m_dev_init() || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, 0) != hipSuccess) return 0;
    return cus;
}

// The (body, head, GPT-2) kinds the persistent kernel is built for: every dtype with a head of its own
// dtype, the mixed heads of the reference's tests (test_engine.py:187-191), an mxfp4 model whose body runs
// as q8_0 (its blocks widened exactly) with its mxfp4 head, and the GPT-2 variant in the dtypes its
// exporter writes (f32, bf16, q8_0, q4_0, each with a head of its own dtype).
#define DECODE_PAIRS(X) \
    X(L3M_F32, L3M_F32, false) X(L3M_BF16, L3M_BF16, false) X(L3M_Q8_0, L3M_Q8_0, false) X(L3M_Q4_0, L3M_Q4_0, false) \
    X(L3M_MXFP4, L3M_MXFP4, false) X(L3M_Q4_0, L3M_Q8_0, false) X(L3M_MXFP4, L3M_Q8_0, false) X(L3M_Q8_0, L3M_BF16, false) \
    X(L3M_Q8_0, L3M_MXFP4, false) X(L3M_F32, L3M_F32, true) X(L3M_BF16, L3M_BF16, true) X(L3M_Q8_0, L3M_Q8_0, true) \
    X(L3M_Q4_0, L3M_Q4_0, true)

int l3m_decode_pair(int dtype, int head_dtype, int gpt2) {
#define PAIR_KNOWN(a, b, g) if (dtype == a && head_dtype == b && !gpt2 == !g) return 1;
    DECODE_PAIRS(PAIR_KNOWN)
#undef PAIR_KNOWN
    return 0;
}

int l3m_decode_fits(int dtype, int head_dtype, int gpt2, int hd, int grid, unsigned lds) {
    if (l3m_dev_init()) return 0;
#define PAIR_FITS(a, b, g) if (dtype == a && head_dtype == b && !gpt2 == !g) return decode_fits<a, b, g>(hd, grid, lds);
    DECODE_PAIRS(PAIR_FITS)
#undef PAIR_FITS
    return 0;
}

// Adds the launch of slot `slot` to the running total once it has finished (its end event waited for).
static int timer_collect(int slot) {
    if (!g_dec_pending[slot]) return 0;
    float ms = 0.f;
    CK(hipEventSynchronize(g_dec_ev[slot][1]));
    CK(hipEventElapsedTime(&ms, g_dec_ev[slot][0], g_dec_ev[slot][1]));
    g_dec_us += 1000.0 * ms;
    g_dec_launches++;
    g_dec_pending[slot] = 0;
    return 0;
}

int l3m_decode_timer_collect(int slot) { return slot < 0 || slot > 1 ? -1 : timer_collect(slot); }

int l3m_decode_timer(int mode, double *us, int *launches) {
    if (l3m_dev_init()) return -1;
    if (mode == 1) {                                   // start: clear and time from now on
        for (int s = 0; s < 2; s++)                   // made here, outside the timed calls
            for (int e = 0; e < 2; e++)
                if (!g_dec_ev[s][e]) CK(hipEventCreate(&g_dec_ev[s][e]));
        g_dec_timing = 1; g_dec_us = 0; g_dec_launches = 0; g_dec_pending[0] = g_dec_pending[1] = 0;
    } else if (mode == 2) {                            // collect the finished launches (their stream has been waited for)
        if (timer_collect(0) || timer_collect(1)) return -1;
    } else {                                           // stop
        g_dec_timing = 0;
    }
    if (us) *us = g_dec_us;
    if (launches) *launches = g_dec_launches;
    return 0;
}

int l3m_decode_placement(int grid, unsigned lds, int *xcc) {
    if (l3m_dev_init()) return -1;
    if (grid <= 0) return fail_msg("placement: empty grid");
    int *d = nullptr;
    CK(hipMalloc(&d, (size_t)grid * 4));
    lds_opt_in(k_where, lds);
    void *args[] = {&d};
    hipError_t e;
    if (g_coop) {
        e = hipLaunchCooperativeKernel((const void *)k_where, dim3(grid), dim3(NTE), args, lds, g_stream);
    } else {
        hipLaunchKernelGGL(k_where, dim3(grid), dim3(NTE), lds, g_stream, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpyAsync(xcc, d, (size_t)grid * 4, hipMemcpyDeviceToHost, g_stream);
    if (e == hipSuccess) e = hipStreamSynchronize(g_stream);
    (void)hipFree(d);
    return e == hipSuccess ? 0 : fail("placement probe", e);
}

int l3m_decode_launch(int dtype, int head_dtype, int gpt2, int hd, const l3m_dmodel *M_dev, const l3m_dlayer *layers_dev, const l3m_run *R_dev,
                      int grid, unsigned lds, void *stream, int slot) {
    hipStream_t st = as_stream(stream);
    if (slot < 0 || slot > 1) return fail_msg("decode: slot out of range");
#define PAIR_LAUNCH(a, b, g) \
    if (dtype == a && head_dtype == b && !gpt2 == !g) return launch_decode<a, b, g>(M_dev, layers_dev, R_dev, hd, grid, lds, st, slot);
    DECODE_PAIRS(PAIR_LAUNCH)
#undef PAIR_LAUNCH
    return fail_msg("decode: no persistent kernel for this pair of dtypes");
}

l3m_graphs *l3m_graphs_build(const l3m_dmodel *M, const l3m_dlayer *layers) {
    l3m_graphs *g = (l3m_graphs *)calloc(1, sizeof *g);
    if (!g) return NULL;
    for (int w = 0; w < 2; w++) {
        if (hipStreamBeginCapture(g_stream, hipStreamCaptureModeThreadLocal) != hipSuccess) { fail_msg("graph capture"); goto bad; }
        int rc = l3m_step_enqueue(M, layers, w, g_stream);
        if (hipStreamEndCapture(g_stream, &g->g[w]) != hipSuccess || rc) { fail_msg("graph capture"); goto bad; }
        if (hipGraphInstantiate(&g->e[w], g->g[w], NULL, NULL, 0) != hipSuccess) { fail_msg("graph instantiate"); goto bad; }
    }
    return g;
bad:
    l3m_graphs_free(g);
    return NULL;
}

int l3m_graphs_launch(l3m_graphs *g, int with_head, void *stream) {
    CK(hipGraphLaunch(g->e[with_head ? 1 : 0], as_stream(stream)));
    return 0;
}

// A prompt length's launches (their grids and arguments depend on P alone, every buffer is the model's own) as a
// graph, for the PF_GRAPHS lengths used last: the first prompt of a length is launched kernel by kernel, its second
// captured, later ones replayed (the loader's rule says for which models). Capture and instantiation cost a call 0.06 ms
// (2 layers) to 0.16 (6), which a length seen once never pays (2 layers of dim 128, 48 tokens: the first call 198 us, the
// second 198, then 133; launched one by one 190, 165, then 157). Captured on a stream
// of its own: other threads' work on the library's stream stays out of it. off: a capture failed, launched one by one
// from then on.
constexpr int PF_GRAPHS = 8;
struct l3m_pfgraphs {
    hipStream_t cap;
    bool off;
    int P[PF_GRAPHS];                 // 0: an empty entry
    hipGraphExec_t e[PF_GRAPHS];      // null: seen once
    unsigned long long used[PF_GRAPHS], tick;
};

l3m_pfgraphs *l3m_pfgraphs_new(void) {
    l3m_pfgraphs *g = (l3m_pfgraphs *)calloc(1, sizeof *g);
    if (g && hipStreamCreateWithFlags(&g->cap, hipStreamNonBlocking) != hipSuccess) {
        (void)hipGetLastError();
        free(g);
        return nullptr;
    }
    return g;
}

void l3m_pfgraphs_free(l3m_pfgraphs *g) {
    if (!g) return;
    for (int i = 0; i < PF_GRAPHS; i++)
        if (g->e[i]) (void)hipGraphExecDestroy(g->e[i]);
    (void)hipStreamDestroy(g->cap);
    free(g);
}

static hipGraphExec_t pf_capture(l3m_pfgraphs *g, const l3m_dmodel *M, const l3m_pflayer *L, const l3m_pfbuf *B, int P) {
    hipGraph_t graph = nullptr;
    hipGraphExec_t e = nullptr;
    const int had = g_has_err;
    if (hipStreamBeginCapture(g->cap, hipStreamCaptureModeThreadLocal) == hipSuccess) {
        const int rc = l3m_prefill(M, L, B, P, g->cap);
        if (hipStreamEndCapture(g->cap, &graph) != hipSuccess || rc || hipGraphInstantiate(&e, graph, NULL, NULL, 0) != hipSuccess) e = nullptr;
        if (graph) (void)hipGraphDestroy(graph);
    }
    if (!e) {                                          // launched one by one instead: no error of the call's
        g->off = true;
        (void)hipGetLastError();
        if (!had) l3m_dev_clear_error();
    }
    return e;
}

int l3m_prefill_graph(l3m_pfgraphs *g, const l3m_dmodel *M, const l3m_pflayer *L, const l3m_pfbuf *B, int P) {
    if (P < 1) return 0;
    int k = -1, lru = 0;
    for (int i = 0; i < PF_GRAPHS; i++) {
        if (g->P[i] == P) k = i;
        if (g->used[i] < g->used[lru]) lru = i;
    }
    if (k < 0) {
        k = lru;
        if (g->e[k]) { (void)hipGraphExecDestroy(g->e[k]); g->e[k] = nullptr; }
        g->P[k] = P;
    } else if (!g->e[k] && !g->off)
        g->e[k] = pf_capture(g, M, L, B, P);
    g->used[k] = ++g->tick;
    if (!g->e[k]) return l3m_prefill(M, L, B, P, g_stream);
    CK(hipGraphLaunch(g->e[k], g_stream));
    return 0;
}

// Mean microseconds per launch of iters launches queued back to back, after one untimed launch: one pair
// of events around them all (events around each launch would add their own markers' time to every
// figure). For a kernel shorter than the launch interval (l3m_time_launch_interval) this is the launch rate.
static double time_launches(int iters, int (*launch)(void *ctx, int i), void *ctx) {
    hipEvent_t a, b;
    if (hipEventCreate(&a) != hipSuccess || hipEventCreate(&b) != hipSuccess) { fail_msg("hipEventCreate"); return -1; }
    double us = -1;
    int rc = launch(ctx, 0);                                   // untimed first launch
    if (!rc && hipEventRecord(a, g_stream) == hipSuccess) {
        for (int i = 0; i < iters && !rc; i++) rc = launch(ctx, i);
        float ms = 0;
        if (!rc && hipEventRecord(b, g_stream) == hipSuccess && hipEventSynchronize(b) == hipSuccess &&
            hipEventElapsedTime(&ms, a, b) == hipSuccess)
            us = 1e3 * ms / iters;
    }
    (void)hipEventDestroy(a);
    (void)hipEventDestroy(b);
    return rc ? -1 : us;
}

static int dummy_one(void *, int) {
    hipLaunchKernelGGL(k_dummy, dim3(1), dim3(NT), 0, g_stream);
    CKL("k_dummy");
    return 0;
}

struct GemvCtx { const l3m_dmat *mats; int n; const void *act; int k; float *y; };
static int gemv_one(void *c, int i) {
    GemvCtx *g = (GemvCtx *)c;
    return l3m_k_gemv(&g->mats[i % g->n], g->act, g->k, g->y, g_stream);
}

double l3m_time_launch_interval(int iters) {
    if (l3m_dev_init() || iters < 1) return -1;
    return time_launches(iters, dummy_one, nullptr);
}

double l3m_time_gemv(const l3m_dmat *mats, int n_mats, const void *act, int k, float *y, int iters) {
    if (l3m_dev_init() || n_mats < 1 || iters < 1) return -1;
    GemvCtx c{mats, n_mats, act, k, y};
    return time_launches(iters, gemv_one, &c);
}

// The measured roofline of a matvec: one streaming read of the same number of bytes, in the same
// residency (the same buffer again: warm; round robin over buffers totalling more than the Infinity
// Cache: cold). Each launch reads one buffer with enough workgroups for every CU.
struct ReadCtx { void *const *bufs; int n; size_t bytes; unsigned grid; };
static int read_one(void *c, int i) {
    ReadCtx *r = (ReadCtx *)c;
    void *b = r->bufs[i % r->n];
    hipLaunchKernelGGL(k_read, dim3(r->grid), dim3(NT), 0, g_stream, (const u32x4 *)b, r->bytes / 16 - 1, (unsigned *)((u32x4 *)b + r->bytes / 16 - 1));
    CKL("k_read");
    return 0;
}

double l3m_time_read(void *const *bufs, int n_bufs, size_t bytes, int iters) {
    if (l3m_dev_init() || n_bufs < 1 || iters < 1 || bytes < 32 || bytes % 16) return -1;
    const size_t n16 = bytes / 16 - 1, want = (n16 + NT - 1) / NT;             // a word per thread, up to 8 workgroups per CU
    const size_t cap = 8 * (size_t)l3m_dev_cus();
    ReadCtx c{bufs, n_bufs, bytes, (unsigned)(want < cap ? want : cap)};
    return time_launches(iters, read_one, &c);
}

struct StepCtx { const l3m_dmodel *M; const l3m_dlayer *L; int kind, layer; };
static int step_one(void *c, int) {
    StepCtx *s = (StepCtx *)c;
    const l3m_dmodel &M = *s->M;
    hipStream_t st = g_stream;
    switch (s->kind) {
    case 0: DISPATCH(M.body_dtype, launch_attn, M, s->L[s->layer], s->layer, st); break;
    case 1: DISPATCH(M.body_dtype, launch_ffn, M, s->L[s->layer], 0, st); break;
    case 2: DISPATCH(M.head.dtype, launch_head, M, 0, st); break;
    default: return fail_msg("bad kernel kind");
    }
    CKL("timed kernel");
    return 0;
}

double l3m_time_step_kernel(const l3m_dmodel *M, const l3m_dlayer *layers, int kind, int layer, int iters) {
    if (l3m_dev_init() || layer < 0 || layer >= M->n_layers || iters < 1) return -1;
    StepCtx c{M, layers, kind, layer};
    return time_launches(iters, step_one, &c);
}

void l3m_graphs_free(l3m_graphs *g) {
    if (!g) return;
    for (int w = 0; w < 2; w++) {
        if (g->e[w]) (void)hipGraphExecDestroy(g->e[w]);
        if (g->g[w]) (void)hipGraphDestroy(g->g[w]);
    }
    free(g);
}

// ------------------------------------------------------------------ probes (host)

int l3m_probe_stream(size_t bytes_per_wg, int xcds, int per_xcd, int passes, double *gbs) {
    if (l3m_dev_init()) return -1;
    if (bytes_per_wg < 16 || bytes_per_wg % 16 || xcds < 1 || xcds > 8 || per_xcd < 1 || per_xcd > 32 || passes < 1)
        return fail_msg("probe_stream: bad arguments");
    const size_t n16 = bytes_per_wg / 16, total = bytes_per_wg * (size_t)xcds * per_xcd;
    void *buf = nullptr;
    unsigned *aux = nullptr;
    CK(hipMalloc(&buf, total));
    if (hipMalloc(&aux, 64 * 4) != hipSuccess) { (void)hipFree(buf); return fail_msg("probe_stream: out of memory"); }
    hipError_t e = hipMemsetAsync(buf, 0x5A, total, g_stream);
    hipEvent_t a = nullptr, b = nullptr;
    if (e == hipSuccess) e = hipEventCreate(&a);
    if (e == hipSuccess) e = hipEventCreate(&b);
    const int grid = l3m_dev_cus();
    float ms = 0.f;
    for (int rep = 0; rep < 2 && e == hipSuccess; rep++) {   // the first launch warms the caches
        e = hipMemsetAsync(aux, 0, 64 * 4, g_stream);
        if (e == hipSuccess && rep) e = hipEventRecord(a, g_stream);
        if (e == hipSuccess) {
            hipLaunchKernelGGL(k_probe_stream, dim3(grid), dim3(NTE), 0, g_stream, (const u32x4 *)buf, n16, passes, xcds, per_xcd, aux, aux + 32);
            e = hipGetLastError();
        }
        if (e == hipSuccess && rep) e = hipEventRecord(b, g_stream);
    }
    if (e == hipSuccess) e = hipEventSynchronize(b);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, a, b);
    unsigned got[8] = {0};
    if (e == hipSuccess) e = hipMemcpy(got, aux, sizeof got, hipMemcpyDeviceToHost);
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
    (void)hipFree(buf); (void)hipFree(aux);
    if (e != hipSuccess) return fail("probe_stream", e);
    for (int x = 0; x < xcds; x++)
        if ((int)got[x] < per_xcd) return fail_msg("probe_stream: an XCD has fewer CUs than requested");
    *gbs = (double)total * passes / (ms * 1e6);
    return 0;
}

int l3m_probe_exchange(int n, int same_xcd, int dim, int rounds, double *us_per_round) {
    if (l3m_dev_init()) return -1;
    if (n < 1 || n > 32 || dim < n || dim > (1 << 20) || rounds < 2) return fail_msg("probe_exchange: bad arguments");
    float *vec = nullptr;
    unsigned *aux = nullptr;
    unsigned long long *out = nullptr;
    CK(hipMalloc(&vec, 2 * (size_t)dim * 4));
    if (hipMalloc(&aux, 256 * 4) != hipSuccess || hipMalloc(&out, 16) != hipSuccess) {
        (void)hipFree(vec); (void)hipFree(aux); return fail_msg("probe_exchange: out of memory");
    }
    hipError_t e = hipMemsetAsync(aux, 0, 256 * 4, g_stream);
    if (e == hipSuccess) e = hipMemsetAsync(out, 0, 16, g_stream);
    unsigned *flags = aux, *tickets = aux + 128;
    unsigned long long limit = 100000000ull, host_out[2] = {0, 0};
    int grid = l3m_dev_cus();
    void *args[] = {&vec, &dim, &n, &same_xcd, &rounds, &flags, &tickets, &out, &limit};
    if (e == hipSuccess && g_coop) e = hipLaunchCooperativeKernel((const void *)k_probe_exchange, dim3(grid), dim3(NTE), args, 0, g_stream);
    if (e == hipSuccess && !g_coop) {                  // L3M_COOP=0: the same grid as an ordinary dispatch
        hipLaunchKernelGGL(k_probe_exchange, dim3(grid), dim3(NTE), 0, g_stream, vec, dim, n, same_xcd, rounds, flags, tickets, out, limit);
        e = hipGetLastError();
    }
    unsigned abort_word = 0;
    if (e == hipSuccess) e = hipMemcpyAsync(host_out, out, 16, hipMemcpyDeviceToHost, g_stream);
    if (e == hipSuccess) e = hipMemcpyAsync(&abort_word, flags + 64, 4, hipMemcpyDeviceToHost, g_stream);
    if (e == hipSuccess) e = hipStreamSynchronize(g_stream);
    (void)hipFree(vec); (void)hipFree(aux); (void)hipFree(out);
    if (e != hipSuccess) return fail("probe_exchange", e);
    if (abort_word || !host_out[0]) return fail_msg("probe_exchange: a wait timed out (not enough workgroups on the XCDs asked for)");
    *us_per_round = (double)host_out[0] * 0.01 / (rounds - 1);
    return 0;
}

int l3m_probe_graph_node(int nodes, int reps, double *us_per_node) {
    if (l3m_dev_init()) return -1;
    if (nodes < 1 || nodes > 4096 || reps < 1) return fail_msg("probe_graph_node: bad arguments");
    hipGraph_t g = nullptr;
    hipGraphExec_t ge = nullptr;
    hipStream_t cs = nullptr;
    hipEvent_t a = nullptr, b = nullptr;
    float ms = 0.f;
    hipError_t e = hipStreamCreateWithFlags(&cs, hipStreamNonBlocking);
    if (e == hipSuccess) e = hipStreamBeginCapture(cs, hipStreamCaptureModeThreadLocal);
    if (e == hipSuccess) {
        for (int i = 0; i < nodes; i++) hipLaunchKernelGGL(k_probe_empty, dim3(1), dim3(64), 0, cs);
        e = hipStreamEndCapture(cs, &g);
    }
    if (e == hipSuccess) e = hipGraphInstantiate(&ge, g, nullptr, nullptr, 0);
    if (e == hipSuccess) e = hipEventCreate(&a);
    if (e == hipSuccess) e = hipEventCreate(&b);
    if (e == hipSuccess) e = hipGraphLaunch(ge, g_stream);                 // warm
    if (e == hipSuccess) e = hipEventRecord(a, g_stream);
    for (int r = 0; r < reps && e == hipSuccess; r++) e = hipGraphLaunch(ge, g_stream);
    if (e == hipSuccess) e = hipEventRecord(b, g_stream);
    if (e == hipSuccess) e = hipEventSynchronize(b);
    if (e == hipSuccess) e = hipEventElapsedTime(&ms, a, b);
    if (a) (void)hipEventDestroy(a);
    if (b) (void)hipEventDestroy(b);
    if (ge) (void)hipGraphExecDestroy(ge);
    if (g) (void)hipGraphDestroy(g);
    if (cs) (void)hipStreamDestroy(cs);
    if (e != hipSuccess) return fail("probe_graph_node", e);
    *us_per_node = 1e3 * ms / ((double)reps * nodes);
    return 0;
}

int l3m_probe_latency(int which, int threads, double *clocks) {
    if (l3m_dev_init()) return -1;
    if (which < 0 || which > 6 || threads < 64 || threads > NTE || (threads & (threads - 1)))
        return fail_msg("probe_latency: bad arguments (which 0-6, threads a power of two from 64 to 1024)");
    void (*const kernels[7])(unsigned long long *, float *, int) = {k_probe_latency<0>, k_probe_latency<1>, k_probe_latency<2>,
                                                                    k_probe_latency<3>, k_probe_latency<4>, k_probe_latency<5>,
                                                                    k_probe_latency<6>};
    unsigned long long *out = nullptr;
    float *sink = nullptr;
    CK(hipMalloc(&out, 8));
    if (hipMalloc(&sink, NTE * sizeof(float)) != hipSuccess) { (void)hipFree(out); return fail_msg("probe_latency: out of memory"); }
    const int iters = 1000;
    unsigned long long got[2] = {0, 0};
    hipError_t e = hipSuccess;
    for (int k = 0; k < 2 && e == hipSuccess; k++) {
        hipLaunchKernelGGL(kernels[which], dim3(1), dim3(threads), 0, g_stream, out, sink, (k + 1) * iters);
        e = hipGetLastError();
        if (e == hipSuccess) e = hipMemcpyAsync(got + k, out, 8, hipMemcpyDeviceToHost, g_stream);
        if (e == hipSuccess) e = hipStreamSynchronize(g_stream);
    }
    (void)hipFree(out); (void)hipFree(sink);
    if (e != hipSuccess) return fail("probe_latency", e);
    *clocks = ((double)got[1] - (double)got[0]) / iters;
    return 0;
}

}  // extern "C"
