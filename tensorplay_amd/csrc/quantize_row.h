// The arithmetic of the row-wise int8 quantizer, shared by its own kernels and by those that quantize an activation row on its
// way into a product: the same codes and scales wherever a row is quantized.
#pragma once

#include "tpq_common.h"

namespace tpq {
namespace {

constexpr int kVec = 8;  // elements per lane per chunk

struct QParams {
    float eps, divisor;
    int qmin, qmax, sign_mode;
    int no_clamp;  // no quotient |v| / scale, |v| <= absmax, can round outside [qmin, qmax]
};

// (apart from the sign mode's form: asked for together with it, eight comparisons and selections of that form were made in front of
// every branch)
__device__ __forceinline__ int quantize_divided(float v, float scale, const QParams& p) {
    // __fdiv_rn: correctly rounded division regardless of compiler flags
    float q = rintf(__fdiv_rn(v, scale));
    q = fminf(fmaxf(q, static_cast<float>(p.qmin)), static_cast<float>(p.qmax));
    return static_cast<int>(q);
}
__device__ __forceinline__ int quantize_one(float v, float scale, const QParams& p) {
    if (p.sign_mode) return v >= 0.0f ? p.qmax : p.qmin;
    return quantize_divided(v, scale, p);
}

// Eight codes with one reciprocal instead of eight divisions, same bits as quantize_one.
// q = v * (1/scale) is within 2^-21 relative of the true quotient, |quotient| <= 128 here, so its
// absolute error is below 2^-14.  If q lies at least 2^-13 inside (c - 1/2, c + 1/2), so does the
// correctly rounded quotient, and both round to c.  Otherwise (about one element in a few thousand;
// also NaN and infinities) the element is redone with the IEEE division.
// The codes leave as two packed words.  v_cvt_pk_u8_f32 converts a float to an unsigned byte (saturating at 0 and
// 255) and drops it into one byte of a register: the rounded quotient c is an integer already, so c + 128 converts
// exactly, the upper clamp is the saturation when qmax = 127, and one xor takes the 128 off the four bytes again.
// Four instructions per code less than clamp, convert, mask, shift, or.
__device__ __forceinline__ void quantize_eight_packed(const float (&v)[kVec], float scale, float inv_scale, const QParams& p,
                                                      uint32_t& lo, uint32_t& hi) {
    bool redo = false;
    uint32_t word[2] = {0u, 0u};
    const float qmin = static_cast<float>(p.qmin), qmax = static_cast<float>(p.qmax);
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const float q = v[i] * inv_scale;
        const float c = rintf(q);
        redo |= !(fabsf(q - c) <= 0.5f - 0x1p-13f);
        const float biased = fminf(fmaxf(c, qmin), qmax) + 128.0f;  // 0 .. 255, an integer
        word[i >> 2] = __builtin_amdgcn_cvt_pk_u8_f32(biased, i & 3, word[i >> 2]);
    }
    lo = word[0] ^ 0x80808080u;
    hi = word[1] ^ 0x80808080u;
    // Rare (one element in a few thousand).  Behind a branch the whole wavefront takes or skips, and with the divisor
    // passed through a statement the compiler may not move: as a plain "if", the eight divisions were hoisted above the
    // branch, computed for every chunk and selected away.
    if (__builtin_amdgcn_ballot_w64(redo) != 0) {
        float divisor = scale;
        asm volatile("; elements redone with the division" : "+v"(divisor));
        if (redo) {
            lo = hi = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo |= (static_cast<uint32_t>(quantize_divided(v[i], divisor, p)) & 0xFFu) << (8 * i);
                hi |= (static_cast<uint32_t>(quantize_divided(v[i + 4], divisor, p)) & 0xFFu) << (8 * i);
            }
        }
    }
}

// The same codes with fewer instructions, for parameters under which no quotient can leave the code range
// (rint(divisor (1 + 2^-20)) <= qmax and >= -qmin, true for the usual divisor = qmax = -qmin = 127): no clamp is
// needed, and the code is read off the mantissa.  t = fma(v, 1/scale, 1.5 * 2^23) rounds the exact product to the
// nearest integer (ties to even) and leaves it in two's complement in the low mantissa bits; c = t - 1.5 * 2^23 is that
// integer, r = fma(v, 1/scale, -c) its distance from the product, rounded by 2^-25 at most.  The product is within 2^-16 of the
// correctly rounded quotient the reference rounds (two roundings of 2^-24 relative, |quotient| <= 128), so |r| <= 1/2 - 2^-15 proves both
// round to c; anything else (also NaN) is redone with the division: one element in 16 000, a wavefront in 30 where a limit of 2^-13 sent one in 8.  Five instructions per code and three byte permutes per four codes.
__device__ __forceinline__ void quantize_eight_lean(const float (&v)[kVec], float scale, float inv_scale, const QParams& p,
                                                    uint32_t& lo, uint32_t& hi) {
    constexpr float kMagic = 12582912.0f;  // 1.5 * 2^23
    bool redo = false;
    uint32_t t[kVec];
#pragma unroll
    for (int i = 0; i < kVec; ++i) {
        const float tf = __builtin_fmaf(v[i], inv_scale, kMagic);
        const float c = tf - kMagic;
        const float r = __builtin_fmaf(v[i], inv_scale, -c);
        redo |= !(fabsf(r) <= 0.5f - 0x1p-15f);
        t[i] = __builtin_bit_cast(uint32_t, tf);
    }
    // v_perm_b32(a, b, sel): selector bytes 0..3 take bytes of b, 4..7 of a, 0x0c a zero byte
    lo = __builtin_amdgcn_perm(t[1], t[0], 0x0c0c0400u) | __builtin_amdgcn_perm(t[3], t[2], 0x04000c0cu);
    hi = __builtin_amdgcn_perm(t[5], t[4], 0x0c0c0400u) | __builtin_amdgcn_perm(t[7], t[6], 0x04000c0cu);
    // Rare (one element in 16 000).  Behind a branch the whole wavefront takes or skips, and with the divisor
    // passed through a statement the compiler may not move: as a plain "if", the eight divisions were hoisted above the
    // branch, computed for every chunk and selected away.
    if (__builtin_amdgcn_ballot_w64(redo) != 0) {
        float divisor = scale;
        asm volatile("; elements redone with the division" : "+v"(divisor));
        if (redo) {
            lo = hi = 0;
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                lo |= (static_cast<uint32_t>(quantize_divided(v[i], divisor, p)) & 0xFFu) << (8 * i);
                hi |= (static_cast<uint32_t>(quantize_divided(v[i + 4], divisor, p)) & 0xFFu) << (8 * i);
            }
        }
    }
}

// What a row's maximum makes of its parameters
struct RowScale {
    float scale, inverse;
    bool shortcut, lean;
};
__device__ __forceinline__ RowScale scale_of_row(float absmax, const QParams& p) {
    RowScale r;
    r.scale = __fdiv_rn(fmaxf(absmax, p.eps), p.divisor);
    // the shortcut needs |quotient| <= 128 and a finite reciprocal: true for every scale the formula
    // above produces from finite inputs with divisor <= 128; anything else takes the divisions
    r.inverse = __fdiv_rn(1.0f, r.scale);
    r.shortcut = !p.sign_mode && p.divisor <= 128.0f && r.inverse < 3.0e38f && absmax <= 3.0e38f;
    r.lean = r.shortcut && p.no_clamp;
    return r;
}
__device__ __forceinline__ void quantize_eight(const float (&v)[kVec], const RowScale& r, const QParams& p, uint32_t& lo, uint32_t& hi) {
    lo = hi = 0;
    if (r.lean) {
        quantize_eight_lean(v, r.scale, r.inverse, p, lo, hi);
    } else if (r.shortcut) {
        quantize_eight_packed(v, r.scale, r.inverse, p, lo, hi);
    } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            lo |= (static_cast<uint32_t>(quantize_one(v[i], r.scale, p)) & 0xFFu) << (8 * i);
            hi |= (static_cast<uint32_t>(quantize_one(v[i + 4], r.scale, p)) & 0xFFu) << (8 * i);
        }
    }
}

// Where a row's chunk of eight that would start at k0 starts: the last eight elements in place of a chunk that reaches past the
// end.  With K % 8 == 4 the last one overlaps the one before it (the same codes are stored twice).
__device__ __forceinline__ int chunk_start(int k0, int K) { return k0 + kVec <= K ? k0 : K - kVec; }

// 16 bytes from a dword-aligned address, non-temporal
__device__ __forceinline__ uint4 nt_load_dword_aligned(const void* p) {
    typedef uint32_t u4 __attribute__((ext_vector_type(4), aligned(4)));
    const u4 v = __builtin_nontemporal_load(static_cast<const u4*>(p));
    return make_uint4(v.x, v.y, v.z, v.w);
}

// eight elements as they lie; NT: non-temporal, for rows that one workgroup reads once
template <int DT>
struct RawChunk { uint4 w[DT == TPQ_DTYPE_F32 ? 2 : 1]; };
template <int DT, bool NT = true>
__device__ __forceinline__ RawChunk<DT> load_raw(const typename Elem<DT>::storage* p) {
    const uint4* const q = reinterpret_cast<const uint4*>(p);
    if constexpr (DT == TPQ_DTYPE_F32) return {{NT ? nt_load(q) : q[0], NT ? nt_load(q + 1) : q[1]}};
    else return {{NT ? nt_load_dword_aligned(p) : q[0]}};  // NT: rows of K % 8 == 4 start on 8 bytes
}
template <int DT>
__device__ __forceinline__ void unpack_chunk(const RawChunk<DT>& raw, float (&v)[kVec]) {
#pragma unroll
    for (int h = 0; h < (DT == TPQ_DTYPE_F32 ? 2 : 1); ++h) {
        const uint32_t w[4] = {raw.w[h].x, raw.w[h].y, raw.w[h].z, raw.w[h].w};
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            if constexpr (DT == TPQ_DTYPE_F32) {
                v[4 * h + i] = __builtin_bit_cast(float, w[i]);
            } else {
                v[2 * i] = Elem<DT>::load(static_cast<uint16_t>(w[i] & 0xFFFFu));
                v[2 * i + 1] = Elem<DT>::load(static_cast<uint16_t>(w[i] >> 16));
            }
        }
    }
}
template <int DT, bool NT = true>
__device__ __forceinline__ void load_chunk(const typename Elem<DT>::storage* p, float (&v)[kVec]) {
    unpack_chunk<DT>(load_raw<DT, NT>(p), v);
}

// The greatest of the wavefronts' maxima over a workgroup of THREADS threads; every thread gets the result.
template <int THREADS>
__device__ __forceinline__ float block_max(float v, float* smem) {
    const int lane = threadIdx.x & (kWave - 1), wave = threadIdx.x >> 6;
    if (lane == 0) smem[wave] = v;
    __syncthreads();
    float r = smem[0];
#pragma unroll
    for (int w = 1; w < THREADS / kWave; ++w) r = fmaxf(r, smem[w]);
    return r;
}

// eight codes to a dword-aligned address
__device__ __forceinline__ void store_codes(int8_t* p, uint32_t lo, uint32_t hi) {
    typedef uint32_t u2 __attribute__((ext_vector_type(2), aligned(4)));
    *reinterpret_cast<u2*>(p) = u2{lo, hi};
}

#ifndef TPQ_QUANT_STAMP  // readings of the clock, in a measuring build of the quantizer's own kernels
#define TPQ_QUANT_STAMP(I) do { } while (0)
#endif

// One row by a workgroup of THREADS threads, kept in registers between the maximum and the codes: CHUNKS * THREADS * 8 >= K >= 8, K % 4 == 0.
template <int DT, int CHUNKS, int THREADS>
__device__ __forceinline__ void quantize_row_cached(const typename Elem<DT>::storage* __restrict__ xr, int8_t* __restrict__ cr,
                                                    float* __restrict__ scale_out, int K, const QParams& p, float* smem) {
#ifdef TPQ_QUANT_STAMPS
    if (threadIdx.x == 0 && blockIdx.x < kStampRows) g_quant_stamps[blockIdx.x * kStampSlots + 6] = __builtin_amdgcn_s_memrealtime();
#endif
    TPQ_QUANT_STAMP(0);
    float v[CHUNKS][kVec];
    float absmax = 0.0f;
    // No branch around the loads: at the join of a branch the compiler waits for every outstanding load, which made
    // the chunks one round trip to memory each.  A chunk past the end re-reads the last chunk of the row: the same
    // elements again do not change the maximum, and nothing is stored for it.
    RawChunk<DT> raw[CHUNKS];
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) raw[c] = load_raw<DT>(xr + chunk_start((c * THREADS + threadIdx.x) * kVec, K));
    // The first use stays behind the last request: left to itself the compiler converted a chunk, and waited for it, between two
    // requests (2048 x 4096 bfloat16 9.4 -> 10.9 us).
    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) unpack_chunk<DT>(raw[c], v[c]);
    TPQ_QUANT_STAMP(1);
#pragma unroll
    for (int c = 0; c < CHUNKS; ++c)
#pragma unroll
        for (int i = 0; i < kVec; ++i) absmax = fmaxf(absmax, fabsf(v[c][i]));
    absmax = wave_max(absmax);
    TPQ_QUANT_STAMP(2);
    absmax = block_max<THREADS>(absmax, smem);
    TPQ_QUANT_STAMP(3);
    const RowScale r = scale_of_row(absmax, p);
    if (threadIdx.x == 0) *scale_out = r.scale;

#pragma unroll
    for (int c = 0; c < CHUNKS; ++c) {
        const int k0 = (c * THREADS + threadIdx.x) * kVec;
        if (k0 < K) {
            uint32_t lo, hi;
            quantize_eight(v[c], r, p, lo, hi);
            store_codes(cr + chunk_start(k0, K), lo, hi);
        }
    }
#ifdef TPQ_QUANT_STAMPS
    TPQ_QUANT_STAMP(4);
    __builtin_amdgcn_s_waitcnt(0);  // every store of this wavefront acknowledged
    TPQ_QUANT_STAMP(5);
    if (threadIdx.x == 0 && blockIdx.x < kStampRows) g_quant_stamps[blockIdx.x * kStampSlots + 7] = __builtin_amdgcn_s_memrealtime();
#endif
}

// the parameters of a quantizer: divisor 127, codes -127 .. 127 and its lower-bit relatives
inline QParams row_quantizer(float eps, float divisor, int qmin, int qmax, int sign_mode) {
    // |v| / scale <= divisor (1 + 2^-22) for every element of the row, whatever the rounding of scale and of the quotient
    const float reach = rintf(divisor * (1.0f + 0x1p-20f));
    const int no_clamp = divisor <= 127.0f && reach <= static_cast<float>(qmax) && -reach >= static_cast<float>(qmin);
    return QParams{eps, divisor, qmin, qmax, sign_mode ? 1 : 0, no_clamp};
}

}  // namespace
}  // namespace tpq
