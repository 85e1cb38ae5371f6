// Loads of a weight span (256 values of a row: 8 blocks of 32) of the types with Q8_0 activations straight from an expert
// matrix, as the register-staged grouped GEMM takes them: what lane quarter q needs of the span at blk.  The last span of
// the last expert ends the allocation, so no load may leave the span.  Nothing here but v_alignbyte is GPU code:
// the sanitizer test (span_loads.cpp) compiles these loads for the CPU and runs them over spans that end an allocation.
#pragma once
#include "hy_types.h"

namespace hy {

__device__ __forceinline__ uint16_t ld_u16(const uint8_t *p) { return *(const uint16_t *) p; }

// Branch-free loads from 2-byte aligned addresses (a fixed instruction count per step lets the compiler count
// the loads in flight): whole dwords from the aligned-down address, joined with v_alignbyte.
__device__ __forceinline__ uint32_t join_b(uint32_t hi, uint32_t lo, uint32_t sb) { return __builtin_amdgcn_alignbyte(hi, lo, sb); }
// 8 bytes at p (2-byte aligned); reads the dwords at p & ~3 .. + 11, all of which must lie in the buffer
// (the aligned-down pointer is formed by pointer arithmetic on p, so that an LDS pointer stays an LDS pointer)
__device__ __forceinline__ uint2 ld8_2a(const uint8_t *p) {
    const uint32_t *w = (const uint32_t *) (p - ((uintptr_t) p & 3));
    const uint32_t sb = (uint32_t) ((uintptr_t) p & 3);
    const uint32_t d0 = w[0], d1 = w[1], d2 = w[2];
    return make_uint2(join_b(d1, d0, sb), join_b(d2, d1, sb));
}

// qv[c]: 8 bytes of block c's quants -- Q8_0 qs[8 q ..], the others qs[8 (q & 1) ..] (values 8 q .. + 7 are their nibbles
// q >> 1); dd / ee / dm: the blocks' scales; hb: byte q of the blocks' fifth bits.
template <int T> struct SpanBytes;

// 18 B a block.  The span is 16-byte aligned (rows of 144 n / 256 bytes), so block c's qs sit at 2 mod 4 for even c and at
// 0 mod 4 for odd c.
template <> struct SpanBytes<IQ4_NL> {
    uint2 qv[8]; uint32_t dd[4];
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint8_t *p = blk + 18 * c + 2 + 8 * (q & 1);
            if (c & 1) qv[c] = *(const uint2 *) p;
            else {
                const uint32_t *w = (const uint32_t *) (p - 2);
                const uint32_t d0 = w[0], d1 = w[1], d2 = w[2];
                qv[c] = make_uint2(join_b(d1, d0, 2), join_b(d2, d1, 2));
            }
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) dd[i] = (uint32_t) ld_u16(blk + 36 * i) | ((uint32_t) ld_u16(blk + 36 * i + 18) << 16);
    }
};
// 34 B a block.  The spans are 16-byte aligned, so block c's qs (34 c + 2) are 2 mod 4 for even c, read by ld8_2a whose 12
// bytes end at most at blk + 239, and dword-aligned for odd c, read as they are: block 7's last 8 bytes end the span.
template <> struct SpanBytes<Q8_0> {
    uint2 qv[8]; uint32_t dd[4];
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint8_t *p = blk + 34 * c + 2 + 8 * q;
            qv[c] = (c & 1) ? *(const uint2 *) p : ld8_2a(p);
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) dd[i] = (uint32_t) ld_u16(blk + 68 * i) | ((uint32_t) ld_u16(blk + 68 * i + 34) << 16);
    }
};
// 17 B a block.  Spans of 136 bytes are 8-byte aligned, so block c's qs at 17 c + 1 sit at offset (17 c + 1) mod 4 = 1 2 3
// 0 1 2 3 0: the dword-aligned ones (c = 3, 7) are read as they are, the others by ld8_2a, whose 12 bytes end at most at
// blk + 119.
template <> struct SpanBytes<MXFP4> {
    uint2 qv[8]; uint32_t ee[2];
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint8_t *p = blk + 17 * c + 1 + 8 * (q & 1);
            qv[c] = (c & 3) == 3 ? *(const uint2 *) p : ld8_2a(p);
        }
        ee[0] = ee[1] = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) ee[c >> 2] |= (uint32_t) blk[17 * c] << (8 * (c & 3));
    }
};
// 24 B a block: every field dword-aligned.
template <> struct SpanBytes<Q5_1> {
    uint2 qv[8]; uint32_t hb[2], dm[8];
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            qv[c] = *(const uint2 *) (blk + 24 * c + 8 + 8 * (q & 1));
            dm[c] = *(const uint32_t *) (blk + 24 * c);
        }
        hb[0] = hb[1] = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) hb[c >> 2] |= (uint32_t) blk[24 * c + 4 + q] << (8 * (c & 3));
    }
};
// 22 B a block.  Block c's qs (22 c + 6) and qh (22 c + 2) are 2 mod 4 for even c, read by ld8_2a whose 12 bytes end at
// most at blk + 155, and dword-aligned for odd c, read as they are.
template <> struct SpanBytes<Q5_0> {
    uint2 qv[8]; uint32_t hb[2], dd[4];
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint8_t *p = blk + 22 * c + 6 + 8 * (q & 1);
            qv[c] = (c & 1) ? *(const uint2 *) p : ld8_2a(p);
        }
        hb[0] = hb[1] = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) hb[c >> 2] |= (uint32_t) blk[22 * c + 2 + q] << (8 * (c & 3));
#pragma unroll
        for (int i = 0; i < 4; ++i) dd[i] = (uint32_t) ld_u16(blk + 44 * i) | ((uint32_t) ld_u16(blk + 44 * i + 22) << 16);
    }
};

} // namespace hy
