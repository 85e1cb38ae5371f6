// Prefill / speculative-verify grouped expert GEMMs on int8 MFMA (gfx950 v_mfma_i32_16x16x32_i8 / 16x16x64_i8).
//
// Work item = (active expert, chunk of up to 64 of its tokens); k_gemm's blocks of 8 or 16 waves walk the items of their
// slot, a wave owning 16 weight rows (gate/up: half of the waves in gate, half in up, SwiGLU after an LDS exchange).
// Replaces k_moe_gemm / k_moe_gemm2, src/kernels4.cu:1354-1467, :1521-1631, which dequantize to fp16 and run fp16 MMA.
// Per 256-value span of the K dimension:
//   A (16 tokens x 32 or 64 k): the tokens' int8 values, staged through LDS for all waves;
//   B (k x 16 rows):            one weight row per lane of a quarter, decoded to int8 in registers from the staged tile;
//   D = A B, exact int32: the type's scales are either carried by B (Q4_K, Q6_K, IQ2_XS, as two int8 planes) or applied to
//   D a 32-value chunk at a time (24-bit v_mad: |D| < 2^23, |scale| < 2^8), the mins by a chained MFMA against the chunk's
//   min; the span's integers then fold into the fp32 accumulator with the contract's formula.  Types with Q8_0
//   activations fold every 32-value block on its own.
// Operand layouts (16x16x32 i8): A lane l holds token l % 16, k = 8 (l / 16) .. + 7; B lane l holds weight row l % 16 with
// the same k; D lane l holds row l % 16 for tokens 4 (l / 16) + v, v = 0..3.  The order of k inside an MFMA is free, as
// long as A and B agree.
#include "hy_internal.h"
#include "hy_blocks.cuh"

#include <algorithm>
#include <type_traits>

namespace hy {

typedef int v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ v4i mfma16(long a, long b, v4i c) { return __builtin_amdgcn_mfma_i32_16x16x32_i8(a, b, c, 0, 0, 0); }
__device__ __forceinline__ long mk_long(uint32_t lo, uint32_t hi) { return (long) (((unsigned long long) hi << 32) | lo); }
// The raw bytes of one weight row's 256-value block that lane quarter q needs, and their decoding per 32-value
// chunk c: B operand words b0/b1 (8 int8 values), scale(s), min.
template <int T> struct Raw;

template <> struct Raw<Q5_K> {   // 176 B: + qh[32] @16 (bit c of qh[l] is bit 4 of chunk c's value l), qs @48
    static constexpr bool mins = true, g16 = false;
    uint2 qv[4], qh; uint32_t dm, sl, sh, ml, mh;   // scales and mins of chunks 0..3 and 4..7, a byte each
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
        const uint4 hd = load16_a4(blk);
        dm = hd.x;
        sl = hd.y & 0x3F3F3F3Fu;
        ml = hd.z & 0x3F3F3F3Fu;
        sh = (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u);
        mh = ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
        qh = *(const uint2 *) (blk + 16 + 8 * q);
#pragma unroll
        for (int jp = 0; jp < 4; ++jp) qv[jp] = *(const uint2 *) (blk + 48 + 32 * jp + 8 * q);
    }
    static __device__ __forceinline__ uint32_t bit4(uint32_t h, int c) { return c <= 4 ? h << (4 - c) : h >> (c - 4); }   // bit c to bit 4 (of every byte, after the mask)
    __device__ __forceinline__ void chunk(int c, int, const uint2 *, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const int n = 4 * (c & 1);
        b0 = (bit4(qh.x, c) & 0x10101010u) | ((qv[c >> 1].x >> n) & 0x0F0F0F0Fu);
        b1 = (bit4(qh.y, c) & 0x10101010u) | ((qv[c >> 1].y >> n) & 0x0F0F0F0Fu);
        s0 = (int) (((c < 4 ? sl : sh) >> (8 * (c & 3))) & 255);
        mn = (int) (((c < 4 ? ml : mh) >> (8 * (c & 3))) & 255);
        s1 = 0;
    }
    __device__ __forceinline__ float fold(int si, int sm) const {
        return __builtin_fmaf(h2f(dm & 0xffff), (float) si, -(h2f(dm >> 16) * (float) sm));
    }
};
// Q2_K (84 B: scales[16], qs[64] @16, d @80, dmin @82): chunk c = values 32 c ..: 2-bit fields 2 (c & 3) of qs bytes
// 32 (c >> 2) + 8 q ..; the chunk's 16-groups 2 c (lanes q < 2) and 2 c + 1 (q >= 2): scales s0 / s1, and the lane's
// own group's min (the mins MFMA takes each lane quarter's bytes, so each 8-value piece carries its group's min).
template <> struct Raw<Q2_K> {
    static constexpr bool mins = true, g16 = true;
    uint4 scv; uint2 qv[2]; uint32_t dm;
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
        scv = load16_a4(blk);
        qv[0] = *(const uint2 *) (blk + 16 + 8 * q);
        qv[1] = *(const uint2 *) (blk + 48 + 8 * q);
        dm = *(const uint32_t *) (blk + 80);
    }
    __device__ __forceinline__ void chunk(int c, int q, const uint2 *, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const int sh = 2 * (c & 3);
        b0 = (qv[c >> 2].x >> sh) & 0x03030303u;
        b1 = (qv[c >> 2].y >> sh) & 0x03030303u;
        const uint32_t w = (c < 2 ? scv.x : c < 4 ? scv.y : c < 6 ? scv.z : scv.w) >> (16 * (c & 1));   // bytes 2 c, 2 c + 1
        s0 = (int) (w & 15);
        s1 = (int) ((w >> 8) & 15);
        mn = (int) ((w >> (q < 2 ? 4 : 12)) & 15);
    }
    __device__ __forceinline__ float fold(int si, int sm) const {
        return __builtin_fmaf(h2f(dm & 0xffff), (float) si, -(h2f(dm >> 16) * (float) sm));
    }
};
// IQ3_XXS (98 B): chunk c = 32-group c; lane q takes 8-group q: grid indices qs[8 c + 2 q], qs[8 c + 2 q + 1] (a
// halfword at 2 + 8 c + 2 q), sign index bits 7 q .. of the word at 66 + 4 c, the chunk's scale 2 sc + 1 (bits 28 ..)
// (src/kernels4.cu:613-627; ggml's vec_dot_iq3_xxs_q8_K integers).
template <> struct Raw<IQ3_XXS> {
    static constexpr bool mins = false, g16 = false;
    uint32_t gi[4], a[8], d;   // gi: the lane's index pair of chunk c in halfword c % 2 of gi[c / 2]
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
#pragma unroll
        for (int c = 0; c < 8; c += 2)
            gi[c >> 1] = (uint32_t) ld_u16(blk + 2 + 8 * c + 2 * q) | ((uint32_t) ld_u16(blk + 10 + 8 * c + 2 * q) << 16);
#pragma unroll
        for (int c = 0; c < 8; ++c) a[c] = (uint32_t) ld_u16(blk + 66 + 4 * c) | ((uint32_t) ld_u16(blk + 68 + 4 * c) << 16);
        d = ld_u16(blk);
    }
    __device__ __forceinline__ void chunk(int c, int q, const uint2 *grid, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const uint32_t ip = gi[c >> 1] >> (16 * (c & 1));
        const uint2 m = grid[256 + ((a[c] >> (7 * q)) & 127)];
        b0 = apply_mask(grid[ip & 255].x, m.x);
        b1 = apply_mask(grid[(ip >> 8) & 255].x, m.y);
        s0 = 2 * (int) (a[c] >> 28) + 1;
        s1 = 0; mn = 0;
    }
    __device__ __forceinline__ float fold(int si, int) const { return (h2f(d) * 0.25f) * (float) si; }
};
// IQ1_S (50 B): chunk c = 32-group c; lane q takes 8-group q: grid row qs[4 c + q] | 3 bits (3 q) of qh[c] << 8 (int8
// -1 / 0 / 1), the chunk's scale ls; the delta term rides on the mins MFMA with the chunk's ls * (+-1) as its "min", so
// sm = sum_ib ls sign sum_32 y and the fold is (d / 8) (8 si + sm) (src/kernels4.cu:650-659; src/iq1s_dot.h:26-64).
template <> struct Raw<IQ1_S> {
    static constexpr bool mins = true, g16 = false;
    uint32_t gq[2], qh[4], d;   // gq: the lane's index byte of chunk c in byte c % 4 of gq[c / 4]; qh[c] in halfwords
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
        gq[0] = gq[1] = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) gq[c >> 2] |= (uint32_t) blk[2 + 4 * c + q] << (8 * (c & 3));
#pragma unroll
        for (int i = 0; i < 4; ++i) qh[i] = (uint32_t) ld_u16(blk + 34 + 4 * i) | ((uint32_t) ld_u16(blk + 36 + 4 * i) << 16);
        d = ld_u16(blk);
    }
    __device__ __forceinline__ void chunk(int c, int q, const uint2 *grid, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const uint32_t h = (qh[c >> 1] >> (16 * (c & 1))) & 0xffff;
        const uint2 g = grid[((gq[c >> 2] >> (8 * (c & 3))) & 255) | (((h >> (3 * q)) & 7) << 8)];
        b0 = g.x; b1 = g.y;
        s0 = 2 * (int) ((h >> 12) & 7) + 1;
        s1 = 0;
        mn = h & 0x8000 ? -s0 : s0;
    }
    __device__ __forceinline__ float fold(int si, int sm) const { return (h2f(d) * 0.125f) * (float) (8 * si + sm); }
};
// IQ2_S (82 B): chunk c = 32-group c; lane q takes 8-group q: grid row qs[4 c + q] | bits 2 q, 2 q + 1 of qh[c] << 8,
// sign byte signs[4 c + q], the chunk's 16-group scales 2 sc + 1 from the nibbles of scales[c] (s0 for lanes q < 2)
// (src/kernels4.cu:602-613; ggml's vec_dot_iq2_s_q8_K integers).
template <> struct Raw<IQ2_S> {
    static constexpr bool mins = false, g16 = true;
    uint32_t gq[2], sg[2], qh[2], sc[2], d;   // byte c % 4 of [c / 4]: the lane's index byte, its sign byte, qh[c], scales[c]
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
        gq[0] = gq[1] = sg[0] = sg[1] = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            gq[c >> 2] |= (uint32_t) blk[2 + 4 * c + q] << (8 * (c & 3));
            sg[c >> 2] |= (uint32_t) blk[34 + 4 * c + q] << (8 * (c & 3));
        }
#pragma unroll
        for (int i = 0; i < 2; ++i) {
            qh[i] = (uint32_t) ld_u16(blk + 66 + 4 * i) | ((uint32_t) ld_u16(blk + 68 + 4 * i) << 16);
            sc[i] = (uint32_t) ld_u16(blk + 74 + 4 * i) | ((uint32_t) ld_u16(blk + 76 + 4 * i) << 16);
        }
        d = ld_u16(blk);
    }
    __device__ __forceinline__ void chunk(int c, int q, const uint2 *grid, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const int sh = 8 * (c & 3);
        const uint32_t idx = ((gq[c >> 2] >> sh) & 255) | (((qh[c >> 2] >> (sh + 2 * q)) & 3) << 8);
        const uint2 g = grid[idx], m = grid[1024 + ((sg[c >> 2] >> sh) & 255)];
        b0 = apply_mask(g.x, m.x);
        b1 = apply_mask(g.y, m.y);
        const uint32_t s = (sc[c >> 2] >> sh) & 255;
        s0 = 2 * (int) (s & 15) + 1;
        s1 = 2 * (int) (s >> 4) + 1;
        mn = 0;
    }
    __device__ __forceinline__ float fold(int si, int) const { return (h2f(d) * 0.125f) * (float) si; }
};
// IQ3_S (110 B): chunk c = 32-group c; lane q takes 8-group q: grid indices qs[8 c + 2 q], qs[8 c + 2 q + 1] with bits
// 2 q, 2 q + 1 of qh[c] as their 9th bits, sign byte signs[4 c + q], the chunk's scale 2 sc + 1 (nibble c & 1 of
// scales[c / 2]) (src/kernels4.cu:682-695; src/iq3s_dot.h:48-76 integers).
template <> struct Raw<IQ3_S> {
    static constexpr bool mins = false, g16 = false;
    uint32_t gi[4], qh[2], sg[2], sc, d;   // gi: index pairs (halfword c % 2 of gi[c / 2]); qh, sg: byte c % 4 of [c / 4]
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
#pragma unroll
        for (int c = 0; c < 8; c += 2)
            gi[c >> 1] = (uint32_t) ld_u16(blk + 2 + 8 * c + 2 * q) | ((uint32_t) ld_u16(blk + 10 + 8 * c + 2 * q) << 16);
        qh[0] = (uint32_t) ld_u16(blk + 66) | ((uint32_t) ld_u16(blk + 68) << 16);
        qh[1] = (uint32_t) ld_u16(blk + 70) | ((uint32_t) ld_u16(blk + 72) << 16);
        sg[0] = sg[1] = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) sg[c >> 2] |= (uint32_t) blk[74 + 4 * c + q] << (8 * (c & 3));
        sc = (uint32_t) ld_u16(blk + 106) | ((uint32_t) ld_u16(blk + 108) << 16);
        d = ld_u16(blk);
    }
    __device__ __forceinline__ void chunk(int c, int q, const uint2 *grid, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const uint32_t ip = gi[c >> 1] >> (16 * (c & 1)), h = qh[c >> 2] >> (8 * (c & 3));
        const uint32_t i1 = (ip & 255) | (((h >> (2 * q)) & 1) << 8), i2 = ((ip >> 8) & 255) | (((h >> (2 * q + 1)) & 1) << 8);
        const uint2 m = grid[512 + ((sg[c >> 2] >> (8 * (c & 3))) & 255)];
        b0 = apply_mask(grid[i1].x, m.x);
        b1 = apply_mask(grid[i2].x, m.y);
        s0 = 2 * (int) ((sc >> (4 * c)) & 15) + 1;
        s1 = 0; mn = 0;
    }
    __device__ __forceinline__ float fold(int si, int) const { return h2f(d) * (float) si; }
};
// Q3_K (110 B: hmask[32], qs[64] @32, scales[12] @96, d @108): chunk c = values 32 c .., hf = c >> 2, j = c & 3; lane
// values l = 8 q .. + 7: 2-bit fields 2 j of qs bytes 32 + 32 hf + l, each byte OR 0xFC where bit 4 hf + j of hmask[l]
// is clear (q - 4 as int8); 16-groups 2 c (lanes q < 2) and 2 c + 1 with their signed 6-bit scales.  Blocks are 2-byte
// aligned: ld8_2a's 12-byte reads end by byte 99.
__device__ __forceinline__ int q3k_scale(const uint32_t (&s)[3], int is) {
    auto byte = [&](int i) { return (int) ((s[i >> 2] >> (8 * (i & 3))) & 255); };
    return (((byte(is & 7) >> (4 * (is >> 3))) & 15) | (((byte(8 + (is & 3)) >> (2 * (is >> 2))) & 3) << 4)) - 32;
}
template <> struct Raw<Q3_K> {
    static constexpr bool mins = false, g16 = true;
    uint2 qv[2], hm; uint32_t sc[3], d;
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
        qv[0] = ld8_2a(blk + 32 + 8 * q);
        qv[1] = ld8_2a(blk + 64 + 8 * q);
        hm = ld8_2a(blk + 8 * q);
#pragma unroll
        for (int i = 0; i < 3; ++i) sc[i] = (uint32_t) ld_u16(blk + 96 + 4 * i) | ((uint32_t) ld_u16(blk + 98 + 4 * i) << 16);
        d = ld_u16(blk + 108);
    }
    __device__ __forceinline__ void chunk(int c, int, const uint2 *, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const int s2 = 2 * (c & 3), hb = 4 * (c >> 2) + (c & 3);
        b0 = ((qv[c >> 2].x >> s2) & 0x03030303u) | fill_fc((~hm.x >> hb) & 0x01010101u);
        b1 = ((qv[c >> 2].y >> s2) & 0x03030303u) | fill_fc((~hm.y >> hb) & 0x01010101u);
        s0 = q3k_scale(sc, 2 * c);
        s1 = q3k_scale(sc, 2 * c + 1);
        mn = 0;
    }
    __device__ __forceinline__ float fold(int si, int) const { return h2f(d) * (float) si; }
};
// IQ4_XS (136 B): chunk c = 32-group c; lane values 8 q .. + 7 are nibbles (q >> 1) of qs[16 c + 8 (q & 1) ..]
template <> struct Raw<IQ4_XS> {
    static constexpr bool mins = false, g16 = false;
    uint2 qv[8]; uint32_t dsh, sl;
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
#pragma unroll
        for (int c = 0; c < 8; ++c) qv[c] = *(const uint2 *) (blk + 8 + 16 * c + 8 * (q & 1));
        dsh = *(const uint32_t *) blk;
        sl = *(const uint32_t *) (blk + 4);
    }
    __device__ __forceinline__ void chunk(int c, int q, const uint2 *, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const int s = 4 * (q >> 1);
        b0 = kv4((qv[c].x >> s) & 0x0F0F0F0Fu);
        b1 = kv4((qv[c].y >> s) & 0x0F0F0F0Fu);
        s0 = (((sl >> (8 * (c >> 1) + 4 * (c & 1))) & 0xF) | ((((dsh >> 16) >> (2 * c)) & 3) << 4)) - 32;
        s1 = 0; mn = 0;
    }
    __device__ __forceinline__ float fold(int si, int) const { return h2f(dsh & 0xffff) * (float) si; }
};
// IQ2_XXS (66 B): chunk c = 32-group c, two words at 2 + 8 c (grid rows a byte each, then 4 x 7 sign bits and the
// 4-bit scale); lane q takes 8-group q: grid row byte q of the first word, signs bits 7 q .. of the second, the chunk's
// scale 2 sc + 1 (src/kernels4.cu:578-589; ggml's vec_dot_iq2_xxs_q8_K integers).
template <> struct Raw<IQ2_XXS> {
    static constexpr bool mins = false, g16 = false;
    uint32_t gi[2], a1[8], d;   // gi: the lane's grid row of chunk c in byte c % 4 of gi[c / 4]
    __device__ __forceinline__ void load(const uint8_t *blk, int q) {
        gi[0] = gi[1] = 0;
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const uint8_t *p = blk + 2 + 8 * c;
            a1[c] = (uint32_t) ld_u16(p + 4) | ((uint32_t) ld_u16(p + 6) << 16);
            gi[c >> 2] |= (uint32_t) p[q] << (8 * (c & 3));
        }
        d = ld_u16(blk);
    }
    __device__ __forceinline__ void chunk(int c, int q, const uint2 *grid, uint32_t &b0, uint32_t &b1, int &s0, int &s1, int &mn) const {
        const uint2 g = grid[(gi[c >> 2] >> (8 * (c & 3))) & 255], m = grid[256 + ((a1[c] >> (7 * q)) & 127)];
        b0 = apply_mask(g.x, m.x);
        b1 = apply_mask(g.y, m.y);
        s0 = 2 * (int) (a1[c] >> 28) + 1;
        s1 = 0; mn = 0;
    }
    __device__ __forceinline__ float fold(int si, int) const { return (h2f(d) * 0.125f) * (float) si; }
};

constexpr int GM_TOK = 64, GM_TILES = GM_TOK / 16, GM_ROWS = 64, GM_LD = 264;   // LDS row stride of staged activations

// Direct global -> LDS loads and the epilogue's stores, issued from inline asm so that the compiler's wait
// bookkeeping sees only the weight loads of the stream.  (Its bookkeeping treats LDS loads, register loads and
// stores as possibly completing out of order and would then wait for all of them at every step.)  Vector memory
// operations of a wave complete in issue order, so waiting for a step's weight registers also covers every DMA
// issued before them.  M0 holds the LDS address of a DMA; it is saved and restored around it.
__device__ __forceinline__ void store_f32(float *g, float v) { asm volatile("global_store_dword %0, %1, off" ::"v"(g), "v"(v) : "memory"); }

// ------------------------------------------------------------------ the grouped GEMM stream
// A block of W waves owns 16 W weight rows -- gate/up: 8 W gate rows (the first half of the waves) and the up rows of the
// same outputs; down: 16 W rows -- and the work items of its slot (up to 64 tokens of an expert each).  Its steps, (item,
// 256-value span b) in order, form one stream.  Every operand reaches LDS by DMA: a stage holds the waves' 16-row weight
// tiles of span b (each one contiguous run of the tiled layout) and the item's 64 activation rows of span b.  D stages
// rotate: step s computes from stage s % D while the DMAs of steps s + 1 .. s + D - 1 are in flight.
//
// Waits are explicit.  Each wave issues the same L DMA instructions per step, and loads complete in issue order, so
// "vmcnt <= (D - 2) L" at the end of step s - 1, before step s + D - 1 is issued, means this wave's step-s DMAs have
// landed; a barrier then makes the whole stage visible and frees stage (s - 1) % D for the next issue.  Nothing in the
// stream is a compiler-visible global load, so the compiler adds no waits of its own.  The epilogue's stores are not
// counted: a store still in flight only makes a later wait stricter (loads cannot overtake the loads before them).
// Geometry of the stream kernel for weight type T, W waves (8 or 16) per block and B blocks per CU (1 or 2): the
// stages get what is left of the CU's 160 KB LDS after the item tables.
//
// Types with Q8_0 activations (A0): their 34-byte blocks are 2-byte aligned, and an LDS read off its natural alignment
// costs about 60 cycles of the CU's LDS pipe, so a span's rows (272 bytes each) land as they are in a buffer of their own
// and are copied into an aligned one (Relay) a step before they are used.  Two weight stages, two raw and two aligned
// activation buffers: step s computes from weights s and aligned rows s while weights s + 1 and raw rows s + 2 are in
// flight and rows s + 1 are copied; every wait is for all of a wave's DMAs.  509 tokens, 288 experts, d 4096, ff 1536,
// top-8 in IQ4_NL: the layer call 2270 us with both operands staged through registers (k_gemm_nl: one step ahead, 4
// waves, a 7-operation codebook and a 3-operation fold) -> 1004 us; bound by VALU issue (71 and 75 % of the cycles of
// gate/up and down).  8 waves of 32 rows instead of 16 of 16 share each activation read but hide less latency: 1196
// against 1115 us at the time.
template <int T, int W, int B> struct G5 {
    static constexpr bool A0 = vec_dot_type(T) == Q8_0;
    static constexpr int WAVES = W, THREADS = 64 * W, ROWS = 16 * W;   // a wave owns 16 weight rows
    static constexpr int HALF = W / 2;                          // gate/up: waves 0 .. HALF - 1 in gate, the rest in up
    static constexpr int TPW = GM_TOK / W;                      // activation rows each wave fetches per step
    static constexpr int AROW = A0 ? 8 * Q8_0_BYTES : Q8K_BYTES;   // activation bytes of a row and span
    static constexpr int NA = A0 ? (TPW * 17 + 63) / 64 : TPW / 4;  // their DMA instructions (1 KB; A0: 17 16-byte pieces a row)
    static constexpr int PER = 1024 / THREADS;                  // expert groups per thread in the item scan
    static constexpr int ITEMS = B == 1 ? 16 : 8;               // items per segment (their tables live in LDS)
    static constexpr int LDS_STAGES = B == 1 ? 150 * 1024 : 72 * 1024;
    static constexpr int BB = span_bytes(T);                    // weight bytes per row and 256 values
    static constexpr int TB = 16 * BB;                          // one wave's 16-row tile of a span
    static constexpr int WB = W * TB;                           // weights of a stage
    static constexpr int AB = A0 ? 0 : GM_TOK * 256;            // activation values of a stage (64 rows of 256)
    static constexpr int SB = WB + AB + (A0 ? 0 : 4 * GM_TOK);  // + the rows' Q8_K d
    static constexpr int RAW = GM_TOK * 8 * Q8_0_BYTES;         // A0: a raw buffer
    static constexpr int AL = GM_TOK * 256 + 8 * GM_TOK * 2;    // A0: an aligned buffer: values, then fp16 d [block][token]
    static constexpr int D = A0 ? 2 : 4 * SB <= LDS_STAGES ? 4 : 3 * SB <= LDS_STAGES ? 3 : 2;   // stages
    static constexpr int SMEM = D * SB + (A0 ? 2 * RAW + 2 * AL : 0);
    static constexpr int N4 = TB / 1024, NR = TB - 1024 * N4, N1 = (NR + 255) / 256;   // tile DMAs: 1 KB, then 256 B
    static constexpr int L = N4 + N1 + NA + 1;                  // DMA instructions per wave and step
    static constexpr int XCH = WB + AB;                         // bytes of a consumed stage the epilogue's exchange takes
    static_assert(W == 8 || W == 16, "8 or 16 waves");
    static_assert(TB % 16 == 0 && NR % 4 == 0, "DMA granules");
    static_assert(WB % 256 == 0 && SB % 256 == 0 && RAW % 256 == 0 && AL % 256 == 0, "activation rows at multiples of 256 (lds_at)");
    static_assert(SMEM <= LDS_STAGES, "stages fit");
    static_assert((D - 2) * L <= 63, "vmcnt range");
};
// Q4_K and IQ4_XS gate/up (whose steps fit 128 registers): two blocks of 8 waves per CU, each block's stream running
// independently of the other's; IQ2_XS, and Q6_K and IQ4_XS down: one block of 16 waves (256 weight rows share every
// activation read; the steps fit 128 registers); the rest: one block of 8 waves (up to 256 registers, deeper rings).
// IQ4_XS, the 1000-token layer call on one card: 1185 us with 16 waves for both, 1125 as here, 1136 with 2 x 8 waves for
// both; IQ2_XS: 3511 us with 16 waves, 3508 with 2 x 8.  Small grids take 8 waves instead of 16: launch_k_gemm_fit.
template <int T, bool GU> constexpr int g5_blocks() { return GU && (T == Q4_K || T == IQ4_XS) ? 2 : 1; }
template <int T, bool GU> constexpr int g5_waves() { return T == IQ2_XS || (!GU && (T == Q6_K || T == IQ4_XS)) ? 16 : 8; }

__device__ __forceinline__ v4i mfma64(v4i a, v4i b, v4i c) { return __builtin_amdgcn_mfma_i32_16x16x64_i8(a, b, c, 0, 0, 0); }
// Operand reads of the activation rows.  Row t (256 bytes, at a multiple of 256) holds its 16-byte pieces at piece ^ (t %
// 16), so the piece p ^ k of a lane's row, p its first one and k compile-time, sits at the first one's address ^ 16 k: one
// operation a read where piece, row and stage take three.
template <typename V> __device__ __forceinline__ V lds_at(uint32_t addr) { return *(const __attribute__((address_space(3))) V *) (uintptr_t) addr; }
typedef unsigned short v2u16 __attribute__((ext_vector_type(2)));
// byte `b` of x in both 16-bit halves / in all four bytes
__device__ __forceinline__ uint32_t bcast16(uint32_t x, int b) { return __builtin_amdgcn_perm(0u, x, 0x0C000C00u | (uint32_t) b | ((uint32_t) b << 16)); }
__device__ __forceinline__ uint32_t bcast8(uint32_t x, int b) { return __builtin_amdgcn_perm(0u, x, 0x01010101u * (uint32_t) b); }
// four bytes of q (each < 16) times the small factor f (< 8) held in both 16-bit halves: products < 128 stay in their bytes
__device__ __forceinline__ int mul_bytes(uint32_t q, uint32_t f) {
    const v2u16 r = __builtin_bit_cast(v2u16, q) * __builtin_bit_cast(v2u16, f);
    return (int) __builtin_bit_cast(uint32_t, r);
}

// Q4_K step on the 16x16x64 MFMA.  The dot products are exact integers, so the K order inside an MFMA is free: in MFMA
// j (values 64 j .. 64 j + 63 of the span) lane quarter q holds values 64 j + 16 q .. + 15, one contiguous 16-byte
// piece of the token row (A: a single LDS read straight into the operand registers) and, for B, the same values of the
// weight row: the low nibbles of qs[32 j + 16 q ..] (chunk 2j) for q < 2, the high nibbles of qs[32 j + 16 (q - 2) ..]
// (chunk 2j + 1) for q >= 2.  Every lane's 16 values lie in one chunk, so its 6-bit scale s = 8 a + b (a, b < 8) is
// applied inside B: D1 = sum a_c dot_c and D2 = sum b_c dot_c (a q, b q < 128 fit int8), sum_c s_c dot_c = 8 D1 + D2
// exactly; a third MFMA against the chunk mins gives sum_c m_c sum(x_c).
// Token tiles 0 .. NT - 1 (compile-time: straight-line code, accumulators only for the tiles present)
// The lane's constants (quarter, row, offsets, selectors) are derived in the step from a lane id the compiler cannot
// hoist: recomputing them costs a few instructions, keeping them live across the stream would cost registers.
__device__ __forceinline__ int lane_id_here() {
    int l;
    asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(l));
    return l;
}
template <int NT, bool FIRST>
__device__ __forceinline__ void step_q4k(const uint8_t *wl0, const int8_t *as, const float *yd, float (&acc)[GM_TILES][4]) {
    // the tiles past NT hold nothing this item reads (a tile count is fixed for an item, and an item's first span
    // writes its tiles without reading them): marking them redefined frees their registers in this step
#pragma unroll
    for (int t = NT; t < GM_TILES; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) asm volatile("" : "=v"(acc[t][v]));
    const int lid = lane_id_here(), q = lid >> 4, rr = lid & 15;
    const uint8_t *wl = wl0 + rr * block_bytes(Q4_K);
    const uint4 hd = *(const uint4 *) wl;   // d | dmin, scales[12]
    const uint32_t s_lo = hd.y & 0x3F3F3F3Fu, m_lo = hd.z & 0x3F3F3F3Fu;   // chunks 0..3, one per byte
    const uint32_t s_hi = (hd.w & 0x0F0F0F0Fu) | ((hd.y >> 2) & 0x30303030u);         // chunks 4..7
    const uint32_t m_hi = ((hd.w >> 4) & 0x0F0F0F0Fu) | ((hd.z >> 2) & 0x30303030u);
    const int hs = q >> 1;                   // 1: this lane takes the odd chunk of each pair (the high nibbles)
    const uint32_t nsh = 4u * (uint32_t) hs;
    const uint32_t a0 = lds_addr(as) + rr * 256 + 16 * (q ^ rr);   // token row rr of tile 0, piece q
    const v4i z = {0, 0, 0, 0};
    v4i d1[NT], d2[NT], dm[NT];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint4 w = *(const uint4 *) (wl + 16 + 32 * j + 16 * (q & 1));
        const uint32_t sp = j < 2 ? s_lo : s_hi, mp = j < 2 ? m_lo : m_hi;
        const int c = ((2 * j) & 3) + hs;    // this lane's chunk, as a byte of sp / mp
        const uint32_t a = bcast16((sp >> 3) & 0x07070707u, c), b = bcast16(sp & 0x07070707u, c);
        const uint32_t n0 = (w.x >> nsh) & 0x0F0F0F0Fu, n1 = (w.y >> nsh) & 0x0F0F0F0Fu;
        const uint32_t n2 = (w.z >> nsh) & 0x0F0F0F0Fu, n3 = (w.w >> nsh) & 0x0F0F0F0Fu;
        const v4i B1 = {mul_bytes(n0, a), mul_bytes(n1, a), mul_bytes(n2, a), mul_bytes(n3, a)};
        const v4i B2 = {mul_bytes(n0, b), mul_bytes(n1, b), mul_bytes(n2, b), mul_bytes(n3, b)};
        const int mm = (int) bcast8(mp, c);
        const v4i Bm = {mm, mm, mm, mm};
        const uint32_t aj = a0 ^ (64 * j);   // piece 4 j + q
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const v4i A = lds_at<v4i>(aj + t * 16 * 256);
            d1[t] = mfma64(A, B1, j ? d1[t] : z);
            d2[t] = mfma64(A, B2, j ? d2[t] : z);
            dm[t] = mfma64(A, Bm, j ? dm[t] : z);
            asm volatile("");   // a scheduling-region boundary: operands are not hoisted across tiles (register pressure)
        }
    }
    const float d = h2f(hd.x & 0xffff), dmin = h2f(hd.x >> 16);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int si = (d1[t][v] << 3) + d2[t][v];
            acc[t][v] = __builtin_fmaf(yd[t * 16 + 4 * q + v], __builtin_fmaf(d, (float) si, -(dmin * (float) dm[t][v])), FIRST ? 0.0f : acc[t][v]);
        }
    }
}

// 16 bytes at p, which is 2-byte aligned (sb = p & 3 is 0 or 2, the same for every call of a lane): five dwords from
// p - sb, joined; reads at most p + 18
__device__ __forceinline__ uint4 ld16_u2(const uint8_t *p, uint32_t sb) {
    const uint32_t *w = (const uint32_t *) (p - sb);
    const uint32_t d0 = w[0], d1 = w[1], d2 = w[2], d3 = w[3], d4 = w[4];
    return make_uint4(__builtin_amdgcn_alignbyte(d1, d0, sb), __builtin_amdgcn_alignbyte(d2, d1, sb),
                      __builtin_amdgcn_alignbyte(d3, d2, sb), __builtin_amdgcn_alignbyte(d4, d3, sb));
}
typedef short v2i16 __attribute__((ext_vector_type(2)));

// Q6_K step on the 16x16x64 MFMA.  In MFMA j (values 64 j .. + 63 of the span) lane quarter q holds values
// 64 j + 16 q .. + 15, which are exactly scale group g = 4 j + q: A is one contiguous 16-byte piece of the token row,
// B carries the group's scale, B = sc_g (q6 - 32) in [-4064, 4096], as two int8 planes B = 64 H + L (H = B >> 6 in
// [-64, 64], L = B & 63): D_H = X.H and D_L = X.L give sum_g sc_g dot_g = 64 D_H + D_L exactly.  The lane's values sit
// in ql[64 (j / 2) + 16 q ..] (nibble j % 2) and qh[32 (j / 2) + 16 (q % 2) ..] (bits 4 (j % 2) + 2 (q / 2)); rows of
// the 210-byte blocks are 2-byte aligned in LDS, so 16-byte reads go through ld16_u2.
template <int NT, bool FIRST>
__device__ __forceinline__ void step_q6k(const uint8_t *wt0, const int8_t *as, const float *yd, float (&acc)[GM_TILES][4]) {
    // the tiles past NT hold nothing this item reads (a tile count is fixed for an item, and an item's first span
    // writes its tiles without reading them): marking them redefined frees their registers in this step
#pragma unroll
    for (int t = NT; t < GM_TILES; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) asm volatile("" : "=v"(acc[t][v]));
    const int lid = lane_id_here(), q = lid >> 4, rr = lid & 15;
    const uint8_t *blk = wt0 + rr * block_bytes(Q6_K);
    const uint32_t sb = 2u * (uint32_t) (rr & 1);   // the tile starts dword-aligned; a 210-byte row shifts by 2
    const uint4 scq = ld16_u2(blk + 192, sb);       // the 16 group scales (int8)
    const float d = h2f(ld_u16(blk + 208));
    const uint32_t a0 = lds_addr(as) + rr * 256 + 16 * (q ^ rr);   // token row rr of tile 0, piece q
    const v4i z = {0, 0, 0, 0};
    v4i dh[NT], dl[NT];
    uint4 ql, qh;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        if ((j & 1) == 0) {
            ql = ld16_u2(blk + 64 * (j >> 1) + 16 * q, sb);
            qh = ld16_u2(blk + 128 + 32 * (j >> 1) + 16 * (q & 1), sb);
        }
        const uint32_t scw = j == 0 ? scq.x : j == 1 ? scq.y : j == 2 ? scq.z : scq.w;
        const int sc = __builtin_amdgcn_sbfe((int) scw, 8 * q, 8);   // scale of group 4 j + q
        const uint32_t sc16 = ((uint32_t) sc & 0xffffu) * 0x10001u, off16 = ((uint32_t) (-32 * sc) & 0xffffu) * 0x10001u;
        const uint32_t hsh = 4u * (uint32_t) (j & 1) + 2u * (uint32_t) (q >> 1);
        const uint32_t qlw[4] = {ql.x, ql.y, ql.z, ql.w}, qhw[4] = {qh.x, qh.y, qh.z, qh.w};
        int H[4], L[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const uint32_t nib = ((j & 1) ? qlw[i] >> 4 : qlw[i]) & 0x0F0F0F0Fu;
            const uint32_t qv = nib | (((qhw[i] >> hsh) & 0x03030303u) << 4);   // four 6-bit values, one per byte
            // values 0, 1 and 2, 3 in 16-bit lanes: B = q sc - 32 sc, exact in 16 bits
            const v2u16 e = __builtin_bit_cast(v2u16, __builtin_amdgcn_perm(0u, qv, 0x0C010C00u));
            const v2u16 o = __builtin_bit_cast(v2u16, __builtin_amdgcn_perm(0u, qv, 0x0C030C02u));
            const v2u16 s2 = __builtin_bit_cast(v2u16, sc16), c2 = __builtin_bit_cast(v2u16, off16);
            const v2u16 be = e * s2 + c2, bo = o * s2 + c2;
            const uint32_t ube = __builtin_bit_cast(uint32_t, be), ubo = __builtin_bit_cast(uint32_t, bo);
            L[i] = (int) (__builtin_amdgcn_perm(ubo, ube, 0x06040200u) & 0x3F3F3F3Fu);
            const v2i16 he = __builtin_bit_cast(v2i16, be) >> (short) 6, ho = __builtin_bit_cast(v2i16, bo) >> (short) 6;
            H[i] = (int) __builtin_amdgcn_perm(__builtin_bit_cast(uint32_t, ho), __builtin_bit_cast(uint32_t, he), 0x06040200u);
        }
        const v4i Bh = {H[0], H[1], H[2], H[3]}, Bl = {L[0], L[1], L[2], L[3]};
        const uint32_t aj = a0 ^ (64 * j);   // piece 4 j + q
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const v4i A = lds_at<v4i>(aj + t * 16 * 256);
            dh[t] = mfma64(A, Bh, j ? dh[t] : z);
            dl[t] = mfma64(A, Bl, j ? dl[t] : z);
            asm volatile("");   // a scheduling-region boundary: operands are not hoisted across tiles (register pressure)
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int si = (dh[t][v] << 6) + dl[t][v];
            acc[t][v] = __builtin_fmaf(yd[t * 16 + 4 * q + v], d * (float) si, FIRST ? 0.0f : acc[t][v]);
        }
    }
    asm volatile("");   // keeps the tile-count variants from being merged (which moved the accumulators to memory)
}

// IQ2_XS step on the 16x16x64 MFMA.  Lane quarter q's 16 values of MFMA j (64 j + 16 q ..) are scale group 4 j + q: the
// two 8-groups of the 32-bit word qs[8 j + 2 q], qs[8 j + 2 q + 1] (9 bits of grid row, 7 of sign index each), scale
// s = 2 nibble + 1 in 1 .. 31.  The codebook has three levels, 8, 25 and 43, so a value of the group is one of the six v =
// +-s level, |v| <= 1333, and B = v splits into two int8 planes, v = 16 P + Q with |P| <= 83 and -8 <= Q < 8: sum_g s_g
// dot_g = 16 X.P + X.Q exactly.  A plane's six bytes per scale come from a 16-entry LDS table (one read without bank
// conflicts; multiplied and negated in registers they cost seven more operations a group), and v_perm picks four at a
// time: the selector table gives each 8-group's levels and signs as nibbles (iq2_sel_table: entry g the levels of row g,
// entry 512 + i the signs of sign index i in bit 2 of each nibble; value v of the 8-group in byte v % 4, nibble v / 4),
// OR-ed into the selectors.  Both tables lie in the first 64 KB of LDS, so that a lookup's base is the instruction's
// offset and not an addition.  It replaced the generic step (two masked 16x16x32 MFMAs a 32-value chunk, eight 24-bit
// multiply-adds an output column, 8-byte codebook and sign rows): the 2048-token, 384-expert layer call of d 7168, ff
// 2048, top-6: 6.29 -> 3.51 ms, and 3473 -> 3294 us with the plane table, the 16 : 1 split and the offsets (55 of 290
// operations a wave and step less).  Of the cycles VALU issue takes 64 %, the LDS pipe 58 %, the matrix cores 22 %.
constexpr int IQ2_SEL = 512 + 128, IQ2_TAB = 4 * IQ2_SEL + 16 * 16;   // selectors (dwords); bytes with the plane table
static_assert(IQ2_TAB % 256 == 0, "the stages behind it stay at multiples of 256");
__device__ __forceinline__ void iq2_sel_table(uint32_t *sel) {
    for (int i = threadIdx.x; i < IQ2_SEL; i += blockDim.x) {
        uint32_t v = 0, c = i < 512 ? c_iq2xs_code[i] : ksign((uint32_t) i - 512);
#pragma unroll
        for (int j = 0; j < 8; ++j) {
            const uint32_t n = i < 512 ? c % 3 : (c & 1) << 2;
            c = i < 512 ? c / 3 : c >> 1;
            v |= n << (8 * (j & 3) + 4 * (j >> 2));
        }
        sel[i] = v;
    }
    if (const int i = threadIdx.x; i < 16) {   // plane bytes of scale nibble i: P of the levels, of their negatives, Q likewise
        uint32_t e[4] = {0, 0, 0, 0};
#pragma unroll
        for (int n = 0; n < 6; ++n) {
            const int l = n % 3, v = (n < 3 ? 1 : -1) * (2 * i + 1) * (l == 0 ? 8 : l == 1 ? 25 : 43), P = (v + 8) >> 4;
            e[n / 3] |= (uint32_t) (P & 255) << (8 * l);
            e[2 + n / 3] |= (uint32_t) ((v - 16 * P) & 255) << (8 * l);
        }
        ((uint4 *) (sel + IQ2_SEL))[i] = make_uint4(e[0], e[1], e[2], e[3]);
    }
}
// 4 bytes at p, which is 2-byte aligned (sb = p & 3 is 0 or 2): two aligned dwords from p - sb, joined.  (One unaligned
// LDS read costs about 60 cycles of the CU's LDS pipe: SQ_LDS_UNALIGNED_STALL.)
__device__ __forceinline__ uint32_t ld4_u2(const uint8_t *p, uint32_t sb) {
    const uint32_t *w = (const uint32_t *) (p - sb);
    return __builtin_amdgcn_alignbyte(w[1], w[0], sb);
}
template <int NT, bool FIRST>
__device__ __forceinline__ void step_iq2xs(const uint8_t *wt0, const int8_t *as, const float *yd, const uint32_t *sel, float (&acc)[GM_TILES][4]) {
    // the tiles past NT hold nothing this item reads: marking them redefined frees their registers (as in step_q4k)
#pragma unroll
    for (int t = NT; t < GM_TILES; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) asm volatile("" : "=v"(acc[t][v]));
    const int lid = lane_id_here(), q = lid >> 4, rr = lid & 15;
    const uint8_t *blk = wt0 + rr * block_bytes(IQ2_XS);
    const uint32_t al = 2u * (uint32_t) (~rr & 1);   // the tile starts dword-aligned: qs and scales of even rows are 2 mod 4
    uint32_t w[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) w[j] = ld4_u2(blk + 2 + 16 * j + 4 * q, al);
    const uint32_t sc0 = ld4_u2(blk + 66, al), sc1 = ld4_u2(blk + 70, al);   // group 4 j + q: nibble 4 (j & 1) + q
    const float d = h2f(ld_u16(blk)) * 0.125f;
    const uint32_t a0 = lds_addr(as) + rr * 256 + 16 * (q ^ rr);   // token row rr of tile 0, piece q
    const v4i z = {0, 0, 0, 0};
    v4i dp[NT], dq[NT];
    uint32_t ga[4], sa[4], gb[4], sb[4];   // every lookup of the step goes out before the first MFMA
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        ga[j] = sel[__builtin_amdgcn_ubfe(w[j], 0, 9)];
        sa[j] = sel[512 + __builtin_amdgcn_ubfe(w[j], 9, 7)];
        gb[j] = sel[__builtin_amdgcn_ubfe(w[j], 16, 9)];
        sb[j] = sel[512 + (w[j] >> 25)];
    }
    auto planes = [&](int j) { return ((const uint4 *) (sel + IQ2_SEL))[__builtin_amdgcn_ubfe(j < 2 ? sc0 : sc1, 4 * q + 16 * (j & 1), 4)]; };
    uint4 pl = planes(0);
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        const uint32_t ca = ga[j] | sa[j], cb = gb[j] | sb[j];
        const uint32_t Pp = pl.x, Pn = pl.y, Qp = pl.z, Qn = pl.w;
        if (j < 3) pl = planes(j + 1);
        const uint32_t i0 = ca & 0x07070707u, i1 = (ca >> 4) & 0x07070707u, i2 = cb & 0x07070707u, i3 = (cb >> 4) & 0x07070707u;
        const v4i BP = {(int) __builtin_amdgcn_perm(Pn, Pp, i0), (int) __builtin_amdgcn_perm(Pn, Pp, i1),
                        (int) __builtin_amdgcn_perm(Pn, Pp, i2), (int) __builtin_amdgcn_perm(Pn, Pp, i3)};
        const v4i BQ = {(int) __builtin_amdgcn_perm(Qn, Qp, i0), (int) __builtin_amdgcn_perm(Qn, Qp, i1),
                        (int) __builtin_amdgcn_perm(Qn, Qp, i2), (int) __builtin_amdgcn_perm(Qn, Qp, i3)};
        const uint32_t aj = a0 ^ (64 * j);   // piece 4 j + q
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const v4i A = lds_at<v4i>(aj + t * 16 * 256);
            dp[t] = mfma64(A, BP, j ? dp[t] : z);
            dq[t] = mfma64(A, BQ, j ? dq[t] : z);
            asm volatile("");   // a scheduling-region boundary: operands are not hoisted across tiles (register pressure)
        }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t) {
#pragma unroll
        for (int v = 0; v < 4; ++v) {
            const int si = (dp[t][v] << 4) + dq[t][v];
            acc[t][v] = __builtin_fmaf(yd[t * 16 + 4 * q + v], d * (float) si, FIRST ? 0.0f : acc[t][v]);
        }
    }
    asm volatile("");   // keeps the tile-count variants from being merged
}

// The step of the other types: per 32-value chunk a 16x16x32 MFMA a tile (16-value scale groups: two, each with the other
// group's lanes of B zeroed), si += scale D with 24-bit multiply-adds, the mins chained in an MFMA against the chunk's min.
// Straight-line code per tile count; with one or two tiles the MFMAs of chunk c + 1 go out before chunk c is scaled.  (A
// run-time tile loop took its branches at every chunk; without the empty asm on each sum the compiler regrouped the
// chunks' sums and spilled.)  IQ4_XS, 1000 tokens, 288 experts, d 4096, ff 1536, top-8: the layer call 1252 -> 1125 us on
// one card, with the lds_at addresses and the geometry of g5_waves; bound by VALU issue (82 % of the cycles in gate/up).
// One tile of a type with 16-value groups (G1) leaves most of the 256 registers free and is bound by latency: its operand
// reads go out together and its chunks are scheduled as one piece; with one chunk in flight at a time a layer call of 37
// tokens (d 2048, 64 experts, ff 768, top-8) took 130.5 us in Q2_K, 133 in Q3_K and 141 in IQ2_S, here 125, 124 and 131
// (the run-time tile loop: 120, 127 and 136).
template <int T, int NT, bool FIRST>
__device__ __forceinline__ void step_gen(const uint8_t *wt, const uint2 *grid, const int8_t *as, const float *yd, float (&acc)[GM_TILES][4]) {
#pragma unroll
    for (int t = NT; t < GM_TILES; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) asm volatile("" : "=v"(acc[t][v]));
    constexpr bool G = Raw<T>::g16, MN = Raw<T>::mins, G1 = G && NT == 1;
    const int lid = G ? (int) (threadIdx.x & 63) : lane_id_here(), q = lid >> 4, rr = lid & 15;
    Raw<T> w;
    w.load(wt + rr * span_bytes(T), q);
    const uint32_t a0 = lds_addr(as) + rr * 256 + 16 * ((q >> 1) ^ rr) + 8 * (q & 1);   // row rr of tile 0, chunk 0
    const v4i z = {0, 0, 0, 0};
    // the MFMAs of chunk c + 1 ahead of chunk c's scaling: not for two tiles of 16-value groups (512 tokens in IQ2_S 241
    // instead of 238 us) nor for one whose values come from a table in LDS (37 tokens in IQ2_S 139 instead of 131)
    constexpr int AHEAD = G ? G1 && !iq2_type(T) : NT <= 2;
    v4i D[1 + AHEAD][NT], E[1 + AHEAD][NT], sm[NT];
    int s0[1 + AHEAD], s1[1 + AHEAD], si[NT][4];
    constexpr int UP = G1 ? 8 : 1;   // chunks whose operands are read together
    long Ac[UP][NT];
    auto read = [&](int c) {
#pragma unroll
        for (int t = 0; t < NT; ++t) Ac[c % UP][t] = lds_at<long>((a0 ^ (32 * c)) + t * 16 * 256);
    };
    if constexpr (G1) {
#pragma unroll
        for (int c = 0; c < 8; ++c) read(c);
    }
    auto mul = [&](int c) {
        const int s = AHEAD ? c & 1 : 0;
        if constexpr (!G1) read(c);
        const long (&A)[NT] = Ac[c % UP];
        uint32_t b0, b1;
        int mn;
        w.chunk(c, q, grid, b0, b1, s0[s], s1[s], mn);
        const uint32_t mb = __builtin_amdgcn_perm(0u, (uint32_t) mn, 0u);   // the min in all four bytes
        const bool lo = q < 2;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            if constexpr (G) {
                D[s][t] = mfma16(A[t], mk_long(lo ? b0 : 0u, lo ? b1 : 0u), z);
                E[s][t] = mfma16(A[t], mk_long(lo ? 0u : b0, lo ? 0u : b1), z);
            } else {
                D[s][t] = mfma16(A[t], mk_long(b0, b1), z);
            }
            if constexpr (MN) sm[t] = mfma16(A[t], mk_long(mb, mb), c ? sm[t] : z);
        }
    };
    auto scale = [&](int c) {
        const int s = AHEAD ? c & 1 : 0;
#pragma unroll
        for (int t = 0; t < NT; ++t)
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                int x = c ? si[t][v] : 0;
                x += __mul24(s0[s], D[s][t][v]);
                if constexpr (G) x += __mul24(s1[s], E[s][t][v]);
                if constexpr (!G1) asm volatile("" : "+v"(x));   // the chain of chunks is not regrouped (which kept every chunk's D live)
                si[t][v] = x;
            }
    };
    if constexpr (AHEAD) mul(0);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        if constexpr (AHEAD) { if (c < 7) mul(c + 1); } else mul(c);
        scale(c);
        if constexpr (!G1) asm volatile("");   // a scheduling-region boundary per chunk (register pressure)
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v)
            acc[t][v] = __builtin_fmaf(yd[t * 16 + 4 * q + v], w.fold(si[t][v], MN ? sm[t][v] : 0), FIRST ? 0.0f : acc[t][v]);
    asm volatile("");   // keeps the tile-count variants from being merged
}

// ------------------------------------------------------------------ Q8_0 activations
// One 256-value span of the staged rows from the raw buffer (row t at 272 t: blocks of fp16 d and 32 int8) into the
// aligned one: block c of token t in 16-byte pieces 2 c and 2 c + 1 of row t, a piece stored at piece ^ (t % 16), the
// block's dwords reordered so that lane quarter q's 8 values of the MFMA (4 q .. + 3 and 16 + 4 q .. + 3, the two nibbles
// of weight bytes 4 q .. + 3) are 8 contiguous bytes; d at [c][t].  A wave takes block c = wave % 8 of 32 (8 waves: 64)
// tokens: 16 tokens x 4 quarters a pass, the block's alignment uniform over the wave.  Raw reads end 4 bytes past the raw
// row at most (inside LDS; those bytes are shifted out).
template <int W> struct Relay {
    static constexpr int N = GM_TOK / W / 2;
    uint32_t w[N][4];
    uint16_t d;
    static __device__ __forceinline__ int tok0(int wave) { return W == 16 ? 32 * (wave >> 3) : 0; }
    __device__ __forceinline__ void load(const uint8_t *raw, int wave) {
        const int lid = lane_id_here(), c = wave & 7, t0 = tok0(wave);
        const uint32_t sb = 2u * (uint32_t) (~c & 1);   // 34 c + 2 is 2 mod 4 for even c
        const uint8_t *p = raw + (t0 + (lid >> 2)) * 272 + 34 * c + 2 + 4 * (lid & 3) - sb;
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const uint32_t *v = (const uint32_t *) (p + 16 * 272 * i);
            w[i][0] = v[0]; w[i][1] = v[1]; w[i][2] = v[4]; w[i][3] = v[5];
        }
        d = ld_u16(raw + (t0 + (W == 16 ? lid & 31 : lid)) * 272 + 34 * c);
    }
    __device__ __forceinline__ void store(uint8_t *al, int wave) const {
        const int lid = lane_id_here(), q = lid & 3, c = wave & 7, t0 = tok0(wave), t = t0 + (lid >> 2);
        const uint32_t sb = 2u * (uint32_t) (~c & 1);
        uint8_t *p = al + t * 256 + 16 * ((2 * c + (q >> 1)) ^ (t & 15)) + 8 * (q & 1);
#pragma unroll
        for (int i = 0; i < N; ++i)
            *(uint2 *) (p + 16 * 256 * i) = make_uint2(__builtin_amdgcn_alignbyte(w[i][1], w[i][0], sb), __builtin_amdgcn_alignbyte(w[i][3], w[i][2], sb));
        *(uint16_t *) (al + GM_TOK * 256 + 2 * (GM_TOK * c + t0 + (W == 16 ? lid & 31 : lid))) = d;
    }
};

// A weight row's span (in LDS) as lane quarter q needs it: per block c the B words of values 4 q .. + 3 and 16 + 4 q ..,
// and the block's scale.  Block offsets are compile-time, so every read is a dword at its natural alignment (two joined
// where the block's quants are not).  magic: the fold's product d D may be taken as fma(D + 1.5 2^23, d, -1.5 2^23 d) (see
// step_a0), which needs d with at most 12 significant bits (fp16).
template <int T> struct A0Row;
__device__ __forceinline__ uint32_t ld4_off(const uint8_t *p, int off) {   // off & 3: compile-time after unrolling
    const uint32_t *w = (const uint32_t *) (p - (off & 3));
    return (off & 3) ? __builtin_amdgcn_alignbyte(w[1], w[0], (uint32_t) (off & 3)) : w[0];
}
template <> struct A0Row<IQ4_NL> {
    static constexpr bool magic = true;
    uint32_t w[8];
    __device__ __forceinline__ void load(const uint8_t *row, int q, float (&d)[8]) {
#pragma unroll
        for (int c = 0; c < 8; ++c) { w[c] = ld4_off(row + 18 * c + 2 + 4 * q, 18 * c + 2); d[c] = h2f(ld_u16(row + 18 * c)); }
    }
    __device__ __forceinline__ long b(int c, int) const { return mk_long(kv4(w[c] & 0x0F0F0F0Fu), kv4((w[c] >> 4) & 0x0F0F0F0Fu)); }
};
template <> struct A0Row<MXFP4> {
    static constexpr bool magic = false;   // d up to 2^127
    uint32_t w[8];
    __device__ __forceinline__ void load(const uint8_t *row, int q, float (&d)[8]) {
#pragma unroll
        for (int c = 0; c < 8; ++c) { w[c] = ld4_off(row + 17 * c + 1 + 4 * q, 17 * c + 1); d[c] = e8m0_half(row[17 * c]); }
    }
    __device__ __forceinline__ long b(int c, int) const { return mk_long(kvfp4(w[c] & 0x0F0F0F0Fu), kvfp4((w[c] >> 4) & 0x0F0F0F0Fu)); }
};
template <> struct A0Row<Q8_0> {
    static constexpr bool magic = true;
    uint32_t lo[8], hi[8];
    __device__ __forceinline__ void load(const uint8_t *row, int q, float (&d)[8]) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            lo[c] = ld4_off(row + 34 * c + 2 + 4 * q, 34 * c + 2);
            hi[c] = ld4_off(row + 34 * c + 18 + 4 * q, 34 * c + 18);
            d[c] = h2f(ld_u16(row + 34 * c));
        }
    }
    __device__ __forceinline__ long b(int c, int) const { return mk_long(lo[c], hi[c]); }
};
template <> struct A0Row<Q5_0> {
    static constexpr bool magic = true;
    uint32_t w[8], h[8];   // h: the fifth bits of values 0..15 and 16..31
    __device__ __forceinline__ void load(const uint8_t *row, int q, float (&d)[8]) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            w[c] = ld4_off(row + 22 * c + 6 + 4 * q, 22 * c + 6);
            h[c] = (uint32_t) ld_u16(row + 22 * c + 2) | ((uint32_t) ld_u16(row + 22 * c + 4) << 16);
            d[c] = h2f(ld_u16(row + 22 * c));
        }
    }
    __device__ __forceinline__ long b(int c, int q) const {
        const uint32_t nh = ~h[c] >> (4 * q);
        return mk_long((w[c] & 0x0F0F0F0Fu) | fill_f0(nh & 15), ((w[c] >> 4) & 0x0F0F0F0Fu) | fill_f0((nh >> 16) & 15));
    }
};
template <> struct A0Row<Q5_1> {
    static constexpr bool magic = false;
    uint32_t w[8], h[8], dm[8];
    __device__ __forceinline__ void load(const uint8_t *row, int q, float (&d)[8]) {
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            w[c] = *(const uint32_t *) (row + 24 * c + 8 + 4 * q);
            h[c] = *(const uint32_t *) (row + 24 * c + 4);
            dm[c] = *(const uint32_t *) (row + 24 * c);
            d[c] = h2f(dm[c] & 0xffff);
        }
    }
    __device__ __forceinline__ long b(int c, int q) const {
        const uint32_t hh = h[c] >> (4 * q);
        return mk_long((w[c] & 0x0F0F0F0Fu) | (spread4(hh & 15) << 4), ((w[c] >> 4) & 0x0F0F0F0Fu) | (spread4((hh >> 16) & 15) << 4));
    }
};
typedef _Float16 v4h __attribute__((ext_vector_type(4)));

// One span's step for 16 weight rows and NT token tiles: per block c one 16x16x32 MFMA a tile, folded at once, acc =
// fma(x_d, t, acc) with t = d D (Q5_1: fma(d, D, m S), S the token block's sum from an MFMA against ones).  MAGIC: the
// MFMA starts from 0x4B400000, so its result read as a float is D + 1.5 2^23 exactly (|D| < 2^22), and t = fma(that, d,
// -1.5 2^23 d) is d D rounded once -- 1.5 2^23 d is exact for a finite fp16 d -- in one operation where a conversion and
// a product take two: the fold is what bounds these types (VALU).
template <int T, int NT, bool FIRST, bool MAGIC>
__device__ __forceinline__ void step_a0(const A0Row<T> &w, const float (&d)[8], const uint8_t *al, float (&acc)[GM_TILES][4]) {
#pragma unroll
    for (int t = NT; t < GM_TILES; ++t)
#pragma unroll
        for (int v = 0; v < 4; ++v) asm volatile("" : "=v"(acc[t][v]));
    const int lid = lane_id_here(), q = lid >> 4, rr = lid & 15;
    const uint32_t a0 = lds_addr(al) + rr * 256 + 16 * ((q >> 1) ^ rr) + 8 * (q & 1);   // row rr of tile 0, block 0
    const uint8_t *yrow = al + GM_TOK * 256 + 8 * q;
    constexpr int M = MAGIC ? 0x4B400000 : 0;
    const v4i z = {M, M, M, M};
    // the MFMAs of block c + 1 go out before block c is folded (with one or two tiles: more cover their latency themselves)
    constexpr int AHEAD = NT <= 2 ? 1 : 0;
    v4i D[1 + AHEAD][NT], S[1 + AHEAD][NT];
    v4h y[1 + AHEAD][NT];
    auto mul = [&](int c) {
        const int s = AHEAD ? c & 1 : 0;
        const uint32_t ac = a0 ^ (32 * c);
        long A[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) A[t] = lds_at<long>(ac + t * 16 * 256);
#pragma unroll
        for (int t = 0; t < NT; ++t) y[s][t] = *(const v4h *) (yrow + 2 * (GM_TOK * c + 16 * t));
        const long B = w.b(c, q);
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            D[s][t] = mfma16(A[t], B, z);
            if constexpr (ysum_type(T)) S[s][t] = mfma16(A[t], mk_long(0x01010101u, 0x01010101u), z);
        }
    };
    auto fold = [&](int c) {
        const int s = AHEAD ? c & 1 : 0;
#pragma unroll
        for (int t = 0; t < NT; ++t) {
#pragma unroll
            for (int v = 0; v < 4; ++v) {
                float x;
                if constexpr (ysum_type(T)) x = __builtin_fmaf(d[c], (float) D[s][t][v], h2f(w.dm[c] >> 16) * (float) S[s][t][v]);
                else if constexpr (MAGIC) x = __builtin_fmaf(__int_as_float(D[s][t][v]), d[c], -12582912.0f * d[c]);
                else x = d[c] * (float) D[s][t][v];
                acc[t][v] = __builtin_fmaf((float) y[s][t][v], x, FIRST && c == 0 ? 0.0f : acc[t][v]);
            }
        }
    };
    if constexpr (AHEAD) mul(0);
#pragma unroll
    for (int c = 0; c < 8; ++c) {
        if constexpr (AHEAD) { if (c < 7) mul(c + 1); } else mul(c);
        fold(c);
        asm volatile("");   // a scheduling-region boundary per block (register pressure)
    }
}
// The step of wave's tile `wt` for ntile token tiles.  MAGIC needs finite scales: a span with an infinite or NaN scale in
// any of the wave's rows (checked with 0 * d, NaN exactly then) takes the plain product.
template <int T>
__device__ __forceinline__ void span_a0(const uint8_t *wt, const uint8_t *al, int ntile, bool first, float (&acc)[GM_TILES][4]) {
    const int lid = lane_id_here();
    A0Row<T> w;
    float d[8];
    w.load(wt + (lid & 15) * span_bytes(T), lid >> 4, d);
    constexpr bool M = A0Row<T>::magic;
    if constexpr (M) {
        float chk = 0.0f;
#pragma unroll
        for (int c = 0; c < 8; ++c) chk = __builtin_fmaf(d[c], 0.0f, chk);
        if (__builtin_expect(__ballot(chk != 0.0f) != 0, 0)) {
            if (first) {
#pragma unroll
                for (int t = 0; t < GM_TILES; ++t)
#pragma unroll
                    for (int v = 0; v < 4; ++v) acc[t][v] = 0.0f;
            }
            step_a0<T, GM_TILES, false, false>(w, d, al, acc);
            return;
        }
    }
    if (first) {
        switch (ntile) {
        case 1: step_a0<T, 1, true, M>(w, d, al, acc); break;
        case 2: step_a0<T, 2, true, M>(w, d, al, acc); break;
        case 3: step_a0<T, 3, true, M>(w, d, al, acc); break;
        default: step_a0<T, 4, true, M>(w, d, al, acc); break;
        }
    } else {
        switch (ntile) {
        case 1: step_a0<T, 1, false, M>(w, d, al, acc); break;
        case 2: step_a0<T, 2, false, M>(w, d, al, acc); break;
        case 3: step_a0<T, 3, false, M>(w, d, al, acc); break;
        default: step_a0<T, 4, false, M>(w, d, al, acc); break;
        }
    }
}

__host__ __device__ constexpr int xcd_gcd8(int n) { return (n & 7) == 0 ? 8 : (n & 3) == 0 ? 4 : (n & 1) == 0 ? 2 : 1; }


// floor(p / a) as a multiply-high, with a_mul = ceil(2^32 / a): exact while p * (a_mul * a - 2^32) < 2^32, which
// p * a < 2^32 guarantees (the launchers check it)
__device__ __forceinline__ uint32_t div_by_mul(uint32_t p, uint64_t a_mul) { return (uint32_t) (((uint64_t) p * a_mul) >> 32); }
static inline uint64_t div_mul_of(int a) { return ((1ull << 32) + (uint64_t) a - 1) / (uint64_t) a; }

template <int T, bool GU, int W, int B>
__global__ __launch_bounds__(64 * W, B * W / 4) void k_gemm(hy_moe_dev m, const uint8_t *__restrict__ aq, uint64_t a_mul, const int *__restrict__ order,
                                                        const int *__restrict__ order_n, const int *__restrict__ egrp, const float *__restrict__ wts,
                                                        float *__restrict__ out) {
    using C = G5<T, W, B>;
    constexpr bool A0 = C::A0;
    constexpr int D = C::D, AQ = C::AROW;
    // stage s at s * SB: weights [wave][TB], activations [64][256], d [64]; A0: weights only, then the raw and aligned buffers
    // IQ2_XS: its tables first, where an LDS instruction's 16-bit offset reaches them (a lookup's address is then its index)
    constexpr int TAB = T == IQ2_XS ? IQ2_TAB : 0;
    __shared__ __align__(256) uint8_t smem[TAB + C::SMEM];
    __shared__ uint64_t s_scan[1024 + C::WAVES];                // per expert group: exclusive prefix of its items per tile class
    __shared__ int s_item[C::ITEMS][3];                  // first pair in order, tokens, weight slot
    __shared__ int s_pair[C::ITEMS][GM_TOK];             // pair index of each token of the segment's items
    __shared__ float s_wt[GU ? 1 : C::ITEMS][GM_TOK];    // down: their route weights
    __shared__ uint2 grid[T == IQ2_XS ? 1 : iq2_lds(T)];   // the codebook
    const int tid = threadIdx.x, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63, rr = lane & 15, q = lane >> 4;
    const int na = order_n[1];
    // ---- items.  Expert group g (cnt tokens) owns ceil(cnt / 64) items: full ones of 4 token tiles and a last one of
    // ceil(rem / 16) tiles.  Items are ordered by tile count (class 4: full items and last items of 4 tiles, expert by
    // expert; then the last items of 3, 2 and 1 tiles) and dealt to the gridDim.y item slots in snake order (slot y
    // takes positions k S + y for even k and k S + S - 1 - y for odd k), which evens out the slots' work.
    // s_scan holds each group's exclusive prefix of the four class counts, 16 bits each (item totals stay below 2^16).
    {
        uint64_t c2[C::PER], loc = 0;
#pragma unroll
        for (int i = 0; i < C::PER; ++i) {
            const int g = C::PER * tid + i;
            uint64_t c = 0;
            if (g < na) {
                const int cnt = egrp[3 * g + 2], n = (cnt + GM_TOK - 1) / GM_TOK, cl = (cnt - GM_TOK * (n - 1) + 15) >> 4;
                c = (uint64_t) (n - 1 + (cl == 4)) | ((uint64_t) (cl == 3) << 16) | ((uint64_t) (cl == 2) << 32) | ((uint64_t) (cl == 1) << 48);
            }
            c2[i] = c;
            loc += c;
        }
        uint64_t inc = loc;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const uint64_t t = __shfl_up(inc, o); if (lane >= o) inc += t; }
        if (lane == 63) s_scan[1024 + wave] = inc;
        __syncthreads();
        uint64_t base = 0;
        for (int w = 0; w < wave; ++w) base += s_scan[1024 + w];
        uint64_t ex = base + inc - loc;
#pragma unroll
        for (int i = 0; i < C::PER; ++i) { s_scan[C::PER * tid + i] = ex; ex += c2[i]; }
        if constexpr (T == IQ2_XS) iq2_sel_table((uint32_t *) smem);
        else if constexpr (iq2_type(T)) expand_iq2_grid<T>(grid);
        __syncthreads();
    }
    uint64_t tot = 0;
    for (int w = 0; w < C::WAVES; ++w) tot += s_scan[1024 + w];
    // (scalar registers: every loop below runs on counts derived from these, and the compiler cannot see that values
    // read from LDS are uniform)
    const uint32_t tlo = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) tot), thi = (uint32_t) __builtin_amdgcn_readfirstlane((int) (uint32_t) (tot >> 32));
    const int n4 = (int) (tlo & 0xffff), n3 = (int) (tlo >> 16), n2 = (int) (thi & 0xffff), n1 = (int) (thi >> 16);
    const int total = n4 + n3 + n2 + n1;
    // Block (x, y) runs on XCD (x + gridDim.x y) % 8, and each XCD has its own L2.  This block's logical row block
    // bx and item slot y0: with gridDim.y a multiple of 8 (the host's choice from 8 slots up), XCD c takes the slots
    // c ys / 8 .. (c + 1) ys / 8 - 1, each with all its row blocks -- an item's activation rows are fetched into one
    // L2 and read there by every row block, and runs of consecutive item positions (mostly one expert's items) share
    // their weight tiles there.  Fewer slots: logical slots l, l + 1, ... sit P = 8 / gcd(gridDim.x, 8) physical
    // slots apart (P = 1 unless gridDim.y is a multiple of it): the same XCD for every row block, the weights shared.
    const int ys = gridDim.y;
    int bx, y0;
    if (ys % 8 == 0) {
        const int b = (int) blockIdx.x + (int) gridDim.x * (int) blockIdx.y;
        bx = (b >> 3) % (int) gridDim.x;
        y0 = (b & 7) * (ys / 8) + (b >> 3) / (int) gridDim.x;
    } else {
        const int P0 = 8 / xcd_gcd8((int) gridDim.x), P = ys % P0 == 0 ? P0 : 1;
        bx = blockIdx.x;
        y0 = ((int) blockIdx.y % P) * (ys / P) + (int) blockIdx.y / P;
    }
    const int rounds = total / ys, rem_items = total - rounds * ys;
    const int my_items = rounds + (((rounds & 1) ? ys - 1 - y0 : y0) < rem_items ? 1 : 0);
    if (my_items == 0) return;   // uniform over the block
    const int in_dim = GU ? m.n : m.ff, nsb = in_dim / 256;
    const size_t mbytes = GU ? m.gate_bytes : m.down_bytes;
    // this wave's 16 rows: tile index (rows / 16) in its matrix, and the output row of each lane
    const int tile_row = GU ? bx * C::HALF + wave % C::HALF : bx * C::WAVES + wave;
    const int row = 16 * tile_row + rr;
    const uint8_t *Wmat = (GU ? (wave < C::HALF ? m.gate : m.up) : m.down) + (size_t) tile_row * nsb * C::TB;
    const size_t arow = (size_t) nsb * AQ;
    // (offsets from the array itself: through a pointer variable behind the tables the types without tables were scheduled
    // anew as well, and the 509-token IQ4_NL layer call took 1064 us instead of 1004)
    auto stage_w = [&](int s) { return smem + TAB + s * C::SB; };
    auto stage_a = [&](int s) { return (int8_t *) (smem + TAB + s * C::SB + C::WB); };
    auto stage_d = [&](int s) { return (const float *) (smem + TAB + s * C::SB + C::WB + C::AB); };
    auto raw_a = [&](int s) { return smem + TAB + D * C::SB + (s & 1) * C::RAW; };
    auto al_a = [&](int s) { return smem + TAB + D * C::SB + 2 * C::RAW + (s & 1) * C::AL; };

    for (int seg = 0; seg < my_items; seg += C::ITEMS) {
        const int nit = min(C::ITEMS, my_items - seg);
        __syncthreads();   // readers of the previous segment's tables are done
        // IQ4_NL and Q4_K: a thread id that the compiler cannot hoist out of the segment loop.  Kept live across the stream,
        // the table addresses made from it went to scratch there, and a scratch reload is a vector memory operation that
        // the compiler waits for by draining the stream.
        int ts = tid;
        if constexpr (T == IQ4_NL || T == Q4_K) asm volatile("" : "+v"(ts));
        for (int i = ts; i < nit; i += C::THREADS) {
            const int k = seg + i;
            int pos = k * ys + ((k & 1) ? ys - 1 - y0 : y0);   // position in the class order
            int cls = 0;                                        // field of s_scan: 0 = 4 tiles, 1 = 3, 2 = 2, 3 = 1
            if (pos >= n4) { pos -= n4; cls = 1; if (pos >= n3) { pos -= n3; cls = 2; if (pos >= n2) { pos -= n2; cls = 3; } } }
            int lo = 0, hi = na - 1;   // last group whose prefix in the class <= pos: the group that owns the item
            while (lo < hi) {
                const int mid = (lo + hi + 1) >> 1;
                if ((int) ((s_scan[mid] >> (16 * cls)) & 0xffff) <= pos) lo = mid; else hi = mid - 1;
            }
            const int cnt = egrp[3 * lo + 2];
            const int chunk = cls == 0 ? pos - (int) (s_scan[lo] & 0xffff) : (cnt - 1) / GM_TOK;
            const int tok0 = chunk * GM_TOK;
            s_item[i][0] = egrp[3 * lo + 1] + tok0;
            s_item[i][1] = min(GM_TOK, cnt - tok0);
            s_item[i][2] = m.slot[egrp[3 * lo]];
        }
        __syncthreads();
        for (int i = ts; i < nit * GM_TOK; i += C::THREADS) {
            const int it = i / GM_TOK, tk = i - it * GM_TOK;
            const int pr = tk < s_item[it][1] ? order[s_item[it][0] + tk] : -1;
            s_pair[it][tk] = pr;
            if (!GU) s_wt[GU ? 0 : it][tk] = pr >= 0 ? wts[pr] : 0.0f;
        }
        __syncthreads();
        const int nsteps = nit * nsb;

        // ---- issue: the DMAs of the next step of each stream (weights; activation rows, with the weights, or for A0 one
        // step ahead of them), then advance.  What an item fixes is read at its first span: the weight and activation
        // addresses (scalar pointers that advance by a span) and the lanes' byte offsets from the latter, NO for lanes
        // that sit out: absent tokens are not fetched (their LDS rows keep stale bytes, whose MFMA columns are never
        // stored).  The caller's activations stay below 4 GB.
        constexpr uint32_t NO = 0xFFFFFFFFu;
        const uint32_t lane16 = 16 * lane, lane4 = 4 * lane;
        auto row_off = [&](int it, int t, int ntok) -> uint32_t {   // the activation row of token t of an item
            const int pr = t < ntok ? s_pair[it][t] : s_pair[it][0];
            return (GU ? div_by_mul((uint32_t) pr, a_mul) : (uint32_t) pr) * (uint32_t) arow;
        };
        int w_it = 0, w_b = 0, w_step = 0;
        const uint8_t *w_src = nullptr;
        auto issue_w = [&](int stage) {
            if (w_b == 0) w_src = Wmat + (size_t) __builtin_amdgcn_readfirstlane(s_item[w_it][2]) * mbytes;
            const uint32_t wdst = lds_addr(stage_w(stage) + wave * C::TB);
#pragma unroll
            for (int i = 0; i < C::N4; ++i) dma_s128(w_src + 1024 * i, lane16, wdst + 1024 * i);
#pragma unroll
            for (int j = 0; j < C::N1; ++j)
                if (256 * j + 4 * lane < C::NR) dma_s32(w_src + 1024 * C::N4 + 256 * j, lane4, wdst + 1024 * C::N4 + 256 * j);
        };
        auto next_w = [&]() { ++w_step; w_src += C::TB; if (++w_b == nsb) { w_b = 0; ++w_it; } };
        uint32_t aoff[C::NA], doff = NO;
        int a_it = 0, a_b = 0;
        const uint8_t *a_src = nullptr;
        // this wave's tokens TPW wave + 4 i + lane / 16: lane l fetches 16-byte piece (l % 16) ^ (t % 16) of token t, the
        // conflict-free layout the MFMA reads use, and, on the first TPW lanes, the d of token TPW wave + lane; lane 0
        // of every instruction fetches something, so that every instruction issues (the waits count them)
        auto issue_a = [&](int stage) {
            if (a_b == 0) {
                const int ntok = __builtin_amdgcn_readfirstlane(s_item[a_it][1]);
                a_src = aq;
#pragma unroll
                for (int i = 0; i < C::NA; ++i) {
                    const int t = C::TPW * wave + 4 * i + (lane >> 4);
                    aoff[i] = t < ntok || lane == 0 ? row_off(a_it, t, ntok) + 4 + 16 * ((lane & 15) ^ (t & 15)) : NO;
                }
                const int td = C::TPW * wave + lane;
                doff = lane < C::TPW && (td < ntok || lane == 0) ? row_off(a_it, td, ntok) : NO;
            }
            const uint32_t adst = lds_addr(stage_a(stage) + C::TPW * wave * 256);
#pragma unroll
            for (int i = 0; i < C::NA; ++i)
                if (aoff[i] != NO) dma_s128(a_src, aoff[i], adst + 1024 * i);
            if (doff != NO) dma_s32(a_src, doff, lds_addr(stage_d(stage) + C::TPW * wave));
        };
        // A0: lane l of DMA i takes 16-byte piece 64 i + l of the wave's TPW rows of 17
        auto issue_raw = [&](int buf) {
            if (a_b == 0) {
                const int ntok = __builtin_amdgcn_readfirstlane(s_item[a_it][1]);
                a_src = aq;
#pragma unroll
                for (int i = 0; i < C::NA; ++i) {
                    const int pc = 64 * i + lane, t = C::TPW * wave + pc / 17;
                    aoff[i] = pc < 17 * C::TPW && t < ntok ? row_off(a_it, t, ntok) + 16 * (pc % 17) : NO;
                }
            }
            const uint32_t adst = lds_addr(raw_a(buf) + 272 * C::TPW * wave);
#pragma unroll
            for (int i = 0; i < C::NA; ++i)
                if (aoff[i] != NO) dma_s128(a_src, aoff[i], adst + 1024 * i);
        };
        auto next_a = [&]() { a_src += AQ; if (++a_b == nsb) { a_b = 0; ++a_it; } };

        float acc[GM_TILES][4];
#pragma unroll
        for (int i = 0; i < GM_TILES; ++i)
#pragma unroll
            for (int v = 0; v < 4; ++v) acc[i][v] = 0.0f;
        auto compute = [&](int it, int b, int stage, int ntok) {
            const int ntile = (ntok + 15) >> 4;
            const int8_t *as = stage_a(stage);
            const float *yd = stage_d(stage);
            if constexpr (A0) {
                span_a0<T>(stage_w(stage) + wave * C::TB, al_a(stage), ntile, b == 0, acc);
            } else if constexpr (T == Q4_K) {
                // straight-line code per tile count
                const uint8_t *wt = stage_w(stage) + wave * C::TB;
                static_assert(GM_TILES == 4, "one case per tile count");
                // an item's first span starts its accumulators (fmaf with +0, the bits of a sum begun at 0): no reset
                // after the epilogue, so the accumulators stay in the same registers on every path through the loop
                if (b == 0) {
                    switch (ntile) {
                    case 1: step_q4k<1, true>(wt, as, yd, acc); break;
                    case 2: step_q4k<2, true>(wt, as, yd, acc); break;
                    case 3: step_q4k<3, true>(wt, as, yd, acc); break;
                    default: step_q4k<4, true>(wt, as, yd, acc); break;
                    }
                } else {
                    switch (ntile) {
                    case 1: step_q4k<1, false>(wt, as, yd, acc); break;
                    case 2: step_q4k<2, false>(wt, as, yd, acc); break;
                    case 3: step_q4k<3, false>(wt, as, yd, acc); break;
                    default: step_q4k<4, false>(wt, as, yd, acc); break;
                    }
                }
            } else if constexpr (T == Q6_K) {
                const uint8_t *wt = stage_w(stage) + wave * C::TB;
                if (b == 0) {
                    switch (ntile) {
                    case 1: step_q6k<1, true>(wt, as, yd, acc); break;
                    case 2: step_q6k<2, true>(wt, as, yd, acc); break;
                    case 3: step_q6k<3, true>(wt, as, yd, acc); break;
                    default: step_q6k<4, true>(wt, as, yd, acc); break;
                    }
                } else {
                    switch (ntile) {
                    case 1: step_q6k<1, false>(wt, as, yd, acc); break;
                    case 2: step_q6k<2, false>(wt, as, yd, acc); break;
                    case 3: step_q6k<3, false>(wt, as, yd, acc); break;
                    default: step_q6k<4, false>(wt, as, yd, acc); break;
                    }
                }
            } else if constexpr (T == IQ2_XS) {
                const uint8_t *wt = stage_w(stage) + wave * C::TB;
                const uint32_t *sel = (const uint32_t *) smem;
                if (b == 0) {
                    switch (ntile) {
                    case 1: step_iq2xs<1, true>(wt, as, yd, sel, acc); break;
                    case 2: step_iq2xs<2, true>(wt, as, yd, sel, acc); break;
                    case 3: step_iq2xs<3, true>(wt, as, yd, sel, acc); break;
                    default: step_iq2xs<4, true>(wt, as, yd, sel, acc); break;
                    }
                } else {
                    switch (ntile) {
                    case 1: step_iq2xs<1, false>(wt, as, yd, sel, acc); break;
                    case 2: step_iq2xs<2, false>(wt, as, yd, sel, acc); break;
                    case 3: step_iq2xs<3, false>(wt, as, yd, sel, acc); break;
                    default: step_iq2xs<4, false>(wt, as, yd, sel, acc); break;
                    }
                }
            } else {
                const uint8_t *wt = stage_w(stage) + wave * C::TB;
                if (b == 0) {
                    switch (ntile) {
                    case 1: step_gen<T, 1, true>(wt, grid, as, yd, acc); break;
                    case 2: step_gen<T, 2, true>(wt, grid, as, yd, acc); break;
                    case 3: step_gen<T, 3, true>(wt, grid, as, yd, acc); break;
                    default: step_gen<T, 4, true>(wt, grid, as, yd, acc); break;
                    }
                } else {
                    switch (ntile) {
                    case 1: step_gen<T, 1, false>(wt, grid, as, yd, acc); break;
                    case 2: step_gen<T, 2, false>(wt, grid, as, yd, acc); break;
                    case 3: step_gen<T, 3, false>(wt, grid, as, yd, acc); break;
                    default: step_gen<T, 4, false>(wt, grid, as, yd, acc); break;
                    }
                }
            }
            // the next step's stage has landed (this wave's DMAs; the barrier at its top covers the others'): waited for
            // here, ahead of the item's stores, so that no step waits for stores just issued (waited for at the next
            // step's top: 131 MXFP4 tokens, d 2048, 64 experts, ff 1024, top-8, 116 us, here 113; 2048 Q5_K/Q6_K tokens 654, 645)
            wait_vm<(D - 2) * C::L>();
            if (b != nsb - 1) return;
            // ---- the item's outputs, through this stage (every wave has finished reading it after a barrier), TOKP
            // tokens a pass: the waves' accumulators go there token-major -- rows padded by one float against bank
            // conflicts -- and wave w finishes tokens w, w + WAVES, ... of the pass: one output row per lane (SwiGLU
            // of the gate and up values, or the route weight times the down value), stored as whole rows.
            constexpr int OR = GU ? 16 * C::HALF : C::ROWS;   // output rows of the block
            constexpr int LD = OR + 1;                         // floats per token in LDS
            constexpr int NCOPY = GU ? 2 : 1;
            constexpr int TOKP = NCOPY * 64 * LD * 4 <= C::XCH ? 64 : NCOPY * 32 * LD * 4 <= C::XCH ? 32 : 16;
            static_assert(NCOPY * TOKP * LD * 4 <= C::XCH, "the exchange fits in a stage");
            float *s_o = (float *) stage_w(stage);             // gate (or down) values
            float *s_u = s_o + TOKP * LD;                      // up values
            const int row0 = bx * OR;
            // IQ4_NL and MXFP4 are at their 128 registers: the epilogue makes its lane constants here instead of keeping
            // them live across the stream (the other kernels have the registers, and are 1-3 % slower this way)
            const int el = T == IQ4_NL || T == MXFP4 ? lane_id_here() : lane, er = el & 15, eq = el >> 4;
            for (int p0 = 0; p0 < ntok; p0 += TOKP) {
                lds_barrier();   // the stage (or the previous pass) is no longer read
                {
                    float *dst = GU && wave >= C::HALF ? s_u : s_o;
                    const int orow = (GU ? wave % C::HALF : wave) * 16 + er;
#pragma unroll
                    for (int tile = 0; tile < GM_TILES; ++tile) {
                        if (tile >= ntile) break;
                        if (tile * 16 < p0 || tile * 16 >= p0 + TOKP) continue;
#pragma unroll
                        for (int v = 0; v < 4; ++v) dst[(tile * 16 - p0 + 4 * eq + v) * LD + orow] = acc[tile][v];
                    }
                }
                lds_barrier();
                for (int tok = p0 + wave; tok < min(ntok, p0 + TOKP); tok += C::WAVES) {
                    float *o = out + (size_t) s_pair[it][tok] * (GU ? m.ff : m.n) + row0;
                    const float wt = GU ? 0.0f : s_wt[GU ? 0 : it][tok];
                    const float *so = s_o + (tok - p0) * LD, *su = s_u + (tok - p0) * LD;
#pragma unroll
                    for (int r = el; r < OR; r += 64) store_f32(o + r, GU ? hy_swiglu(so[r], su[r], m.clamp) : wt * so[r]);
                }
            }
        };

        int ntok = __builtin_amdgcn_readfirstlane(s_item[0][1]);   // of the item in progress
        if constexpr (A0) {
            Relay<W> rl;
            issue_w(0);
            next_w();
            issue_raw(0);
            next_a();
            wait_vm<0>();
            lds_barrier();
            if (nsteps > 1) { issue_raw(1); next_a(); }
            rl.load(raw_a(0), wave);
            rl.store(al_a(0), wave);
            wait_vm<0>();
            for (int st = 0, it = 0, b = 0; st < nsteps; ++st) {
                lds_barrier();   // weights st, raw rows st + 1 and aligned rows st are in place; step st - 1 is done with its own
                const bool more = st + 1 < nsteps;
                if (more) {
                    issue_w(st + 1 & 1);
                    next_w();
                    if (st + 2 < nsteps) { issue_raw(st); next_a(); }
                    rl.load(raw_a(st + 1), wave);   // (its LDS reads land while the step's weights are decoded)
                }
                compute(it, b, st & 1, ntok);
                if (more) rl.store(al_a(st + 1), wave);
                if (++b == nsb) {
                    b = 0;
                    ++it;
                    if (it < nit) ntok = __builtin_amdgcn_readfirstlane(s_item[it][1]);
                }
            }
            continue;
        }
        // the stream: steps 0 .. D - 2 issued ahead; past the end, the last step is issued again (into the stage
        // of step s - 1, which nobody reads any more) so that every wait counts the same instructions
        int istage = 0;
        auto issue = [&]() {
            issue_w(istage);
            issue_a(istage);
            if (w_step < nsteps - 1) { next_w(); next_a(); }
            istage = istage == D - 1 ? 0 : istage + 1;
        };
#pragma unroll
        for (int s = 0; s < D - 1; ++s) issue();
        wait_vm<(D - 2) * C::L>();
        for (int st = 0, it = 0, b = 0, stage = 0; st < nsteps; ++st) {
            lds_barrier();
            issue();
            compute(it, b, stage, ntok);
            if (++b == nsb) {
                b = 0;
                ++it;
                if (it < nit) ntok = __builtin_amdgcn_readfirstlane(s_item[it][1]);
            }
            stage = stage == D - 1 ? 0 : stage + 1;
        }
        wait_vm<0>();   // no DMA into this block's LDS may outlive the segment
    }
}

// A lane's bytes of a span (SpanBytes) as its B words of 32-value block c -- values 8 q .. + 7 -- and the block's fold of the
// exact integer d (and, Q5_1, the token block's sum of quants s).
template <int T> struct Staged;
template <> struct Staged<IQ4_NL> : SpanBytes<IQ4_NL> {
    __device__ __forceinline__ long b(int c, int q) const {
        const int s = 4 * (q >> 1);
        return mk_long(kv4((qv[c].x >> s) & 0x0F0F0F0Fu), kv4((qv[c].y >> s) & 0x0F0F0F0Fu));
    }
    __device__ __forceinline__ float fold(int c, int d, int) const { return h2f((dd[c >> 1] >> (16 * (c & 1))) & 0xffff) * (float) d; }
};
template <> struct Staged<Q8_0> : SpanBytes<Q8_0> {
    __device__ __forceinline__ long b(int c, int) const { return mk_long(qv[c].x, qv[c].y); }
    __device__ __forceinline__ float fold(int c, int d, int) const { return h2f((dd[c >> 1] >> (16 * (c & 1))) & 0xffff) * (float) d; }
};
template <> struct Staged<MXFP4> : SpanBytes<MXFP4> {
    __device__ __forceinline__ long b(int c, int q) const {
        const int s = 4 * (q >> 1);
        return mk_long(kvfp4((qv[c].x >> s) & 0x0F0F0F0Fu), kvfp4((qv[c].y >> s) & 0x0F0F0F0Fu));
    }
    __device__ __forceinline__ float fold(int c, int d, int) const { return e8m0_half((ee[c >> 2] >> (8 * (c & 3))) & 255) * (float) d; }
};
template <> struct Staged<Q5_1> : SpanBytes<Q5_1> {   // x = nibble | bit << 4, 0..31
    __device__ __forceinline__ long b(int c, int q) const {
        const int s = 4 * (q >> 1);
        const uint32_t h = hb[c >> 2] >> (8 * (c & 3));
        return mk_long(((qv[c].x >> s) & 0x0F0F0F0Fu) | (spread4(h & 15) << 4), ((qv[c].y >> s) & 0x0F0F0F0Fu) | (spread4((h >> 4) & 15) << 4));
    }
    __device__ __forceinline__ float fold(int c, int d, int s) const {
        return __builtin_fmaf(h2f(dm[c] & 0xffff), (float) d, h2f(dm[c] >> 16) * (float) s);
    }
};
template <> struct Staged<Q5_0> : SpanBytes<Q5_0> {   // each byte nibble | 0xF0 where the fifth bit is clear (x - 16 as int8)
    __device__ __forceinline__ long b(int c, int q) const {
        const int s = 4 * (q >> 1);
        const uint32_t nh = ~(hb[c >> 2] >> (8 * (c & 3)));
        return mk_long(((qv[c].x >> s) & 0x0F0F0F0Fu) | fill_f0(nh & 15), ((qv[c].y >> s) & 0x0F0F0F0Fu) | fill_f0((nh >> 4) & 15));
    }
    __device__ __forceinline__ float fold(int c, int d, int) const { return h2f((dd[c >> 1] >> (16 * (c & 1))) & 0xffff) * (float) d; }
};

// one block's MFMA per tile, folded straight into the fp32 accumulators (Yc: 8 block scales per token)
template <int T>
__device__ __forceinline__ void chunk_fold(const Staged<T> &w, int c, int q, const int8_t *As, const float *Yc, int rr, int ntile,
                                           float (&acc)[GM_TILES][4]) {
    const v4i z = {0, 0, 0, 0};
    const long b = w.b(c, q);
#pragma unroll
    for (int tile = 0; tile < GM_TILES; ++tile) {
        if (tile >= ntile) break;
        const long a = *(const long *) (As + (tile * 16 + rr) * GM_LD + 32 * c + 8 * q);
        const v4i d = mfma16(a, b, z);
        v4i s = z;
        if constexpr (ysum_type(T)) s = mfma16(a, mk_long(0x01010101u, 0x01010101u), z);   // each token's block sum: A against ones
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[tile][v] = __builtin_fmaf(Yc[(tile * 16 + 4 * q + v) * 8 + c], w.fold(c, d[v], s[v]), acc[tile][v]);
    }
}

// The types with Q8_0 activations in launches beyond k_gemm's 32-bit activation offsets or 16-bit item counts: a
// register-staged stream, one step ahead.  A block walks the work items it, it + gridDim.y, ...; the (item, block) steps
// form one stream in which the next step's weight and activation bytes are loaded while the current step computes, across
// item boundaries.
template <int T, bool GU>
__global__ __launch_bounds__(256) void k_gemm_nl(hy_moe_dev m, const uint8_t *__restrict__ aq, int a_div, const int *__restrict__ order,
                                              const int *__restrict__ order_n, const int *__restrict__ egrp, const float *__restrict__ wts,
                                              float *__restrict__ out) {
    __shared__ __align__(16) int8_t As[2][GM_TOK * GM_LD];
    static_assert(vec_dot_type(T) == Q8_0, "Q8_0 activations, a fold per 32-value block");
    __shared__ float Yd[2][GM_TOK * 8];
    __shared__ int s_scan[1024 + 8];
    __shared__ float s_up[GU ? 32 * GM_TOK : 1];
    const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, rr = lane & 15, q = lane >> 4;
    const int na = order_n[1];
    // ---- items: expert group g owns ceil(cnt_g / GM_TOK) of them; s_scan = exclusive prefix (block-wide)
    {
        int c4[4], loc = 0;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
            const int g = 4 * tid + i;
            c4[i] = g < na ? (egrp[3 * g + 2] + GM_TOK - 1) / GM_TOK : 0;
            loc += c4[i];
        }
        int inc = loc;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) { const int t = __shfl_up(inc, o); if (lane >= o) inc += t; }
        if (lane == 63) s_scan[1024 + wave] = inc;
        __syncthreads();
        int base = 0;
        for (int w = 0; w < wave; ++w) base += s_scan[1024 + w];
        int ex = base + inc - loc;
#pragma unroll
        for (int i = 0; i < 4; ++i) { s_scan[4 * tid + i] = ex; ex += c4[i]; }
        __syncthreads();
    }
    const int total = s_scan[1024] + s_scan[1025] + s_scan[1026] + s_scan[1027];
    int it = blockIdx.y;
    if (it >= total) return;
    const int rows = GU ? m.ff : m.n, in_dim = GU ? m.n : m.ff, nsb = in_dim / 256;
    const int orows = GU ? 32 : GM_ROWS;
    const int row = blockIdx.x * orows + (GU ? (wave & 1) : wave) * 16 + rr;
    const bool row_ok = row < rows;
    const size_t mbytes = GU ? m.gate_bytes : m.down_bytes;
    const uint8_t *Wbase = (GU ? (wave < 2 ? m.gate : m.up) : m.down) + tiled_off(row_ok ? row : rows - 1, 0, nsb, span_bytes(T));
    constexpr int AB = 8 * Q8_0_BYTES;   // activation bytes per 256 values
    const size_t arow = (size_t) nsb * AB;
    constexpr int BB = 8 * block_bytes(T);   // weight bytes per 256 values
    const int st_tok = tid >> 2, st_part = tid & 3;   // staging: 64 bytes of token st_tok per thread

    // item -> (first pair in order, tokens, weight pointer); the staging thread's activation row
    struct ItemState { int start, ntok; const uint8_t *W; const uint8_t *src; };
    auto locate = [&](int item) {
        int lo = 0, hi = na - 1;   // last group whose prefix <= item
        while (lo < hi) { const int mid = (lo + hi + 1) >> 1; if (s_scan[mid] <= item) lo = mid; else hi = mid - 1; }
        const int tok0 = (item - s_scan[lo]) * GM_TOK;
        ItemState st;
        st.start = egrp[3 * lo + 1] + tok0;
        st.ntok = min(GM_TOK, egrp[3 * lo + 2] - tok0);
        st.W = Wbase + (size_t) m.slot[egrp[3 * lo]] * mbytes;
        st.src = nullptr;
        if (st_tok < st.ntok) {
            const int p = order[st.start + st_tok];
            st.src = aq + (size_t) (GU ? p / a_div : p) * arow;
        }
        return st;
    };
    auto load_a = [&](const uint8_t *src, int b, uint4 (&a)[4], float (&yd)[2]) {
        if (src) {
            const uint8_t *s = src + (size_t) b * AB;
            // Q8_0 blocks 2 st_part, 2 st_part + 1: qs at 68 p + 2 (2 mod 4) and 68 p + 36
            const uint8_t *p0 = s + 2 * Q8_0_BYTES * st_part;
            a[0] = load16_a2(p0 + 2); a[1] = load16_a2(p0 + 18);
            a[2] = load16_a4(p0 + 36); a[3] = load16_a4(p0 + 52);
            yd[0] = h2f(ld_u16(p0)); yd[1] = h2f(ld_u16(p0 + Q8_0_BYTES));
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) a[i] = make_uint4(0, 0, 0, 0);
            yd[0] = yd[1] = 0.0f;
        }
    };

    ItemState cur = locate(it);
    Staged<T> w;
    w.load(cur.W, q);
    uint4 a[4];
    float yd[2];
    load_a(cur.src, 0, a, yd);
    float acc[GM_TILES][4];
#pragma unroll
    for (int i = 0; i < GM_TILES; ++i)
#pragma unroll
        for (int v = 0; v < 4; ++v) acc[i][v] = 0.0f;
    int b = 0, buf = 0;
    for (;;) {
        {
            uint4 *dst = (uint4 *) (As[buf] + st_tok * GM_LD + 64 * st_part);
#pragma unroll
            for (int i = 0; i < 4; ++i) dst[i] = a[i];
            Yd[buf][st_tok * 8 + 2 * st_part] = yd[0]; Yd[buf][st_tok * 8 + 2 * st_part + 1] = yd[1];
        }
        // the next step: block b + 1 of this item, or block 0 of the next item
        const bool last_b = b + 1 == nsb;
        const int nit = last_b ? it + (int) gridDim.y : it;
        const bool more = nit < total;
        ItemState nxt = cur;
        Staged<T> nw;
        if (more) {
            if (last_b) nxt = locate(nit);
            const int nb = last_b ? 0 : b + 1;
            nw.load(nxt.W + (size_t) nb * (HY_TILE * BB), q);
            load_a(nxt.src, nb, a, yd);
        }
        __syncthreads();
        const int ntile = (cur.ntok + 15) / 16;
#pragma unroll
        for (int c = 0; c < 8; ++c) chunk_fold<T>(w, c, q, As[buf], Yd[buf], rr, ntile, acc);
        if (last_b) {   // the item's outputs
            if (GU && wave >= 2) {
#pragma unroll
                for (int tile = 0; tile < GM_TILES; ++tile)
#pragma unroll
                    for (int v = 0; v < 4; ++v) s_up[((wave & 1) * 16 + rr) * GM_TOK + tile * 16 + 4 * q + v] = acc[tile][v];
            }
            if (GU) __syncthreads();
            if (!GU || wave < 2) {
#pragma unroll
                for (int tile = 0; tile < GM_TILES; ++tile) {
                    if (tile >= ntile) break;
#pragma unroll
                    for (int v = 0; v < 4; ++v) {
                        const int tok = tile * 16 + 4 * q + v;
                        if (tok < cur.ntok && row_ok) {
                            const int p = order[cur.start + tok];
                            if (GU) out[(size_t) p * m.ff + row] = hy_swiglu(acc[tile][v], s_up[((wave & 1) * 16 + rr) * GM_TOK + tok], m.clamp);
                            else out[(size_t) p * m.n + row] = wts[p] * acc[tile][v];
                        }
                    }
                }
            }
#pragma unroll
            for (int i = 0; i < GM_TILES; ++i)
#pragma unroll
                for (int v = 0; v < 4; ++v) acc[i][v] = 0.0f;
        }
        if (!more) break;
        cur = nxt;
        it = nit;
        b = last_b ? 0 : b + 1;
        buf ^= 1;
        w = nw;
    }
}

#define HY_GEMM_SWITCH(T, ...)                                                                    \
    switch (T) {                                                                                   \
    case Q4_K: { constexpr int TT = Q4_K; __VA_ARGS__; }                                                 \
    case Q5_K: { constexpr int TT = Q5_K; __VA_ARGS__; }                                                 \
    case Q6_K: { constexpr int TT = Q6_K; __VA_ARGS__; }                                                 \
    case IQ4_XS: { constexpr int TT = IQ4_XS; __VA_ARGS__; }                                             \
    case IQ2_XS: { constexpr int TT = IQ2_XS; __VA_ARGS__; }                                             \
    case IQ2_XXS: { constexpr int TT = IQ2_XXS; __VA_ARGS__; }                                           \
    case Q2_K: { constexpr int TT = Q2_K; __VA_ARGS__; }                                                 \
    case Q3_K: { constexpr int TT = Q3_K; __VA_ARGS__; }                                                 \
    case IQ3_XXS: { constexpr int TT = IQ3_XXS; __VA_ARGS__; }                                           \
    case IQ3_S: { constexpr int TT = IQ3_S; __VA_ARGS__; }                                               \
    case IQ2_S: { constexpr int TT = IQ2_S; __VA_ARGS__; }                                               \
    case IQ1_S: { constexpr int TT = IQ1_S; __VA_ARGS__; }                                               \
    default: set_error("grouped GEMM: unsupported expert type %d", (int) (T)); return HY_EUNSUPPORTED_TYPE; \
    }

// k_gemm keeps each expert group's item prefix per tile class in a 16-bit field of s_scan: the item total of a launch
// must stay below 2^16 (checked against the upper bound below, from the host)
constexpr int GM_MAX_ITEMS = 1 << 16;
// upper bound of the work items: sum over active experts of ceil(cnt / GM_TOK) <= ceil(P / GM_TOK) + active
constexpr int max_items(int n_pairs, int max_active) { return (n_pairs + GM_TOK - 1) / GM_TOK + max_active; }
// the current device's CU count (an attribute query: cheap, thread-safe, and right for each device)
static int cu_count() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    return cus;
}
// item slots per row tile: enough blocks for about `per_cu` resident blocks on every CU.  k_gemm (`xcd`) groups its
// slots by XCD when they are a multiple of 8, else places consecutive items P slots apart: from 8 slots up a
// multiple of 8, else of P where there are that many.  A multiple of 8 that leaves an eighth of the CUs without a block is
// not worth its locality: 20 slots instead of 16 for 12 row blocks, 512 tokens (d 2048, 64 experts, ff 768, top-8) in
// Q2_K 283 -> 252 us, in Q5_1 354 -> 314; the 509-token IQ4_NL call (288 experts) 1118 -> 1005.
static int item_slots(int row_tiles, int n_pairs, int max_active, int per_cu, bool xcd = false) {
    const int want = cu_count() * per_cu / row_tiles;   // every block resident at once
    const int n = std::max(1, std::min(max_items(n_pairs, max_active), want));
    if (xcd && n >= 8 && n / 8 * 8 * 8 > n * 7) return n / 8 * 8;
    const int P = 8 / xcd_gcd8(row_tiles);
    return n >= P ? n / P * P : n;
}

// the types with Q8_0 activations
#define HY_A0_SWITCH(T, ...)                                                                       \
    switch (T) {                                                                                   \
    case IQ4_NL: { constexpr int TT = IQ4_NL; __VA_ARGS__; }                                             \
    case MXFP4: { constexpr int TT = MXFP4; __VA_ARGS__; }                                               \
    case Q5_0: { constexpr int TT = Q5_0; __VA_ARGS__; }                                                 \
    case Q5_1: { constexpr int TT = Q5_1; __VA_ARGS__; }                                                 \
    default: { constexpr int TT = Q8_0; __VA_ARGS__; }                                                   \
    }
// their waves a block: 16 where two weight stages of 256 rows leave room for the activation buffers, else 8
constexpr int a0_waves(int t) { return 2 * 256 * span_bytes(t) + 4 * (GM_TOK * 8 * Q8_0_BYTES) <= 150 * 1024 ? 16 : 8; }
// k_gemm's 32-bit activation offsets, its pair / k by multiply-high and its 16-bit item counts hold (larger launches take
// k_gemm_nl).  k: pairs a row of activations, so gate/up's offsets reach (n_pairs - 1) / k rows.
constexpr bool a0_fits(int n_pairs, int k, int in_dim, int max_active) {
    return (size_t) ((n_pairs - 1) / k + 1) * (in_dim / 256) * (8 * Q8_0_BYTES) < 0xFFFF0000u &&
           (uint64_t) n_pairs * (uint64_t) k < (1ull << 32) && max_items(n_pairs, max_active) < GM_MAX_ITEMS;
}
static_assert(a0_fits(131072 * 8, 8, 28672, 1024), "4.0e9 bytes of activation rows, each of eight pairs");
static_assert(!a0_fits(1024 * 1024, 1, 28672, 1024) && !a0_fits(142000 * 8, 8, 28672, 1024), "rows past 32-bit offsets");
static_assert(!a0_fits(1 << 28, 64, 256, 1) && !a0_fits(64 * 65536, 8, 256, 1), "pairs past the multiply-high; items past 16 bits");

// One k_gemm launch: W waves a block, B blocks a CU (8 W output rows a block for gate/up, 16 W for down; ff and n are
// multiples of 256, so 8 and 16 waves both tile them).
template <int T, bool GU, int W, int B>
static int launch_k_gemm(const hy_moe_dev &m, const void *a, int k, int n_pairs, const int *order, const int *order_n, const int *egrp,
                         int max_active, const float *wts, float *out, hipStream_t s) {
    const int rb = GU ? m.ff / (8 * W) : m.n / (16 * W);
    dim3 grid(rb, item_slots(rb, n_pairs, max_active, B, B == 1));   // two blocks a CU: every slot counts
    hipLaunchKernelGGL((k_gemm<T, GU, W, B>), grid, dim3(64 * W), 0, s, m, (const uint8_t *) a, div_mul_of(k), order, order_n, egrp, wts, out);
    return check_launch(GU ? "hy_moe_gemm_gate_up" : "hy_moe_gemm_down");
}
// The same, in 8-wave blocks where blocks of 16 waves would take at most half of the CUs: twice the blocks then still run
// at once, each with half of the weight rows to stream and decode.  d 2048, ff 1024, one expert and 64 tokens: IQ4_NL 97
// -> 76 us, MXFP4 100 -> 79, IQ2_XS 81 -> 69, IQ4_XS 72 -> 68; 8 experts, top-2, 64 tokens: 81 -> 65, 80 -> 67, 72 -> 61
// and 64 -> 61, Q4_K/Q6_K 68 -> 63.  Past the half the 16-wave blocks win: 512 of those tokens (192 blocks of 16 waves)
// in IQ2_XS 91 us, in 8-wave blocks 96.
template <int T, bool GU, int W, int B>
static int launch_k_gemm_fit(const hy_moe_dev &m, const void *a, int k, int n_pairs, const int *order, const int *order_n, const int *egrp,
                             int max_active, const float *wts, float *out, hipStream_t s) {
    if constexpr (W == 16) {
        if (2 * max_items(n_pairs, max_active) * (GU ? m.ff / 128 : m.n / 256) <= cu_count())
            return launch_k_gemm<T, GU, 8, B>(m, a, k, n_pairs, order, order_n, egrp, max_active, wts, out, s);
    }
    return launch_k_gemm<T, GU, W, B>(m, a, k, n_pairs, order, order_n, egrp, max_active, wts, out, s);
}

int launch_gemm_gate_up(const hy_moe_dev &m, const void *xq, int k, int n_pairs, const int *order, const int *order_n, const int *egrp,
                        int max_active, float *h, hipStream_t s) {
    if (max_active <= 0 || n_pairs <= 0) return HY_OK;
    if (vec_dot_type(m.tg) == Q8_0) {
        if (a0_fits(n_pairs, k, m.n, max_active)) {
            HY_A0_SWITCH(m.tg, return (launch_k_gemm_fit<TT, true, a0_waves(TT), 1>(m, xq, k, n_pairs, order, order_n, egrp, max_active, nullptr, h, s)));
        }
        const int rt = (m.ff + 31) / 32;
        dim3 grid(rt, item_slots(rt, n_pairs, max_active, 3));
        HY_A0_SWITCH(m.tg, {
            hipLaunchKernelGGL((k_gemm_nl<TT, true>), grid, dim3(256), 0, s, m, (const uint8_t *) xq, k, order, order_n, egrp, nullptr, h);
            return check_launch("hy_moe_gemm_gate_up");
        });
    }
    if ((size_t) n_pairs * (m.n / 256) * Q8K_BYTES >= (1ull << 32)) { set_error("hy_moe_gemm_gate_up: activations of 4 GB or more"); return HY_EBAD_SHAPE; }
    if (k <= 0 || (uint64_t) n_pairs * (uint64_t) k >= (1ull << 32)) { set_error("hy_moe_gemm_gate_up: k out of range for the pair count"); return HY_EBAD_SHAPE; }
    if (max_items(n_pairs, max_active) >= GM_MAX_ITEMS) { set_error("hy_moe_gemm_gate_up: %d pairs make more than %d work items", n_pairs, GM_MAX_ITEMS - 1); return HY_EBAD_SHAPE; }
    // Q5_K: 16-wave blocks (256 weight rows, so every item's activations are read by half as many row blocks, and
    // four waves a SIMD) while that grid still has a block for every CU, and for a single expert: a shared expert's
    // GEMM, which runs beside the routing and the routed GEMMs on a second stream, then takes half the CUs and leaves
    // the rest to them (the 2048-token Q5_K/Q6_K chunk 690 -> 683 us; alone it takes 46 us against 32 at 8 waves and
    // twice the blocks).  Other small grids keep 8 waves.  ff is a multiple of 256, so either size tiles it.
    if (m.tg == Q5_K && (max_items(n_pairs, max_active) * (m.ff / 128) >= cu_count() || max_active == 1)) {
        return launch_k_gemm<Q5_K, true, 16, 1>(m, xq, k, n_pairs, order, order_n, egrp, max_active, nullptr, h, s);
    }
    HY_GEMM_SWITCH(m.tg, return (launch_k_gemm_fit<TT, true, g5_waves<TT, true>(), g5_blocks<TT, true>()>(m, xq, k, n_pairs, order, order_n, egrp, max_active, nullptr, h, s)));
}
int launch_gemm_down(const hy_moe_dev &m, const void *hq, int n_pairs, const int *order, const int *order_n, const int *egrp, int max_active,
                     const float *wts, float *y, hipStream_t s) {
    if (max_active <= 0 || n_pairs <= 0) return HY_OK;
    if (vec_dot_type(m.td) == Q8_0) {
        if (a0_fits(n_pairs, 1, m.ff, max_active)) {
            HY_A0_SWITCH(m.td, return (launch_k_gemm_fit<TT, false, a0_waves(TT), 1>(m, hq, 1, n_pairs, order, order_n, egrp, max_active, wts, y, s)));
        }
        const int rt = (m.n + GM_ROWS - 1) / GM_ROWS;
        dim3 grid(rt, item_slots(rt, n_pairs, max_active, 3));
        HY_A0_SWITCH(m.td, {
            hipLaunchKernelGGL((k_gemm_nl<TT, false>), grid, dim3(256), 0, s, m, (const uint8_t *) hq, 1, order, order_n, egrp, wts, y);
            return check_launch("hy_moe_gemm_down");
        });
    }
    if ((size_t) n_pairs * (m.ff / 256) * Q8K_BYTES >= (1ull << 32)) { set_error("hy_moe_gemm_down: activations of 4 GB or more"); return HY_EBAD_SHAPE; }
    if (max_items(n_pairs, max_active) >= GM_MAX_ITEMS) { set_error("hy_moe_gemm_down: %d pairs make more than %d work items", n_pairs, GM_MAX_ITEMS - 1); return HY_EBAD_SHAPE; }
    HY_GEMM_SWITCH(m.td, return (launch_k_gemm_fit<TT, false, g5_waves<TT, false>(), g5_blocks<TT, false>()>(m, hq, 1, n_pairs, order, order_n, egrp, max_active, wts, y, s)));
}

} // namespace hy
