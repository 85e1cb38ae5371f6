/* The span loads of the register-staged grouped GEMM (hyper_amd/csrc/hy_spans.cuh) on the CPU under AddressSanitizer and
   UBSan: a 16-row tile of spans that fills its allocation exactly, every row and lane quarter.  A load that leaves the
   tile, or a dword load off a dword boundary, is reported; the bytes loaded are checked against the blocks' fields.  Built
   by tests/sanitize/Makefile, run by tests/test_sanitize.py. */
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>

#define __device__
#define __forceinline__ inline
struct uint2 { uint32_t x, y; };
static inline uint2 make_uint2(uint32_t x, uint32_t y) { return uint2{x, y}; }
/* v_alignbyte_b32: the low 32 bits of hi:lo shifted right by s & 3 bytes */
static inline uint32_t alignbyte(uint32_t hi, uint32_t lo, uint32_t s) { return (uint32_t) ((((uint64_t) hi << 32) | lo) >> (8 * (s & 3))); }
#define __builtin_amdgcn_alignbyte alignbyte
#include "../../hyper_amd/csrc/hy_spans.cuh"

using namespace hy;

static int bad = 0;
static void same(const void *got, const uint8_t *want, int n, int type, int row, int q, int c, const char *what) {
    if (std::memcmp(got, want, n)) { std::printf("type %d row %d quarter %d block %d: %s\n", type, row, q, c, what); ++bad; }
}
static const void *scale(const SpanBytes<IQ4_NL> &w, int c) { return (const uint16_t *) w.dd + c; }
static const void *scale(const SpanBytes<Q8_0> &w, int c) { return (const uint16_t *) w.dd + c; }
static const void *scale(const SpanBytes<Q5_0> &w, int c) { return (const uint16_t *) w.dd + c; }
static const void *scale(const SpanBytes<MXFP4> &w, int c) { return (const uint8_t *) w.ee + c; }
static const void *scale(const SpanBytes<Q5_1> &w, int c) { return w.dm + c; }

template <int T> static void tile(int scale_bytes, int high, int quants) {   // byte offsets of the fifth bits (0: none) and quants
    const int bb = block_bytes(T), sb = 8 * bb;
    void *mem = nullptr;
    if (posix_memalign(&mem, 16, 16 * sb)) std::exit(2);   // as expert matrices are: a tile starts 16-byte aligned
    uint8_t *p = (uint8_t *) mem;
    for (int i = 0; i < 16 * sb; ++i) p[i] = (uint8_t) std::rand();
    for (int row = 0; row < 16; ++row)
        for (int q = 0; q < 4; ++q) {
            const uint8_t *blk = p + row * sb;
            SpanBytes<T> w;
            w.load(blk, q);
            for (int c = 0; c < 8; ++c) {
                same(&w.qv[c], blk + bb * c + quants + 8 * (T == Q8_0 ? q : q & 1), 8, T, row, q, c, "quants");
                same(scale(w, c), blk + bb * c, scale_bytes, T, row, q, c, "scale");
                if constexpr (T == Q5_0 || T == Q5_1) same((const uint8_t *) w.hb + c, blk + bb * c + high + q, 1, T, row, q, c, "fifth bits");
            }
        }
    std::free(mem);
}

int main() {
    tile<IQ4_NL>(2, 0, 2);
    tile<Q8_0>(2, 0, 2);
    tile<MXFP4>(1, 0, 1);
    tile<Q5_0>(2, 2, 6);
    tile<Q5_1>(4, 4, 8);
    std::printf("span_loads: %d wrong\n", bad);
    return bad != 0;
}
