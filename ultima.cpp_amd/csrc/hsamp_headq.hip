// The logits producer's quantised heads and its Hadamard fold on gfx950
// (reference src/model/qwen_model.cpp:182-207, src/model/weight_dispatch.cpp:106-146).
//
// k_head_prep, one block per batch row: the final rmsnorm in the reference's
//   order (src/kernels/rmsnorm.cpp:21-52: eight fused chains of x * x, their
//   horizontal sum and tail, mean, 1 / sqrt(mean + eps), (x * scale) * inv),
//   then, for a folded head, the Hadamard fold (src/kernels/hadamard.cpp:9-44:
//   signs, the butterflies a + b / a - b over each block, * fl(1 / sqrt(block)))
//   in LDS; the head's input rows are written to `normed`.
//
// The quantised matvec (k_head_q: up to four batch rows on the vector units;
//   k_head_qm: more, on the matrix cores). The reference's AVX2 kernels fix each
//   row's evaluation order -- for every type a set of partial sums (8 to 64),
//   each a chain of fused multiply-adds over the row in a fixed element order,
//   and a fixed reduction of them. The lanes of a row (two or four) each run
//   the chains of their own bytes of every block, so a row's chains stay in
//   registers, and the reduction crosses lanes once, at the end.
//   The bytes arrive in chunks of whole blocks (270-420 bytes per row):
//   coalesced 16-byte buffer loads of the rows' aligned spans, one chunk ahead
//   in registers, then a row-major LDS tile, from which each lane reads its
//   row's dwords (a byte shift by alignbyte where a block starts inside a
//   dword). The activation's chunk goes through LDS and is read 16 bytes at a
//   time. Values are unpacked a dword at a time into one value per byte (masks
//   and shifts over four values at once) and converted by byte.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>
#include <utility>

#include "hsamp_head.h"
#include "hsamp_wave.h"
#include "ultima_hsamp.h"

#pragma clang fp contract(off)

namespace hsamp {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// IEEE half -> float: exact, subnormals included
__device__ __forceinline__ float half_to_f32(uint32_t h) {
    return (float)__builtin_bit_cast(_Float16, (uint16_t)h);
}

__device__ __forceinline__ float hsum8(const float* p) {
    const float s0 = p[0] + p[4], s1 = p[1] + p[5], s2 = p[2] + p[6], s3 = p[3] + p[7];
    return (s0 + s1) + (s2 + s3);
}

// signed byte e of w (one sign-extending convert), unsigned byte e of w as a
// float (one v_cvt_f32_ubyte)
__device__ __forceinline__ int sbyte(uint32_t w, int e) { return (int)(w << (24 - 8 * e)) >> 24; }
__device__ __forceinline__ float ubytef(uint32_t w, int e) { return (float)((w >> (8 * e)) & 0xFFu); }
// four values, one to a byte: kept as one dword, so that each is one
// v_cvt_f32_ubyte (the compiler otherwise takes the masks apart into a bit-field
// extract per value: one instruction a value more)
__device__ __forceinline__ uint32_t bytes4(uint32_t w) {
    asm("" : "+v"(w));
    return w;
}
// bits 0..3 of t, one to a byte (bit k -> bit 0 of byte k)
__device__ __forceinline__ uint32_t spread4(uint32_t t) { return __umul24(t & 15u, 0x00204081u) & 0x01010101u; }

// ---- the row's bytes in the LDS tile ------------------------------------------
// A row's chunk starts at byte `sh` (0..15) of its tile slot. AL: the rows'
// chunks start on dwords, so a field's place in its dword is known (SC: the
// block's own, 0 or 2 bytes) and a dword is one LDS read, plus an alignbyte by
// a constant where it starts mid-dword; else any byte alignment (two reads and
// an alignbyte by the row's shift).
template <int AL>
struct RowBytes {
    const uint32_t* dw;   // the row's slot + (sh >> 2) dwords (+ the lane's own)
    int s3;               // sh & 3 (AL = 0 only)
    __device__ __forceinline__ RowBytes at(int dwords) const { return {dw + dwords, s3}; }
    template <int SC>
    __device__ __forceinline__ uint32_t ld32(int off) const {
        if (AL) {
            const int o = SC + off;
            const int i = o >> 2, r = o & 3;
            if (r == 0) return dw[i];
            return __builtin_amdgcn_alignbyte(dw[i + 1], dw[i], (uint32_t)r);
        }
        const int o = s3 + off;
        const int i = o >> 2;
        return __builtin_amdgcn_alignbyte(dw[i + 1], dw[i], (uint32_t)(o & 3));
    }
    // byte `off` of the row's chunk (SC added by the caller's offset)
    template <int SC>
    __device__ __forceinline__ int sbyte_at(int off) const {
        return reinterpret_cast<const signed char*>(dw)[(AL ? SC : s3) + off];
    }
};

// ---- the formats -----------------------------------------------------------------
// BE values per block, BB bytes per block; NA chains per row; LPR lanes of a
// row (k_head_q); BPC blocks per chunk of k_head_q (whole dwords), MPC of
// k_head_qm. Formats of 32 or 64 chains: block(rb, t, c, sink) unpacks
// lane t's (0..3) values of the block, and calls sink(slot, off, v) for four
// consecutive chains of the lane and the four consecutive values v at element
// off + (the lane's own offset, XL * t) -- in each chain's order. With 64
// chains, c selects the half of 32 it goes over.

// Q4_1 (matvec_q4_1_f32.cpp:47-75 over dequant_q4_1.cpp:46-54): value j =
// fl(nib * d + m) (fused as GCC compiles it), j + 16 the high nibble; value i
// into partial i. Slots: 4t + i, then 16 + 4t + i.
struct FQ4_1 {
    static constexpr int BE = 32, BB = 20, NA = 32, LPR = 4, BPC = 16, MPC = 8, XL = 4;
    template <int SC, class RB, class S>
    __device__ __forceinline__ static void block(const RB& rb, int t, int, const S& sink) {
        const uint32_t h = rb.template ld32<SC>(0);
        const float d = half_to_f32(h & 0xFFFFu), m = half_to_f32(h >> 16);
        const uint32_t q = rb.at(t).template ld32<SC>(4);
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
            const uint32_t n = bytes4((q >> (4 * hi)) & 0x0F0F0F0Fu);
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(ubytef(n, e), d, m);
            sink(4 * hi, 16 * hi, v);
        }
    }
};

// Q5_0 (matvec_q5_0_f32.cpp:108-150): value i = (nib | bit i of qh << 4) - 16,
// scaled fl(q * d) on its own, into partial i. Slots as Q4_1.
struct FQ5_0 {
    static constexpr int BE = 32, BB = 22, NA = 32, LPR = 4, BPC = 16, MPC = 8, XL = 4;
    template <int SC, class RB, class S>
    __device__ __forceinline__ static void block(const RB& rb, int t, int, const S& sink) {
        const float d8 = half_to_f32(rb.template ld32<SC>(0) & 0xFFFFu) * 0.125f;
        const uint32_t qh = rb.template ld32<SC>(2) >> (4 * t);
        const uint32_t q = rb.at(t).template ld32<SC>(6);
#pragma unroll
        for (int hi = 0; hi < 2; ++hi) {
            // the five-bit values nibble | fifth bit << 4, as the bytes 8 (q - 16):
            // one signed convert each, and 8 (q - 16) * d / 8 is fl((q - 16) * d)
            // (d / 8 is exact: d is a half)
            const uint32_t nib = (hi ? q >> 1 : q << 3) & 0x78787878u;
            const uint32_t n = bytes4((nib | (spread4(qh >> (16 * hi)) << 7)) ^ 0x80808080u);
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) v[e] = (float)sbyte(n, e) * d8;
            sink(4 * hi, 16 * hi, v);
        }
    }
};

// The eight six-bit scales and mins of a Q4_K / Q5_K super-block's 12-byte
// table (bytes 4..15 of the block, in s[0..2]), one to a byte: 0..3 in sc[0]
// and mn[0], 4..7 in sc[1] and mn[1]; matvec_q4k_f32.cpp:45-55
__device__ __forceinline__ void scales_min_k4(const uint32_t* s, uint32_t* sc, uint32_t* mn) {
    sc[0] = bytes4(s[0] & 0x3F3F3F3Fu);
    mn[0] = bytes4(s[1] & 0x3F3F3F3Fu);
    sc[1] = bytes4((s[2] & 0x0F0F0F0Fu) | ((s[0] >> 2) & 0x30303030u));
    mn[1] = bytes4(((s[2] >> 4) & 0x0F0F0F0Fu) | ((s[1] >> 2) & 0x30303030u));
}

// Q4_K (matvec_q4k_f32.cpp:108-160): pair j's low nibbles are values 64j + l
// (partial l), its high nibbles 64j + 32 + l (partial 32 + l); each value
// fl(nib * d1 - m1) fused. Lane t: l = 8t .. 8t + 7; c: low or high.
struct FQ4_K {
    static constexpr int BE = 256, BB = 144, NA = 64, LPR = 4, BPC = 2, MPC = 1, XL = 8;
    template <int SC, class RB, class S>
    __device__ __forceinline__ static void block(const RB& rb, int t, int c, const S& sink) {
        const uint32_t h = rb.template ld32<SC>(0);
        const float d = half_to_f32(h & 0xFFFFu), dmin = half_to_f32(h >> 16);
        uint32_t s[3], sc[2], mn[2];
#pragma unroll
        for (int k = 0; k < 3; ++k) s[k] = rb.template ld32<SC>(4 + 4 * k);
        scales_min_k4(s, sc, mn);
#pragma unroll
        for (int k = 0; k < 2; ++k) {
            sc[k] = bytes4(sc[k] >> (8 * c));
            mn[k] = bytes4(mn[k] >> (8 * c));
        }
        const RB rl = rb.at(2 * t);
#pragma unroll
        for (int j = 0; j < 4; ++j) {
            // scale and min 2j + c
            const float d1 = d * ubytef(sc[j >> 1], 2 * (j & 1)), m1 = dmin * ubytef(mn[j >> 1], 2 * (j & 1));
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t n = bytes4((rl.template ld32<SC>(16 + 32 * j + 4 * k) >> (4 * c)) & 0x0F0F0F0Fu);
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(ubytef(n, e), d1, -m1);
                sink(4 * k, 64 * j + 32 * c + 4 * k, v);
            }
        }
    }
};

// Q5_K (matvec_q5k_f32.cpp:48-80 over dequant_q5k.cpp:57-93): value e of the
// super-block = fl(d1 * q - m1) (fused as GCC compiles it) into partial e % 32,
// in increasing e. Lane t: partials 8t .. 8t + 7.
struct FQ5_K {
    static constexpr int BE = 256, BB = 176, NA = 32, LPR = 4, BPC = 2, MPC = 1, XL = 8;
    template <int SC, class RB, class S>
    __device__ __forceinline__ static void block(const RB& rb, int t, int, const S& sink) {
        const uint32_t h = rb.template ld32<SC>(0);
        const float d = half_to_f32(h & 0xFFFFu), dmin = half_to_f32(h >> 16);
        uint32_t s[3], sc[2], mn[2];
#pragma unroll
        for (int k = 0; k < 3; ++k) s[k] = rb.template ld32<SC>(4 + 4 * k);
        scales_min_k4(s, sc, mn);
        const RB rl = rb.at(2 * t);
        const uint32_t qh[2] = {rl.template ld32<SC>(16), rl.template ld32<SC>(20)};
#pragma unroll
        for (int j = 0; j < 4; ++j)
#pragma unroll
            for (int hi = 0; hi < 2; ++hi) {
                const int g = 2 * j + hi;
                const float d1 = d * ubytef(sc[g >> 2], g & 3), m1 = dmin * ubytef(mn[g >> 2], g & 3);
#pragma unroll
                for (int k = 0; k < 2; ++k) {
                    const uint32_t q = rl.template ld32<SC>(48 + 32 * j + 4 * k);
                    // the five-bit values, one to a byte
                    const uint32_t n = bytes4(((q >> (4 * hi)) & 0x0F0F0F0Fu) | (((qh[k] >> g) & 0x01010101u) << 4));
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = __builtin_fmaf(d1, ubytef(n, e), -m1);
                    sink(4 * k, 32 * g + 4 * k, v);
                }
            }
    }
};

// Q6_K (matvec_q6k_f32.cpp:99-169): per half, runs r = 0..3 of 32 six-bit
// values q - 32, value l of run r scaled fl(q * fl(d * sc[2r + l / 16])) on its
// own and fused into partial (r % 2) * 32 + l, runs in order. Lane t:
// l = 8t .. 8t + 7; c: runs c and c + 2.
struct FQ6_K {
    static constexpr int BE = 256, BB = 210, NA = 64, LPR = 4, BPC = 2, MPC = 1, XL = 8;
    template <int SC, class RB, class S>
    __device__ __forceinline__ static void block(const RB& rb, int t, int c, const S& sink) {
        const float d4 = half_to_f32(rb.template ld32<SC>(208) & 0xFFFFu) * 0.25f;
        const RB rl = rb.at(2 * t);
#pragma unroll
        for (int half = 0; half < 2; ++half) {
            // scales 2c and 2c + 4 of the half, of the lane's sixteen values, over 4:
            // exact (a half times a small integer), so 4 (q - 32) * s / 4 is
            // fl((q - 32) * s)
            const int so = 192 + 8 * half + 2 * c + (t >> 1);
            const float s0 = d4 * (float)rb.template sbyte_at<SC>(so), s1 = d4 * (float)rb.template sbyte_at<SC>(so + 4);
#pragma unroll
            for (int k = 0; k < 2; ++k) {
                const uint32_t l = rl.at(8 * c).template ld32<SC>(64 * half + 4 * k);
                const uint32_t h = rl.template ld32<SC>(128 + 32 * half + 4 * k) >> (2 * c);
                // the six-bit values as the bytes 4 (q - 32): one signed convert each
                const uint32_t q0 = bytes4((((l << 2) & 0x3C3C3C3Cu) | ((h << 6) & 0xC0C0C0C0u)) ^ 0x80808080u);
                const uint32_t q1 = bytes4((((l >> 2) & 0x3C3C3C3Cu) | ((h << 2) & 0xC0C0C0C0u)) ^ 0x80808080u);
                float v[4];
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = (float)sbyte(q0, e) * s0;
                sink(4 * k, 128 * half + 32 * c + 4 * k, v);
#pragma unroll
                for (int e = 0; e < 4; ++e) v[e] = (float)sbyte(q1, e) * s1;
                sink(4 * k, 128 * half + 32 * c + 64 + 4 * k, v);
            }
        }
    }
};

// Q8_0 (matvec_q8_0_f32.cpp:83-117): per block, lane l of a block accumulator
// takes values 8c + l (c = 0..3) from zero; then row partial l += d * it.
struct FQ8_0 {
    static constexpr int BE = 32, BB = 34, NA = 8, LPR = 2, BPC = 8, MPC = 8, XL = 4;
};

// PQ2_0 (matvec_pq2_0_f32.cpp:111-184, its vectorised path): per block, lane
// l of one accumulator takes, for code position j = 0..3 and byte group
// g = 0..3, byte i = 8g + l's code j times x[4i + j] (fused, from zero); the
// row sum += d * (horizontal sum - the block's plain sequential sum of x)
// (fused as GCC compiles it).
struct FPQ2_0 {
    static constexpr int BE = 128, BB = 34, NA = 8, LPR = 2, BPC = 4, XL = 16;
};

template <int T> struct FmtOf;
template <> struct FmtOf<ULTIMA_HSAMP_HEAD_Q4_K> { using F = FQ4_K; };
template <> struct FmtOf<ULTIMA_HSAMP_HEAD_Q5_K> { using F = FQ5_K; };
template <> struct FmtOf<ULTIMA_HSAMP_HEAD_Q6_K> { using F = FQ6_K; };
template <> struct FmtOf<ULTIMA_HSAMP_HEAD_Q8_0> { using F = FQ8_0; };
template <> struct FmtOf<ULTIMA_HSAMP_HEAD_Q4_1> { using F = FQ4_1; };
template <> struct FmtOf<ULTIMA_HSAMP_HEAD_Q5_0> { using F = FQ5_0; };
template <> struct FmtOf<ULTIMA_HSAMP_HEAD_PQ2_0> { using F = FPQ2_0; };

constexpr int kMaxPqBlocks = 512;   // PQ2_0 block sums kept in LDS: H <= 65536

// ---- chunks of rows into LDS -------------------------------------------------------
// R rows' chunks of PC blocks, loaded by NT threads through one buffer
// resource based at the first row (16-byte aligned down; `delta` bytes before
// it): 32-bit offsets (offsets_fit), loads past the rows' end read 0. The slots are NV
// 16-byte vectors padded to S dwords (S = 8 mod 32: the rows' 8-byte reads
// spread over the banks).
template <class F, int PC, int R, int NT>
struct Tile {
    static constexpr int CB = F::BB * PC;                  // bytes per chunk (whole dwords)
    static constexpr bool DW = CB % 4 == 0;                // dword-aligned rows: every chunk starts on a dword
    static constexpr int NV = (CB + 15 + 15) / 16;         // 16-byte vectors of a row's aligned span
    static constexpr int S = (4 * NV + 31 - 8) / 32 * 32 + 8;
    static constexpr int N = (R * NV + NT - 1) / NT;       // vectors per thread
    static constexpr int WORDS = R * S + 4;
    static_assert(S >= 4 * NV, "a slot holds its vectors");
    // chunks of whole 16-byte granules keep their rows' place in a granule, and
    // ask for the NV granules at any place: one addition a vector
    static constexpr bool G16 = CB % 16 == 0;
    __amdgpu_buffer_rsrc_t rs;
    uint32_t delta;
    uint32_t ofs[N];                                       // G16: the vector's offset in chunk 0; else its row's
    int seg[N], at[N];
    u32x4 reg[N];
    // w: the rows' first byte; rows: how many there are (0..R)
    __device__ __forceinline__ void init(const unsigned char* w, int rows, int64_t rb, int tid) {
        const uintptr_t b0 = reinterpret_cast<uintptr_t>(w);
        delta = (uint32_t)(b0 & 15u);
        // rounded up to 16 bytes (a 16-byte load is out of range as a whole
        // when it reaches past the end: the granule holding the rows' last byte
        // is read in full; it lies in that byte's page)
        const int64_t n = rows > 0 ? (delta + rows * rb + 15) & ~(int64_t)15 : 0;
        rs = __builtin_amdgcn_make_buffer_rsrc(reinterpret_cast<void*>(b0 - delta), (short)0, (int)n, 0x00020000);
#pragma unroll
        for (int i = 0; i < N; ++i) {
            const int v = min(tid + NT * i, R * NV - 1), r = v / NV;
            seg[i] = v - r * NV;
            at[i] = r * S + 4 * seg[i];
            ofs[i] = delta + (uint32_t)((int64_t)r * rb);
            if (G16) ofs[i] = (ofs[i] & ~15u) + 16u * (uint32_t)seg[i];
        }
    }
    // With the default cache policy: a span shares its first and last 128-byte
    // lines with the chunks before and after it, which then mostly find them in
    // L2 (from HBM come 1.18 times the bytes with Q6_K, 1.28 with Q8_0).
    // (not G16: only the granules of the rows' spans are asked for; an offset
    // past the range makes the rest read 0 without touching memory)
    __device__ __forceinline__ void load(int c, int nb) {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            uint32_t o = ofs[i] + (uint32_t)c * CB;
            if (!G16) {
                const uint32_t end = o + (uint32_t)(min(PC, nb - c * PC) * F::BB);
                o = (o & ~15u) + 16u * (uint32_t)seg[i];
                o = o < end ? o : 0xFFFFFFF0u;
            }
            reg[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0);
        }
    }
    __device__ __forceinline__ void store(uint32_t* tile, int tid) const {
#pragma unroll
        for (int i = 0; i < N; ++i)
            if ((R * NV) % NT == 0 || tid + NT * i < R * NV) *reinterpret_cast<u32x4*>(tile + at[i]) = reg[i];
    }
    // row r's bytes of chunk c
    template <int AL>
    __device__ __forceinline__ RowBytes<AL> row(const uint32_t* tile, int r, int64_t rb, int c) const {
        const int sh = (int)((delta + (uint32_t)((int64_t)r * rb) + (uint32_t)c * CB) & 15u);
        return {tile + r * S + (sh >> 2), sh & 3};
    }
};

// n rows of H activation values (H a multiple of 4: a 16-byte load lies inside
// the rows or past them): loads past the last row read 0, those past a row's
// end the next row's, which no block uses. 32-bit offsets: n * H * 4 < 2^32
// (offsets_fit).
struct Rows {
    __amdgpu_buffer_rsrc_t rs;
    uint32_t row;   // bytes
    __device__ __forceinline__ Rows(const float* x, int n, int H)
        : rs(__builtin_amdgcn_make_buffer_rsrc(const_cast<float*>(x), (short)0, (int)((uint32_t)n * (uint32_t)H * 4u),
                                               0x00020000)),
          row((uint32_t)H * 4u) {}
    __device__ __forceinline__ uint32_t offset(int j, int k) const { return (uint32_t)j * row + 4u * (uint32_t)k; }
    __device__ __forceinline__ u32x4 load(uint32_t o) const { return __builtin_amdgcn_raw_buffer_load_b128(rs, o, 0, 0); }
};

// a row's fields move by BB bytes per block: the shift class of block j of a chunk
template <class F>
constexpr int shift_class(int j) { return F::BB * j & 3; }

// the sum over the lanes that differ in bit `m` of the lane index (a + b = b + a)
__device__ __forceinline__ float xadd(float v, int m) { return v + __shfl_xor(v, m, 64); }

// NB: batch rows. Four waves, each with its own 64 / LPR vocabulary rows and
// its own tile (no block barrier: a wave's LDS accesses are in order, and
// wave_sync keeps the compiler from moving a chunk's stores over the other
// lanes' reads of the chunk before); the activation's chunk is shared,
// double-buffered, one barrier per chunk.
// Lane LPR r + t: row r's lane t.
//
// Bound by the vector units (4 to 6 instructions a value: unpack, convert,
// scale, multiply-add) with the weights' stream close behind. One wave per 64
// rows with a row per lane left 2.3 waves per SIMD: latency. H = 4096,
// V = 151936, one row, k_head_prep's 6 us included, before -> now, us: Q4_K
// 161 -> 105, Q5_K 159 -> 103, Q6_K 268 -> 119, Q8_0 190 -> 147, Q4_1 147 -> 97,
// Q5_0 203 -> 113, PQ2_0 117 -> 74; four rows, Q4_K 280 -> 162, Q6_K 467 -> 194.
template <int T, int NB, int AL>
__global__ __launch_bounds__(256) void k_head_q(const unsigned char* __restrict__ w, int V, int H, int64_t rb,
                                                const float* __restrict__ xin, int rows, float logit_scale,
                                                float* __restrict__ logits, int64_t lstride) {
    using F = typename FmtOf<T>::F;
    constexpr bool PQ = T == ULTIMA_HSAMP_HEAD_PQ2_0, Q8 = T == ULTIMA_HSAMP_HEAD_Q8_0;
    constexpr int LPR = F::LPR, R = 64 / LPR, CE = F::BE * F::BPC;
    constexpr int NS = PQ ? 1 : F::NA / LPR;               // chains (PQ2_0: row sums) per lane
    constexpr int NX = (CE / 4 * NB + 255) / 256;          // 16-byte vectors of the activation per thread
    using W = Tile<F, F::BPC, R, 64>;
    __shared__ __attribute__((aligned(16))) uint32_t tiles[4][(W::WORDS + 3) / 4 * 4];
    __shared__ __attribute__((aligned(16))) float xl[2][NB][CE];
    __shared__ float bsum[PQ ? NB * kMaxPqBlocks : 1];
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int m0 = (blockIdx.x * 4 + wave) * R;
    const int r = lane / LPR, t = lane % LPR;
    const int b0 = blockIdx.y * NB;
    const int nb = H / F::BE;                              // blocks per row
    const int nC = (nb + F::BPC - 1) / F::BPC;
    auto xrow = [&](int b) { return xin + (int64_t)min(b0 + b, rows - 1) * H; };
    const Rows xr(xin + (int64_t)b0 * H, min(NB, rows - b0), H);

    W tile;
    tile.init(w + (int64_t)min(m0, V) * rb, max(0, min(R, V - m0)), rb, lane);
    u32x4 xv[NX];
    uint32_t xo[NX];
#pragma unroll
    for (int i = 0; i < NX; ++i) {
        const int n = min(tid + 256 * i, CE / 4 * NB - 1);
        xo[i] = xr.offset(n / (CE / 4), n % (CE / 4) * 4);
    }
    auto load_x = [&](int c) {
#pragma unroll
        for (int i = 0; i < NX; ++i) xv[i] = xr.load(xo[i] + (uint32_t)c * (CE * 4));
    };
    auto store_x = [&](int buf) {
#pragma unroll
        for (int i = 0; i < NX; ++i) {
            const int n = tid + 256 * i;
            if (CE / 4 * NB % 256 == 0 || n < CE / 4 * NB)
                reinterpret_cast<u32x4*>(&xl[buf][0][0])[n] = xv[i];
        }
    };
    if (nC > 0) {
        tile.load(0, nb);
        load_x(0);
    }
    if (PQ) {
        // the activation's block sums, plain sequential float sums
        for (int k = tid; k < nb * NB; k += 256) {
            const float* xs = xrow(k / nb) + k % nb * F::BE;
            float sum = 0.0f;
            for (int i = 0; i < F::BE; i += 32) {
                f32x4_a4 v[8];
#pragma unroll
                for (int e = 0; e < 8; ++e) v[e] = *reinterpret_cast<const f32x4_a4*>(xs + i + 4 * e);
#pragma unroll
                for (int e = 0; e < 8; ++e) sum = (((sum + v[e].x) + v[e].y) + v[e].z) + v[e].w;
            }
            bsum[k / nb * kMaxPqBlocks + k % nb] = sum;
        }
    }
    float a[NB][NS];
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
        for (int i = 0; i < NS; ++i) a[b][i] = 0.0f;
    uint32_t* mine = tiles[wave];
    for (int c = 0; c < nC; ++c) {
        wave_sync();                                       // the lanes' reads of the chunk before are done
        tile.store(mine, lane);
        store_x(c & 1);
        __syncthreads();
        const int cn = min(c + 1, nC - 1);
        tile.load(cn, nb);
        load_x(cn);
        __builtin_amdgcn_sched_barrier(0);                 // (the loads stay ahead of the chunk's work)
        const int nblk = min(F::BPC, nb - c * F::BPC);
        const RowBytes<AL> row = tile.template row<AL>(mine, r, rb, c);
        const float* xc = &xl[c & 1][0][0] + F::XL * t;
        auto one = [&](auto jc) {
            constexpr int j = decltype(jc)::value;
            constexpr int SC = AL ? shift_class<F>(j) : 0;
            // (AL: the block's offset less its shift class is whole dwords)
            const RowBytes<AL> rbj = AL ? row.at((j * F::BB - SC) / 4)
                                        : RowBytes<AL>{row.dw + ((row.s3 + j * F::BB) >> 2), (row.s3 + j * F::BB) & 3};
            const float* xj = xc + j * F::BE;
            if constexpr (Q8) {
                const float d = half_to_f32(rbj.template ld32<SC>(0) & 0xFFFFu);
                float bk[NB][4];
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) bk[b][e] = 0.0f;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const uint32_t q = rbj.at(t).template ld32<SC>(2 + 8 * s);
                    float v[4];
#pragma unroll
                    for (int e = 0; e < 4; ++e) v[e] = (float)sbyte(q, e);
#pragma unroll
                    for (int b = 0; b < NB; ++b) {
                        const float4 x = *reinterpret_cast<const float4*>(xj + b * CE + 8 * s);
                        bk[b][0] = __builtin_fmaf(v[0], x.x, bk[b][0]);
                        bk[b][1] = __builtin_fmaf(v[1], x.y, bk[b][1]);
                        bk[b][2] = __builtin_fmaf(v[2], x.z, bk[b][2]);
                        bk[b][3] = __builtin_fmaf(v[3], x.w, bk[b][3]);
                    }
                }
#pragma unroll
                for (int b = 0; b < NB; ++b)
#pragma unroll
                    for (int e = 0; e < 4; ++e) a[b][e] = __builtin_fmaf(d, bk[b][e], a[b][e]);
            } else if constexpr (PQ) {
                const float d = half_to_f32(rbj.template ld32<SC>(0) & 0xFFFFu);
                uint32_t q[4];
#pragma unroll
                for (int g = 0; g < 4; ++g) q[g] = rbj.at(t).template ld32<SC>(2 + 8 * g);
#pragma unroll
                for (int b = 0; b < NB; ++b) {
                    float4 x[4][4];
#pragma unroll
                    for (int g = 0; g < 4; ++g)
#pragma unroll
                        for (int e = 0; e < 4; ++e)
                            x[g][e] = *reinterpret_cast<const float4*>(xj + b * CE + 32 * g + 4 * e);
                    float acc[4] = {0.0f, 0.0f, 0.0f, 0.0f};
                    auto pos = [&](int jp, auto of) {
#pragma unroll
                        for (int g = 0; g < 4; ++g) {
                            const uint32_t cj = bytes4((q[g] >> (2 * jp)) & 0x03030303u);
#pragma unroll
                            for (int e = 0; e < 4; ++e) acc[e] = __builtin_fmaf(ubytef(cj, e), of(x[g][e]), acc[e]);
                        }
                    };
                    pos(0, [](const float4& v) { return v.x; });
                    pos(1, [](const float4& v) { return v.y; });
                    pos(2, [](const float4& v) { return v.z; });
                    pos(3, [](const float4& v) { return v.w; });
                    // p_l + p_{l+4}, then as hsum8 (both lanes of the row)
                    const float s0 = xadd(acc[0], 1), s1 = xadd(acc[1], 1), s2 = xadd(acc[2], 1), s3 = xadd(acc[3], 1);
                    const float hs = (s0 + s1) + (s2 + s3);
                    a[b][0] = __builtin_fmaf(d, hs - bsum[b * kMaxPqBlocks + c * F::BPC + j], a[b][0]);
                }
            } else {
#pragma unroll
                for (int ch = 0; ch < (F::NA == 64 ? 2 : 1); ++ch)
                    F::template block<SC>(rbj, t, ch, [&](int slot, int off, const float (&v)[4]) {
#pragma unroll
                        for (int b = 0; b < NB; ++b) {
                            const float4 x = *reinterpret_cast<const float4*>(xj + b * CE + off);
                            float* p = a[b] + 8 * ch + slot;
                            p[0] = __builtin_fmaf(v[0], x.x, p[0]);
                            p[1] = __builtin_fmaf(v[1], x.y, p[1]);
                            p[2] = __builtin_fmaf(v[2], x.z, p[2]);
                            p[3] = __builtin_fmaf(v[3], x.w, p[3]);
                        }
                    });
            }
        };
        auto all = [&]<int... J>(std::integer_sequence<int, J...>) {
            ((J < nblk ? one(std::integral_constant<int, J>()) : void()), ...);
        };
        all(std::make_integer_sequence<int, F::BPC>());
    }
    const int m = m0 + r;
#pragma unroll
    for (int b = 0; b < NB; ++b) {
        // the reference's reduction of the partials over the row's lanes
        float y;
        if constexpr (PQ) {
            y = a[b][0];
        } else if constexpr (Q8) {
            // lane t holds partials 4t + e
            const float s0 = xadd(a[b][0], 1), s1 = xadd(a[b][1], 1), s2 = xadd(a[b][2], 1), s3 = xadd(a[b][3], 1);
            y = (s0 + s1) + (s2 + s3);
        } else if constexpr (F::BE == 256) {
            // lane t holds partials 8t + e (and 32 + 8t + e): groups of eight
            // summed pairwise, ((0 + 1) + (2 + 3)) + ((4 + 5) + (6 + 7))
            float s[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                s[e] = xadd(xadd(a[b][e], 1), 2);
                if constexpr (F::NA == 64) s[e] = s[e] + xadd(xadd(a[b][8 + e], 1), 2);
            }
            y = hsum8(s);
        } else {
            // lane t holds partials 4t + e and 16 + 4t + e: (0 + 1) + (2 + 3) of
            // groups of eight, then p_e + p_{e+4}
            float s[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) s[e] = xadd(xadd(a[b][e], 2) + xadd(a[b][4 + e], 2), 1);
            y = (s[0] + s[1]) + (s[2] + s[3]);
        }
        if (t != 0 || m >= V || b0 + b >= rows) continue;
        if (logit_scale != 1.0f && logit_scale != 0.0f) y = y * (1.0f / logit_scale);
        logits[(int64_t)(b0 + b) * lstride + m] = y;
    }
}

// More than four batch rows: the chains as f32 matrix instructions with K = 1
// (one fused multiply-add per output, the same bits; hsamp_headm.hip), 16
// vocabulary rows x 16 batch rows x four lanes' chains each. Lane 16 t + i
// unpacks row i's lane t values (the formats' `block`), one register of which
// is one instruction's operand, and reads batch row i's values at the same
// elements. The block's four waves: NC halves of the chains (64-chain formats:
// 128 accumulator registers a wave) by 4 / NC groups of sixteen vocabulary
// rows; tile and activation are shared through LDS.
//
// Bound by the matrix pipe (busy 0.48 of the SIMDs' cycles) and the unpacking,
// which share the SIMD's issue. H = 4096, V = 151936, sixteen rows, passes of four rows through
// the vector units -> now, us: Q4_K 935 -> 295, Q5_K 931 -> 285, Q6_K
// 1638 -> 336, Q8_0 909 -> 350, Q4_1 975 -> 265, Q5_0 1361 -> 287; 64 rows, Q4_K
// 3630 -> 1120. Not faster: two or four batch tiles a block, double buffers,
// interleaved scheduling groups.
template <int T, int AL>
__global__ __launch_bounds__(256, 2) void k_head_qm(const unsigned char* __restrict__ w, int V, int H, int64_t rb,
                                                    const float* __restrict__ xin, int rows, float logit_scale,
                                                    float* __restrict__ logits, int64_t lstride) {
    using F = typename FmtOf<T>::F;
    constexpr bool Q8 = T == ULTIMA_HSAMP_HEAD_Q8_0;
    constexpr int NC = F::NA == 64 ? 2 : 1, VG = 4 / NC, R = 16 * VG;
    constexpr int CE = F::BE * F::MPC, XS = CE + 4;        // (rows padded: 16-byte reads without conflicts)
    constexpr int NSL = Q8 ? 2 : F::NA / (4 * NC);         // chains per lane
    constexpr int NX = 16 * CE / (4 * 256);                // 16-byte vectors of the activation per thread
    using W = Tile<F, F::MPC, R, 256>;
    static_assert(!AL || W::DW, "chunks that start inside a dword: AL = 0");
    __shared__ __attribute__((aligned(16))) uint32_t tl[(W::WORDS + 3) / 4 * 4];
    __shared__ __attribute__((aligned(16))) float xl[16 * XS];
    static_assert(NC == 1 || 16 * XS >= VG * 32 * 64, "the halves' sums fit the activation's buffer");
    const int tid = threadIdx.x, lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int ch = wave % NC, vg = wave / NC;
    const int i = lane & 15, t = lane >> 4;
    const int m0 = blockIdx.x * R;
    const int b0 = blockIdx.y * 16;
    const int nb = H / F::BE;
    const int nC = (nb + F::MPC - 1) / F::MPC;
    W tile;
    tile.init(w + (int64_t)m0 * rb, min(R, V - m0), rb, tid);
    const Rows xr(xin + (int64_t)b0 * H, min(16, rows - b0), H);
    u32x4 xv[NX];
    uint32_t xo[NX];
#pragma unroll
    for (int k = 0; k < NX; ++k) {
        const int n = tid + 256 * k;
        xo[k] = xr.offset(n / (CE / 4), n % (CE / 4) * 4);
    }
    auto load_x = [&](int c) {
#pragma unroll
        for (int k = 0; k < NX; ++k) xv[k] = xr.load(xo[k] + (uint32_t)c * (CE * 4));
    };
    auto store_x = [&]() {
#pragma unroll
        for (int k = 0; k < NX; ++k) {
            const int n = tid + 256 * k, j = n / (CE / 4);
            *reinterpret_cast<u32x4*>(&xl[j * XS + n % (CE / 4) * 4]) = xv[k];
        }
    };
    f32x16 a[NSL];
#pragma unroll
    for (int s = 0; s < NSL; ++s)
#pragma unroll
        for (int e = 0; e < 16; ++e) a[s][e] = 0.0f;
    if (nC > 0) {
        tile.load(0, nb);
        load_x(0);
    }
    for (int c = 0; c < nC; ++c) {
        __syncthreads();                                   // the chunk before is done with
        tile.store(tl, tid);
        store_x();
        __syncthreads();
        const int cn = min(c + 1, nC - 1);
        tile.load(cn, nb);
        load_x(cn);
        __builtin_amdgcn_sched_barrier(0);                 // (the loads stay ahead of the chunk's work)
        const int nblk = min(F::MPC, nb - c * F::MPC);
        const RowBytes<AL> row = tile.template row<AL>(tl, 16 * vg + i, rb, c);
        const float* xj0 = xl + i * XS + (Q8 ? 2 : F::XL) * t;
        auto one = [&](auto jc) {
            constexpr int j = decltype(jc)::value;
            constexpr int SC = AL ? shift_class<F>(j) : 0;
            const RowBytes<AL> rbj = AL ? row.at((j * F::BB - SC) / 4)
                                        : RowBytes<AL>{row.dw + ((row.s3 + j * F::BB) >> 2), (row.s3 + j * F::BB) & 3};
            const float* xj = xj0 + j * F::BE;
            if constexpr (Q8) {
                // lane t: values 8s + 2t and 8s + 2t + 1, partials 2t and 2t + 1
                const float d = half_to_f32(rbj.template ld32<SC>(0) & 0xFFFFu);
                f32x16 bk[2];
#pragma unroll
                for (int e = 0; e < 16; ++e) bk[0][e] = bk[1][e] = 0.0f;
#pragma unroll
                for (int s = 0; s < 4; ++s) {
                    const float2 x = *reinterpret_cast<const float2*>(xj + 8 * s);
                    bk[0] = __builtin_amdgcn_mfma_f32_16x16x1f32((float)rbj.template sbyte_at<SC>(2 + 8 * s + 2 * t), x.x, bk[0], 0, 0, 0);
                    bk[1] = __builtin_amdgcn_mfma_f32_16x16x1f32((float)rbj.template sbyte_at<SC>(3 + 8 * s + 2 * t), x.y, bk[1], 0, 0, 0);
                }
                // the outputs' rows 4t + q: their blocks' scales from lanes 4t + q
#pragma unroll
                for (int q = 0; q < 4; ++q) {
                    const float dq = __shfl(d, 4 * t + q, 64);
#pragma unroll
                    for (int k = 0; k < 4; ++k) {
                        a[0][4 * k + q] = __builtin_fmaf(dq, bk[0][4 * k + q], a[0][4 * k + q]);
                        a[1][4 * k + q] = __builtin_fmaf(dq, bk[1][4 * k + q], a[1][4 * k + q]);
                    }
                }
            } else {
                F::template block<SC>(rbj, t, NC == 2 ? ch : 0, [&](int slot, int off, const float (&v)[4]) {
                    const float4 x = *reinterpret_cast<const float4*>(xj + off);
                    a[slot] = __builtin_amdgcn_mfma_f32_16x16x1f32(v[0], x.x, a[slot], 0, 0, 0);
                    a[slot + 1] = __builtin_amdgcn_mfma_f32_16x16x1f32(v[1], x.y, a[slot + 1], 0, 0, 0);
                    a[slot + 2] = __builtin_amdgcn_mfma_f32_16x16x1f32(v[2], x.z, a[slot + 2], 0, 0, 0);
                    a[slot + 3] = __builtin_amdgcn_mfma_f32_16x16x1f32(v[3], x.w, a[slot + 3], 0, 0, 0);
                });
            }
        };
        auto all = [&]<int... J>(std::integer_sequence<int, J...>) {
            ((J < nblk ? one(std::integral_constant<int, J>()) : void()), ...);
        };
        all(std::make_integer_sequence<int, F::MPC>());
    }
    // Lane 16 t + i holds, for vocabulary rows 4t + q and batch row i, slot s's
    // chain of lane k in a[s][4k + q]: the reference's reduction.
    float s8[4][8];
#pragma unroll
    for (int q = 0; q < 4; ++q)
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            if constexpr (Q8) s8[q][e] = a[e & 1][4 * (e >> 1) + q];
            else if constexpr (F::BE == 256)
                s8[q][e] = (a[e][q] + a[e][4 + q]) + (a[e][8 + q] + a[e][12 + q]);
            else {
                const int k = e >> 2, f = e & 3;           // partials 8g + e: lanes k and k + 2, low and high
                s8[q][e] = (a[f][4 * k + q] + a[f][8 + 4 * k + q]) + (a[4 + f][4 * k + q] + a[4 + f][8 + 4 * k + q]);
            }
        }
    if constexpr (NC == 2) {
        __syncthreads();                                   // the activation is done with
        float* other = xl + vg * 32 * 64 + lane;
        if (ch == 1)
#pragma unroll
            for (int q = 0; q < 4; ++q)
#pragma unroll
                for (int e = 0; e < 8; ++e) other[(8 * q + e) * 64] = s8[q][e];
        __syncthreads();
        if (ch == 1) return;
#pragma unroll
        for (int q = 0; q < 4; ++q)
#pragma unroll
            for (int e = 0; e < 8; ++e) s8[q][e] = s8[q][e] + other[(8 * q + e) * 64];
    }
    const int b = b0 + i;
    if (b >= rows) return;
#pragma unroll
    for (int q = 0; q < 4; ++q) {
        const int m = m0 + 16 * vg + 4 * t + q;
        if (m >= V) continue;
        float y = hsum8(s8[q]);
        if (logit_scale != 1.0f && logit_scale != 0.0f) y = y * (1.0f / logit_scale);
        logits[(int64_t)b * lstride + m] = y;
    }
}

template <int T, int NB>
hipError_t launch_q_nb(const ultima_hsamp_head* h, const float* xin, int64_t rb, bool al, hipStream_t s) {
    constexpr int R = 4 * 64 / FmtOf<T>::F::LPR;           // vocabulary rows per block
    const dim3 grid((h->vocab + R - 1) / R, (h->rows + NB - 1) / NB);
    const unsigned char* wp = static_cast<const unsigned char*>(h->weight);
    if (al)
        hipLaunchKernelGGL((k_head_q<T, NB, 1>), grid, dim3(256), 0, s, wp, h->vocab, h->hidden_dim, rb, xin,
                           h->rows, h->logit_scale, h->logits, h->logits_stride);
    else
        hipLaunchKernelGGL((k_head_q<T, NB, 0>), grid, dim3(256), 0, s, wp, h->vocab, h->hidden_dim, rb, xin,
                           h->rows, h->logit_scale, h->logits, h->logits_stride);
    return hipGetLastError();
}

template <int T>
hipError_t launch_qm(const ultima_hsamp_head* h, const float* xin, int64_t rb, bool al, hipStream_t s) {
    constexpr int R = FmtOf<T>::F::NA == 64 ? 32 : 64;     // vocabulary rows per block
    const dim3 grid((h->vocab + R - 1) / R, (h->rows + 15) / 16);
    const unsigned char* wp = static_cast<const unsigned char*>(h->weight);
    auto go = [&](auto a) {
        hipLaunchKernelGGL((k_head_qm<T, decltype(a)::value>), grid, dim3(256), 0, s, wp, h->vocab, h->hidden_dim,
                           rb, xin, h->rows, h->logit_scale, h->logits, h->logits_stride);
    };
    if constexpr (FmtOf<T>::F::BB * FmtOf<T>::F::MPC % 4 == 0)
        al ? go(std::integral_constant<int, 1>()) : go(std::integral_constant<int, 0>());
    else
        go(std::integral_constant<int, 0>());
    return hipGetLastError();
}

// Whether the kernels' 32-bit offsets reach every byte of a tile: its `rows`
// weight rows of rb bytes (of the V there are; 15 bytes of alignment on either
// side) and nx activation rows.
bool offsets_fit(int64_t rb, int rows, int V, int64_t H, int nx) {
    const int64_t lim = (int64_t)1 << 32;
    return std::min(rows, V) * rb + 30 < lim && nx * H * 4 < lim;
}

// Up to kGemvRows rows (PQ2_0, whose block sums are per batch row: any number,
// four at a time) the vector units, which unpack each value once for all rows;
// more the matrix cores, a tile of sixteen rows costing little more than five:
// H = 4096, V = 151936, us for 4 rows by the first and 5 / 16 by the second: Q4_K
// 148, 283 / 287, Q5_K 154, 273 / 277, Q6_K 187, 321 / 330, Q8_0 197, 336 / 339,
// Q4_1 147, 252 / 258, Q5_0 162, 277 / 280 (five rows are two passes of the
// first); H = 1024, V = 50257 likewise (Q4_K 25, 37 / 38). Hidden sizes
// of 2^26 and more, whose sixteen activation rows pass 32-bit offsets, stay on
// the vector units with as many batch rows at a time as do not.
template <int T>
hipError_t launch_q(const ultima_hsamp_head* h, const float* xin, int64_t rb, bool al, hipStream_t s) {
    using F = typename FmtOf<T>::F;
    const int64_t H = h->hidden_dim;
    auto fits = [&](int nb) { return offsets_fit(rb, 64 / F::LPR, h->vocab, H, nb); };
    if constexpr (T != ULTIMA_HSAMP_HEAD_PQ2_0) {
        constexpr int R = F::NA == 64 ? 32 : 64;           // as launch_qm
        if (h->rows > kGemvRows && offsets_fit(rb, R, h->vocab, H, 16)) return launch_qm<T>(h, xin, rb, al, s);
    }
    if (h->rows > 2 && fits(4)) return launch_q_nb<T, 4>(h, xin, rb, al, s);
    if (h->rows > 1 && fits(2)) return launch_q_nb<T, 2>(h, xin, rb, al, s);
    return launch_q_nb<T, 1>(h, xin, rb, al, s);
}

// ---- the norm and the fold -------------------------------------------------------

constexpr int kPrepThreads = 1024;
constexpr int kPrepPiece = ULTIMA_HSAMP_MAX_FOLD_BLOCK;      // elements of a row in LDS at a time
constexpr int kPrepPer = kPrepPiece / kPrepThreads;          // a thread's share of a piece
constexpr int kPrepChain = kPrepPiece / 8 + 8;               // LDS floats of one chain (8 mod 64: conflict-free)

// 2^R butterfly inputs `len` apart in registers: the stages len, 2 len, .. of
// the fold, the same additions on the same values as one stage at a time.
template <int R>
__device__ __forceinline__ void fold_stages(float* buf, int len, int n) {
    constexpr int N = 1 << R;
    auto at = [](int i) { return i + (i >> 3); };            // padded: every stride used below is conflict-free
    for (int p = threadIdx.x; p < n / N; p += kPrepThreads) {
        const int j = (p / len) * N * len + (p % len);
        float v[N];
#pragma unroll
        for (int e = 0; e < N; ++e) v[e] = buf[at(j + e * len)];
#pragma unroll
        for (int h = 1; h < N; h <<= 1)
#pragma unroll
            for (int e = 0; e < N; ++e)
                if ((e & h) == 0) {
                    const float a = v[e], b = v[e + h];
                    v[e] = a + b;
                    v[e + h] = a - b;
                }
#pragma unroll
        for (int e = 0; e < N; ++e) buf[at(j + e * len)] = v[e];
    }
    __syncthreads();
}

// One block per batch row; bound by the sum of squares' serial order (eight
// chains of H / 8 dependent multiply-adds, ~1.7 us at H = 4096) and three
// round trips to memory. The row comes in pieces of 8192 elements: coalesced
// loads by every thread, stored chain-major in LDS, from which eight lanes
// run the chains, four steps per 16-byte read and the next sixteen steps' reads
// in flight. A fold takes all the fold blocks of a piece at once, three of its
// stages per barrier in registers. H = 4096, one row: 29.3 -> 5.9 us (the
// chains read global memory eight elements at a time before); sixteen rows
// with a 128-block fold: 95.6 -> 9.1 us (a barrier per stage of each fold
// block before).
__global__ __launch_bounds__(kPrepThreads) void k_head_prep(const float* __restrict__ hidden, int64_t hstride,
                                                            const float* __restrict__ scale, float eps, int H,
                                                            int fold_block, const float* __restrict__ signs,
                                                            float* __restrict__ normed) {
    __shared__ float red[8];
    __shared__ __attribute__((aligned(16))) float buf[kPrepPiece + kPrepPiece / 8];
    static_assert(8 * kPrepChain <= kPrepPiece + kPrepPiece / 8, "the chains fit the fold's buffer");
    const int row = blockIdx.x;
    const float* x = hidden + (int64_t)row * hstride;
    float* y = normed + (int64_t)row * H;
    const int tid = threadIdx.x;
    const int H8 = H / 8 * 8;
    const bool fold = fold_block > 0 && H % fold_block == 0;
    // a piece's elements, scales and signs; indices clamped into the row
    float pv[kPrepPer], sv[kPrepPer], gv[kPrepPer];
    // (piece starts are unsigned: the one past the row's end may pass 2^31)
    auto load = [&](uint32_t p0, float* v, const float* from) {
#pragma unroll
        for (int e = 0; e < kPrepPer; ++e) v[e] = from[min(p0 + tid + e * kPrepThreads, (uint32_t)H - 1u)];
    };
    load(0, pv, x);
    load(0, sv, scale);
    if (fold && signs != nullptr) load(0, gv, signs);
    float p = 0.0f;
    for (uint32_t p0 = 0; p0 < (uint32_t)H8; p0 += kPrepPiece) {
        if (p0 > 0) {
            load(p0, pv, x);
            __syncthreads();                                 // the previous piece's chains are done
        }
#pragma unroll
        for (int e = 0; e < kPrepPer; ++e) {
            const int k = tid + e * kPrepThreads;
            buf[(k & 7) * kPrepChain + (k >> 3)] = pv[e];
        }
        __syncthreads();
        if (tid < 8) {
            const int n = min(kPrepPiece, H8 - (int)p0) >> 3;   // steps of this piece
            const float* cf = buf + tid * kPrepChain;
            const float4* cs = reinterpret_cast<const float4*>(cf);
            const int ng = n >> 4;
            float4 v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = cs[i];
            for (int g = 0; g < ng; ++g) {
                float4 w[4];
                const float4* nx = cs + 4 * min(g + 1, ng - 1);
#pragma unroll
                for (int i = 0; i < 4; ++i) w[i] = nx[i];
#pragma unroll
                for (int i = 0; i < 4; ++i) {
                    p = __builtin_fmaf(v[i].x, v[i].x, p);
                    p = __builtin_fmaf(v[i].y, v[i].y, p);
                    p = __builtin_fmaf(v[i].z, v[i].z, p);
                    p = __builtin_fmaf(v[i].w, v[i].w, p);
                }
#pragma unroll
                for (int i = 0; i < 4; ++i) v[i] = w[i];
            }
            for (int j = 16 * ng; j < n; ++j) p = __builtin_fmaf(cf[j], cf[j], p);
        }
    }
    if (tid < 8) red[tid] = p;
    __syncthreads();
    float ss = hsum8(red);
    // the tail as GCC compiles the reference's vectorised loop: the first four
    // products rounded on their own when four or more remain, the rest fused
    {
        const int t = H - H8;
        int i = 0;
        if (t >= 4)
            for (; i < 4; ++i) ss = ss + x[H8 + i] * x[H8 + i];
        for (; i < t; ++i) ss = __builtin_fmaf(x[H8 + i], x[H8 + i], ss);
    }
    const float inv = 1.0f / sqrtf(ss / (float)H + eps);
    const float finv = 1.0f / sqrtf((float)fold_block);
    for (uint32_t p0 = 0; p0 < (uint32_t)H; p0 += kPrepPiece) {
        if (H > kPrepPiece) {                                // (one piece: still in registers)
            load(p0, pv, x);
            load(p0, sv, scale);
            if (fold && signs != nullptr) load(p0, gv, signs);
        }
        const int n = min(kPrepPiece, H - (int)p0);
        if (!fold) {
#pragma unroll
            for (int e = 0; e < kPrepPer; ++e) {
                const int i = tid + e * kPrepThreads;
                if (i < n) y[p0 + i] = (pv[e] * sv[e]) * inv;
            }
            continue;
        }
        // (fold blocks are powers of two up to the piece: n is a whole number of them)
#pragma unroll
        for (int e = 0; e < kPrepPer; ++e) {
            const int i = tid + e * kPrepThreads;
            const float v = (pv[e] * sv[e]) * inv;
            if (i < n) buf[i + (i >> 3)] = signs != nullptr ? v * gv[e] : v;
        }
        __syncthreads();
        for (int len = 1; len < fold_block;) {
            const int left = fold_block / len;
            if (left >= 8) fold_stages<3>(buf, len, n), len *= 8;
            else if (left == 4) fold_stages<2>(buf, len, n), len *= 4;
            else fold_stages<1>(buf, len, n), len *= 2;
        }
#pragma unroll
        for (int e = 0; e < kPrepPer; ++e) {
            const int i = tid + e * kPrepThreads;
            if (i < n) y[p0 + i] = fold_block >= 2 ? buf[i + (i >> 3)] * finv : buf[i + (i >> 3)];
        }
        __syncthreads();
    }
}

// logits of 0 (a hidden size that is not a whole number of the type's blocks)
__global__ void k_head_zero(float* __restrict__ logits, int64_t lstride, int V) {
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < V) logits[(int64_t)blockIdx.y * lstride + i] = 0.0f;
}

}  // namespace

int head_block_values(int dtype) {
    switch (dtype) {
        case ULTIMA_HSAMP_HEAD_Q4_K: case ULTIMA_HSAMP_HEAD_Q5_K: case ULTIMA_HSAMP_HEAD_Q6_K: return 256;
        case ULTIMA_HSAMP_HEAD_Q8_0: case ULTIMA_HSAMP_HEAD_Q4_1: case ULTIMA_HSAMP_HEAD_Q5_0: return 32;
        case ULTIMA_HSAMP_HEAD_PQ2_0: return 128;
        default: return 0;
    }
}

int head_block_bytes(int dtype) {
    switch (dtype) {
        case ULTIMA_HSAMP_HEAD_Q4_K: return 144;
        case ULTIMA_HSAMP_HEAD_Q5_K: return 176;
        case ULTIMA_HSAMP_HEAD_Q6_K: return 210;
        case ULTIMA_HSAMP_HEAD_Q8_0: return 34;
        case ULTIMA_HSAMP_HEAD_Q4_1: return 20;
        case ULTIMA_HSAMP_HEAD_Q5_0: return 22;
        case ULTIMA_HSAMP_HEAD_PQ2_0: return 34;
        default: return 0;
    }
}

bool head_quant_fits(const ultima_hsamp_head* h) {
    const int64_t be = head_block_values(h->weight_dtype), H = h->hidden_dim;
    const bool two = h->weight_dtype == ULTIMA_HSAMP_HEAD_Q8_0 || h->weight_dtype == ULTIMA_HSAMP_HEAD_PQ2_0;
    const int lpr = two ? FQ8_0::LPR : FQ4_K::LPR;
    return H % be != 0 || offsets_fit(H / be * head_block_bytes(h->weight_dtype), 64 / lpr, h->vocab, H, 1);
}

hipError_t launch_head_prep(const ultima_hsamp_head* h, hipStream_t s) {
    hipLaunchKernelGGL(k_head_prep, dim3(h->rows), dim3(kPrepThreads), 0, s, h->hidden, h->hidden_stride,
                       h->norm_scale, h->eps, h->hidden_dim, h->fold_block, h->fold_signs, h->normed);
    return hipGetLastError();
}

hipError_t launch_head_quant(const ultima_hsamp_head* h, hipStream_t s) {
    const int be = head_block_values(h->weight_dtype);
    const int64_t H = h->hidden_dim;
    if (H % be != 0) {
        hipLaunchKernelGGL(k_head_zero, dim3((h->vocab + 255) / 256, h->rows), dim3(256), 0, s, h->logits,
                           h->logits_stride, h->vocab);
        return hipGetLastError();
    }
    const int64_t rb = H / be * head_block_bytes(h->weight_dtype);
    // dword-aligned rows: every chunk starts on a dword
    const bool al = reinterpret_cast<uintptr_t>(h->weight) % 4 == 0 && rb % 4 == 0;
    switch (h->weight_dtype) {
        case ULTIMA_HSAMP_HEAD_Q4_K: return launch_q<ULTIMA_HSAMP_HEAD_Q4_K>(h, h->normed, rb, al, s);
        case ULTIMA_HSAMP_HEAD_Q5_K: return launch_q<ULTIMA_HSAMP_HEAD_Q5_K>(h, h->normed, rb, al, s);
        case ULTIMA_HSAMP_HEAD_Q6_K: return launch_q<ULTIMA_HSAMP_HEAD_Q6_K>(h, h->normed, rb, al, s);
        case ULTIMA_HSAMP_HEAD_Q8_0: return launch_q<ULTIMA_HSAMP_HEAD_Q8_0>(h, h->normed, rb, al, s);
        case ULTIMA_HSAMP_HEAD_Q4_1: return launch_q<ULTIMA_HSAMP_HEAD_Q4_1>(h, h->normed, rb, al, s);
        case ULTIMA_HSAMP_HEAD_Q5_0: return launch_q<ULTIMA_HSAMP_HEAD_Q5_0>(h, h->normed, rb, al, s);
        case ULTIMA_HSAMP_HEAD_PQ2_0: return launch_q<ULTIMA_HSAMP_HEAD_PQ2_0>(h, h->normed, rb, al, s);
        default: return hipErrorInvalidValue;
    }
}

}  // namespace hsamp
