// The logits producer's dense heads over more than four batch rows, on the
// matrix cores (reference src/kernels/matvec_f32_f32.cpp:22-50,
// matvec_bf16_f32.cpp:48-68, one call of them per batch row).
//
// The reference's order is eight chains of fused multiply-adds per output. An
// f32 matrix instruction with K = 1 is one fused multiply-add per output,
// rounded once to nearest, subnormals kept: the same bits as the chain's step.
// v_mfma_f32_16x16x1_4b runs four independent 16 x 16 blocks, so two of them
// are one step of all eight chains of a tile of 16 vocabulary rows x 16 batch
// rows. Its peak is little above v_fma_f32's (142 against 135 TFLOP/s measured
// on independent chains), but one instruction takes 1024 multiply-adds from
// two registers a lane where the vector form issues sixteen, each with its
// operand read from LDS, and the accumulators of 16 x 16 outputs let the
// weights be read once per 64 batch rows instead of once per four.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cstdint>
#include <type_traits>

#include "hsamp_head.h"
#include "ultima_hsamp.h"

#pragma clang fp contract(off)

namespace hsamp {
namespace {

typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef u32x4 u32x4_a2 __attribute__((aligned(2)));      // 16 bytes on any bf16 boundary
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));

// exchanges between the 16-lane rows of a wave: the odd rows of a with the
// even rows of b; the upper half of a with the lower half of b
__device__ __forceinline__ void swap16(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane16_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}
__device__ __forceinline__ void swap32(uint32_t& a, uint32_t& b) {
    const auto r = __builtin_amdgcn_permlane32_swap(a, b, false, false);
    a = r[0];
    b = r[1];
}

// WB: bf16 weights (else f32). NT: batch tiles of 16 rows. Four waves of 16
// vocabulary rows each share the batch rows' values through LDS.
//
// Lane 16 q + i of a wave (q = 0..3) feeds vocabulary row m0 + i's chains 2q
// and 2q + 1 to block q of the two instructions. It loads 16 bytes of the row
// where its neighbours' 16 bytes follow (64 contiguous bytes per row and
// load, any alignment), and the lanes of one row exchange dwords (permlane
// swaps, two or four per load) so that each holds its two chains of every
// step. The batch rows' values come in chunks of KC columns, row-major in
// LDS (rows padded by 2 floats: the 8-byte reads of a step are conflict-free),
// the next chunk's values and weights in flight while one is multiplied.
//
// Bound by the matrix pipe (busy 0.75 of the SIMDs' cycles at 64 rows, where it
// would take 561 us at the rate above) and, up to 16 rows, by the weights'
// stream. H = 4096, V = 151936 bf16, against passes of four rows
// through the lane-per-row kernel: 64 rows 800 us (3200), 32 rows 460 us
// (1650), 16 rows 305 us (877), 5 rows 300 us (455); f32, 16 rows 480 us
// (1667). No change from two vocabulary tiles per wave, reads issued a step
// ahead or 128-column chunks at 64 rows.
template <bool WB, int NT>
__global__ __launch_bounds__(256, 2) void k_head_mm(const void* __restrict__ weight, int V, int H,
                                                    const float* __restrict__ x, int rows, float logit_scale,
                                                    float* __restrict__ logits, int64_t lstride) {
    constexpr int KC = NT == 1 ? 128 : 64;         // columns per chunk
    constexpr int ES = WB ? 2 : 4;
    constexpr int LC = 64 / ES;                    // columns the four lanes of a row load at a time
    constexpr int NL = KC / LC;                    // weight loads per lane per chunk
    constexpr int GS = LC / 8;                     // steps of one load
    constexpr int XS = KC + 2;                     // floats per batch row in LDS
    constexpr int NX = KC * 16 * NT / (4 * 256);   // 16-byte loads of batch values per thread per chunk
    __shared__ __attribute__((aligned(16))) float xl[2][16 * NT * XS];
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int i = lane & 15, q = lane >> 4;
    const int m0 = (blockIdx.x * 4 + wave) * 16;
    const int b0 = blockIdx.y * 16 * NT;
    const int H8 = H / 8 * 8;
    const int nC = H8 / KC + (H8 % KC != 0);
    const unsigned char* wrow = static_cast<const unsigned char*>(weight) + (int64_t)min(m0 + i, V - 1) * H * ES;
    // the lane's place among the LC columns: bf16, step q of four; f32, half
    // q >> 1 of step q & 1 of two
    const int lcol = WB ? 8 * q : 8 * (q & 1) + 4 * (q >> 1);

    // Addresses clamped into the rows: columns past H8 feed steps that are
    // skipped, rows past V and past the batch feed outputs that are not stored.
    // (columns are unsigned: those past the row's end may pass 2^31)
    auto load_w = [&](uint32_t col) {
        col = min(col + (uint32_t)lcol, (uint32_t)(H8 - 16 / ES));
        return (u32x4)*reinterpret_cast<const u32x4_a2*>(wrow + (int64_t)col * ES);
    };
    auto load_x = [&](f32x4_a4 (&v)[NX], int c) {
#pragma unroll
        for (int t = 0; t < NX; ++t) {
            const int n = tid + 256 * t, j = n / (KC / 4), k = n % (KC / 4) * 4;
            v[t] = *reinterpret_cast<const f32x4_a4*>(x + (int64_t)min(b0 + j, rows - 1) * H +
                                                      min((uint32_t)c * KC + k, (uint32_t)H8 - 4u));
        }
    };
    auto store_x = [&](const f32x4_a4 (&v)[NX], int buf) {
#pragma unroll
        for (int t = 0; t < NX; ++t) {
            const int n = tid + 256 * t, j = n / (KC / 4), k = n % (KC / 4) * 4;
            float2* to = reinterpret_cast<float2*>(&xl[buf][j * XS + k]);
            to[0] = make_float2(v[t].x, v[t].y);
            to[1] = make_float2(v[t].z, v[t].w);
        }
    };
    // the lane's weights of chains 2q and 2q + 1 at each step of a load
    auto weights = [&](u32x4 w, float (&a0)[GS], float (&a1)[GS]) {
        uint32_t d[4] = {w.x, w.y, w.z, w.w};
        if (WB) {
            swap32(d[0], d[2]);
            swap32(d[1], d[3]);
            swap16(d[0], d[1]);
            swap16(d[2], d[3]);
#pragma unroll
            for (int s = 0; s < GS; ++s) {
                a0[s] = __uint_as_float(d[s] << 16);
                a1[s] = __uint_as_float(d[s] & 0xFFFF0000u);
            }
        } else {
            swap16(d[0], d[2]);
            swap16(d[1], d[3]);
#pragma unroll
            for (int s = 0; s < GS; ++s) {
                a0[s] = __uint_as_float(d[2 * s]);
                a1[s] = __uint_as_float(d[2 * s + 1]);
            }
        }
    };
    f32x16 acc[NT][2];
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[t][0][e] = acc[t][1][e] = 0.0f;
    const int xlane = i * XS + 2 * q;
    auto step = [&](const float* xs, float a0, float a1) {
#pragma unroll
        for (int t = 0; t < NT; ++t) {
            const float2 b = *reinterpret_cast<const float2*>(xs + t * 16 * XS);
            acc[t][0] = __builtin_amdgcn_mfma_f32_16x16x1f32(a0, b.x, acc[t][0], 0, 0, 0);
            acc[t][1] = __builtin_amdgcn_mfma_f32_16x16x1f32(a1, b.y, acc[t][1], 0, 0, 0);
        }
    };
    u32x4 w[NL];
    f32x4_a4 xv[NX];
    if (nC > 0) {
        load_x(xv, 0);
#pragma unroll
        for (int t = 0; t < NL; ++t) w[t] = load_w(t * LC);
        store_x(xv, 0);
    }
    __syncthreads();
    const int whole = H8 / KC;
    for (int c = 0; c < whole; ++c) {
        u32x4 next[NL];
        load_x(xv, min(c + 1, nC - 1));
#pragma unroll
        for (int t = 0; t < NL; ++t) next[t] = load_w((uint32_t)(c + 1) * KC + t * LC);
        // the loads stay here, a chunk ahead of their use (the compiler moves
        // them down to it otherwise)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int t = 0; t < NL; ++t) {
            float a0[GS], a1[GS];
            weights(w[t], a0, a1);
#pragma unroll
            for (int s = 0; s < GS; ++s) step(xl[c & 1] + xlane + 8 * (t * GS + s), a0[s], a1[s]);
        }
        __builtin_amdgcn_sched_barrier(0);
        store_x(xv, (c + 1) & 1);                           // (past the last chunk: read by nobody)
        __syncthreads();
#pragma unroll
        for (int t = 0; t < NL; ++t) w[t] = next[t];
    }
    // the columns past the last whole chunk, in their own loads
    const int left = (H8 - whole * KC) >> 3;
    for (int n = 0; n < left; n += GS) {
        float a0[GS], a1[GS];
        weights(load_w((uint32_t)whole * KC + 8 * n), a0, a1);
#pragma unroll
        for (int s = 0; s < GS; ++s)
            if (n + s < left) step(xl[whole & 1] + xlane + 8 * (n + s), a0[s], a1[s]);
    }

    // Lane 16 q + j holds, for vocabulary rows m0 + 4q + r and batch row j of
    // each tile, chain 2k + e in acc[t][e][4k + r]: the horizontal sum, the
    // tail and the logit scale, as the reference's kernel ends.
    const int tl = H - H8;
    const bool scaled = logit_scale != 1.0f && logit_scale != 0.0f;
    const float inv = scaled ? 1.0f / logit_scale : 1.0f;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
        const int b = b0 + 16 * t + i;
        if (b >= rows) continue;
        const float* xt = x + (int64_t)b * H + H8;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const int m = m0 + 4 * q + r;
            if (m >= V) continue;
            auto p = [&](int l) { return acc[t][l & 1][4 * (l >> 1) + r]; };
            const float s0 = p(0) + p(4), s1 = p(1) + p(5), s2 = p(2) + p(6), s3 = p(3) + p(7);
            float y = (s0 + s1) + (s2 + s3);
            if (WB) {
                const uint16_t* wt = static_cast<const uint16_t*>(weight) + (int64_t)m * H + H8;
                float tail = 0.0f;
                for (int k = 0; k < tl; ++k) tail = __builtin_fmaf(__uint_as_float((uint32_t)wt[k] << 16), xt[k], tail);
                y = y + tail;
            } else if (tl > 0) {
                const float* wt = static_cast<const float*>(weight) + (int64_t)m * H + H8;
                y = tail_f32(y, [&](int k) { return wt[k]; }, [&](int k) { return xt[k]; }, tl);
            }
            if (scaled) y = y * inv;
            logits[(int64_t)b * lstride + m] = y;
        }
    }
}

template <bool WB>
hipError_t launch_mm(const ultima_hsamp_head* h, hipStream_t s) {
    const int tiles = std::min(4, (h->rows + 15) / 16);
    const dim3 grid((h->vocab + 63) / 64, (h->rows + 16 * tiles - 1) / (16 * tiles));
    auto go = [&](auto nt) {
        hipLaunchKernelGGL((k_head_mm<WB, decltype(nt)::value>), grid, dim3(256), 0, s, h->weight, h->vocab,
                           h->hidden_dim, h->normed, h->rows, h->logit_scale, h->logits, h->logits_stride);
    };
    if (tiles == 1) go(std::integral_constant<int, 1>());
    else if (tiles == 2) go(std::integral_constant<int, 2>());
    else if (tiles == 3) go(std::integral_constant<int, 3>());
    else go(std::integral_constant<int, 4>());
    return hipGetLastError();
}

}  // namespace

hipError_t launch_head_mm(const ultima_hsamp_head* h, hipStream_t s) {
    return h->weight_dtype == ULTIMA_HSAMP_BF16 ? launch_mm<true>(h, s) : launch_mm<false>(h, s);
}

}  // namespace hsamp
