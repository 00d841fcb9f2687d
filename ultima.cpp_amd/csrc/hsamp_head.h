// Launchers and the evaluation order shared by the logits producer's sources
// (hsamp_head.hip: the entry point and the F32 / BF16 heads of up to four rows;
// hsamp_headm.hip: those of more rows; hsamp_headq.hip: the norm / fold kernel
// and the quantised heads).
#pragma once

#include <hip/hip_runtime.h>

#include "ultima_hsamp.h"

namespace hsamp {

// acc + a(0) b(0) + ... + a(t-1) b(t-1) as the reference's vectorised f32 tail
// (t < 8): when t >= 4 the first four products are rounded on their own.
template <class A, class B>
__device__ __forceinline__ float tail_f32(float acc, A a, B b, int t) {
#pragma clang fp contract(off)
    int i = 0;
    if (t >= 4)
        for (; i < 4; ++i) acc = acc + a(i) * b(i);
    for (; i < t; ++i) acc = __builtin_fmaf(a(i), b(i), acc);
    return acc;
}

// Dense heads of up to this many rows take one pass of the lane-per-row kernel
// (bound by the weights' stream, the norm fused in), more rows the matrix-core
// kernel, whose one tile of 16 rows costs the same for 5 as for 16: H = 4096,
// V = 151936 bf16, 4 rows 258 us by the first, 5 rows 455 us by it (two
// passes) and 300 us by the second.
constexpr int kGemvRows = 4;

// values / bytes of one block of a quantised head type (0 for others)
int head_block_values(int dtype);
int head_block_bytes(int dtype);
// whether a quantised head's rows are within the kernels' 32-bit offsets
bool head_quant_fits(const ultima_hsamp_head* h);
// the final rmsnorm (and the fold, when h->fold_block divides H) of every row
// into h->normed
hipError_t launch_head_prep(const ultima_hsamp_head* h, hipStream_t s);
// the F32 / BF16 matvecs of h->normed (more than kGemvRows rows) into h->logits
hipError_t launch_head_mm(const ultima_hsamp_head* h, hipStream_t s);
// the quantised matvec of h->normed into h->logits (with the logit scale)
hipError_t launch_head_quant(const ultima_hsamp_head* h, hipStream_t s);

}  // namespace hsamp
