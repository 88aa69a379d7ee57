// GEMM operands whose K is no whole number of 16-byte vectors (or that are K-major as well), copied to a workspace as K-contiguous rows that
// are, zeros behind K: the instances for whole vectors then take the problem.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

namespace ckx {

struct GemmPack
{
    const void *a, *b;
    void *to_a, *to_b; // 16-byte aligned: M and N rows of pitch elements
    int es;            // bytes of an element
    int M, N, K, lda, ldb;
    bool ta, tb;       // K-major
    int pitch;
};
// (the contiguous extent of both operands is 16 bytes and more)
hipError_t launch_gemm_pack(const GemmPack& g, hipStream_t s);

} // namespace ckx
