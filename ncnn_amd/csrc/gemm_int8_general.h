// The any-shape int8 Gemm / InnerProduct kernel (gemm_int8_general.hip), and how it reads rows that begin and end at any byte.
#ifndef NCNNHIP_GEMM_INT8_GENERAL_H
#define NCNNHIP_GEMM_INT8_GENERAL_H

#include "epilogues.h"
#include "mfma_tile.h"

namespace ncnnhip {

typedef int v4i_any __attribute__((ext_vector_type(4), aligned(1))); // 16 bytes at any address

__device__ __forceinline__ v4i load16(const int8_t* p)
{
    return *reinterpret_cast<const v4i_any*>(p);
}

// 16 bytes without their first `drop` (0..16), zeros behind: the chunk of a row that K ends in, from the row's last 16 bytes
__device__ __forceinline__ v4i drop_bytes(v4i w, int drop)
{
    const int dw = drop >> 2, b = drop & 3;
    int t[5] = {0, 0, 0, 0, 0};
#pragma unroll
    for (int i = 0; i < 4; i++)
#pragma unroll
        for (int j = 0; j < 4; j++)
            if (i + dw == j) t[i] = w[j];
    v4i v;
#pragma unroll
    for (int i = 0; i < 4; i++) v[i] = (int)__builtin_amdgcn_alignbyte((unsigned)t[i + 1], (unsigned)t[i], (unsigned)b);
    return v;
}

// whether the general entry points below take their streaming kernel for this shape (aligned: rows, strides and K in multiples of 16 bytes)
bool gemm_int8_streams(int M, int N, int K, bool aligned);

// any M, N, K >= 1, strides >= K, any alignment, every form of the epilogue
int launch_gemm_int8_general(const int8_t* a, size_t lda, const int8_t* b, size_t ldb, int M, int N, int K, const GemmEpilogue& epi, hipStream_t stream);
int launch_fc_int8_general(const int8_t* x, size_t xs, const int8_t* w, size_t ws, int rows, int num_output, int K, const FcEpilogue& epi, hipStream_t stream);

} // namespace ncnnhip

#endif // NCNNHIP_GEMM_INT8_GENERAL_H
