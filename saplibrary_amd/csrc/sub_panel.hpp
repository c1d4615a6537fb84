// Device helpers of the banded factorizations whose panels are factored in
// sub-panels of 16 columns, one row of L or column of U per lane: broadcasts
// inside a 16-lane row, the elimination steps, and the LDS and buffer accesses
// around them.
#pragma once
#include "sap_internal.hpp"

namespace sap_amd {
namespace {

// acc -= (lane N of the 16-lane row of src) * m.  hipcc does not fold the
// broadcast into the multiply-add, so it is written out; an instruction that
// broadcasts must not follow the one that wrote its source by less than two
// wait states, hence the s_nop that begins every group.
// a[i] -= (lane N of the row of c[i]) * m; in place (c = a); a[i] -= (lane
// N + i of the row of c) * m, for groups of 8, 4, 2 and 1
template <int N>
__device__ __forceinline__ void bc_rows8(float* a, const float* c, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%8, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%9, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %2, -%10, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %3, -%11, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %4, -%12, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %5, -%13, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %6, -%14, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %7, -%15, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7])
                 : "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]), "v"(c[4]), "v"(c[5]), "v"(c[6]), "v"(c[7]), "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_rows8(double* a, const double* c, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%8, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%9, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %2, -%10, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %3, -%11, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %4, -%12, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %5, -%13, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %6, -%14, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %7, -%15, %16 row_newbcast:%17 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7])
                 : "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]), "v"(c[4]), "v"(c[5]), "v"(c[6]), "v"(c[7]), "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_rows4(float* a, const float* c, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%4, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%5, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %2, -%6, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %3, -%7, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
                 : "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]), "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_rows4(double* a, const double* c, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%4, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%5, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %2, -%6, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %3, -%7, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
                 : "v"(c[0]), "v"(c[1]), "v"(c[2]), "v"(c[3]), "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_rows2(float* a, const float* c, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1])
                 : "v"(c[0]), "v"(c[1]), "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_rows2(double* a, const double* c, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1])
                 : "v"(c[0]), "v"(c[1]), "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_rows1(float* a, const float* c, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0])
                 : "v"(c[0]), "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_rows1(double* a, const double* c, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0])
                 : "v"(c[0]), "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_self8(float* a, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%0, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%1, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %2, -%2, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %3, -%3, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %4, -%4, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %5, -%5, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %6, -%6, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %7, -%7, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7])
                 : "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_self8(double* a, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%0, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%1, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %2, -%2, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %3, -%3, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %4, -%4, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %5, -%5, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %6, -%6, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %7, -%7, %8 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7])
                 : "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_self4(float* a, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %2, -%2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %3, -%3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
                 : "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_self4(double* a, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%0, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%1, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %2, -%2, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %3, -%3, %4 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
                 : "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_self2(float* a, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%0, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1])
                 : "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_self2(double* a, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%0, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1])
                 : "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_self1(float* a, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0])
                 : "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_self1(double* a, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%0, %1 row_newbcast:%2 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0])
                 : "v"(m), "n"(N));
}
template <int N>
__device__ __forceinline__ void bc_cols8(float* a, float c, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%8, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%8, %9 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %2, -%8, %9 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %3, -%8, %9 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %4, -%8, %9 row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %5, -%8, %9 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %6, -%8, %9 row_newbcast:%16 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %7, -%8, %9 row_newbcast:%17 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7])
                 : "v"(c), "v"(m), "n"(N + 0), "n"(N + 1), "n"(N + 2), "n"(N + 3), "n"(N + 4), "n"(N + 5), "n"(N + 6), "n"(N + 7));
}
template <int N>
__device__ __forceinline__ void bc_cols8(double* a, double c, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%8, %9 row_newbcast:%10 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%8, %9 row_newbcast:%11 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %2, -%8, %9 row_newbcast:%12 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %3, -%8, %9 row_newbcast:%13 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %4, -%8, %9 row_newbcast:%14 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %5, -%8, %9 row_newbcast:%15 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %6, -%8, %9 row_newbcast:%16 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %7, -%8, %9 row_newbcast:%17 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3]), "+&v"(a[4]), "+&v"(a[5]), "+&v"(a[6]), "+&v"(a[7])
                 : "v"(c), "v"(m), "n"(N + 0), "n"(N + 1), "n"(N + 2), "n"(N + 3), "n"(N + 4), "n"(N + 5), "n"(N + 6), "n"(N + 7));
}
template <int N>
__device__ __forceinline__ void bc_cols4(float* a, float c, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%4, %5 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%4, %5 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %2, -%4, %5 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %3, -%4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
                 : "v"(c), "v"(m), "n"(N + 0), "n"(N + 1), "n"(N + 2), "n"(N + 3));
}
template <int N>
__device__ __forceinline__ void bc_cols4(double* a, double c, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%4, %5 row_newbcast:%6 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%4, %5 row_newbcast:%7 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %2, -%4, %5 row_newbcast:%8 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %3, -%4, %5 row_newbcast:%9 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1]), "+&v"(a[2]), "+&v"(a[3])
                 : "v"(c), "v"(m), "n"(N + 0), "n"(N + 1), "n"(N + 2), "n"(N + 3));
}
template <int N>
__device__ __forceinline__ void bc_cols2(float* a, float c, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%2, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f32_dpp %1, -%2, %3 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1])
                 : "v"(c), "v"(m), "n"(N + 0), "n"(N + 1));
}
template <int N>
__device__ __forceinline__ void bc_cols2(double* a, double c, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%2, %3 row_newbcast:%4 row_mask:0xf bank_mask:0xf\n\t"
                 "v_fmac_f64_dpp %1, -%2, %3 row_newbcast:%5 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0]), "+&v"(a[1])
                 : "v"(c), "v"(m), "n"(N + 0), "n"(N + 1));
}
template <int N>
__device__ __forceinline__ void bc_cols1(float* a, float c, float m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f32_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0])
                 : "v"(c), "v"(m), "n"(N + 0));
}
template <int N>
__device__ __forceinline__ void bc_cols1(double* a, double c, double m)
{
    asm volatile("s_nop 1\n\t"
                 "v_fmac_f64_dpp %0, -%1, %2 row_newbcast:%3 row_mask:0xf bank_mask:0xf"
                 : "+&v"(a[0])
                 : "v"(c), "v"(m), "n"(N + 0));
}

// the same for i = J .. 15
template <int N, int J, class T>
__device__ __forceinline__ void bc_rows(T (&a)[16], const T (&c)[16], T m)
{
    if constexpr (J + 7 < 16) { bc_rows8<N>(a + J, c + J, m); bc_rows<N, J + 8, T>(a, c, m); }
    else if constexpr (J + 3 < 16) { bc_rows4<N>(a + J, c + J, m); bc_rows<N, J + 4, T>(a, c, m); }
    else if constexpr (J + 1 < 16) { bc_rows2<N>(a + J, c + J, m); bc_rows<N, J + 2, T>(a, c, m); }
    else if constexpr (J < 16) { bc_rows1<N>(a + J, c + J, m); }
}
template <int N, int J, class T>
__device__ __forceinline__ void bc_self(T (&a)[16], T m)
{
    if constexpr (J + 7 < 16) { bc_self8<N>(a + J, m); bc_self<N, J + 8, T>(a, m); }
    else if constexpr (J + 3 < 16) { bc_self4<N>(a + J, m); bc_self<N, J + 4, T>(a, m); }
    else if constexpr (J + 1 < 16) { bc_self2<N>(a + J, m); bc_self<N, J + 2, T>(a, m); }
    else if constexpr (J < 16) { bc_self1<N>(a + J, m); }
}
// u[i] -= (lane i of the row of c) * m for i = I .. 15
template <int I, class T>
__device__ __forceinline__ void bc_cols(T (&u)[16], T c, T m)
{
    if constexpr (I + 7 < 16) { bc_cols8<I>(u + I, c, m); bc_cols<I + 8, T>(u, c, m); }
    else if constexpr (I + 3 < 16) { bc_cols4<I>(u + I, c, m); bc_cols<I + 4, T>(u, c, m); }
    else if constexpr (I + 1 < 16) { bc_cols2<I>(u + I, c, m); bc_cols<I + 2, T>(u, c, m); }
    else if constexpr (I < 16) { bc_cols1<I>(u + I, c, m); }
}

template <int N>
__device__ __forceinline__ float row_get(float v)
{
    return __int_as_float(__builtin_amdgcn_update_dpp(0, __float_as_int(v), 0x150 + N, 0xf, 0xf, true));
}
template <int N>
__device__ __forceinline__ double row_get(double v)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)b, 0x150 + N, 0xf, 0xf, true);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), 0x150 + N, 0xf, 0xf, true);
    return __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
}

template <class T>
__device__ inline T buffer_load(__amdgpu_buffer_rsrc_t r, int off, int soff = 0);
template <>
__device__ inline float buffer_load<float>(__amdgpu_buffer_rsrc_t r, int off, int soff)
{
    return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(r, off, soff, 0));
}
template <>
__device__ inline double buffer_load<double>(__amdgpu_buffer_rsrc_t r, int off, int soff)
{
    const auto v = __builtin_amdgcn_raw_buffer_load_b64(r, off, soff, 0);
    return __longlong_as_double((long long)(((unsigned long long)v[1] << 32) | v[0]));
}

template <class T>
__device__ inline void buffer_store(T v, __amdgpu_buffer_rsrc_t r, int off, int soff = 0);
template <>
__device__ inline void buffer_store<float>(float v, __amdgpu_buffer_rsrc_t r, int off, int soff)
{
    __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(v), r, off, soff, 0);
}
template <>
__device__ inline void buffer_store<double>(double v, __amdgpu_buffer_rsrc_t r, int off, int soff)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    typedef unsigned int u2 __attribute__((ext_vector_type(2)));
    const u2 x = {(unsigned)b, (unsigned)(b >> 32)};
    __builtin_amdgcn_raw_buffer_store_b64(x, r, off, soff, 0);
}

// 16 values of a 16-byte aligned LDS row
__device__ inline void lds_get16(const float* p, float (&v)[16])
{
    const float4* q = reinterpret_cast<const float4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        const float4 x = q[i];
        v[4 * i] = x.x; v[4 * i + 1] = x.y; v[4 * i + 2] = x.z; v[4 * i + 3] = x.w;
    }
}
__device__ inline void lds_get16(const double* p, double (&v)[16])
{
    const double2* q = reinterpret_cast<const double2*>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) {
        const double2 x = q[i];
        v[2 * i] = x.x; v[2 * i + 1] = x.y;
    }
}
__device__ inline void lds_get4(const float* p, float (&v)[4])
{
    const float4 x = *reinterpret_cast<const float4*>(p);
    v[0] = x.x; v[1] = x.y; v[2] = x.z; v[3] = x.w;
}
__device__ inline void lds_get4(const double* p, double (&v)[4])
{
    const double2* q = reinterpret_cast<const double2*>(p);
    const double2 x = q[0], y = q[1];
    v[0] = x.x; v[1] = x.y; v[2] = y.x; v[3] = y.y;
}
__device__ inline void lds_put16(float* p, const float (&v)[16])
{
    float4* q = reinterpret_cast<float4*>(p);
#pragma unroll
    for (int i = 0; i < 4; ++i) q[i] = make_float4(v[4 * i], v[4 * i + 1], v[4 * i + 2], v[4 * i + 3]);
}
__device__ inline void lds_put16(double* p, const double (&v)[16])
{
    double2* q = reinterpret_cast<double2*>(p);
#pragma unroll
    for (int i = 0; i < 8; ++i) q[i] = make_double2(v[2 * i], v[2 * i + 1]);
}

__device__ inline float pivot_rcp(float v) { return __builtin_amdgcn_rcpf(v); }
__device__ inline double pivot_rcp(double v) { return 1.0 / v; }

// all ones when x < 0, else 0
__device__ inline int neg_mask(int x) { return __builtin_amdgcn_sbfe(x, 31, 1); }
// x / v from q = x * r, r the reciprocal of v, with one correction
template <class T>
__device__ __forceinline__ T quotient(T q, T x, T v, T r)
{
    return fma(fma(-q, v, x), r, q);
}
// The pivot of step N from the lane row's copy d of the diagonal block (row
// `c` of it in lane c): boosted unless `plain`, kept in pr by lane N; returns
// the reciprocal of the lane's own candidate (lane N's is the pivot's).
template <int N, class T>
__device__ __forceinline__ T sub_panel_pivot(const T (&d)[16], T& pr, int c, bool plain)
{
    const T thr = (T)1e-7, nv = (T)1e-4;
    T piv = d[N];
    if (!(fabs(piv) > thr || plain)) piv = piv < (T)0 ? -nv : nv;
    pr = c == N ? piv : pr;
    return pivot_rcp(piv);
}
// Steps N .. 15 of a 16-column sub-panel: own is the lane's row of L (ROWS) or
// column of U, rl what sub_panel_pivot<N> returned.  d is left with L below
// the diagonal and U above (ROWS; the diagonal itself is in pr).  The next
// pivot's entry is updated first, and its chain (boost, reciprocal, broadcast)
// runs under the rest of the step.  REFINE: the multipliers are corrected once
// with the pivot itself, which leaves them as a division would give them.
template <int N, bool ROWS, bool REFINE, class T>
__device__ __forceinline__ void sub_panel_steps(T (&d)[16], T (&own)[16], T& pr, T rl, int c, bool plain)
{
    asm volatile("" : "+v"(c));   // masks of lane numbers are made where they are used
    const T rp = row_get<N>(rl);
    T l = d[N] * rp, o = own[N] * rp;
    if constexpr (REFINE) {
        const T pv = row_get<N>(pr);
        l = quotient(l, d[N], pv, rp);
        o = quotient(o, own[N], pv, rp);
    }
    l = c > N ? l : (T)0;
    if constexpr (ROWS) own[N] = o;
    if constexpr (N + 1 < 16) {
        bc_self1<N>(d + N + 1, l);
        // row N of d is not changed by this step, so the order of the two is free
        if constexpr (ROWS) bc_rows<N, N + 1, T>(own, d, own[N]);
        else bc_cols<N + 1, T>(own, l, own[N]);
        const T rn = sub_panel_pivot<N + 1, T>(d, pr, c, plain);
        if constexpr (ROWS) d[N] = c > N ? l : d[N];
        if constexpr (sizeof(T) == 4) __builtin_amdgcn_sched_barrier(0);
        bc_self<N, N + 2, T>(d, l);
        sub_panel_steps<N + 1, ROWS, REFINE, T>(d, own, pr, rn, c, plain);
    }
}

}  // namespace
}  // namespace sap_amd
