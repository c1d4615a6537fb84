// Preconditioner apply: z = M^{-1} v (Precond::solve / getSRev,
// sap/precond.h:1392-1528).
//
// SaP-C runs three launches:
//   pass 1  interface values of g = A_D^{-1} v.  The reduced system needs
//           only the bottom k rows of A_i^{-1} v_i and the top k rows of
//           A_{i+1}^{-1} v_{i+1}: the first come from a full L sweep of the
//           LU factors plus a k-row U' sweep, the second from a full U' sweep
//           of the UL factors plus a k-row L' sweep.  The two are
//           independent, so every partition boundary gets two workgroups.
//   iface   reduced solve per boundary with S_i^{-1} and purification
//           (partFullFwdSweep/partFullBckSweep + purifyRHS,
//           sap/precond.h:5418-5530), producing corrections of the rhs rows
//           next to each boundary.
//   pass 2  full L, D^{-1}, U' sweep of (v - corrections) for every
//           partition (partBandedFwdSweep/partBandedBckSweep); the last
//           partition uses its UL factors when factMethod = LU_UL.
// SaP-D (or P = 1) runs pass 2 alone.
//
// Triangular sweeps: one workgroup per (partition, direction) walks the rows
// in blocks; wavefront 0 solves each block's unit-lower diagonal block, the
// other wavefronts apply the block to the next k rows, and the pending
// values live in an LDS ring.  Two variants:
//   MODE 2 (k <= 384 + BS while the staging fits, the default; above
//          192 + BS each far-row lane takes two rows): multipliers, inverted
//          diagonal blocks and right-hand side staged HBM -> LDS by producer
//          wavefronts several blocks ahead;
//   MODE 0 (any k): the plain blocked sweep with blocks of 64.
#include "sap_internal.hpp"

#include <algorithm>
#include <type_traits>

namespace sap_amd {

namespace {

constexpr int NBS = 64;

template <class T>
struct BandView {
    const T* base;
    int64_t origin;
    int64_t w;
    int k;
    int dir;
    __device__ inline T at(int64_t r, int64_t c) const { return base[origin + dir * (c * w + k + r - c)]; }
};

template <class T>
__device__ inline BandView<T> make_view(const T* B, int64_t s, int64_t len, int k, int dir)
{
    BandView<T> v;
    v.base = B;
    v.w = 2 * k + 1;
    v.k = k;
    v.dir = dir;
    v.origin = dir > 0 ? s * v.w : (s + len) * v.w - 1;
    return v;
}

// v if bit j of m is set, else +0 (bitwise: a signed one-bit field extract
// and an AND, so no compare and no scalar mask register per element)
__device__ inline float keep_if(float v, unsigned m, int j)
{
    return __int_as_float(__float_as_int(v) & __builtin_amdgcn_sbfe((int)m, j, 1));
}
__device__ inline double keep_if(double v, unsigned m, int j)
{
    // the 32-bit field mask applied to each half (hipcc drops the sign
    // extension of the field extract when it is widened to 64 bits first)
    const unsigned sm = (unsigned)__builtin_amdgcn_sbfe((int)m, j, 1);
    const long long b = __double_as_longlong(v);
    const unsigned lo = (unsigned)b & sm, hi = (unsigned)(b >> 32) & sm;
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}
// bits 0 .. n-1 set (n clamped to [0, 32])
__device__ inline unsigned bits_below(int n)
{
    return n <= 0 ? 0u : n >= 32 ? ~0u : (1u << n) - 1u;
}

__device__ inline float bcast(float v, int j)
{
    return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), j));
}
__device__ inline double bcast(double v, int j)
{
    const long long b = __double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(b & 0xffffffffLL), j);
    const int hi = __builtin_amdgcn_readlane((int)(b >> 32), j);
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

// y = L^{-1} b over local rows [0, len) of a view (L unit lower, band k).
// in(r) gives b_r; out(r, y_r) receives each final value.
template <class T, class In, class Out>
__device__ void lower_sweep(const BandView<T>& V, int64_t len, In in, Out out, T* pend, int ring_mask, T* xblk)
{
    const int k = V.k;
    const int tid = threadIdx.x;
    const int lane = tid & 63;
    const int wave = tid >> 6;
    const int64_t init = min(len, (int64_t)NBS + k);
    for (int64_t r = tid; r < init; r += blockDim.x) pend[r & ring_mask] = in(r);
    __syncthreads();
    for (int64_t c0 = 0; c0 < len; c0 += NBS) {
        const int nb = (int)min((int64_t)NBS, len - c0);
        if (wave == 0) {
            T Ld[NBS];
#pragma unroll
            for (int j = 0; j < NBS; ++j)
                Ld[j] = (j < lane && lane < nb && lane - j <= k) ? V.at(c0 + lane, c0 + j) : (T)0;
            T x = lane < nb ? pend[(c0 + lane) & ring_mask] : (T)0;
#pragma unroll
            for (int j = 0; j < NBS - 1; ++j) {
                const T xj = bcast(x, j);
                x -= Ld[j] * xj;
            }
            if (lane < nb) {
                xblk[lane] = x;
                out(c0 + lane, x);
            }
        }
        __syncthreads();
        for (int t = tid; t < k; t += blockDim.x) {
            const int64_t r = c0 + nb + t;
            if (r >= len) break;
            const int jlo = max(0, nb + t - k);
            T acc = (T)0;
            for (int j = jlo; j < nb; ++j) acc += V.at(r, c0 + j) * xblk[j];
            pend[r & ring_mask] -= acc;
        }
        {
            const int64_t lo = c0 + nb + k;
            const int64_t hi = min(len, c0 + nb + k + NBS);
            for (int64_t r = lo + tid; r < hi; r += blockDim.x) pend[r & ring_mask] = in(r);
        }
        __syncthreads();
    }
}

// rows per block of the staged sweep
template <class T>
constexpr int sweep_bs() { return sizeof(T) == 4 ? 32 : 16; }

// ---------------------------------------------------------------------------
// LDS-staged variant (768 threads).  A block of BS columns takes
//   its table, made once per factorization by sweep_tables_kernel: the
//     inverse T of the block's unit-lower diagonal block, the sub-diagonal
//     BS x BS block S (zeros outside the band), both in the order the chain's
//     lanes read them, and the pivots;
//   the far rows (2 BS .. BS + k - 1) of its columns, from the band.
// Producer wavefronts copy them HBM -> LDS with global_load_lds_dwordx4 into
// two rings of slots (A: tables, B: far rows, used one step later), several
// blocks ahead; the right-hand side rows stream into an LDS staging ring the
// same way, SW_DIN steps ahead.  No step waits for HBM.
// With x_b = T_b p_b and p_{b+1} -= S_b x_b the dependency chain of a block is
// two BS x BS matrix-vector products of one wavefront instead of a
// substitution of BS dependent steps: each lane holds half a row of the
// matrix, the vector stays in registers (one element per lane, broadcast
// inside the 16-lane rows by DPP), and the halves meet by a swap of lane
// halves.
// In step b:
//   wave 0            S_{b-1} x_{b-1} (while its pending values and T_b come
//                     from LDS), then x_b = T_b p_b;
//   waves 1-3, 5-7    far rows of block b-1, one row per lane, half of the
//                     columns each; the two column halves add into pending
//                     rings of their own, which the chain sums;
//   wave 9            moves the staged right-hand side rows into the pending
//                     ring and streams the next ones;
//   wave 8            writes the results of block b-1 (divided by the pivots
//                     in the first stage);
//   wave 4            producer of ring A, waves 10, 11 of ring B.
// Each producer (and wave 9 for the staging ring) waits with an explicit
// vmcnt count for its own copies before the barrier that publishes them.
// What bounds it: the chain of steps, about 740 cycles each in FP32 against
// 3200 by substitution (32 dependent steps and their multiplier reads), and
// from about k = 120 the 45 to 59 GB/s that one workgroup draws from HBM
// (19 KB a step there).  One application, before and after: n = 200000, k = 50,
// 16 partitions 1054 -> 260 us; n = 1000000, k = 200, 64 partitions (both
// passes and the interface solve) 1644 -> 1063 us.
// ---------------------------------------------------------------------------
// Wavefronts w, w + 4 and w + 8 share a SIMD: the chain's partners are the
// light ones.
constexpr int SW_PROD_A = 4;
constexpr int SW_WRITER = 8;
constexpr int SW_STREAMER = 9;
constexpr int SW_PROD_B = 10;        // .. SW_PROD_B + SW_NPB - 1
constexpr int SW_NPB = 2;
constexpr int SW_FAR = 192;          // far rows per pass (three row groups of 64)
constexpr int SW_MAX_SB = 416;       // widest ring B column (rows)
constexpr int SW_THREADS = 768;
constexpr int SW_DIN = 16;           // right-hand side steps in flight
constexpr int SW_NIN = SW_DIN + 1;   // staging slots of 64 dwords

// widest band the staged sweep takes (two far rows per lane above 192 + BS)
template <class T>
constexpr int sweep_staged_max() { return 2 * SW_FAR + sweep_bs<T>(); }   // (ring B columns: up to 384 far rows)

// Waits until at most n (wave-uniform, 0 .. 63) vector memory operations are
// outstanding.  s_waitcnt takes an immediate, so this jumps into a table of
// 64 (wait, branch) pairs of 8 bytes each, which starts 12 bytes after the
// program counter that s_getpc returns.
__device__ __forceinline__ void wait_vmcnt(int n)
{
    const int off = __builtin_amdgcn_readfirstlane(n) * 8 + 12;
    asm volatile("s_getpc_b64 vcc\n\t"
                 "s_add_u32 vcc_lo, vcc_lo, %0\n\t"
                 "s_addc_u32 vcc_hi, vcc_hi, 0\n\t"
                 "s_setpc_b64 vcc\n\t"
                 ".set .Lwait_i%=, 0\n\t"
                 ".rept 64\n\t"
                 "s_waitcnt vmcnt(.Lwait_i%=)\n\t"
                 "s_branch .Lwait_end%=\n\t"
                 ".set .Lwait_i%=, .Lwait_i%=+1\n\t"
                 ".endr\n"
                 ".Lwait_end%=:"
                 :
                 : "s"(off)
                 : "vcc", "scc", "memory");
}

// the same for a constant count; gfx9 encoding: vmcnt bits [3:0] and [15:14],
// expcnt [6:4] and lgkmcnt [11:8] left at their maxima (no wait)
template <int N>
__device__ __forceinline__ void wait_vmcnt_imm()
{
    __builtin_amdgcn_s_waitcnt((N & 0xF) | ((N >> 4) << 14) | (0x7 << 4) | (0xF << 8));
    asm volatile("" ::: "memory");
}

// one asynchronous copy of 16 (4) bytes per lane, HBM -> LDS (lane l's at
// dst + 16 l (4 l); dst wave-uniform)
__device__ __forceinline__ void copy16_to_lds(const void* src, void* dst)
{
    __builtin_amdgcn_global_load_lds(src, dst, 16, 0, 0);
}
__device__ __forceinline__ void copy4_to_lds(const void* src, void* dst)
{
    __builtin_amdgcn_global_load_lds(src, dst, 4, 0, 0);
}

// The two BS x BS products of the chain.  A "half" of a row is MJ columns.
// The vector x is held one element per lane in one of two arrangements
// (lane l: row r = l / 16, c = l % 16):
//   FP32, BS = 32:  A: rows 0,1 hold x[c], rows 2,3 hold x[16 + c]
//                   B: rows 0,2 hold x[c], rows 1,3 hold x[16 + c]
//   FP64, BS = 16:  A = B: every row holds x[c]
// mul_ab takes A and returns B, mul_ba the reverse.
template <class T>
struct ChainMul;

// The N products of a lane: sum of m[jj] * x[lane jj of its 16-lane row],
// four partial sums.  (hipcc keeps the broadcasts as moves of their own, so
// the multiply-adds are written out; an instruction that broadcasts must not
// follow the one that wrote its source by less than two wait states, hence
// the leading s_nop.)
__device__ __forceinline__ float row_dot(const float (&m)[16], float x)
{
    float s0, s1, s2, s3;
    asm volatile("s_nop 1\n\t"
        "v_mul_f32_dpp %0, %4, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_mul_f32_dpp %1, %4, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_mul_f32_dpp %2, %4, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_mul_f32_dpp %3, %4, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %4, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %4, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %4, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %4, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %4, %13 row_newbcast:8 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %4, %14 row_newbcast:9 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %4, %15 row_newbcast:10 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %4, %16 row_newbcast:11 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %0, %4, %17 row_newbcast:12 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %1, %4, %18 row_newbcast:13 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %2, %4, %19 row_newbcast:14 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f32_dpp %3, %4, %20 row_newbcast:15 row_mask:0xf bank_mask:0xf"
        : "=&v"(s0), "=&v"(s1), "=&v"(s2), "=&v"(s3)
        : "v"(x), "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(m[4]), "v"(m[5]), "v"(m[6]), "v"(m[7]), "v"(m[8]),
          "v"(m[9]), "v"(m[10]), "v"(m[11]), "v"(m[12]), "v"(m[13]), "v"(m[14]), "v"(m[15]));
    return (s0 + s1) + (s2 + s3);
}
__device__ __forceinline__ double row_dot(const double (&m)[8], double x)
{
    double s0 = 0., s1 = 0., s2 = 0., s3 = 0.;
    asm volatile("s_nop 1\n\t"
        "v_fmac_f64_dpp %0, %4, %5 row_newbcast:0 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %4, %6 row_newbcast:1 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %2, %4, %7 row_newbcast:2 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %3, %4, %8 row_newbcast:3 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %0, %4, %9 row_newbcast:4 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %1, %4, %10 row_newbcast:5 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %2, %4, %11 row_newbcast:6 row_mask:0xf bank_mask:0xf\n\t"
        "v_fmac_f64_dpp %3, %4, %12 row_newbcast:7 row_mask:0xf bank_mask:0xf"
        : "+&v"(s0), "+&v"(s1), "+&v"(s2), "+&v"(s3)
        : "v"(x), "v"(m[0]), "v"(m[1]), "v"(m[2]), "v"(m[3]), "v"(m[4]), "v"(m[5]), "v"(m[6]), "v"(m[7]));
    return (s0 + s1) + (s2 + s3);
}

// lanes 0-31 and 32-63 (swap32) or odd and even 16-lane rows (swap16) of v
// added: every lane gets the sum of its value and its counterpart's
__device__ __forceinline__ float add_swap32(float v)
{
    const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ float add_swap16(float v)
{
    const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
    return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}
__device__ __forceinline__ double add_swap32(double v)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const auto lo = __builtin_amdgcn_permlane32_swap((unsigned)b, (unsigned)b, false, false);
    const auto hi = __builtin_amdgcn_permlane32_swap((unsigned)(b >> 32), (unsigned)(b >> 32), false, false);
    return __longlong_as_double((long long)(((unsigned long long)hi[0] << 32) | lo[0])) +
           __longlong_as_double((long long)(((unsigned long long)hi[1] << 32) | lo[1]));
}

template <>
struct ChainMul<float> {
    static constexpr int BS = 32, MJ = 16;
    __device__ static int vec_a(int l) { return (l & 15) + 16 * (l >> 5); }   // element a lane holds in A
    __device__ static int tab_lane(int l) { return l; }
    __device__ static constexpr int lane_of(int e) { return e < 16 ? e : 16 + e; }   // a lane holding element e in A
    __device__ __forceinline__ static float a_to_b(float x)
    {
        // both swapped copies: every row x[0..15], every row x[16..31]
        const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(x), __float_as_uint(x), false, false);
        return __uint_as_float((threadIdx.x & 16) ? r[1] : r[0]);
    }
    // T(0, 0), lane 0's first entry, is 1 in a table that may be used
    __device__ __forceinline__ static bool tab_usable(float t)
    {
        return __builtin_amdgcn_readfirstlane(__float_as_int(t)) == 0x3f800000;
    }
    // position of entry (i, j) of T (multiplied by mul_ab: lane l computes
    // row (l & 15) + 16 ((l >> 4) & 1) over columns 16 (l >> 5) ..) and of S
    // (mul_ba: row (l & 15) + 16 (l >> 5), columns 16 ((l >> 4) & 1) ..) in a
    // block's table: [quad of columns][lane][4]
    __device__ static int tab_pos(int i, int j)
    {
        const int lane = (i & 15) + 16 * (i >> 4) + 32 * (j >> 4), jj = j & 15;
        return (jj >> 2) * 256 + lane * 4 + (jj & 3);
    }
    __device__ static int sub_pos(int i, int j)
    {
        const int lane = (i & 15) + 32 * (i >> 4) + 16 * (j >> 4), jj = j & 15;
        return (jj >> 2) * 256 + lane * 4 + (jj & 3);
    }
    // row i of the block's T
    __device__ __forceinline__ static void lds_row(const float* t, int i, float (&v)[BS])
    {
#pragma unroll
        for (int q = 0; q < BS / 4; ++q) {
            const float4 x = *reinterpret_cast<const float4*>(t + tab_pos(i, 4 * q));
            v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
        }
    }
    __device__ __forceinline__ static float mul_ab(const float (&m)[MJ], float x)
    {
        return add_swap32(row_dot(m, x));
    }
    __device__ __forceinline__ static float mul_ba(const float (&m)[MJ], float x)
    {
        return add_swap16(row_dot(m, x));
    }
};

template <>
struct ChainMul<double> {
    static constexpr int BS = 16, MJ = 8;
    __device__ static int vec_a(int l) { return l & 15; }
    __device__ static int tab_lane(int l) { return (l & 15) + 16 * (l >> 5); }
    __device__ static constexpr int lane_of(int e) { return e; }
    __device__ __forceinline__ static double a_to_b(double x) { return x; }
    __device__ __forceinline__ static bool tab_usable(double t)
    {
        return __builtin_amdgcn_readfirstlane(__double2hiint(t)) == 0x3ff00000;
    }
    // (row l & 15 over columns 8 (l >> 5) .., for T and S alike)
    __device__ static int tab_pos(int i, int j)
    {
        const int jj = j & 7;
        return (jj >> 1) * 64 + (i + 16 * (j >> 3)) * 2 + (jj & 1);
    }
    __device__ static int sub_pos(int i, int j) { return tab_pos(i, j); }
    __device__ __forceinline__ static void lds_row(const double* t, int i, double (&v)[BS])
    {
#pragma unroll
        for (int q = 0; q < BS / 2; ++q) {
            const double2 x = *reinterpret_cast<const double2*>(t + tab_pos(i, 2 * q));
            v[2 * q] = x.x; v[2 * q + 1] = x.y;
        }
    }
    __device__ __forceinline__ static double mul_ab(const double (&m)[MJ], double x)
    {
        // lanes 32-63 take columns 8..15: their row rotated by 8 lanes, so
        // that broadcasting lane jj of a row gives x[8 + jj] there
        const long long b = __double_as_longlong(x);
        const int lo = __builtin_amdgcn_update_dpp((int)b, (int)b, 0x128, 0xc, 0xf, false);
        const int hi = __builtin_amdgcn_update_dpp((int)(b >> 32), (int)(b >> 32), 0x128, 0xc, 0xf, false);
        const double xr = __longlong_as_double(((long long)hi << 32) | (unsigned)lo);
        return add_swap32(row_dot(m, xr));
    }
    __device__ __forceinline__ static double mul_ba(const double (&m)[MJ], double x) { return mul_ab(m, x); }
};

// N values from 16-byte aligned LDS (16-byte reads)
template <int N>
__device__ __forceinline__ void lds_read16(const float* p, float (&v)[N], int stride)
{
#pragma unroll
    for (int q = 0; q < N / 4; ++q) {
        const float4 x = *reinterpret_cast<const float4*>(p + q * stride);
        v[4 * q] = x.x; v[4 * q + 1] = x.y; v[4 * q + 2] = x.z; v[4 * q + 3] = x.w;
    }
}
template <int N>
__device__ __forceinline__ void lds_read16(const double* p, double (&v)[N], int stride)
{
#pragma unroll
    for (int q = 0; q < N / 2; ++q) {
        const double2 x = *reinterpret_cast<const double2*>(p + q * stride);
        v[2 * q] = x.x; v[2 * q + 1] = x.y;
    }
}

// LDS geometry of the staged sweep.  A ring A slot is one block's table: T,
// S and 64 dwords that start with the pivots.  The far rows are copied as
// 16-byte chunks (E elements) covering each column's at any alignment; a
// column of ring B takes sb elements, a multiple of 32, so that the far rows
// are read at compile-time offsets.  A round is 64 chunks, one load of a
// wavefront.
template <class T>
struct SweepGeom {
    static constexpr int E = 16 / sizeof(T);
    static constexpr int BS = sweep_bs<T>();
    static constexpr int RT = 2 * BS * BS / (64 * E);                    // rounds of T and S
    static constexpr int slot_a = 2 * BS * BS + 256 / (int)sizeof(T);    // elements of a table
    int nfar, sb, rb;                                    // far rows; ring B column; its rounds
    __host__ __device__ explicit SweepGeom(int k)
    {
        nfar = k > BS ? k - BS : 0;
        sb = nfar > 0 ? (nfar + E - 1 + 31) / 32 * 32 : 0;
        rb = sb / 8;                                     // BS * sb / E / 64
    }
    __host__ __device__ int slot_b() const { return rb * 64 * E; }
};

// Right-hand side of a sweep: view row r reads element s0 + sdir * r of p
// (FP64 input vector: raw64, else T), less the corrections of the view's
// first k rows (element i at first[cdir * i]) and of its last k rows
// (last[cdir * i]); either may be null.
template <class T>
struct SweepSrc {
    const void* p;
    bool raw64;
    int64_t s0;
    int sdir;
    const T *first, *last;
    int cdir;
    __device__ __forceinline__ T load(int r, int len, int k) const
    {
        const int64_t i = s0 + (int64_t)sdir * r;
        T v = raw64 ? (T) reinterpret_cast<const double*>(p)[i] : reinterpret_cast<const T*>(p)[i];
        if (first && r < k) v -= first[cdir * r];
        if (last && r >= len - k) v -= last[cdir * (r - (len - k))];
        return v;
    }
};

// Where a sweep's results go: view row r to element s0 + sdir * r of p (FP64
// or T).
struct SweepDst {
    void* p;
    bool f64;
    int64_t s0;
    int sdir;
};

// LDS of one staged sweep: pending rings of the two column halves, the
// corrections of the last k rows, the right-hand side staging, the slots of
// rings A and B.
template <class T>
struct SweepLds {
    T *pend0, *pend1, *corr, *a, *b;
    unsigned* stage;
    int ring_mask, na, nb;
};

// all ones where c, kept in a vector register (the compiler would hold a
// pair of scalar registers per mask otherwise, and spill them)
__device__ __forceinline__ int vector_mask(bool c)
{
    int m = c ? -1 : 0;
    asm volatile("" : "+v"(m));
    return m;
}
__device__ __forceinline__ float and_bits(float v, int m) { return __int_as_float(__float_as_int(v) & m); }
__device__ __forceinline__ double and_bits(double v, int m)
{
    const unsigned long long b = (unsigned long long)__double_as_longlong(v);
    const unsigned lo = (unsigned)b & (unsigned)m, hi = (unsigned)(b >> 32) & (unsigned)m;
    return __longlong_as_double((long long)(((unsigned long long)hi << 32) | lo));
}

// The far rows of every block (waves 1-3, 5-7): rows 2 BS + t of block b - 1
// in step b, columns jh .. jh + BS/2 - 1.  MASKED: some of the wavefront's
// rows leave the band (2 BS + t - j > k).
template <class T, int SB, bool MASKED>
__device__ __forceinline__ void sweep_far_loop(int k, int dir, int len, int nblk, int t, int jh, int al0, int al1,
                                               const SweepLds<T>& S, T* pend, const T* xblk2)
{
    constexpr int E = SweepGeom<T>::E, BS = SweepGeom<T>::BS, HC = BS / 2;
    constexpr int slot = SB / 8 * 64 * E;
    const int nfar = k - BS;
    int mk[HC];
    if constexpr (MASKED) {
#pragma unroll
        for (int j = 0; j < HC; ++j) mk[j] = vector_mask(2 * BS + t - jh - j <= k);
    }
    const int pos = jh * SB + (dir > 0 ? t : nfar - 1 - t);
    const T* const q0 = S.b + pos + al0;
    const T* const q1 = S.b + pos + al1 + SB;
    const T* const xq = xblk2 + jh;
    const int end = S.nb * slot;
    int base = 0, r = (2 * BS + t) & S.ring_mask, left = t < nfar ? len - 2 * BS - t : 0;
    lds_barrier();   // step 0: nothing to apply yet
    for (int b = 1; b <= nblk; ++b) {
        if (left > 0) {   // (then block b - 1 is a full block)
            T xp[HC], m[HC];
            const T old = pend[r];
            lds_read16<HC>(xq + ((b - 1) & 1) * BS, xp, E);
#pragma unroll
            for (int j = 0; j < HC; j += 2) {
                m[j] = q0[base + j * SB];
                m[j + 1] = q1[base + j * SB];
            }
            T s0 = 0, s1 = 0;
#pragma unroll
            for (int j = 0; j < HC; j += 2) {
                if constexpr (MASKED) {
                    m[j] = and_bits(m[j], mk[j]);
                    m[j + 1] = and_bits(m[j + 1], mk[j + 1]);
                }
                s0 = fma(m[j], xp[j], s0);
                s1 = fma(m[j + 1], xp[j + 1], s1);
            }
            pend[r] = old - (s0 + s1);
        }
        left -= BS;
        r = (r + BS) & S.ring_mask;
        base = base + slot == end ? 0 : base + slot;
        lds_barrier();
    }
}

// The same for bands above SW_FAR + BS: the wavefront's rows in two passes,
// SW_FAR apart.
template <class T, int SB>
__device__ __forceinline__ void sweep_far_wide(int k, int dir, int len, int nblk, int t0, int jh, int al0, int al1,
                                               const SweepLds<T>& S, T* pend, const T* xblk2)
{
    constexpr int E = SweepGeom<T>::E, BS = SweepGeom<T>::BS, HC = BS / 2;
    constexpr int slot = SB / 8 * 64 * E;
    const int nfar = k - BS;
    lds_barrier();
    int base = 0;
    for (int b = 1; b <= nblk; ++b) {
        const int row0 = (b - 1) * BS + 2 * BS;
        for (int t = t0; t < nfar; t += SW_FAR) {
            if (row0 + t < len) {
                T xp[HC];
                lds_read16<HC>(xblk2 + ((b - 1) & 1) * BS + jh, xp, E);
                const int r = (row0 + t) & S.ring_mask;
                const T old = pend[r];
                const int pos = base + jh * SB + (dir > 0 ? t : nfar - 1 - t);
                const T* p0 = S.b + pos + al0;
                const T* p1 = S.b + pos + al1 + SB;
                T s0 = 0, s1 = 0;
                unsigned m = ~bits_below(2 * BS + t - jh - k);
                asm volatile("" : "+v"(m));   // (no scalar mask per column kept across the loop)
#pragma unroll
                for (int j = 0; j < HC; j += 2) {
                    s0 = fma(keep_if(p0[j * SB], m, j), xp[j], s0);
                    s1 = fma(keep_if(p1[j * SB], m, j + 1), xp[j + 1], s1);
                }
                pend[r] = old - (s0 + s1);
            }
        }
        base = base + slot == S.nb * slot ? 0 : base + slot;
        lds_barrier();
    }
}

template <class T, int SB>
__device__ __forceinline__ void sweep_far(int sb, int k, int dir, int len, int nblk, int t0, int jh, int al0, int al1,
                                          const SweepLds<T>& S, T* pend, const T* xblk2)
{
    if constexpr (SB <= SW_MAX_SB) {
        if (sb != SB) {
            sweep_far<T, SB + 32>(sb, k, dir, len, nblk, t0, jh, al0, al1, S, pend, xblk2);
            return;
        }
        constexpr int BS = SweepGeom<T>::BS;
        if constexpr (SB > SW_FAR) {
            if (k - BS > SW_FAR) {
                sweep_far_wide<T, SB>(k, dir, len, nblk, t0, jh, al0, al1, S, pend, xblk2);
                return;
            }
        }
        if constexpr (SB <= SW_FAR + 32) {
            // is the wavefront's last row inside the band?
            if (__builtin_amdgcn_readfirstlane(2 * BS + (t0 | 63) - jh <= k))
                sweep_far_loop<T, SB, false>(k, dir, len, nblk, t0, jh, al0, al1, S, pend, xblk2);
            else
                sweep_far_loop<T, SB, true>(k, dir, len, nblk, t0, jh, al0, al1, S, pend, xblk2);
        }
    }
}

// Element (row c0 + r, column c0 + j) of block b = c0 / BS sits at V.origin +
// dir * ((c0 + j) * w + k + r - j).  In ring B column j starts at its lowest
// address (row 2 BS, or the last far row when dir < 0) rounded down to a
// chunk, far_al(j) elements below it; that depends on j's parity only (rows
// are one element apart, columns 2 k).
template <class T>
__device__ __forceinline__ int far_al(const BandView<T>& V, int j)
{
    constexpr int BS = SweepGeom<T>::BS;
    const int64_t lo = V.origin + V.dir * ((int64_t)V.k + (int64_t)j * 2 * V.k) + (V.dir > 0 ? 2 * BS : -(BS + V.k - 1));
    return (int)(lo & (SweepGeom<T>::E - 1));
}

// tab: the view's tables; scale: the results are divided by the pivots.
template <class T>
__device__ __forceinline__ void lower_sweep_lds(const BandView<T>& V, const T* __restrict__ tab, int64_t len64,
                                                const SweepSrc<T>& src, const SweepDst& dst, bool scale,
                                                const SweepLds<T>& S, T* xblk2)
{
    using CM = ChainMul<T>;
    using GM = SweepGeom<T>;
    constexpr int BS = CM::BS, MJ = CM::MJ, E = GM::E;
    static_assert(BS == sweep_bs<T>(), "block rows");
    const GM G(V.k);
    const int k = V.k;
    const int dir = V.dir;
    const int len = (int)len64;
    // (opaque: nothing derived from the lane is kept across the stages)
    int tid = threadIdx.x;
    asm volatile("" : "+v"(tid));
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int nblk = (len + BS - 1) / BS;
    const int na = S.na, nb = S.nb, ring_mask = S.ring_mask;

    const int H = BS + max(BS, k);   // rows [c0 + H, ..) are first touched after step b
    const int init = min(len, H);
    for (int r = threadIdx.x; r < init; r += blockDim.x) {
        S.pend0[r & ring_mask] = src.load(r, len, k);
        S.pend1[r & ring_mask] = (T)0;
    }
    // (in LDS: the streamer's waits count its own copies, so it loads nothing else)
    if (src.last)
        for (int i = threadIdx.x; i < k; i += blockDim.x) S.corr[i] = src.last[src.cdir * i];

    // Every role walks the same nblk + 1 steps, one barrier each, after the
    // barrier that follows its prologue.
    if (wave == 0) {
        lds_barrier();
        const int vi = CM::vec_a(lane);
        const int tl = CM::tab_lane(lane) * E;
        T* const px = xblk2 + (lane & (BS - 1));   // (lanes BS .. 63 hold copies of lanes 0 .. BS-1)
        T sm[MJ];
#pragma unroll
        for (int jj = 0; jj < MJ; ++jj) sm[jj] = (T)0;
        T x = (T)0;
        // (what the next step reads is addressed before the barrier, and the
        // empty asm keeps each group of reads where it is)
        int base = 0, ri = vi, rows = len - vi;
        int tp = tl;
        for (int b = 0; b < nblk; ++b) {
            const T q0 = S.pend0[ri], q1 = S.pend1[ri];
            T tm[MJ];
            lds_read16<MJ>(S.a + tp, tm, BS * BS / (MJ / E));
            asm volatile("" ::: "memory");
            const T carry = CM::mul_ba(sm, x);   // S_{b-1} x_{b-1}, the element vi of block b
            lds_read16<MJ>(S.a + tp + BS * BS, sm, BS * BS / (MJ / E));
            asm volatile("" ::: "memory");
            const T p = rows > 0 ? (q0 + q1) - carry : (T)0;
            if (__builtin_expect(CM::tab_usable(tm[0]), 1)) {
                x = CM::mul_ab(tm, p);
            } else {
                // the block's inverse grew too large to multiply with, and
                // the table holds its multipliers (0 from a row's own column
                // on): substitute, element vi in each lane.  (The row comes
                // to registers first: with a read per step of the chain, a
                // band of n = 100000, k = 20, 16 partitions whose blocks mostly
                // grow took 628 us in FP32, 550 in FP64; 225 and 330 so, 119
                // and 217 where none grows.)
                T l[BS], y = p;
                CM::lds_row(S.a + base, vi, l);
#pragma unroll
                for (int j = 0; j < BS - 1; ++j) y = fma(-l[j], bcast(y, CM::lane_of(j)), y);
                x = CM::a_to_b(y);
            }
            px[(b & 1) * BS] = x;
            base = base + GM::slot_a == na * GM::slot_a ? 0 : base + GM::slot_a;
            tp = tl + base;
            ri = (ri + BS) & ring_mask;
            rows -= BS;
            asm volatile("" : "+v"(tp), "+v"(ri));
            lds_barrier();
        }
        lds_barrier();
    } else if (wave < 8 && wave != SW_PROD_A) {
        const int half = wave >> 2, t0 = ((wave & 3) - 1) * 64 + lane;
        lds_barrier();
        if (G.nfar > 0) {
            sweep_far<T, 32>(G.sb, k, dir, len, nblk, t0, half * (BS / 2), far_al(V, 0), far_al(V, 1), S,
                             half ? S.pend1 : S.pend0, xblk2);
        } else {
            for (int b = 0; b <= nblk; ++b) lds_barrier();
        }
    } else if (wave == SW_STREAMER) {
        // step st carries rows [st*BS + H, st*BS + H + BS)
        const int nstream = len > H ? (len - H + BS - 1) / BS : 0;
        auto run = [&](auto raw) {
            using R = decltype(raw);
            constexpr int SH = sizeof(R) == 8 ? 1 : 0;   // dwords per row: 1 << SH
            const int str = (lane >> SH) % BS, word = lane & ((1 << SH) - 1);
            const unsigned* p0 = reinterpret_cast<const unsigned*>(reinterpret_cast<const R*>(src.p) + src.s0) + word;
            auto stream = [&](int st, int slot) {
                const int r = min(st * BS + H + str, len - 1);
                const int64_t off = (int64_t)(src.sdir * r) * (1 << SH);
                copy4_to_lds(p0 + off, S.stage + slot * 64);
            };
            for (int st = 0; st < min(nstream, SW_DIN); ++st) stream(st, st);
            lds_barrier();
            // In step b the rows of stream step b (read from the staging ring
            // in the step before) go to the pending ring, and those of step
            // b + 1 are read.
            const bool have_last = src.last != nullptr;
            const R* sg = reinterpret_cast<const R*>(S.stage);
            const int ln = lane & (BS - 1);
            R raw_v = (R)0;
            if (nstream > 0) {
                wait_vmcnt(min(SW_DIN, nstream) - 1);
                raw_v = sg[ln];
            }
            int sl = 0;     // b % SW_NIN
            int rr = H + lane;
            for (int b = 0; b <= nblk; ++b) {
                if (b < nstream) {
                    if (b + SW_DIN < nstream) stream(b + SW_DIN, sl == 0 ? SW_NIN - 1 : sl - 1);
                    sl = sl + 1 == SW_NIN ? 0 : sl + 1;
                    T v = (T)raw_v;
                    // the next step's rows: every copy but the SW_DIN - 1
                    // after them has arrived
                    if (b + SW_DIN < nstream) {
                        wait_vmcnt_imm<SW_DIN - 1>();
                        raw_v = sg[sl * (256 / (int)sizeof(R)) + ln];
                    } else if (b + 1 < nstream) {
                        wait_vmcnt(nstream - 2 - b);
                        raw_v = sg[sl * (256 / (int)sizeof(R)) + ln];
                    }
                    if (lane < BS && rr < len) {
                        if (have_last && rr >= len - k) v -= S.corr[rr - (len - k)];
                        S.pend0[rr & ring_mask] = v;
                        S.pend1[rr & ring_mask] = (T)0;
                    }
                    rr += BS;
                }
                lds_barrier();
            }
        };
        if (src.raw64) run(double{});
        else run(T{});
    } else if (wave == SW_WRITER) {
        lds_barrier();
        // block b - 1's results in step b; its pivots were read in the step
        // before (their slot is refilled)
        auto run = [&](auto o, auto sc) {
            using O = decltype(o);
            constexpr bool SC = decltype(sc)::value;
            const T* const pd = S.a + 2 * BS * BS + (lane & (BS - 1));
            const T* const px = xblk2 + (lane & (BS - 1));
            O* to = reinterpret_cast<O*>(dst.p) + (dst.s0 + (int64_t)dst.sdir * lane);
            int left = lane < BS ? len - lane : 0, base = 0;
            for (int b = 0; b < nblk; ++b) {
                T d = (T)1;
                if constexpr (SC) d = pd[base];
                base = base + GM::slot_a == na * GM::slot_a ? 0 : base + GM::slot_a;
                lds_barrier();
                const T x = px[(b & 1) * BS];
                if (left > 0) *to = (O)(SC ? x / d : x);
                to += dst.sdir * BS;
                left -= BS;
            }
            lds_barrier();
        };
        if (dst.f64) {
            if (scale) run(double{}, std::true_type{});
            else run(double{}, std::false_type{});
        } else {
            if (scale) run(T{}, std::true_type{});
            else run(T{}, std::false_type{});
        }
    } else if (wave == SW_PROD_A) {
        constexpr int NI = GM::RT + 1;
        auto produce = [&](int b, int slot) {
            T* dst = S.a + slot * GM::slot_a;
            const char* st = reinterpret_cast<const char*>(tab + (int64_t)b * GM::slot_a);
#pragma unroll
            for (int i = 0; i < GM::RT; ++i)
                copy16_to_lds(st + (unsigned)(i * 64 + lane) * 16, dst + i * 64 * E);
            copy4_to_lds(st + (unsigned)(GM::RT * 64 * 16 + lane * 4), dst + 2 * BS * BS);
        };
        // Block b is in LDS when step b starts; step b refills the slot of
        // block b - 1.  While blocks are still requested, na - 2 of them may be
        // outstanding.
        auto run = [&](auto c) -> void {
            constexpr int W = decltype(c)::value;
            for (int b = 0; b < min(nblk, na - 1); ++b) produce(b, b);
            wait_vmcnt((min(nblk, na - 1) - 1) * NI);
            lds_barrier();
            int slot = na - 1, b = 0;   // slot (b + na - 1) % na
            for (; b + na - 1 < nblk; ++b) {
                produce(b + na - 1, slot);
                slot = slot + 1 == na ? 0 : slot + 1;
                wait_vmcnt_imm<W * NI>();
                lds_barrier();
            }
            for (; b <= nblk; ++b) {
                if (b + 1 < nblk) wait_vmcnt((nblk - 2 - b) * NI);
                lds_barrier();
            }
        };
        static_assert(6 * NI <= 63, "outstanding loads");
        switch (na) {
        case 3: run(std::integral_constant<int, 1>{}); break;
        case 4: run(std::integral_constant<int, 2>{}); break;
        case 5: run(std::integral_constant<int, 3>{}); break;
        case 6: run(std::integral_constant<int, 4>{}); break;
        case 7: run(std::integral_constant<int, 5>{}); break;
        default: run(std::integral_constant<int, 6>{}); break;   // 8
        }
    } else {
        constexpr int NIM = (SW_MAX_SB / 8 + SW_NPB - 1) / SW_NPB;
        const int pw = wave - SW_PROD_B;
        const int ni = G.rb > 0 ? (G.rb - pw + SW_NPB - 1) / SW_NPB : 0;
        const int nch = G.sb / E;
        // Chunk ch of column j, from row 2 BS of the block (its last far row
        // when dir < 0) rounded down to a chunk.  Chunks without a band entry
        // of the column (never used) copy the nearest one that has: in bounds.
        // Byte offset from `low`, the lowest band entry of block 0 rounded
        // down to a chunk; it is the same in every block (a block is BS * w
        // elements, a multiple of E).
        const int r0 = 2 * BS, r1 = BS + k - 1;
        const int64_t e00 = V.origin + (int64_t)dir * k;   // element (0, 0)
        const int64_t low = (dir > 0 ? e00 : e00 - (int64_t)(BS - 1) * V.w - k) & ~(int64_t)(E - 1);
        const int64_t blk_bytes = (int64_t)dir * V.w * BS * (int64_t)sizeof(T);
        auto chunk_off = [&](int g) -> unsigned {
            const int j = g / nch;
            const int64_t lo = e00 + dir * ((int64_t)j * 2 * k) + (dir > 0 ? r0 : -r1);
            const int al = (int)(lo & (E - 1));
            const int last = min(r1, j + k);               // last band row of the column in the slot
            int x0 = dir > 0 ? 0 : r1 - last, x1 = dir > 0 ? last - r0 : r1 - r0;
            if (r0 > last) x0 = x1 = dir > 0 ? j + k - r0 : r1 - (j + k);
            const int sh = E == 4 ? 2 : 1;
            const int ch = min(max(g - j * nch, (x0 + al) >> sh), (x1 + al) >> sh);
            return (unsigned)(((lo - al) + (int64_t)ch * E - low) * (int64_t)sizeof(T));
        };
        unsigned off[NIM];
#pragma unroll
        for (int i = 0; i < NIM; ++i) {
            if (i >= ni) break;
            off[i] = chunk_off((i * SW_NPB + pw) * 64 + lane);
            asm volatile("" : "+v"(off[i]));   // (one after the other: fewer registers)
        }
        auto produce = [&](int b, int slot) {
            T* dst = S.b + slot * G.slot_b() + pw * 64 * E;
            const char* sb = reinterpret_cast<const char*>(V.base + low) + b * blk_bytes;
            int nl = ni;
            asm volatile("" : "+s"(nl));   // (no scalar mask per unrolled comparison kept across the loop)
#pragma unroll
            for (int i = 0; i < NIM; ++i) {
                if (i >= nl) break;
                copy16_to_lds(sb + off[i], dst + i * SW_NPB * 64 * E);
            }
        };
        // Block b is in LDS when step b + 1 starts; step b refills the slot of
        // block b - 2.  Only full blocks are copied.  While blocks are still
        // requested, (nb - 2) * ni loads may be outstanding; the wait takes
        // the next lower count it has an immediate for.
        const int nfull = ni > 0 ? len / BS : 0;
        auto run = [&](auto c) -> void {
            constexpr int W = decltype(c)::value;
            for (int b = 0; b < min(nfull, nb - 2); ++b) produce(b, b);
            lds_barrier();
            int slot = nb - 2, b = 0;   // slot (b + nb - 2) % nb
            for (; b + nb - 2 < nfull; ++b) {
                produce(b + nb - 2, slot);
                slot = slot + 1 == nb ? 0 : slot + 1;
                wait_vmcnt_imm<W>();
                lds_barrier();
            }
            for (; b <= nblk; ++b) {
                if (b < nfull) wait_vmcnt(min((nfull - 1 - b) * ni, 63));
                lds_barrier();
            }
        };
        const int w = min((nb - 2) * ni, 63);
        if (w >= 48) run(std::integral_constant<int, 48>{});
        else if (w >= 36) run(std::integral_constant<int, 36>{});
        else if (w >= 28) run(std::integral_constant<int, 28>{});
        else if (w >= 24) run(std::integral_constant<int, 24>{});
        else if (w >= 20) run(std::integral_constant<int, 20>{});
        else if (w >= 16) run(std::integral_constant<int, 16>{});
        else if (w >= 12) run(std::integral_constant<int, 12>{});
        else if (w >= 8) run(std::integral_constant<int, 8>{});
        else run(std::integral_constant<int, 0>{});
    }
}

// ---------------------------------------------------------------------------
// The tables of the staged sweeps (SweepGeom::slot_a elements per block of BS
// columns): for every factored range (FactorJob) and both sweep directions
// (stage 1 the factorization's own, stage 2 the other) T, S and the pivots of
// each block of the view.  Rows past the range's end are rows of the identity
// in T, zero in S.  One BS-lane group per block: lane j solves for column j
// of T with the block's multipliers broadcast from LDS.  A block of whose
// inverse an entry passes SW_GROWTH (or is no number) keeps its multipliers
// instead, T(0, 0) = 0 telling the sweeps to substitute: the product with T has
// no small residual in the block's own equations, which the following blocks
// then amplify.  The limit is where the error of a whole application (against
// the same factors in higher precision) is still that of substituting
// everywhere: the ratio of the two, geometric mean of 240 bands each with n =
// 800, k = 20, 50 and 90 (+- 0.04), by the band's dominance:
//               FP32 0.04   0.07   0.1    FP64 0.04   0.07   0.1
//   limit 4          1.00   1.00   0.87        0.97   1.04   0.96
//         8          0.99   1.05   0.86        0.99   1.04   0.97
//        16          1.06   1.21   0.99        1.14   1.21   1.14
// The error is smaller than substitution's where nothing grows (0.6 in FP32
// and 0.8 in FP64 from 0.3 on, at every limit), and T in twice the precision
// changes nothing.  A lower limit costs time on growing bands only: 211 us at
// 16, 225 at 8, 228 at 4 (dominance 0.1, n = 100000, k = 20, FP32).
// Bound by bytes, 264 written a row and direction and the lines that hold the
// diagonal blocks read: 0.62 ms at n = 1000000, k = 200 with both
// factorizations (1.06 GB written, 1.6 GB read), 52 us at n = 200000, k = 50.
// That is paid once a setup and won back about with the first application
// (0.58 and 0.79 ms saved on each).
// ---------------------------------------------------------------------------
constexpr int TAB_THREADS = 256;
constexpr double SW_GROWTH = 8.0;

template <class T>
__global__ __launch_bounds__(TAB_THREADS) void sweep_tables_kernel(const T* __restrict__ B0, const T* __restrict__ B1,
                                                                   int k_all, const FactorJob* __restrict__ jobs,
                                                                   T* __restrict__ tab0, T* __restrict__ tab1,
                                                                   int64_t stage_stride)
{
    using CM = ChainMul<T>;
    constexpr int BS = CM::BS, NB = TAB_THREADS / BS, LS = BS + 16 / (int)sizeof(T), E = 16 / (int)sizeof(T);
    __shared__ alignas(16) T lb[NB * BS * LS];   // per block: column m of L in row m; then T, then S
    const FactorJob J = jobs[blockIdx.y];
    const int k = J.kb > 0 ? J.kb : k_all;
    if (k > sweep_staged_max<T>()) return;   // swept without tables
    const int stage = blockIdx.z;
    const int nblk = (int)((J.len + BS - 1) / BS);
    if ((int)blockIdx.x * NB >= nblk) return;
    const BandView<T> V = make_view((J.buf ? B1 : B0) + J.boff, J.start, J.len, k, stage ? -J.dir : J.dir);
    const int grp = threadIdx.x / BS, lane = threadIdx.x % BS;
    const int b = blockIdx.x * NB + grp;
    const int64_t c0 = (int64_t)b * BS;
    const int nb = (int)min((int64_t)BS, J.len - c0);              // <= 0: no such block
    const int ns = (int)min((int64_t)BS, J.len - c0 - BS);         // rows of S
    T* L = lb + grp * BS * LS;
    T sub[BS];
#pragma unroll
    for (int m = 0; m < BS; ++m) {
        L[m * LS + lane] = (lane > m && lane < nb && lane - m <= k) ? V.at(c0 + lane, c0 + m) : (T)0;
        sub[m] = lane < ns && BS + lane - m <= k ? V.at(c0 + BS + lane, c0 + m) : (T)0;
    }
    const T piv = lane < nb ? V.at(c0 + lane, c0 + lane) : (T)1;
    __syncthreads();
    T x[BS];
#pragma unroll
    for (int i = 0; i < BS; ++i) x[i] = i == lane ? (T)1 : (T)0;
#pragma unroll
    for (int m = 0; m < BS - 1; ++m) {
        T l[BS];
        lds_read16<BS>(L + m * LS, l, E);
#pragma unroll
        for (int i = m + 1; i < BS; ++i) x[i] = fma(-l[i], x[m], x[i]);
    }
    bool big = false;
#pragma unroll
    for (int i = 0; i < BS; ++i) big |= !(x[i] <= (T)SW_GROWTH && x[i] >= (T)-SW_GROWTH);
    // any lane of this block's group
    const unsigned long long any = __ballot(big) >> ((threadIdx.x & 63) / BS * BS);
    if ((any & ((1ull << BS) - 1)) != 0) {
        // column `lane` of L instead
#pragma unroll
        for (int i = 0; i < BS; ++i) x[i] = L[lane * LS + i];
    }
    // each block's table, BS * BS entries at a time through LDS
    T* out = (J.buf ? tab1 : tab0) + stage * stage_stride + (J.tab + (int64_t)blockIdx.x * NB) * SweepGeom<T>::slot_a;
    const int nhere = min(NB, nblk - (int)blockIdx.x * NB);
    auto store = [&](int part) {
        for (int e = threadIdx.x * E; e < nhere * BS * BS; e += TAB_THREADS * E)
            *reinterpret_cast<uint4*>(out + (int64_t)(e / (BS * BS)) * SweepGeom<T>::slot_a + part * BS * BS +
                                      e % (BS * BS)) = *reinterpret_cast<const uint4*>(lb + e);
    };
    __syncthreads();
#pragma unroll
    for (int i = 0; i < BS; ++i) lb[grp * BS * BS + CM::tab_pos(i, lane)] = x[i];
    __syncthreads();
    store(0);
    __syncthreads();
#pragma unroll
    for (int m = 0; m < BS; ++m) lb[grp * BS * BS + CM::sub_pos(lane, m)] = sub[m];
    __syncthreads();
    store(1);
    if (nb > 0) {
        T* d = out + (int64_t)grp * SweepGeom<T>::slot_a + 2 * BS * BS;
        for (int e = lane; e < 256 / (int)sizeof(T); e += BS) d[e] = e < BS ? piv : (T)0;
    }
}

inline int ring_size(int k)
{
    int r = 1;
    while (r < 2 * NBS + k) r <<= 1;
    return r;
}

template <class T>
__device__ inline T* lds_ring()
{
    extern __shared__ unsigned char smem_raw[];
    return reinterpret_cast<T*>(smem_raw);
}

// elements kept for the corrections (whole 16-byte chunks)
__host__ __device__ inline int sweep_corr_elems(int k) { return (k + 3) / 4 * 4; }

// dynamic LDS of the staged sweep: two pending rings, the corrections, the
// right-hand side staging, the slots of the rings
template <class T>
__device__ inline SweepLds<T> sweep_lds_of(T* pend, int ring_mask, int k, int nbuf)
{
    const SweepGeom<T> G(k);
    SweepLds<T> S;
    S.pend0 = pend;
    S.pend1 = pend + ring_mask + 1;
    S.corr = S.pend1 + ring_mask + 1;
    S.stage = reinterpret_cast<unsigned*>(S.corr + sweep_corr_elems(k));
    S.na = nbuf & 255;
    S.nb = nbuf >> 8;
    S.a = reinterpret_cast<T*>(S.stage + SW_NIN * 64);
    S.b = S.a + S.na * G.slot_a;
    S.ring_mask = ring_mask;
    return S;
}

// first element of the tables of partition p, whose first row is s
template <class T>
__device__ inline int64_t sweep_tab_pos(int64_t s, int p)
{
    return (s / sweep_bs<T>() + p) * SweepGeom<T>::slot_a;
}

// Several right-hand sides: workgroup -> (job, right-hand side) for nj jobs
// and nr right-hand sides.  The nr workgroups of one job get ids that are
// equal mod 8, and workgroup ids are dealt to the 8 XCDs round-robin, so the
// sweeps of one partition for all right-hand sides run on one XCD and read
// its factors through that XCD's L2.  With nr = 1 the job is blockIdx.x.
// Grid: ceil(nj / 8) * 8 * nr workgroups; false for the padding ones.
__device__ inline bool job_and_rhs(int nj, int nr, int& job, int& r)
{
    const int b = blockIdx.x;
    const int q = b >> 3;
    r = q % nr;
    job = (q / nr) * 8 + (b & 7);
    return job < nj;
}

inline unsigned job_rhs_grid(int nj, int nr) { return (unsigned)(((nj + 7) / 8) * 8 * nr); }

// ---------------------------------------------------------------------------
// pass 1 (LU_UL): blockIdx.x = 2*i + side, i = boundary.
//   side 0: partition i, LU factors (B), bottom k rows of A_i^{-1} v_i
//   side 1: partition i+1, UL factors (Bul), top k rows of A_{i+1}^{-1} v_{i+1}
// g receives those 2k values per boundary at their row positions;
// scr is a length-n scratch vector per side.
// ---------------------------------------------------------------------------
// MODE: 0 simple blocked sweep, 2 LDS-staged (SW_THREADS threads; nbuf =
// slots of ring A + 256 * slots of ring B).
template <class T, int MODE>
__global__ __launch_bounds__(MODE == 2 ? SW_THREADS : 256) void sweep_interface_kernel(
    const T* __restrict__ B, const T* __restrict__ Bul, SweepTabs<T> tabs, int k, PartInfo pi,
    const double* __restrict__ v, T* __restrict__ g, T* __restrict__ scr0, T* __restrict__ scr1, int ring_mask, int nbuf, int nr, int64_t ldv,
    const int* __restrict__ gate)
{
    T* pend = lds_ring<T>();
    __shared__ T xblk[NBS];
    __shared__ alignas(16) T xblk2[2 * NBS];
    int job, rh;
    if (!job_and_rhs(2 * (pi.P - 1), nr, job, rh)) return;
    if (gate && !gate[rh]) return;
    v += rh * ldv;
    g += rh * pi.n;
    scr0 += rh * pi.n;
    scr1 += rh * pi.n;
    const int i = job >> 1;
    const int side = job & 1;
    const int p = i + side;
    int64_t s, len;
    pi.bounds(p, s, len);
    const T* F = side == 0 ? B : Bul;
    T* scr = side == 0 ? scr0 : scr1;
    const int d1 = side == 0 ? 1 : -1;       // stage-1 direction
    // local row r of a view with direction d -> global row
    auto grow = [&](int d, int64_t r) -> int64_t { return d > 0 ? s + r : s + len - 1 - r; };

    const int64_t kl = min((int64_t)k, len);
    if constexpr (MODE == 2) {
        const int64_t tp = sweep_tab_pos<T>(s, p);
        const SweepLds<T> S = sweep_lds_of<T>(pend, ring_mask, k, nbuf);
#pragma nounroll
        for (int stage = 0; stage < 2; ++stage) {
            const int d = stage ? -d1 : d1;
            const T* tab = (side == 0 ? (stage ? tabs.lu2 : tabs.lu1) : (stage ? tabs.ul2 : tabs.ul1)) + tp;
            T* to = stage ? g : scr;
            const SweepSrc<T> src{stage ? (const void*)scr : v, stage == 0, grow(d, 0), d, nullptr, nullptr, 1};
            const SweepDst dst{to, sizeof(T) == 8, grow(d, 0), d};
            lower_sweep_lds<T>(make_view(F, s, len, k, d), tab, stage ? kl : len, src, dst, stage == 0, S, xblk2);
            __syncthreads();
        }
    } else {
        const BandView<T> V1 = make_view(F, s, len, k, d1);
        const BandView<T> V2 = make_view(F, s, len, k, -d1);
        auto in1 = [&](int64_t r) -> T { return (T)v[grow(d1, r)]; };
        auto in2 = [&](int64_t r) -> T { return scr[grow(-d1, r)]; };
        auto out2 = [&](int64_t r, T y) { g[grow(-d1, r)] = y; };
        lower_sweep<T>(V1, len, in1, [&](int64_t r, T y) { scr[grow(d1, r)] = y / V1.at(r, r); }, pend, ring_mask,
                       xblk);
        __syncthreads();
        lower_sweep<T>(V2, kl, in2, out2, pend, ring_mask, xblk);
    }
}

// ---------------------------------------------------------------------------
// pass 2: blockIdx.x = partition.  out = A_p^{-1} (v - corr) with the LU
// factors (stage 1 forward L with D^{-1}, stage 2 backward U'), or for the
// UL-factored last partition the mirror order.  corr (2k per boundary) may
// be null.  Output FP64 (outd) or preconditioner precision (outt).
// ---------------------------------------------------------------------------
// The full sweep of partition p for one right-hand side (pointers already
// at that column), shared by the per-system and the job-table kernels.
template <class T, int MODE>
__device__ __forceinline__ void sweep_full_body(const T* __restrict__ B, const T* __restrict__ Bul,
                                                const SweepTabs<T>& tabs, int k, PartInfo pi, int last_is_ul,
                                                int p, const double* __restrict__ v, const T* __restrict__ corr, double* __restrict__ outd,
                                                T* __restrict__ outt, T* __restrict__ scr, int ring_mask, int nbuf,
                                                T* pend, T* xblk, T* xblk2, int half = -1,
                                                int64_t s_ovr = 0, int64_t len_ovr = 0)
{
    // len_ovr > 0: the rows [s_ovr, s_ovr + len_ovr) of the band instead of
    // partition p (a block of a partition; tabs then point at its own blocks)
    int64_t s, len, tp = 0;
    if (len_ovr > 0) { s = s_ovr; len = len_ovr; }
    else { pi.bounds(p, s, len); tp = sweep_tab_pos<T>(s, p); }
    // half 0: rows [s + len/2, s + len) from the LU factors (stage 2 from
    // the bottom up to the middle); half 1: rows [s, s + len/2) from the UL
    // factors (stage 2 from the top down to the middle); -1: all rows
    const bool ul = half >= 0 ? half == 1 : (last_is_ul && p == pi.P - 1);
    const int64_t mid = len / 2;
    const int64_t len2 = half < 0 ? len : (half == 1 ? mid : len - mid);
    const T* F = ul ? Bul : B;
    const int d1 = ul ? -1 : 1;
    auto grow = [&](int d, int64_t r) -> int64_t { return d > 0 ? s + r : s + len - 1 - r; };
    const bool has_top = corr && p > 0;
    const bool has_bot = corr && p < pi.P - 1;
    if constexpr (MODE == 2) {
        const T* t1 = ul ? tabs.ul1 : tabs.lu1;
        const T* t2 = ul ? tabs.ul2 : tabs.lu2;
        const SweepLds<T> S = sweep_lds_of<T>(pend, ring_mask, k, nbuf);
#pragma nounroll
        for (int stage = 0; stage < 2; ++stage) {
            const int d = stage ? -d1 : d1;
            const T* tab = (stage ? t2 : t1) + tp;
            // stage 1 right-hand side: v minus the corrections of the
            // partition's first and last k rows
            SweepSrc<T> src{stage ? (const void*)scr : v, stage == 0, grow(d, 0), d, nullptr, nullptr, d};
            if (stage == 0) {
                const T* top = has_top ? corr + (size_t)(p - 1) * 2 * k + k : nullptr;
                const T* bot = has_bot ? corr + (size_t)p * 2 * k : nullptr;
                src.first = d > 0 ? top : bot ? bot + k - 1 : nullptr;
                src.last = d > 0 ? bot : top ? top + k - 1 : nullptr;
            }
            const bool wide = stage == 1 && outd;   // FP64 results
            const SweepDst dst{stage == 0 ? (void*)scr : outd ? (void*)outd : (void*)outt, wide || sizeof(T) == 8,
                               grow(d, 0), d};
            lower_sweep_lds<T>(make_view(F, s, len, k, d), tab, stage ? len2 : len, src, dst, stage == 0, S, xblk2);
            __syncthreads();
        }
    } else {
        const BandView<T> V1 = make_view(F, s, len, k, d1);
        const BandView<T> V2 = make_view(F, s, len, k, -d1);
        auto rhs = [&](int64_t r) -> T {
            const int64_t gr = grow(d1, r);
            T val = (T)v[gr];
            const int64_t lr = gr - s;
            if (has_top && lr < k) val -= corr[(size_t)(p - 1) * 2 * k + k + lr];
            if (has_bot && lr >= len - k) val -= corr[(size_t)p * 2 * k + (lr - (len - k))];
            return val;
        };
        auto in2 = [&](int64_t r) -> T { return scr[grow(-d1, r)]; };
        lower_sweep<T>(V1, len, rhs, [&](int64_t r, T y) { scr[grow(d1, r)] = y / V1.at(r, r); }, pend, ring_mask,
                       xblk);
        __syncthreads();
        if (outd)
            lower_sweep<T>(V2, len2, in2, [&](int64_t r, T y) { outd[grow(-d1, r)] = (double)y; }, pend, ring_mask,
                           xblk);
        else
            lower_sweep<T>(V2, len2, in2, [&](int64_t r, T y) { outt[grow(-d1, r)] = y; }, pend, ring_mask, xblk);
    }
}

template <class T, int MODE>
__global__ __launch_bounds__(MODE == 2 ? SW_THREADS : 256) void sweep_full_kernel(
    const T* __restrict__ B, const T* __restrict__ Bul, SweepTabs<T> tabs, int k, PartInfo pi, int last_is_ul,
    const double* __restrict__ v, const T* __restrict__ corr, double* __restrict__ outd, T* __restrict__ outt,
    T* __restrict__ scr, int ring_mask, int nbuf, int nr, int64_t ldv, int64_t ldo, const int* __restrict__ gate,
    int split, T* __restrict__ scr_alt)
{
    T* pend = lds_ring<T>();
    __shared__ T xblk[NBS];
    __shared__ alignas(16) T xblk2[2 * NBS];
    // split: two workgroups per partition, the bottom half of its rows from
    // the LU factors and the top half from the UL factors (scratch scr_alt)
    int job, rh;
    if (!job_and_rhs(split ? 2 * pi.P : pi.P, nr, job, rh)) return;
    if (gate && !gate[rh]) return;
    const int p = split ? job >> 1 : job;
    const int half = split ? (job & 1) : -1;
    v += rh * ldv;
    if (corr) corr += rh * (int64_t)2 * k * (pi.P - 1);
    if (outd) outd += rh * ldo;
    if (outt) outt += rh * pi.n;
    T* sc = (half == 1 ? scr_alt : scr) + rh * pi.n;
    sweep_full_body<T, MODE>(B, Bul, tabs, k, pi, last_is_ul, p, v, corr, outd, outt, sc, ring_mask, nbuf, pend, xblk,
                             xblk2, half);
}

// Full sweeps of several systems in one launch: workgroup b takes job b of
// a table (one partition of one system for one right-hand side; null B:
// padding), with that system's band, width, staging depth and LDS ring;
// the input column is V + voff and the output Z + ooff.
template <class T, int MODE>
__global__ __launch_bounds__(MODE == 2 ? SW_THREADS : 256) void sweep_full_jobs_kernel(
    const SweepJob* __restrict__ jobs, const double* __restrict__ V, double* __restrict__ Z,
    const int* __restrict__ gate)
{
    T* pend = lds_ring<T>();
    __shared__ T xblk[NBS];
    __shared__ alignas(16) T xblk2[2 * NBS];
    const SweepJob J = jobs[blockIdx.x];
    if (!J.B) return;
    if (gate && !gate[J.gate]) return;
    const PartInfo pi{J.n, J.P};
    const SweepTabs<T> tabs{(const T*)J.t1, (const T*)J.t2, (const T*)J.t1, (const T*)J.t2};
    sweep_full_body<T, MODE>((const T*)J.B, (const T*)J.B, tabs, J.k, pi, 0, J.part, V + J.voff, nullptr, Z + J.ooff, nullptr, (T*)J.scr, J.ring_mask, J.nbuf, pend, xblk, xblk2,
                          -1, J.s0, J.len0);
}

// ---------------------------------------------------------------------------
// Reduced solve and purification per boundary i (one workgroup):
//   zt' = g_t - W g_b ;  x_t = S^{-1} zt' ;  x_b = g_b - V x_t
//   corr_b = B_i x_t (rows e0-k..e0-1),  corr_t = C_{i+1} x_b (rows s1..s1+k-1)
// All k x k matrices column-major.
// ---------------------------------------------------------------------------
template <class T>
__device__ void gemv_cm(const T* __restrict__ M, int k, const T* x, T* y, T beta_src_sign, const T* src)
{
    // y[a] = src[a] + sign * sum_b M(a, b) x[b]   (src may be null -> 0)
    for (int a = threadIdx.x; a < k; a += blockDim.x) {
        T acc = (T)0;
        for (int b = 0; b < k; ++b) acc += M[(size_t)b * k + a] * x[b];
        y[a] = (src ? src[a] : (T)0) + beta_src_sign * acc;
    }
}

// The same with 1024 threads: thread (a mod 256, q) sums columns
// [q k / 4, (q + 1) k / 4) in order, and the four partial sums are added as
// (p0 + p1) + (p2 + p3) through part[4][256] in LDS, so each output row
// has four times the loads in flight.  Ends with a barrier (y is complete).
template <class T>
__device__ void gemv_cm4(const T* __restrict__ M, int k, const T* x, T* y, T beta_src_sign, const T* src, T* part)
{
    const int t = threadIdx.x & 255, q = threadIdx.x >> 8;
    const int b0 = (k * q) / 4, b1 = (k * (q + 1)) / 4;
    for (int a0 = 0; a0 < k; a0 += 256) {
        const int a = a0 + t;
        T acc = (T)0;
        if (a < k) {
            // eight loads issued together, then added in column order
            int b = b0;
            for (; b + 8 <= b1; b += 8) {
                T m[8];
#pragma unroll
                for (int u = 0; u < 8; ++u) m[u] = M[(size_t)(b + u) * k + a];
#pragma unroll
                for (int u = 0; u < 8; ++u) acc += m[u] * x[b + u];
            }
            for (; b < b1; ++b) acc += M[(size_t)b * k + a] * x[b];
        }
        part[q * 256 + t] = acc;
        __syncthreads();
        if (q == 0 && a < k)
            y[a] = (src ? src[a] : (T)0) + beta_src_sign * ((part[t] + part[256 + t]) + (part[512 + t] + part[768 + t]));
        __syncthreads();
    }
}

template <class T>
__global__ __launch_bounds__(256) void interface_kernel(const T* __restrict__ WV, const T* __restrict__ Sinv,
                                                        const T* __restrict__ offB, const T* __restrict__ offC, int k,
                                                        PartInfo pi, const T* __restrict__ g, T* __restrict__ corr,
                                                        const int* __restrict__ gate)
{
    extern __shared__ unsigned char smem_raw[];
    T* gb = reinterpret_cast<T*>(smem_raw);
    T* gt = gb + k;
    T* zt = gt + k;
    T* xt = zt + k;
    T* xb = xt + k;
    const int i = blockIdx.x;
    if (gate && !gate[blockIdx.y]) return;
    g += blockIdx.y * pi.n;
    corr += blockIdx.y * (int64_t)2 * k * (pi.P - 1);
    int64_t s1, l1;
    pi.bounds(i + 1, s1, l1);
    const size_t kk = (size_t)k * k;
    for (int a = threadIdx.x; a < k; a += blockDim.x) {
        gb[a] = g[s1 - k + a];
        gt[a] = g[s1 + a];
    }
    __syncthreads();
    gemv_cm<T>(WV + (2 * i + 1) * kk, k, gb, zt, (T)-1, gt);   // zt = gt - W gb
    __syncthreads();
    gemv_cm<T>(Sinv + i * kk, k, zt, xt, (T)1, nullptr);        // xt = S^{-1} zt
    __syncthreads();
    gemv_cm<T>(WV + 2 * i * kk, k, xt, xb, (T)-1, gb);          // xb = gb - V xt
    __syncthreads();
    T* c = corr + (size_t)i * 2 * k;
    gemv_cm<T>(offB + i * kk, k, xt, c, (T)1, nullptr);         // B_i xt
    gemv_cm<T>(offC + i * kk, k, xb, c + k, (T)1, nullptr);     // C_{i+1} xb
}

// interface_kernel with 1024 threads and gemv_cm4
template <class T>
__global__ __launch_bounds__(1024) void interface4_kernel(const T* __restrict__ WV, const T* __restrict__ Sinv,
                                                          const T* __restrict__ offB, const T* __restrict__ offC,
                                                          int k, PartInfo pi, const T* __restrict__ g,
                                                          T* __restrict__ corr, const int* __restrict__ gate)
{
    extern __shared__ unsigned char smem_raw[];
    T* part = reinterpret_cast<T*>(smem_raw);
    T* gb = part + 1024;
    T* gt = gb + k;
    T* zt = gt + k;
    T* xt = zt + k;
    T* xb = xt + k;
    const int i = blockIdx.x;
    if (gate && !gate[blockIdx.y]) return;
    g += blockIdx.y * pi.n;
    corr += blockIdx.y * (int64_t)2 * k * (pi.P - 1);
    int64_t s1, l1;
    pi.bounds(i + 1, s1, l1);
    const size_t kk = (size_t)k * k;
    for (int a = threadIdx.x; a < k; a += blockDim.x) {
        gb[a] = g[s1 - k + a];
        gt[a] = g[s1 + a];
    }
    __syncthreads();
    gemv_cm4<T>(WV + (2 * i + 1) * kk, k, gb, zt, (T)-1, gt, part);   // zt = gt - W gb
    gemv_cm4<T>(Sinv + i * kk, k, zt, xt, (T)1, nullptr, part);        // xt = S^{-1} zt
    gemv_cm4<T>(WV + 2 * i * kk, k, xt, xb, (T)-1, gb, part);          // xb = gb - V xt
    T* c = corr + (size_t)i * 2 * k;
    gemv_cm4<T>(offB + i * kk, k, xt, c, (T)1, nullptr, part);         // B_i xt
    gemv_cm4<T>(offC + i * kk, k, xb, c + k, (T)1, nullptr, part);     // C_{i+1} xb
}

template <class T>
__global__ void diag_divide_kernel(const T* __restrict__ B, int64_t n, const double* __restrict__ v,
                                   double* __restrict__ out, int64_t ldv, int64_t ldo, const int* __restrict__ gate)
{
    if (gate && !gate[blockIdx.y]) return;
    v += blockIdx.y * ldv;
    out += blockIdx.y * ldo;
    const int64_t stride = (int64_t)gridDim.x * blockDim.x;
    for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = (double)((T)v[i] / B[i]);
}

template <class T>
size_t sweep_lds(int k)
{
    return sizeof(T) * (size_t)ring_size(k);
}

}  // namespace

// Sweep configuration: mode and (mode 2) slots of the rings (nbuf as the
// kernels take it, depth the slots of the deeper one), as many as fit next to
// the pending rings (at most 8: the loads a producer may have outstanding).
struct SweepCfg { int mode, nbuf; size_t lds; int threads, depth; };

// tabs_ok: the factorization's T blocks exist; depth_req: at most so many
// slots (0: as many as fit).  As many as fit also where there are more
// workgroups than CUs (several columns, job tables): three wavefronts of 121
// to 126 registers per SIMD leave no CU room for a second workgroup, whatever
// its LDS.  One sweep of 16 partitions, 16 columns with at most four slots and
// with all: 271 and 149 us at k = 50 (n = 200000, FP32), 152 and 152 at k = 80,
// 188 and 151 at k = 20 (n = 100000, FP64), 171 and 175 at k = 150.
template <class T>
SweepCfg sweep_cfg(int k, bool tabs_ok, int depth_req = 0)
{
    constexpr size_t LDS_MAX = 160 * 1024 - 4096;   // static LDS of the kernels + margin
    const size_t ring = sweep_lds<T>(k);
    if (!tabs_ok || k > sweep_staged_max<T>()) return {0, 0, ring, 256, 0};
    const SweepGeom<T> G(k);
    const size_t sa = G.slot_a * sizeof(T), sb = (size_t)G.slot_b() * sizeof(T);
    const size_t fixed = 2 * ring + sweep_corr_elems(k) * sizeof(T) + SW_NIN * 64 * 4;
    const int want = depth_req >= 4 ? std::min(depth_req, 8) : 8;
    // ring A holds the block in use and those on their way; ring B also the
    // one before.  Wide bands: ring B with three or two slots (with two, the
    // far rows' loads complete within the step that issues them, still far
    // faster than the plain blocked sweep).
    int na = 3, nb = 4;
    while (nb > 2 && fixed + na * sa + nb * sb > LDS_MAX) --nb;
    if (fixed + na * sa + nb * sb > LDS_MAX) return {0, 0, ring, 256, 0};
    if (nb == 4) {
        if (fixed + (na + 1) * sa + nb * sb <= LDS_MAX) ++na;
        while (na == nb && na < want && fixed + (na + 1) * (sa + sb) <= LDS_MAX) { ++na; ++nb; }
    }
    return {2, na + 256 * nb, fixed + na * sa + nb * sb, SW_THREADS, nb};
}

template <class T, int MODE>
void launch_sweep_interface_t(const T* B, const T* Bul, const SweepTabs<T>& tabs, int k, PartInfo pi, const double* v, T* g, T* scr0, T* scr1,
                              const SweepCfg& c, const Rhs& rh, hipStream_t st)
{
    set_lds_limit((const void*)sweep_interface_kernel<T, MODE>, c.lds);
    hipLaunchKernelGGL((sweep_interface_kernel<T, MODE>), dim3(job_rhs_grid(2 * (pi.P - 1), rh.nr)), dim3(c.threads),
                       c.lds, st, B, Bul, tabs, k, pi, v, g, scr0, scr1, ring_size(k) - 1, c.nbuf, rh.nr, rh.ldv, rh.gate);
    SAP_LAUNCH_CHECK();
}

template <class T>
void launch_sweep_interface(const T* B, const T* Bul, const SweepTabs<T>& tabs, int k, PartInfo pi, const double* v,
                            T* g, T* scr0, T* scr1, hipStream_t st, const Rhs& rh)
{
    if (pi.P < 2) return;
    const SweepCfg c = sweep_cfg<T>(k, tabs.lu1 != nullptr, rh.nbuf);
    if (c.mode == 2) launch_sweep_interface_t<T, 2>(B, Bul, tabs, k, pi, v, g, scr0, scr1, c, rh, st);
    else launch_sweep_interface_t<T, 0>(B, Bul, tabs, k, pi, v, g, scr0, scr1, c, rh, st);
}

template <class T>
void launch_interface_solve(const T* WV, const T* Sinv, const T* offB, const T* offC, int k, PartInfo pi, const T* g,
                            T* corr, hipStream_t st, const Rhs& rh)
{
    if (pi.P < 2) return;
    const size_t lds4 = sizeof(T) * (1024 + 5 * (size_t)k);
    if (lds4 <= 64 * 1024) {
        hipLaunchKernelGGL(interface4_kernel<T>, dim3(pi.P - 1, rh.nr), dim3(1024), lds4, st, WV, Sinv, offB, offC, k,
                           pi, g, corr, rh.gate);
    } else {
        const size_t lds = sizeof(T) * 5 * (size_t)k;
        hipLaunchKernelGGL(interface_kernel<T>, dim3(pi.P - 1, rh.nr), dim3(256), lds, st, WV, Sinv, offB, offC, k,
                           pi, g, corr, rh.gate);
    }
    SAP_LAUNCH_CHECK();
}

template <class T, int MODE>
void launch_sweep_full_t(const T* B, const T* Bul, const SweepTabs<T>& tabs, int k, PartInfo pi, int last_is_ul,
                         const double* v, const T* corr, double* outd, T* outt, T* scr, const SweepCfg& c,
                         const Rhs& rh, hipStream_t st)
{
    set_lds_limit((const void*)sweep_full_kernel<T, MODE>, c.lds);
    const int split = rh.split_scr != nullptr;
    hipLaunchKernelGGL((sweep_full_kernel<T, MODE>), dim3(job_rhs_grid(split ? 2 * pi.P : pi.P, rh.nr)),
                       dim3(c.threads), c.lds, st, B, Bul, tabs, k, pi, last_is_ul, v, corr, outd, outt, scr,
                       ring_size(k) - 1, c.nbuf, rh.nr, rh.ldv, rh.ldo, rh.gate, split, (T*)rh.split_scr);
    SAP_LAUNCH_CHECK();
}

template <class T>
void launch_sweep_full(const T* B, const T* Bul, const SweepTabs<T>& tabs, int k, PartInfo pi, int last_is_ul,
                       const double* v, const T* corr, double* outd, T* outt, T* scr, hipStream_t st, const Rhs& rh)
{
    const SweepCfg c = sweep_cfg<T>(k, tabs.lu1 != nullptr, rh.nbuf);
    if (c.mode == 2) launch_sweep_full_t<T, 2>(B, Bul, tabs, k, pi, last_is_ul, v, corr, outd, outt, scr, c, rh, st);
    else launch_sweep_full_t<T, 0>(B, Bul, tabs, k, pi, last_is_ul, v, corr, outd, outt, scr, c, rh, st);
}

template <class T>
void launch_diag_divide(const T* B, int64_t n, const double* v, double* out, hipStream_t st, const Rhs& rh)
{
    int64_t g = (n + 255) / 256;
    if (g > 8192) g = 8192;
    hipLaunchKernelGGL(diag_divide_kernel<T>, dim3((unsigned)g, rh.nr), dim3(256), 0, st, B, n, v, out, rh.ldv,
                       rh.ldo, rh.gate);
    SAP_LAUNCH_CHECK();
}

template <class T>
bool sweep_jobs_append(std::vector<SweepJob>& jobs, size_t& lds, const T* B, const SweepTabs<T>& tabs, int k,
                       PartInfo pi, T* scr, int64_t voff, int64_t ldv, int64_t ooff, int64_t ldo, int nr, int gate0,
                       int* mode_out)
{
    const SweepCfg c = sweep_cfg<T>(k, tabs.lu1 != nullptr);
    if (k == 0) return false;
    if (mode_out) *mode_out = c.mode;
    else if (c.mode != 2) return false;
    lds = std::max(lds, c.lds);
    // the kernel's (job, right-hand side) order per system: the nr
    // workgroups of a partition 8 ids apart (one XCD), padded to whole
    // groups of 8 partitions
    const int groups = (pi.P + 7) / 8;
    for (int q = 0; q < groups * 8 * nr; ++q) {
        const int r = (q >> 3) % nr;
        const int part = ((q >> 3) / nr) * 8 + (q & 7);
        SweepJob J{};
        if (part < pi.P) {
            J.B = B;
            J.t1 = tabs.lu1;
            J.t2 = tabs.lu2;
            J.scr = scr + (int64_t)r * pi.n;
            J.voff = voff + r * ldv;
            J.ooff = ooff + r * ldo;
            J.n = pi.n;
            J.P = pi.P;
            J.k = k;
            J.part = part;
            J.gate = gate0 + r;
            J.ring_mask = ring_size(k) - 1;
            J.nbuf = c.nbuf;
        }
        jobs.push_back(J);
    }
    return true;
}

template <class T>
int sweep_range_job_append(std::vector<SweepJob>& jobs, size_t& lds, const T* B, const SweepTabs<T>& tabs, int k,
                           int64_t s0, int64_t len0, T* scr, int64_t n, int64_t ldv, int64_t ldo, int nr)
{
    const SweepCfg c = sweep_cfg<T>(k, tabs.lu1 != nullptr);
    lds = std::max(lds, c.lds);
    for (int r = 0; r < nr; ++r) {
        SweepJob J{};
        J.B = B;
        J.t1 = tabs.lu1;
        J.t2 = tabs.lu2;
        J.scr = scr + (int64_t)r * n;
        J.voff = r * ldv;
        J.ooff = r * ldo;
        J.n = n;
        J.P = 1;
        J.k = k;
        J.part = 0;
        J.gate = r;
        J.ring_mask = ring_size(k) - 1;
        J.nbuf = c.nbuf;
        J.s0 = s0;
        J.len0 = len0;
        jobs.push_back(J);
    }
    return c.mode;
}

template <class T, int MODE>
void launch_sweep_full_jobs_t(const SweepJob* d_jobs, int njobs, size_t lds, const double* V, double* Z,
                              const int* gate, hipStream_t st)
{
    set_lds_limit((const void*)sweep_full_jobs_kernel<T, MODE>, lds);
    hipLaunchKernelGGL((sweep_full_jobs_kernel<T, MODE>), dim3(njobs), dim3(MODE == 2 ? SW_THREADS : 256), lds, st,
                       d_jobs, V, Z, gate);
    SAP_LAUNCH_CHECK();
}

template <class T>
void launch_sweep_full_jobs(const SweepJob* d_jobs, int njobs, size_t lds, const double* V, double* Z,
                            const int* gate, hipStream_t st, int mode)
{
    if (njobs <= 0) return;
    if (mode == 2) launch_sweep_full_jobs_t<T, 2>(d_jobs, njobs, lds, V, Z, gate, st);
    else launch_sweep_full_jobs_t<T, 0>(d_jobs, njobs, lds, V, Z, gate, st);
}

template <class T>
int sweep_max_nbuf(int k)
{
    const SweepCfg c = sweep_cfg<T>(k, true);
    return c.mode == 2 ? c.depth : 0;
}

template <class T>
int64_t sweep_tab_elems(int64_t n, int ranges)
{
    return (n / sweep_bs<T>() + ranges) * SweepGeom<T>::slot_a;
}

template <class T>
int64_t sweep_tab_block(int64_t start, int range)
{
    return start / sweep_bs<T>() + range;
}

template <class T>
void launch_sweep_tables(const T* B0, const T* B1, int k, const FactorJob* d_jobs, int njobs, int64_t max_len, T* tab0,
                         T* tab1, int64_t stage_stride, hipStream_t st)
{
    if (njobs <= 0) return;
    const int nb = TAB_THREADS / sweep_bs<T>();
    const int64_t nblk = (max_len + sweep_bs<T>() - 1) / sweep_bs<T>();
    hipLaunchKernelGGL(sweep_tables_kernel<T>, dim3((unsigned)((nblk + nb - 1) / nb), njobs, 2), dim3(TAB_THREADS), 0,
                       st, B0, B1, k, d_jobs, tab0, tab1, stage_stride);
    SAP_LAUNCH_CHECK();
}

#define SAP_INST(T)                                                                                               \
    template int sweep_max_nbuf<T>(int);                                                                           \
    template int64_t sweep_tab_elems<T>(int64_t, int);                                                             \
    template int64_t sweep_tab_block<T>(int64_t, int);                                                             \
    template void launch_sweep_tables<T>(const T*, const T*, int, const FactorJob*, int, int64_t, T*, T*, int64_t, \
                                         hipStream_t);                                                             \
    template bool sweep_jobs_append<T>(std::vector<SweepJob>&, size_t&, const T*, const SweepTabs<T>&, int,        \
                                       PartInfo, T*, int64_t, int64_t, int64_t, int64_t, int, int, int*);           \
    template void launch_sweep_full_jobs<T>(const SweepJob*, int, size_t, const double*, double*, const int*,      \
                                            hipStream_t, int);                                                     \
    template int sweep_range_job_append<T>(std::vector<SweepJob>&, size_t&, const T*, const SweepTabs<T>&, int,    \
                                           int64_t, int64_t, T*, int64_t, int64_t, int64_t, int);                  \
    template void launch_sweep_interface<T>(const T*, const T*, const SweepTabs<T>&, int, PartInfo, const double*, \
                                            T*, T*, T*, hipStream_t, const Rhs&);                                  \
    template void launch_interface_solve<T>(const T*, const T*, const T*, const T*, int, PartInfo, const T*, T*,   \
                                            hipStream_t, const Rhs&);                                              \
    template void launch_sweep_full<T>(const T*, const T*, const SweepTabs<T>&, int, PartInfo, int, const double*, \
                                       const T*, double*, T*, T*, hipStream_t, const Rhs&);                        \
    template void launch_diag_divide<T>(const T*, int64_t, const double*, double*, hipStream_t, const Rhs&);
SAP_INST(float)
SAP_INST(double)
#undef SAP_INST

}  // namespace sap_amd
