// Blocked MFMA banded LU/UL of the partitions with the active window in global
// memory (L2): the bands wider than the register-resident kernel takes, up to
// k = 480 in FP32 and 224 in FP64, and partitions of any size.
#include "mfma.hpp"
#include "sap_internal.hpp"
#include "sub_panel.hpp"

#include <climits>

namespace sap_amd {

namespace {

// ---------------------------------------------------------------------------
// One workgroup per partition, 32-column panels, the window of panel p being
// rows and columns [32p, 32p + 16 KT) with KT = ceil((k + 32) / 16).  Band
// layout and directions as in the register-resident kernel.  Per panel:
//   A.  the panel's 32 columns and its 32 U rows go from the band to LDS, a
//       column and 64 rows (two columns and 32 rows) per load, all in flight
//       together;
//   B.  two sub-panels of 16 columns, as in the register-resident kernel, with
//       the multipliers corrected to what a division gives;
//   C.  the panel's factors go out, and the trailing tiles are read, updated on
//       the matrix cores and written back, two per wavefront at a time while
//       the next two are loading.
// What bounds it, FP64 at k = 150, of 62k cycles a panel with a clock read
// between the phases (57k without): A 14k (latency of the L2), B 23k (issue of
// the broadcast multiply-adds, two wavefronts on a SIMD), C 25k (the matrix
// cores need 13.2k of it).  The columns that enter next are read ahead from
// HBM during B (without: 6.8 ms instead of 5.9).  29 registers spill in FP32
// (128 for each of 16 wavefronts) and 28 in FP64 (256 for each of 8), 120 and
// 116 bytes of scratch a lane.  A thread per panel row with a barrier per
// column, as this was done before, took 13.4 ms for LU and UL (n = 250007, k =
// 150, 32 partitions, FP64); this takes 5.9.  FP32, n = 100000, 16 partitions:
// 13.1 -> 4.8 ms at k = 230, 25.9 -> 11.9 at k = 480.
// ---------------------------------------------------------------------------
template <class T>
struct WinGeom {
    static constexpr int NW = sizeof(T) == 4 ? 16 : 8;        // wavefronts
    static constexpr int KMAX = sizeof(T) == 4 ? 480 : 224;   // 16 + 16 (KT - 2) rows of L on half the threads
    static constexpr int PS = sizeof(T) == 4 ? 36 : 34;       // LDS row stride: 16-byte aligned rows, few bank conflicts
    static constexpr int HRMAX = (KMAX + 32 + 15) / 16 * 16;
    static size_t bytes(int k)
    {
        const int hr = (k + 32 + 15) / 16 * 16;
        return sizeof(T) * ((size_t)(2 * hr - 32) * PS + 64);
    }
};

template <class T>
__global__ __launch_bounds__(64 * WinGeom<T>::NW) void band_factor_window_kernel(T* __restrict__ B0, T* __restrict__ B1,
                                                                               int k_all,
                                                                               const FactorJob* __restrict__ jobs)
{
    using MF = Mfma16<T>;
    using acc_t = typename MF::acc_t;
    using WG = WinGeom<T>;
    constexpr int NW = WG::NW, PS = WG::PS, SZ = sizeof(T);
    constexpr int NG = (WG::HRMAX + 63) / 64, NCW = 32 / NW, NUW = (WG::HRMAX - 32 + 2 * NW - 1) / (2 * NW);
    constexpr int CS = sizeof(T) == 4 ? 1 : 4;   // columns between a lane's elements of a tile
    const FactorJob job = jobs[blockIdx.x];
    const int k = job.kb > 0 ? job.kb : k_all;
    T* __restrict__ base = (job.buf ? B1 : B0) + job.boff;
    const int w = 2 * k + 1, wm1 = 2 * k;
    const int64_t len = job.len;
    const int dir = job.dir;
    const int KT = (k + 32 + 15) / 16;

    extern __shared__ unsigned char smem_raw[];
    T* const Pn = reinterpret_cast<T*>(smem_raw);   // [HR][PS]: panel rows; after B rows >= 32 hold -L21
    T* const UbT = Pn + 16 * KT * PS;               // [NTR][PS]: U block, one column per row
    T* const pivs = UbT + 16 * (KT - 2) * PS;       // pivots [32]
    T* const rpiv = pivs + 32;                      // their reciprocals [32], 0 past the partition's end
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);

    for (int64_t j0 = 0; j0 < len; j0 += 32) {
        // re-materialised every panel: lane values and the many uniform
        // conditions on HR and NTR would otherwise be kept over the loop
        int tid = threadIdx.x, HR = 16 * KT;
        asm volatile("" : "+v"(tid), "+s"(HR));
        const int NTR = HR - 32, RW = (NTR + 16 + 63) / 64;   // RW: wavefronts of the L rows in B, and of the U columns
        const int lane = tid & 63, lr = lane & 15, lg = lane >> 4;
        const int rem = (int)min(len - j0, (int64_t)(1 << 30));   // partition rows left
        const int nb = min(32, rem);
        // The window's columns as one buffer: element (dr, dc) of the window is
        // at element offset ob + dir * (dc * 2k + dr); a column past the
        // partition's end is past the end of the buffer, reads zero there and
        // drops what is written.
        const int nc = min(rem, HR);
        const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
            (void*)(base + (dir > 0 ? job.start + j0 : job.start + len - j0 - nc) * w), 0, nc * w * SZ, 0x00020000);
        const int ob = dir > 0 ? k : nc * w - 1 - k;
        const int rl = dir > 0 ? lane : 63 - lane;
        const int half = lane >> 5, um = dir > 0 ? lane & 31 : 31 - (lane & 31);
        const int ctop = min(min(NTR, rem - 32), k);   // columns of the U block
        // byte offset of row 64 g + rl of panel column c, -1 off the band
        auto pn_off = [&](int c, int g) {
            const int lo = max(c - k, 0), top = c < nb ? min(min(HR, rem), c + k + 1) : lo;
            const bool in = (unsigned)(rl + 64 * g - lo) < (unsigned)(top - lo);
            return in ? (ob + dir * (c * wm1 + rl + 64 * g)) * SZ : -1;
        };
        // the same of row um of U column c0 + half
        auto ub_off = [&](int c0) {
            const int cc = c0 + half;
            const bool in = um < nb && cc < ctop && um >= 32 + cc - k;
            return in ? (ob + dir * ((32 + cc) * wm1 + um)) * SZ : -1;
        };

        // A. panel columns and U rows to LDS
        {
            T v[NCW][NG], u[NUW];
#pragma unroll
            for (int i = 0; i < NCW; ++i)
#pragma unroll
                for (int g = 0; g < NG; ++g)
                    if (64 * g < HR) v[i][g] = buffer_load<T>(rsrc, pn_off(wave + NW * i, g));
#pragma unroll
            for (int i = 0; i < NUW; ++i)
                if (2 * (wave + NW * i) < NTR) u[i] = buffer_load<T>(rsrc, ub_off(2 * (wave + NW * i)));
#pragma unroll
            for (int i = 0; i < NCW; ++i)
#pragma unroll
                for (int g = 0; g < NG; ++g)
                    if (64 * g < HR && 64 * g + rl < HR) Pn[(64 * g + rl) * PS + wave + NW * i] = v[i][g];
#pragma unroll
            for (int i = 0; i < NUW; ++i)
                if (2 * (wave + NW * i) < NTR) UbT[(2 * (wave + NW * i) + half) * PS + um] = u[i];
        }
        lds_barrier();

        // The 32 columns that enter the window with the next panel, read once
        // from HBM here so that its loads find them in the L2: one word of
        // every 128 bytes.
        constexpr int NPF = (32 * (2 * WG::KMAX + 1) * SZ + 128 * 64 * NW - 1) / (128 * 64 * NW);
        unsigned pf[NPF];
        {
            const int np = min(max(rem - HR, 0), 32);
            const __amdgpu_buffer_rsrc_t rp = __builtin_amdgcn_make_buffer_rsrc(
                (void*)(base + (dir > 0 ? job.start + j0 + (np ? HR : 0) : job.start + max(len - j0 - HR - np, (int64_t)0)) * w),
                0, np * w * SZ, 0x00020000);
#pragma unroll
            for (int i = 0; i < NPF; ++i)
                pf[i] = __builtin_amdgcn_raw_buffer_load_b32(rp, 128 * (tid + 64 * NW * i), 0, 0);
        }

        // B. the two sub-panels (columns O .. O + 15).  Threads 0 .. 15 + NTR - O
        //    hold rows 16 + O .. of the panel, threads 64 RW .. the columns
        //    16 + O .. (the first 16 of sub-panel 0 are the panel's own columns
        //    16 .. 31, in Pn; the rest UbT).
        const int boosted = job.boost ? (job.boost_last ? 32 : min(32, rem - 1)) : 0;
#pragma unroll 1
        for (int O = 0; O < 32; O += 16) {
            int c16 = lane & 15;
            asm volatile("" : "+v"(c16));
            T d[16], own[16], pr = (T)0;
            lds_get16(Pn + (O + c16) * PS + O, d);
            const bool urow = wave < RW;
            const int t = urow ? tid : tid - 64 * RW;      // row 16 + O + t, or column t
            const bool on = t < 16 + NTR - O;
            const bool incol = O == 0 && !urow && t < 16;  // a column of the panel itself
            T* const mine = urow ? Pn + (16 + O + t) * PS + O : UbT + (t - (16 - O)) * PS + O;
            if (incol) {
#pragma unroll
                for (int i = 0; i < 16; ++i) own[i] = Pn[i * PS + 16 + t];
            } else if (on) {
                lds_get16(mine, own);
            } else {
#pragma unroll
                for (int i = 0; i < 16; ++i) own[i] = (T)0;
            }
            lds_barrier();   // every copy of the diagonal block is read before it is overwritten
            const bool live = O + c16 < nb, plain = O + c16 >= boosted;
            if (nb < 32) {   // a unit pivot makes the steps past the partition's end exact no-ops
                int cd = live ? -1 : c16;
                asm volatile("" : "+v"(cd));
#pragma unroll
                for (int i = 0; i < 16; ++i) d[i] = i == cd ? (T)1 : d[i];
            }
            if (wave < 2 * RW) {
                const T r0 = sub_panel_pivot<0, T>(d, pr, c16, plain);
                if (urow) sub_panel_steps<0, true, true, T>(d, own, pr, r0, c16, plain);
                else sub_panel_steps<0, false, true, T>(d, own, pr, r0, c16, plain);
            }
            if (incol) {
#pragma unroll
                for (int i = 0; i < 16; ++i) Pn[i * PS + 16 + t] = own[i];
            } else if (on) {
                if (urow && 16 + O + t >= 32) {            // L21 is kept negated: the trailing update adds
#pragma unroll
                    for (int i = 0; i < 16; ++i) own[i] = -own[i];
                }
                lds_put16(mine, own);
            }
            if (tid < 16) {
                lds_put16(Pn + (O + tid) * PS + O, d);
                Pn[(O + tid) * PS + O + tid] = pr;
                pivs[O + tid] = pr;
                rpiv[O + tid] = live ? pivot_rcp(pr) : (T)0;
            }
            lds_barrier();
            if (O == 0) {
                // columns 16 .. 31 of the rows below (A = -L_a, B = rows 0 .. 15 of
                // U, columns 16 .. 31), and rows 16 .. 31 of the columns right
                // (A = -U_a^T, B = L_ba^T), 16 x 16 tiles
#pragma unroll 1
                for (int f = wave; f < 2 * KT - 3; f += NW) {
                    const bool lside = f < KT - 1;
                    T* const rows = lside ? Pn + (16 + 16 * f) * PS : UbT + 16 * (f - (KT - 1)) * PS;
                    const bool neg = f == 0 || !lside;   // operands not kept negated
                    T* const at = rows + MF::row(lane, 0) * PS + 16 + c16;
                    acc_t ac;
                    T av[4], bv[4];
#pragma unroll
                    for (int q = 0; q < 4; ++q) {
                        ac[q] = at[CS * q * PS];
                        const T x = rows[c16 * PS + 4 * q + lg];
                        av[q] = neg ? -x : x;
                        bv[q] = lside ? Pn[(4 * q + lg) * PS + 16 + c16] : Pn[(16 + c16) * PS + 4 * q + lg];
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q) ac = MF::mma(av[q], bv[q], ac);
#pragma unroll
                    for (int q = 0; q < 4; ++q) at[CS * q * PS] = ac[q];
                }
                lds_barrier();
            }
        }

#pragma unroll
        for (int i = 0; i < NPF; ++i) asm volatile("" :: "v"(pf[i]));   // the reads stay, and have long arrived

        // C. the panel's factors out: L, D and U' of its 32 columns (U' of the
        //    diagonal block divided by the row's pivot, L21 kept negated in
        //    LDS), and its U' rows
        {
            const T p0 = pivs[rl & 31], r0 = rpiv[rl & 31];
#pragma unroll 1
            for (int c = wave; c < nb; c += NW) {
#pragma unroll
                for (int g = 0; g < NG; ++g) {
                    if (64 * g >= HR) break;
                    const T x = Pn[min(64 * g + rl, HR - 1) * PS + c];
                    T v = -x;
                    if (g == 0) v = rl >= 32 ? -x : (rl < c ? quotient(x * r0, x, p0, r0) : x);
                    buffer_store<T>(v, rsrc, pn_off(c, g));
                }
            }
            const T pu = pivs[um], ru = rpiv[um];
#pragma unroll 2
            for (int c0 = 2 * wave; c0 < ctop; c0 += 2 * NW) {
                const T x = UbT[(c0 + half) * PS + um];
                buffer_store<T>(quotient(x * ru, x, pu, ru), rsrc, ub_off(c0));
            }
        }
        // and the trailing tiles, held transposed: register q of lane l is
        // window element (dr0 + l % 16, dc0 + row(l, q)); acc^T += U12^T (-L21)^T
        const int nt = rem > 32 ? min(KT - 2, (rem - 32 + 15) / 16) : 0, ne = nt * nt;
        const int inv = nt ? (65536 + nt - 1) / nt : 0;   // e / nt = e * inv >> 16: exact while e (nt - 1) < 65536
        const int e0 = lr - MF::row(lane, 0);
        const int so_rev = dir < 0 ? (15 * wm1 + 15) * SZ : 0, cstep = dir * CS * wm1 * SZ;
        const int lp0 = so_rev + dir * (MF::row(lane, 0) * wm1 + lr) * SZ;   // from the tile's lowest address
        int lp[4];
#pragma unroll
        for (int q = 0; q < 4; ++q) lp[q] = lp0 + q * cstep;
        // tile e: its place, the byte offset of its lowest address and whether
        // it is inside the band and the partition (no masks)
        struct Tile { int dr0, dc0, so; bool inside; };
        auto tile = [&](int e) {
            Tile t;
            const int rn = (e * inv) >> 16, cn = e - rn * nt;
            t.dr0 = 32 + 16 * rn;
            t.dc0 = 32 + 16 * cn;
            t.so = (ob + dir * (t.dc0 * wm1 + t.dr0)) * SZ - so_rev;
            t.inside = 16 * max(rn - cn, cn - rn) + 15 <= k && max(t.dr0, t.dc0) + 16 <= rem;
            return t;
        };
        auto tile_off = [&](const Tile& t, int q) {
            const int x = lr < rem - t.dr0 ? e0 + t.dr0 - t.dc0 + k : INT_MIN;
            return (unsigned)(x - CS * q) <= (unsigned)wm1 ? lp[q] + t.so : -1;
        };
        auto fetch = [&](int e, acc_t (&a)[2]) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (e + NW * i >= ne) return;
                const Tile t = tile(e + NW * i);
                if (t.inside) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) a[i][q] = buffer_load<T>(rsrc, lp[q], t.so);
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q) a[i][q] = buffer_load<T>(rsrc, tile_off(t, q));
                }
            }
        };
        auto update = [&](int e, acc_t (&a)[2]) {
#pragma unroll
            for (int i = 0; i < 2; ++i) {
                if (e + NW * i >= ne) return;
                const Tile t = tile(e + NW * i);
                const T* const ap = Pn + (t.dr0 + lr) * PS + 8 * lg;
                const T* const bp = UbT + (t.dc0 - 32 + lr) * PS + 8 * lg;
                T a0[4], b0[4], a1[4], b1[4];
                lds_get4(ap, a0); lds_get4(bp, b0); lds_get4(ap + 4, a1); lds_get4(bp + 4, b1);
#pragma unroll
                for (int q = 0; q < 4; ++q) a[i] = MF::mma(b0[q], a0[q], a[i]);
#pragma unroll
                for (int q = 0; q < 4; ++q) a[i] = MF::mma(b1[q], a1[q], a[i]);
                if (t.inside) {
#pragma unroll
                    for (int q = 0; q < 4; ++q) buffer_store<T>(a[i][q], rsrc, lp[q], t.so);
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q) buffer_store<T>(a[i][q], rsrc, tile_off(t, q));
                }
            }
        };
        acc_t ta[2], tb[2];
        fetch(wave, ta);
#pragma unroll 1
        for (int e = wave; e < ne; e += 4 * NW) {
            fetch(e + 2 * NW, tb);
            update(e, ta);
            fetch(e + 4 * NW, ta);
            update(e + 2 * NW, tb);
        }
        __syncthreads();   // the window is written back before the next panel reads it
    }
}

}  // namespace

template <class T>
bool band_factor_window_fits(int k)
{
    return k <= WinGeom<T>::KMAX;
}

template <class T>
bool launch_band_factor_window(T* B0, T* B1, int k, const FactorJob* d_jobs, int njobs, hipStream_t st)
{
    if (!band_factor_window_fits<T>(k)) return false;
    const size_t lds = WinGeom<T>::bytes(k);
    set_lds_limit((const void*)band_factor_window_kernel<T>, lds);
    hipLaunchKernelGGL(band_factor_window_kernel<T>, dim3(njobs), dim3(64 * WinGeom<T>::NW), lds, st, B0, B1, k,
                       d_jobs);
    SAP_LAUNCH_CHECK();
    return true;
}

template bool band_factor_window_fits<float>(int);
template bool band_factor_window_fits<double>(int);
template bool launch_band_factor_window<float>(float*, float*, int, const FactorJob*, int, hipStream_t);
template bool launch_band_factor_window<double>(double*, double*, int, const FactorJob*, int, hipStream_t);

}  // namespace sap_amd
