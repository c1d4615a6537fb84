// Register-resident MFMA banded LU/UL of the partitions (the factorization
// used for half-bandwidths up to 224 in FP32 and 112 in FP64).
//
// Band layout (column-major, as the reference's m_B, sap/device/
// data_transfer.cuh:440-447): A(r, c) at B[c*(2k+1) + k + r - c]; a UL
// factorization is the LU factorization of the same storage read backwards.
#include "mfma.hpp"
#include "sap_internal.hpp"
#include "sub_panel.hpp"

#include <climits>
#include <type_traits>

namespace sap_amd {

namespace {

// ---------------------------------------------------------------------------
// Register-resident blocked banded LU, 512 threads (8 wavefronts) per
// partition, 32-column panels, 16 x 16 MFMA tiles.
// The active region of panel p, rows and columns [32p, 32p + 16 KT) with
// KT = ceil((k + 32) / 16), stays in the MFMA accumulators of the eight
// wavefronts for the whole factorization: tile (R, C) of the partition (tile
// row R, tile column C) lives in slot (R mod KT, C mod KT), and slot s
// belongs to wavefront s mod 8.  When the elimination moves down the diagonal
// by 32 rows, the tiles that leave the region are exactly the next panel's
// columns and U rows, and the slots they free take the tiles that enter, so
// every band entry is read from HBM once and every factor entry written once.
// Per panel:
//   A.  the slots of the panel's columns and U rows are copied to LDS, and
//       start loading the entering tiles (first used one panel later);
//   B.  the panel is factored in two sub-panels of 16 columns.  The first
//       wavefronts hold the rows below the sub-panel's diagonal block, one
//       per lane (L), as many others the columns right of it (U), and every
//       16-lane row of every wavefront holds a copy of the diagonal block
//       itself, one row per lane: each factors its copy (boosting at pivot
//       time) and applies every elimination step to its own row or column at
//       once, with the pivot row (the multipliers) broadcast from the copy
//       inside the lane row by DPP.  So the diagonal block's LU and both
//       triangular solves are one pass of 16 steps, with no exchange between
//       wavefronts.  Between the sub-panels the first one's contribution to
//       the second's columns and rows goes through the matrix cores;
//   C.  trailing tiles += (-L21) U12 on the matrix cores
//       (v_mfma_f32_16x16x4f32 / v_mfma_f64_16x16x4f64, the 32 panel columns
//       split over the four lane groups), and the panel's factors go out;
//       wavefronts w and w + 4 share a SIMD, and one does its stores while
//       the other multiplies.  Tiles are kept transposed in the accumulators
//       (the update is acc^T += U12^T (-L21)^T), which makes each tile load
//       read whole 16-row column segments.
// Outside the band every stored value is an exact zero, so the padded tiles
// never create fill-in.  The wavefronts exchange data only through LDS (each
// tile load is consumed by the wavefront that issued it; factor stores are
// not read back), so the barriers do not wait for global memory.  Factors are
// stored as L (unit), D, U' like the other factorization kernels; the
// multipliers use the pivot's reciprocal.
// What bounds it: two wavefronts on a SIMD, each running a chain of dependent
// instructions (8 cycles apiece, 12 while the other one multiplies), so time
// goes with the instructions per panel, not with bytes (k = 200: 0.6 TB/s) and
// only for the widest windows with the matrix cores (k = 200: 9.2k of 40k
// cycles a panel).  Both triangular solves in one pass over register-held rows
// and columns, instead of a diagonal LU by one wavefront followed by solves
// out of LDS, took the factorizations of both directions from 3.15 to 2.58 ms
// (n = 200000, k = 50, 16 partitions, FP32), 8.53 to 8.28 ms (n = 1000000,
// k = 200, 64 partitions), and in FP64 (n = 100000, 8 partitions) from 5.80
// to 2.75 ms at k = 16 and 8.65 to 5.54 ms at k = 100.
// ---------------------------------------------------------------------------
template <class T, int KT>
struct ResLds {
    static constexpr int PS = 36;                         // row stride: 16-byte aligned rows, few bank conflicts
    static constexpr int NTR = 16 * (KT - 2);             // trailing rows / columns
    // two panel buffers, used by alternate panels (a wavefront may copy the
    // next panel's tiles while another still stores this one's factors):
    static constexpr int pn_off = 0;                      // Pn [16 KT][PS]: panel rows; after B rows >= 32 hold -L21
    static constexpr int ub_off = pn_off + 16 * KT * PS;  // UbT [NTR][PS]: U block, one column per row
    static constexpr int rp_off = ub_off + NTR * PS;      // pivot reciprocals [32]
    static constexpr int buf_elems = rp_off + 32;
    static constexpr size_t bytes = sizeof(T) * (size_t)(2 * buf_elems);
};

template <class T, int KT, int NW>
__global__ __launch_bounds__(64 * NW) void band_factor_resident_kernel(T* __restrict__ B0, T* __restrict__ B1,
                                                                   const T* __restrict__ Bin, int k_all,
                                                                   const FactorJob* __restrict__ jobs)
{
    using MF = Mfma16<T>;
    using acc_t = typename MF::acc_t;
    using LY = ResLds<T, KT>;
    constexpr int PS = LY::PS, NTR = LY::NTR, NS = KT * KT, SPW = (NS + NW - 1) / NW, HR = 32 + NTR;
    constexpr int RW = (16 + NTR + 63) / 64;   // wavefronts of the L rows in B, and of the U columns
    constexpr int UOFF = 64 * RW;              // first thread of the U columns
    constexpr int UT = sizeof(T) == 4 ? 2 : 1; // tiles in flight in the update between sub-panels (registers)
    static_assert(2 * RW <= NW, "B thread ranges");
    static_assert(SPW <= 32, "slot class masks are 32-bit");
    const FactorJob job = jobs[blockIdx.x];
    const int k = job.kb > 0 ? job.kb : k_all;
    T* __restrict__ base = (job.buf ? B1 : B0) + job.boff;
    const int64_t w = 2 * k + 1;
    const int64_t len = job.len;
    const int dir = job.dir;
    const int wm1 = 2 * k;   // next column, same row

    extern __shared__ unsigned char smem_raw[];
    T* const sm = reinterpret_cast<T*>(smem_raw);
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);   // uniform: slot logic stays scalar

    // Tile loads are buffer loads over the partition's storage: every element
    // is one unconditional load, and entries outside the band or the
    // partition use an offset past the end of the buffer, which reads zero.
    // (A register only ever written by loads needs no wait for an earlier
    // load into it.)  rem = len - j0 is the number of partition rows left.  Element (j0 + dr, j0 + dc) is at element offset
    // ob + dir * (dc * 2k + dr) with ob = rel0 + dir * (j0 * (2k + 1) + k).
    // The band is read from Bin when given (the LU and UL factorizations of
    // one partition then share one unfactored copy) and the factors are
    // written to the job's band; without Bin the factorization is in place.
    const __amdgpu_buffer_rsrc_t rsrc = __builtin_amdgcn_make_buffer_rsrc(
        (void*)(base + job.start * w), 0, (int)(len * w * (int64_t)sizeof(T)), 0x00020000);
    const __amdgpu_buffer_rsrc_t rsrc_in = __builtin_amdgcn_make_buffer_rsrc(
        (void*)((Bin ? Bin + job.boff : base) + job.start * w), 0, (int)(len * w * (int64_t)sizeof(T)), 0x00020000);
    const int rel0 = dir > 0 ? 0 : (int)(len * w - 1);
    // Tiles are held transposed: accumulator register q of lane l holds
    // A(dr0 + l % 16, dc0 + row(l, q)), so for each register the 16 lanes of
    // a group read 16 consecutive rows of one column (one contiguous segment
    // per lane group).
    // A lane's first element of the tile with its lowest address at byte
    // offset so is lp0 bytes above it, its row less its column is e0 more
    // than the tile's, and each further element is one column step on.
    // sk = dr0 - dc0 + k, rr = rem - dr0 (rows of the tile in the partition;
    // a column past its end is past the end of the buffer).
    constexpr int CS = sizeof(T) == 4 ? 1 : 4;       // columns between a lane's elements
    const int so_rev = dir < 0 ? (15 * wm1 + 15) * (int)sizeof(T) : 0;
    const int cstep = dir * CS * wm1 * (int)sizeof(T);
    const int lr0 = threadIdx.x & 15, lc0 = MF::row(threadIdx.x & 63, 0);
    const int lp0 = so_rev + dir * (lc0 * wm1 + lr0) * (int)sizeof(T), e0 = lr0 - lc0;
    auto load_tile = [&](acc_t& t, int so, int sk, int rr) {
        const int e = lr0 < rr ? e0 + sk : INT_MIN;
#pragma unroll
        for (int q = 0; q < 4; ++q)
            t[q] = buffer_load<T>(rsrc_in, (unsigned)(e - CS * q) <= (unsigned)wm1 ? lp0 + so + q * cstep : -1);
    };
    // so of the tile at (dr0, dc0) of the panel whose window begins at element ob
    auto tile_off = [&](int ob, int dr0, int dc0) {
        return (ob + dir * (dc0 * wm1 + dr0)) * (int)sizeof(T) - so_rev;
    };
    // Factors of panel pp from panel buffer bq: its 32 columns (rows 0 .. HR-1:
    // L, D, U' of the diagonal block and L21), a column and 64 rows at a time,
    // and its 32 U' rows, two columns at a time.  Lanes run up the addresses;
    // entries outside the band get an offset past the end of the buffer and
    // are dropped.
    auto store_panel = [&](int64_t pp, const T* bq, int lane) {
        constexpr int NG = (HR + 63) / 64;
        const int64_t pj0 = 32 * pp;
        const int obq = rel0 + dir * (int)(pj0 * w + k);
        const int prem = (int)min(len - pj0, (int64_t)(1 << 30));
        const int pnb = min(32, prem);
        const T* qPn = bq + LY::pn_off;
        const T* qUb = bq + LY::ub_off;
        const T* qrp = bq + LY::rp_off;   // pivot reciprocals (0 past the partition's end)
        const int rl = dir > 0 ? lane : 63 - lane;
        const T f0 = qrp[rl & 31];
#pragma unroll 1
        for (int c = wave; c < pnb; c += NW) {
            T v[NG];
#pragma unroll
            for (int g = 0; g < NG; ++g) v[g] = qPn[min(64 * g + rl, HR - 1) * PS + c];
            // U' of the diagonal block is scaled by 1 / pivot; L21 rows are
            // kept negated in LDS
            v[0] = rl >= 32 ? -v[0] : (rl < c ? v[0] * f0 : v[0]);
            const int lo = max(c - k, 0), top = min(min(HR, prem), c + k + 1);   // rows [lo, top) are stored
            const int oc = (obq + dir * (c * wm1 + rl)) * (int)sizeof(T);
#pragma unroll
            for (int g = 0; g < NG; ++g) {
                const bool in = (unsigned)(rl + 64 * g - lo) < (unsigned)(top - lo);
                buffer_store<T>(g == 0 ? v[g] : -v[g], rsrc, in ? oc + dir * 64 * g * (int)sizeof(T) : -1);
            }
        }
        const int half = lane >> 5, um = dir > 0 ? lane & 31 : 31 - (lane & 31);
        const T fu = qrp[um];
        const int ul = (obq + dir * ((32 + half) * wm1 + um)) * (int)sizeof(T);
        const int ctop = min(min(NTR, prem - 32), k);
#pragma unroll 1
        for (int c0 = 2 * wave; c0 < ctop; c0 += 8 * NW) {
            T v[4];
#pragma unroll
            for (int i = 0; i < 4; ++i) v[i] = qUb[min(c0 + half + 2 * NW * i, NTR - 1) * PS + um];
#pragma unroll
            for (int i = 0; i < 4; ++i) {
                const int cc = c0 + half + 2 * NW * i;
                const bool in = um < pnb && cc < ctop && um >= 32 + cc - k;
                buffer_store<T>(v[i] * fu, rsrc, in ? ul + dir * (c0 + 2 * NW * i) * wm1 * (int)sizeof(T) : -1);
            }
        }
    };

    acc_t acc[SPW];
    {
        const int ob = rel0 + dir * k;
        const int rem = (int)min(len, (int64_t)(1 << 30));
#pragma unroll
        for (int j = 0; j < SPW; ++j) {
            const int s = wave + NW * j, dr0 = 16 * (s / KT), dc0 = 16 * (s % KT);
            if (s < NS) load_tile(acc[j], tile_off(ob, dr0, dc0), dr0 - dc0 + k, rem - dr0);
        }
    }

    const int64_t npan = (len + 31) / 32;
    for (int64_t p = 0; p < npan; ++p) {
        // lane-derived values are re-materialised every panel (keeps the
        // per-lane predicates of the unrolled loops out of the registers)
        int tid = threadIdx.x, zoff = 0;
        asm volatile("" : "+v"(tid), "+v"(zoff));
        const int lane = tid & 63, lr = lane & 15, lg = lane >> 4;
        const int cur = (int)(p & 1);
        // LDS addresses from an opaque zero fold into the ds_* immediate
        // offsets instead of living in scalar registers across the loop
        T* bcur = sm + zoff + cur * LY::buf_elems;
        T* Pn = bcur + LY::pn_off;
        T* UbT = bcur + LY::ub_off;
        T* rpiv = bcur + LY::rp_off;
        const int64_t j0 = 32 * p;
        const int rem = (int)min(len - j0, (int64_t)(1 << 30));
        const int nb = min(32, rem);
        const int sh = (int)((2 * p) % KT);
        const int obp = rel0 + dir * (int)(j0 * w + k);
        // Slot bookkeeping, lane-parallel: lane j holds, for slot j of this
        // wavefront (s = wave + NW j, clamped to NS - 1 past the last slot)
        // with rotated tile coordinates (rl, gl), the LDS offset it is copied
        // to, the place of the tile it loads next and the LDS offsets of its
        // operands; three ballots give the slot classes: panel column
        // (gl < 2), U row (rl < 2 <= gl) and trailing (both >= 2).  Each
        // unrolled slot step then costs a mask bit test and a few readlanes
        // instead of its own scalar index arithmetic: the panel loop has to
        // stay well inside the 64 KiB instruction cache that two compute
        // units share.
        unsigned pm, um, tm;
        int cpo, lso, lsk, lrr, mao, mbo;
        {
            const int sl = min(wave + NW * lane, NS - 1);
            int rl = sl / KT - sh, gl = sl % KT - sh;
            rl += KT & neg_mask(rl);
            gl += KT & neg_mask(gl);
            const bool okl = lane < SPW && wave + NW * lane < NS;
            pm = (unsigned)__builtin_amdgcn_ballot_w64(okl && gl < 2);
            um = (unsigned)__builtin_amdgcn_ballot_w64(okl && gl >= 2 && rl < 2);
            tm = (unsigned)__builtin_amdgcn_ballot_w64(okl && gl >= 2 && rl >= 2);
            mao = 16 * PS * rl;
            mbo = LY::ub_off + 16 * PS * (gl - 2);
            cpo = gl < 2 ? mao + 16 * gl : mbo + 16 * rl;
            const int dr0 = 16 * (rl < 2 ? rl + KT : rl), dc0 = 16 * (gl < 2 ? gl + KT : gl);
            lso = tile_off(obp, dr0, dc0);
            lsk = dr0 - dc0 + k;
            lrr = rem - dr0;
        }
        auto of_slot = [&](int v, int j) { return __builtin_amdgcn_readlane(v, j); };   // j a compile-time constant

        // A. the leaving tiles to LDS, then their slots load the entering
        //    tiles.  (All copies to LDS come first: reading a slot that may
        //    still be loading waits for every load issued before it.)
#pragma unroll
        for (int j = 0; j < SPW; ++j) {
            if ((pm >> j) & 1) {
                T* const pt = bcur + of_slot(cpo, j) + lr * PS;
                if constexpr (sizeof(T) == 4) {   // four consecutive columns
                    *reinterpret_cast<acc_t*>(pt + 4 * lg) = acc[j];
                } else {
#pragma unroll
                    for (int q = 0; q < 4; ++q) pt[MF::row(lane, q)] = acc[j][q];
                }
            } else if ((um >> j) & 1) {
                T* const pt = bcur + of_slot(cpo, j) + lr;
#pragma unroll
                for (int q = 0; q < 4; ++q) pt[MF::row(lane, q) * PS] = acc[j][q];
            }
        }
        lds_barrier();
#pragma unroll
        for (int j = 0; j < SPW; ++j)
            if (((pm | um) >> j) & 1) load_tile(acc[j], of_slot(lso, j), of_slot(lsk, j), of_slot(lrr, j));

        // B. the two sub-panels (columns O .. O + 15).  Threads 0 .. 15 + NTR - O
        //    hold rows 16 + O .. of the panel, threads UOFF .. the columns 16 + O ..
        //    (the first 16 of sub-panel 0 are the panel's own columns 16 .. 31,
        //    in Pn; the rest UbT).
        const int boosted = job.boost ? (job.boost_last ? 32 : min(32, rem - 1)) : 0;
#pragma unroll 1
        for (int O = 0; O < 32; O += 16) {
            int c16 = lane & 15;
            asm volatile("" : "+v"(c16));
            T d[16], own[16], pr = (T)0;
            lds_get16(Pn + (O + c16) * PS + O, d);
            const bool urow = wave < RW;
            const int t = urow ? tid : tid - UOFF;         // row 16 + O + t, or column t
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
                const T rl = sub_panel_pivot<0, T>(d, pr, c16, plain);
                if (urow) sub_panel_steps<0, true, false, T>(d, own, pr, rl, c16, plain);
                else sub_panel_steps<0, false, false, T>(d, own, pr, rl, c16, plain);
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
                rpiv[O + tid] = live ? pivot_rcp(pr) : (T)0;
            }
            lds_barrier();
            if (O == 0) {
                // columns 16 .. 31 of the rows below (A = -L_a, B = rows 0 .. 15 of
                // U, columns 16 .. 31), and rows 16 .. 31 of the columns right
                // (A = -U_a^T, B = L_ba^T), 16 x 16 tiles
                const int g = lane >> 4;
#pragma unroll 1
                for (int f0 = wave; f0 < 2 * KT - 3; f0 += UT * NW) {
                    T* at[UT];
                    acc_t ac[UT];
                    T av[UT][4], bv[UT][4];
#pragma unroll
                    for (int i = 0; i < UT; ++i) {
                        const int f = min(f0 + NW * i, 2 * KT - 4);
                        const bool lside = f < KT - 1;
                        const T* const rows = lside ? Pn + (16 + 16 * f) * PS : UbT + 16 * (f - (KT - 1)) * PS;
                        const bool neg = f == 0 || !lside;   // operands not kept negated
                        at[i] = const_cast<T*>(rows) + MF::row(lane, 0) * PS + 16 + c16;
#pragma unroll
                        for (int q = 0; q < 4; ++q) ac[i][q] = at[i][CS * q * PS];
#pragma unroll
                        for (int q = 0; q < 4; ++q) {
                            const T x = rows[c16 * PS + 4 * q + g];
                            av[i][q] = neg ? -x : x;
                            bv[i][q] = lside ? Pn[(4 * q + g) * PS + 16 + c16] : Pn[(16 + c16) * PS + 4 * q + g];
                        }
                    }
#pragma unroll
                    for (int q = 0; q < 4; ++q)
#pragma unroll
                        for (int i = 0; i < UT; ++i) ac[i] = MF::mma(av[i][q], bv[i][q], ac[i]);
#pragma unroll
                    for (int i = 0; i < UT; ++i)
                        if (f0 + NW * i < 2 * KT - 3) {
#pragma unroll
                            for (int q = 0; q < 4; ++q) at[i][CS * q * PS] = ac[i][q];
                        }
                }
                lds_barrier();
            }
        }

        // C. trailing update on the matrix cores and the panel's factors out.
        //    The next panel writes the other buffer, so no barrier is needed
        //    after this phase.
        // Every tile load of this panel has long completed (B ran since);
        // saying so with an explicit wait before the stores are issued clears
        // the compiler's record of loads pending across the loop back-edge,
        // which would otherwise make each slot of the next phase A wait for
        // the loads just issued by the slots before it, and for the stores
        // (vmcnt bits [3:0] and [15:14] = 0, expcnt and lgkmcnt at their
        // maxima).
        __builtin_amdgcn_s_waitcnt((0x7 << 4) | (0xF << 8));
        if (wave >= NW / 2) store_panel(p, bcur, lane);
        if (tm) {
            // Each slot's operands are two rows of 8 values (lane group lg
            // takes k = 8 lg .. 8 lg + 7), in two halves; each half of the
            // next trailing slot's is fetched while the other half of this
            // one's is multiplied.  Lane j holds the operand offsets of the
            // slot after trailing slot j (its own again for the last), so
            // that both are in one basic block.
            const T* const al = bcur + lr * PS + 8 * lg;
            const unsigned after = tm & (~1u << (lane & 31));
            const int nj = 4 * (after ? __builtin_ctz(after) : 31 - __builtin_clz(tm)), first = __builtin_ctz(tm);
            const int nma = __builtin_amdgcn_ds_bpermute(nj, mao), nmb = __builtin_amdgcn_ds_bpermute(nj, mbo);
            T a0[4], b0[4], a1[4], b1[4];
            {
                const T* const ap = al + __builtin_amdgcn_readlane(mao, first);
                const T* const bp = al + __builtin_amdgcn_readlane(mbo, first);
                lds_get4(ap, a0); lds_get4(bp, b0); lds_get4(ap + 4, a1); lds_get4(bp + 4, b1);
            }
#pragma unroll
            for (int j = 0; j < SPW; ++j) {
                if ((tm >> j) & 1) {
                    const T* const ap = al + of_slot(nma, j);
                    const T* const bp = al + of_slot(nmb, j);
                    // transposed tiles: acc^T += U12^T (-L21)^T
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[j] = MF::mma(b0[q], a0[q], acc[j]);
                    __builtin_amdgcn_sched_barrier(0);
                    lds_get4(ap, a0); lds_get4(bp, b0);
                    __builtin_amdgcn_sched_barrier(0);
#pragma unroll
                    for (int q = 0; q < 4; ++q) acc[j] = MF::mma(b1[q], a1[q], acc[j]);
                    __builtin_amdgcn_sched_barrier(0);
                    lds_get4(ap + 4, a1); lds_get4(bp + 4, b1);
                }
            }
        }
        if (wave < NW / 2) store_panel(p, bcur, lane);
    }
}

// Wavefronts per workgroup.  Sixteen leave 128 registers each: no faster where
// the tiles fit (k = 50: 2.59 against 2.58 ms for LU and UL, n = 200000), and
// from k = 100 they spill (k = 120: 8.97 against 8.41 ms, k = 200: 10.4
// against 8.28).
template <class T, int KT>
constexpr int resident_waves() { return 8; }

template <class T, int KT>
void launch_factor_resident(T* B0, T* B1, const T* Bin, int k, const FactorJob* jobs, int njobs, hipStream_t st)
{
    constexpr int NW = resident_waves<T, KT>();
    const size_t lds = ResLds<T, KT>::bytes;
    set_lds_limit((const void*)band_factor_resident_kernel<T, KT, NW>, lds);
    hipLaunchKernelGGL((band_factor_resident_kernel<T, KT, NW>), dim3(njobs), dim3(64 * NW), lds, st, B0, B1, Bin,
                       k, jobs);
    SAP_LAUNCH_CHECK();
}

// Largest window (in 16-row tiles) kept in registers: FP32 up to k = 224,
// FP64 (twice the registers and LDS per tile) up to k = 112.  The two widest
// FP64 windows spill (7 registers at k = 81 .. 96, 78 at k = 97 .. 112: 32 and
// 124 bytes of scratch a lane) and are still faster than the kernel with the
// window in the L2: 4.7 against 5.6 ms and 5.6 against 6.6 (n = 100000, 8
// partitions); the next does not fit.
template <class T>
constexpr int resident_max_kt() { return sizeof(T) == 4 ? 16 : 9; }

template <class T, int KT>
bool dispatch_resident(int kt, T* B0, T* B1, const T* Bin, int k, const FactorJob* jobs, int njobs,
                       hipStream_t st)
{
    if constexpr (KT > resident_max_kt<T>()) {
        return false;
    } else {
        if (kt == KT) { launch_factor_resident<T, KT>(B0, B1, Bin, k, jobs, njobs, st); return true; }
        return dispatch_resident<T, KT + 1>(kt, B0, B1, Bin, k, jobs, njobs, st);
    }
}

}  // namespace

template <class T>
bool band_factor_resident_fits(int k, int64_t max_len)
{
    // buffer offsets are 32-bit: a partition's storage must stay below 2 GiB
    if (max_len * (2 * (int64_t)k + 1) * (int64_t)sizeof(T) >= ((int64_t)1 << 31)) return false;
    return (k + 32 + 15) / 16 <= resident_max_kt<T>();
}

template <class T>
bool launch_band_factor_resident(T* B0, T* B1, const T* Bin, int k, const FactorJob* d_jobs, int njobs,
                                 int64_t max_len, hipStream_t st)
{
    if (!band_factor_resident_fits<T>(k, max_len)) return false;
    return dispatch_resident<T, 3>((k + 32 + 15) / 16, B0, B1, Bin, k, d_jobs, njobs, st);
}

template bool band_factor_resident_fits<float>(int, int64_t);
template bool band_factor_resident_fits<double>(int, int64_t);
template bool launch_band_factor_resident<float>(float*, float*, const float*, int, const FactorJob*, int, int64_t,
                                                 hipStream_t);
template bool launch_band_factor_resident<double>(double*, double*, const double*, int, const FactorJob*, int,
                                                  int64_t, hipStream_t);

}  // namespace sap_amd
