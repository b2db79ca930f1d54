// The helicity chain over column-contiguous profiles, read where they lie.
//
// Almost all of the chain's arithmetic -- a level's virtual temperature and
// its height above the level below: two FP64 logarithms, an exponential, five
// divisions -- depends on that level and the one below only.  A block takes 64
// columns and their levels in windows of SRH_KC:
//
//  * three of its waves compute the heights' increments of a window's (column,
//    level) pairs, consecutive lanes on consecutive levels of a column, so the
//    reads are contiguous as the profiles lie and nothing waits for a level
//    below (its virtual temperature comes from the neighbouring lane); the
//    increments and the winds go to LDS, level by level;
//  * the fourth, a lane per column, walks the window before (SrhWalk: the sum
//    of the heights, the Bunkers brackets, the helicity sum).  Which wave that
//    is changes from block to block, so that the CU's four SIMDs share the
//    walks.
//
// When every column of the block has its outputs' levels behind it (above
// 6 km and the helicity's depth), the rest of the levels is only checked for
// rising heights, as srh_column does; a column that fails the check, whose
// heights fall anywhere, or with a level outside the straight-line kernels'
// range, is done again by srh_column.  The arithmetic is srh_column's
// operation for operation, so the results are its bit for bit.
//
// A lane per column over transposed copies, with the whole chain in one walk,
// took for 1024 x 512 columns of 137 levels 490 us for the copies and 4 x 240
// us for the walks, which waited for their own chains of FP64 operations (one
// VALU instruction in 24 cycles per wave); this takes 713 us for the call, at
// one VALU instruction in 6.6 cycles per SIMD.  It fetches 5.05 GB for 1.45 of
// profiles (read requests, all of 128 bytes): a window is part of a cache
// line, and the columns in flight are more than the L2 keeps.  Windows of
// whole lines fetched less and were slower: more levels computed past the
// outputs' (32 levels to a window), or too few columns in flight.
#pragma once
#include "cape_launch.h"
#include "srh_column.h"

namespace xcape {
namespace XC_NS {

constexpr int SRH_KC = 8;         // levels per window (16: as fast on 137 levels, slower on 37)
constexpr int SRH_COLS = 64;      // columns per block
constexpr int SRH_PITCH = 65;     // elements per level row in LDS (distinct banks)

template <typename TI> struct SrhLds {
    // by window parity
    double dh[2][SRH_KC * SRH_PITCH];
    TI u[2][SRH_KC * SRH_PITCH], v[2][SRH_KC * SRH_PITCH];
    // of the level below the next window (first the surface): its virtual
    // temperature and pressure
    double tv[SRH_COLS], P[SRH_COLS];
    int first[SRH_COLS];          // a column's first level (0-based)
    int fail[SRH_COLS];
    // every column complete, by window parity (a slot is written again two
    // windows on, with a barrier in between)
    int complete[2];
};

// A column by srh_column: the columns a block's walk cannot do.
template <typename TB, typename TI>
__device__ __forceinline__ void srh_column_again(const CapeGridArgs &a, int64_t col)
{
    SigmaCol<uint64_t, TI> c{};
    int nk = 0;
    if (!column_at(a, col, c, nk)) return;
    c.us = in_arr<TI>(a.us)[col];
    c.vs = in_arr<TI>(a.vs)[col];
    SrhOutT<TB> so;
    srh_column<TB>(c, nk, a.depth, 2.0, so);
    store_srh(a, col, so);
}

template <typename TB, typename TI>
__global__ void __launch_bounds__(256) srh_slab_kernel(CapeGridArgs a)
{
    __shared__ SrhLds<TI> L;
    const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
    const int64_t c0 = (int64_t)blockIdx.x * SRH_COLS;
    const int nc = a.ncol - c0 < SRH_COLS ? (int)(a.ncol - c0) : SRH_COLS;
    const int nk = (int)a.nk_in;
    // the block's slab of each profile array: column c0 + c's level k at
    // c * nk + k (shared pressure levels: at k)
    const int64_t slab = c0 * nk;
    const TI *p = a.p1d ? in_arr<TI>(a.p1d) : in_arr<TI>(a.p) + slab;
    const int pc = a.p1d ? 0 : nk;
    const TI *t = in_arr<TI>(a.t) + slab, *td = in_arr<TI>(a.td) + slab;
    const TI *u = in_arr<TI>(a.u) + slab, *v = in_arr<TI>(a.v) + slab;
    const double hs = 2.0;
    const TB zsurf = (TB)hs;
    // makers 0, 1, 2 and the walker
    const int role = (wave + 3 - (int)(blockIdx.x & 3)) & 3;
    const bool walker = role == 3;
    // the walker's lane: column c0 + lane
    double us = 0.0, vs = 0.0;
    SrhWalk<TB> w;
    if (walker) {
        L.first[lane] = nk;       // no levels
        if (lane < nc) {
            SigmaCol<uint64_t, TI> col{};
            int nk_col = 0;
            column_at(a, c0 + lane, col, nk_col);
            L.tv[lane] = std_tv((double)col.ts, (double)col.tds, (double)col.ps);
            L.P[lane] = (double)col.ps;
            L.first[lane] = nk + 1 - nk_col;
            us = (double)in_arr<TI>(a.us)[c0 + lane];
            vs = (double)in_arr<TI>(a.vs)[c0 + lane];
        }
        L.fail[lane] = 0;
        if (lane < 2) L.complete[lane] = 0;
        w.init(hs, us, vs);
    }
    __syncthreads();
    // the makers' shares of a window's columns, CW columns at a time
    constexpr int CW = 64 / SRH_KC, GROUPS = SRH_COLS / CW, SHARE = (GROUPS + 2) / 3;
    const int c_begin = role * SHARE * CW;
    const int c_stop = c_begin + SHARE * CW;
    const int c_end = walker ? 0 : (c_stop < nc ? c_stop : nc);
    // window i is computed while window i - 1 is walked
    const int windows = (nk + SRH_KC - 1) / SRH_KC;
    int walked = 0;               // windows walked
    bool complete = false;
    for (int i = 0; i <= windows; ++i) {
        const int buf = i & 1;
        if (!walker && i < windows) {
            const int kk = lane & (SRH_KC - 1), k = i * SRH_KC + kk;
            const auto load = [&](int c, TI &pk, TI &tk, TI &tdk, TI &uk, TI &vk) {
                c = c < nc ? c : nc - 1;
                // a level of the column, where this lane has none
                const int f = L.first[c], kq = k < f ? f : (k < nk ? k : nk - 1);
                const uint32_t e = (uint32_t)(c * nk + kq);
                pk = p[(uint32_t)(c * pc + kq)];
                tk = t[e];
                tdk = td[e];
                uk = u[e];
                vk = v[e];
            };
            TI pn, tn, tdn, un, vn;
            load(c_begin + lane / SRH_KC, pn, tn, tdn, un, vn);
#pragma unroll 1
            for (int cb = c_begin; cb < c_end; cb += CW) {
                const TI pk = pn, tk = tn, tdk = tdn, uk = un, vk = vn;
                const int cw = cb + lane / SRH_KC, c = cw < nc ? cw : nc - 1;
                load(cw + CW, pn, tn, tdn, un, vn);   // in flight meanwhile
                const int first = L.first[c];
                const bool on = cw < nc && k >= first && k < nk;
                const double Pk = (double)pk;
                // the level below: the lane below's, or (at the window's first
                // level, and at the column's, whose level below is the surface)
                // the carried one
                const bool carry = kk == 0 || k == first;
                double Pb = __shfl_up(Pk, 1, SRH_KC);
                if (carry) Pb = L.P[c];
                double tv, lnr;
                bool ok;
                std_level_raw((double)tk, (double)tdk, Pk, Pb, tv, lnr, ok);
                double tvb = __shfl_up(tv, 1, SRH_KC);
                if (carry) tvb = L.tv[c];
                const double dh = std_dh_raw(tv, tvb, lnr);
                if (on) {
                    // outside the straight-line kernels' range (a lane below
                    // that is fails itself)
                    if (!(ok && __builtin_isfinite(dh))) L.fail[c] = 1;
                    L.dh[buf][kk * SRH_PITCH + c] = dh;
                    L.u[buf][kk * SRH_PITCH + c] = uk;
                    L.v[buf][kk * SRH_PITCH + c] = vk;
                    // (a column's lanes are in one wave, in every window)
                    if (kk == SRH_KC - 1) {
                        L.tv[c] = tv;
                        L.P[c] = Pk;
                    }
                }
            }
        } else if (walker && i > 0) {
            const int first = L.first[lane], kw = (i - 1) * SRH_KC;
            const int kn = nk - kw < SRH_KC ? nk - kw : SRH_KC;
            const double *dh = L.dh[buf ^ 1] + lane;
            const TI *lu = L.u[buf ^ 1] + lane, *lv = L.v[buf ^ 1] + lane;
            for (int q = 0; q < kn; ++q) {
                if (kw + q < first) continue;
                w.level(dh[q * SRH_PITCH], (double)lu[q * SRH_PITCH], (double)lv[q * SRH_PITCH],
                        a.depth);
            }
            const bool done = lane >= nc || (first < kw + kn && w.complete(zsurf));
            if (__builtin_amdgcn_ballot_w64(!done) == 0 && lane == 0) L.complete[buf] = 1;
        }
        __syncthreads();
        walked = i;
        complete = L.complete[buf] != 0;
        if (complete) break;
    }
    // the levels from k0 on are only checked (k0 - 1: the last one walked)
    const int k0 = walked * SRH_KC;
    if (complete && k0 < nk) {
        for (int c = wave; c < nc; c += 4) {
            for (int k = k0 - 1 + lane; k < nk; k += 64) {
                const uint32_t e = (uint32_t)(c * nk + k), ep = (uint32_t)(c * pc + k);
                const float pk = (float)p[ep], pb = (float)p[k >= k0 ? ep - 1 : ep];
                const bool ok = std_tv_sign((float)t[e], (float)td[e], pk) > 1.0f;
                if (!(ok && (k < k0 || pk < pb))) L.fail[c] = 1;
            }
        }
        __syncthreads();
    }
    if (!walker || lane >= nc) return;
    // done here: heights that rise throughout the walk, and either through the
    // rest too or, the whole column walked, ending above the surface
    if (L.fail[lane] == 0 && w.mono && (complete || !(zsurf > w.z_prev))) {
        SrhOutT<TB> so;
        w.finish_b();
        w.finish(us, vs, so);
        store_srh(a, c0 + lane, so);
    } else {
        srh_column_again<TB, TI>(a, c0 + lane);
    }
}

}  // namespace XC_NS
}  // namespace xcape
