// fdga_local.h -- BSE_K2!, BSE_L_K2! and the SDE L-vertices of the local solver as sums of strided dot
// products, for gfx950.
//
// Each of these is a sum over the bubble mesh of a vertex evaluation times a weight, and a vertex evaluation
// is a sum of classes (src/channel.jl:220-339): in a channel reached by the conversion (src/convention.jl:4-37)
// K1(Ω') + K2(Ω', ν1) + K2(Ω', ν2) + K3(Ω', ν1, ν2), each where its arguments lie in its box.  Ω', ν1 and ν2
// are linear in the summed ω with slopes -1, 0 or 1, so each class is nonzero on one interval of ω and runs
// through its array with a constant stride there: Σ_ω F(...) W(ω) = Σ_classes Σ_{ω in interval} X[b + s ω] W[ω].
// A class's loop is a load of each side and a complex multiply-add, where evaluating F(Ω, ν, ω) point by point
// over the window tests every box of every class at every ω (some 150 instructions per point).  The K2
// classes whose Ω' and ν move together read a copy of K2 stored along that diagonal (k_seg_prep), so that
// the lanes of a wave, on consecutive ω, load whole lines; the K3 classes (at most the K3 box's Ω range
// of terms) are read in place.
#pragma once
#include "fdga_kernels.h"

namespace fdga {

// one channel's classes; S: K2 along its diagonals, S[ν + n2f + 2 n2f row] with row = Ω + ν (t, a) or
// Ω - ν (p) counted from its smallest value, zero outside the box (null: K2 is read in place)
struct SegCh {
    const double2 *K1, *K2, *K3;
    double2* S;
    int n1, n2b, n2f, n3b, n3f;
    __host__ __device__ __forceinline__ int rows() const { return 2 * (n2b + n2f) - 2; }
};
struct SegVtx { SegCh p, t, a; };
template <int CH>
__device__ __forceinline__ const SegCh& seg_ch(const SegVtx& v) { return CH == PCH ? v.p : CH == TCH ? v.t : v.a; }

// K2 along the diagonals of up to six channels, and for BSE_L_K2! the weights Π0(Ω, ω) F0(Ω, ω~, ∞) of up
// to three, on the band (the layout of k_bse_w)
struct SegPrep {
    SegCh ch[6];
    int plus[6];             // row = Ω + ν, else Ω - ν
    unsigned blk[6];         // first block of the channel's copy
    int nch;
    double2* W[3];
    const double2* Pi0[3];
    int wch[3];              // their channels
    unsigned wblk;           // first block of the weights, per channel
    unsigned wper;
    F0V f0;
    int n2b, nWP, nVP, wb;
};
__global__ __launch_bounds__(256) void k_seg_prep(SegPrep a) {
    if (blockIdx.x < a.wblk) {
        int k = 0;
        while (k + 1 < a.nch && blockIdx.x >= a.blk[k + 1]) ++k;
        const SegCh& c = a.ch[k];
        const int NV2 = 2 * c.n2f, e = (int)(blockIdx.x - a.blk[k]) * 256 + (int)threadIdx.x;
        if (e >= NV2 * c.rows()) return;
        const int v = e % NV2 - c.n2f, row = e / NV2;
        const int m = a.plus[k] ? row - (c.n2b - 1) - c.n2f - v : row - (c.n2b - 1) - (c.n2f - 1) + v;
        c.S[e] = in_b(m, c.n2b) ? c.K2[(size_t)(m + c.n2b - 1) + (size_t)(2 * c.n2b - 1) * (v + c.n2f)] : czero();
        return;
    }
    const unsigned q = blockIdx.x - a.wblk;
    const int k = (int)(q / a.wper);
    const size_t e = (size_t)(q - k * a.wper) * 256 + threadIdx.x;
    const int per = 2 * a.wb, NW2 = 2 * a.n2b - 1;
    if (e >= (size_t)per * NW2) return;
    const int t = (int)(e % per), m = (int)(e / per) - (a.n2b - 1), w = t - a.wb, ch = a.wch[k];
    const double2 f = ch == PCH ? a.f0.eval(m, bmf(m, w), FDGA_INF, PCH, PSP)
                      : ch == TCH ? a.f0.eval(m, w, FDGA_INF, TCH, DSP)
                                  : a.f0.eval(m, w, FDGA_INF, ACH, PSP);
    a.W[k][e] = cmul(a.Pi0[k][(size_t)(w + a.nVP) + (size_t)(2 * a.nVP) * (m + a.nWP - 1)], f);
}

// the wave's number in its block, in a scalar register: a class's bounds and base are the same for all lanes,
// and the scalar unit then forms them
__device__ __forceinline__ int seg_wave() { return __builtin_amdgcn_readfirstlane((int)threadIdx.x / WAVE); }
// acc(X[s ω], ω) over ω = l + lane, l + lane + 64, ... <= h
template <class ACC>
__device__ __forceinline__ void seg_run(const double2* X, int s, int l, int h, int lane, ACC&& acc) {
    for (int w = l + lane; w <= h; w += WAVE) acc(X[(ptrdiff_t)s * w], w);
}
// the classes of channel TO in the evaluation F(m, v, ω) of channel CH (CH != TO) on the mesh wl <= ω <= wh; DIAG: K2
// along its diagonals from S, else in place
template <int CH, int TO, bool DIAG, class ACC>
__device__ __forceinline__ void seg_cross(const SegCh& g, int m, int v, int wl, int wh, int lane, ACC&& acc) {
    // Ω' = al (ω - w0); ν1 = f1 fixed (F1) or ω + f1, ν2 likewise
    constexpr int al = (TO == PCH || CH == TCH) ? 1 : -1;
    constexpr bool F1 = (CH == PCH && TO == ACH) || (CH == TCH && TO == ACH), F2 = (CH != ACH && TO != ACH) || (CH == TCH && TO == ACH);
    const int w0 = CH == PCH && TO == TCH ? m - v - 1 : TO == PCH ? -(m + v + 1) : v;
    const int f1 = CH == PCH && TO == ACH ? m - v - 1 : CH == TCH && TO == ACH ? m + v : CH == ACH && TO == PCH ? m : 0;
    const int f2 = F2 ? v : CH == ACH && TO == TCH ? m : 0;
    seg_run(g.K1 + (g.n1 - 1) - (ptrdiff_t)al * w0, al, max(wl, w0 - (g.n1 - 1)), min(wh, w0 + (g.n1 - 1)), lane, acc);
    const int l2 = max(wl, w0 - (g.n2b - 1)), h2 = min(wh, w0 + (g.n2b - 1)), NW2 = 2 * g.n2b - 1, NV2 = 2 * g.n2f;
    auto k2 = [&](bool fixed, int f) {
        const double2* K2 = g.K2 + (g.n2b - 1) - (ptrdiff_t)al * w0 + (ptrdiff_t)NW2 * (f + g.n2f);
        if (fixed) {
            if (in_f(f, g.n2f)) seg_run(K2, al, l2, h2, lane, acc);
            return;
        }
        const int l = max(l2, -g.n2f - f), h = min(h2, g.n2f - 1 - f);
        if (!DIAG) {
            seg_run(K2, al + NW2, l, h, lane, acc);
        } else {   // Ω' + ν = w0 + f (al = -1) or Ω' - ν = -w0 - f (al = 1) along the class
            const int row = al < 0 ? w0 + f + (g.n2b - 1) + g.n2f : -w0 - f + (g.n2b - 1) + (g.n2f - 1);
            if (row >= 0 && row < g.rows()) seg_run(g.S + (ptrdiff_t)NV2 * row + (g.n2f + f), 1, l, h, lane, acc);
        }
    };
    k2(F1, f1);
    k2(F2, f2);
    int l3 = max(wl, w0 - (g.n3b - 1)), h3 = min(wh, w0 + (g.n3b - 1));
    const int N = 2 * g.n3f;
    if (F1) { if (!in_f(f1, g.n3f)) return; }
    else { l3 = max(l3, -g.n3f - f1); h3 = min(h3, g.n3f - 1 - f1); }
    if (F2) { if (!in_f(f2, g.n3f)) return; }
    else { l3 = max(l3, -g.n3f - f2); h3 = min(h3, g.n3f - 1 - f2); }
    seg_run(g.K3 + (f1 + g.n3f) + (ptrdiff_t)N * ((f2 + g.n3f) + (ptrdiff_t)N * (g.n3b - 1 - al * w0)),
            (F1 ? 0 : 1) + (F2 ? 0 : N) + al * N * N, l3, h3, lane, acc);
}
// the channel's own K3(m, v, ω)
template <class ACC>
__device__ __forceinline__ void seg_own(const SegCh& g, int m, int v, int wl, int wh, int lane, ACC&& acc) {
    if (!in_b(m, g.n3b) || !in_f(v, g.n3f)) return;
    const int N = 2 * g.n3f;
    seg_run(g.K3 + (v + g.n3f) + (ptrdiff_t)N * (g.n3f + (ptrdiff_t)N * (m + g.n3b - 1)), N, max(wl, -g.n3f),
            min(wh, g.n3f - 1), lane, acc);
}
// a RefVertex table's entries along ω: (Ω, ν, ω) or, swapped, (Ω, ω, ν)
template <class ACC>
__device__ __forceinline__ void seg_tab(const RefV& r, int k, bool swapped, int m, int v, int wl, int wh, int lane,
                                        ACC&& acc) {
    if (!in_b(m, r.tb) || !in_f(v, r.tf)) return;
    const int NB = 2 * r.tb - 1, NF = 2 * r.tf;
    const ptrdiff_t o = (ptrdiff_t)(m + r.tb - 1) + (ptrdiff_t)NB * (swapped ? r.tf + (ptrdiff_t)NF * (v + r.tf)
                                                                              : (v + r.tf) + (ptrdiff_t)NF * r.tf);
    seg_run(r.tab[k] + o, swapped ? NB : NB * NF, max(wl, -r.tf), min(wh, r.tf - 1), lane, acc);
}

// Arguments of BSE_K2! (src/BSEa/BSEa_K2.jl:43-100) and BSE_L_K2! (BSEa_K2.jl:1-41)
struct SegK2 {
    SegVtx F, F0;                // F0: the local Vertex of the reference system (vtx0)
    RefV ref;
    const double2 *Wp, *Wt, *Wa; // weights on the band
    const double2* ws;           // their sums over the mesh (BSE_K2!; the layout of K1Args)
    const double2 *Lp, *Lt, *La; // FL.K2 (BSE_K2!)
    const double2 *L1p, *L1t, *L1a;                                              // ROWS: FL.K1,
    const double2 *Ppp, *Ppp0, *Pph, *Pph0, *Spp, *Spp0, *Sph, *Sph0;            // Π, Π0 and their sums
    int nWP, nVP, vtx0;
    double2 *Kp, *Kt, *Ka;       // results
    int n2b, n2f, wb;
    double T;
    SymCls sp, sat;
    int np, nat;                 // classes of the p channel, and of the a and t channels
    int bat;                     // blocks per XCD of the latter, the first ones
    int at;                      // of those, 1: a is computed, 2: t (from a, or from the finished Ka without 1)
};
// the part of Σ_ω [F(Ω, ν, ω) - F(Ω, ∞, ω)] W(ω) that depends on ω under the sum (LEFT: of Σ Γ W with Γ free of
// F0 and of the own channel)
template <bool LEFT, bool REF, int CH, bool DIAG, class ACC>
__device__ __forceinline__ void seg_term(const SegK2& A, int m, int v, int wl, int wh, int lane, ACC&& acc) {
    constexpr int C1 = CH == PCH ? TCH : PCH, C2 = CH == ACH ? TCH : ACH;
    seg_cross<CH, C1, DIAG>(seg_ch<C1>(A.F), m, v, wl, wh, lane, acc);
    seg_cross<CH, C2, DIAG>(seg_ch<C2>(A.F), m, v, wl, wh, lane, acc);
    if (LEFT) return;
    seg_own(seg_ch<CH>(A.F), m, v, wl, wh, lane, acc);
    if (REF) {
        seg_cross<CH, C1, DIAG>(seg_ch<C1>(A.F0), m, v, wl, wh, lane, acc);
        seg_cross<CH, C2, DIAG>(seg_ch<C2>(A.F0), m, v, wl, wh, lane, acc);
        seg_own(seg_ch<CH>(A.F0), m, v, wl, wh, lane, acc);
    }
    if (A.ref.tb) {
        if (CH == ACH)
            seg_tab(A.ref, 3, true, m, v, wl, wh, lane, [&](double2 x, int w) { acc(cneg(x), w); });
        else
            seg_tab(A.ref, CH == PCH ? 0 : 2, false, m, v, wl, wh, lane, acc);
    }
}
// the part that does not depend on ω, K2(Ω, ν) of the channel in F and F0
template <bool REF, int CH>
__device__ __forceinline__ double2 seg_const(const SegK2& A, int m, int v) {
    const SegCh& g = seg_ch<CH>(A.F);
    double2 x = g.K2[(size_t)(m + g.n2b - 1) + (size_t)(2 * g.n2b - 1) * (v + g.n2f)];
    if (REF) {
        const SegCh& h = seg_ch<CH>(A.F0);
        if (in_b(m, h.n2b) && in_f(v, h.n2f))
            x = cadd(x, h.K2[(size_t)(m + h.n2b - 1) + (size_t)(2 * h.n2b - 1) * (v + h.n2f)]);
    }
    return x;
}
// threads of a block, and the largest band of the one-launch form
constexpr int seg_nt(bool rows) { return rows ? 256 : 512; }
constexpr int SEG_WB = 128;
__device__ __forceinline__ double2 seg_k1(const SegCh& g, const double2* K1, int m) {
    return in_b(m, g.n1) ? K1[m + g.n1 - 1] : czero();
}
__device__ __forceinline__ double2 seg_k2(const SegCh& g, const double2* K2, int m, int n) {
    return in_b(m, g.n2b) && in_f(n, g.n2f) ? K2[(size_t)(m + g.n2b - 1) + (size_t)(2 * g.n2b - 1) * (n + g.n2f)] : czero();
}
// A wave's row of weights in LDS: the terms of k_bse_w (LEFT: Π0(Ω, ω) F0(Ω, ω~, ∞)) at the class's Ω; returns Σ W
// over the mesh (BSE_K2!)
template <bool LEFT, int CH>
__device__ __forceinline__ double2 seg_row(const SegK2& A, int m, int lane, double2* row) {
    const SegCh &f0 = seg_ch<CH>(A.F0), &g = seg_ch<CH>(A.F);
    const double2 *L1 = CH == PCH ? A.L1p : CH == TCH ? A.L1t : A.L1a, *L2 = CH == PCH ? A.Lp : CH == TCH ? A.Lt : A.La;
    double2 c = A.ref.U, l = czero();   // F0 and FL without their K2
    if (A.vtx0) {
        c = cadd(c, CH == TCH ? csub(cscale(seg_k1(f0, f0.K1, m), 2.0), seg_k1(A.F0.a, A.F0.a.K1, m)) : seg_k1(f0, f0.K1, m));
    }
    if (!LEFT) l = CH == TCH ? csub(cscale(seg_k1(g, L1, m), 2.0), seg_k1(g, A.L1a, m)) : seg_k1(g, L1, m);
    const size_t r = (size_t)(m + A.nWP - 1), o = (size_t)(2 * A.nVP) * r + A.nVP;
    const double2 *P = (CH == PCH ? A.Ppp : A.Pph) + o, *P0 = (CH == PCH ? A.Ppp0 : A.Pph0) + o;
    double2 s = czero();
    for (int t = lane; t < 2 * A.wb; t += WAVE) {
        const int w = t - A.wb, wc = crossing(m, w, CH);
        double2 f = c, x = P0[w];
        if (A.vtx0) {
            double2 k = seg_k2(f0, f0.K2, m, wc);
            if (CH == TCH) k = csub(cscale(k, 2.0), seg_k2(A.F0.a, A.F0.a.K2, m, wc));
            f = cadd(f, k);
        }
        if (LEFT) {
            x = cmul(x, f);
        } else {
            double2 k = seg_k2(g, L2, m, wc);
            if (CH == TCH) k = csub(cscale(k, 2.0), seg_k2(g, A.La, m, wc));
            const double2 p = P[w];
            x = cadd(cmul(csub(p, x), f), cmul(p, cadd(l, k)));
            s = cadd(s, x);
        }
        row[t] = x;
    }
    if (LEFT) return s;
    const double2 *S = (CH == PCH ? A.Spp : A.Sph) + 3 * r, *S0 = (CH == PCH ? A.Spp0 : A.Sph0) + 3 * r;
    auto far = [&](int q) { return cadd(cmul(csub(S[q], S0[q]), c), cmul(S[q], l)); };
    return cadd(wave_sum2(s), cadd(far(0), far(1)));
}
// One wave per output class, lanes over ω.  The t channel is summed in the density component 2 F(t) - F(a)
// next to the a channel, whose terms both share.
// Blocks of 8 waves on consecutive ν of one Ω (shared lines of W), each XCD on a range of Ω of its own.  Bound
// by the L1: a chunk of 64 ω loads 1 KB of each side.  SIAM boxes 128, (64, 64), (32, 64), mesh 1536, alone on
// the card, without symmetry groups BSE_L_K2! 92 us and BSE_K2! 125 us (point by point: 240 and 292), with them
// 31 and 58 (61 and 164).  Tried: loops unrolled twice (the registers cost more occupancy than the second load
// in flight gives: 160 -> 209 us), the wave's number in a vector register (160 against 92 us).
// ROWS: each wave forms its weights in LDS and K2 is read in place, so that nothing has to be prepared: one launch
// instead of two (BSE_L_K2!) or three, for boxes whose kernels are not longer than a launch.  Called alone, p
// channel, SIAM boxes 33, (16, 16): BSE_K2! 8.1 us (prepared 15.2), BSE_L_K2! 7.1 (9.0).  Blocks of four waves, so that
// few classes spread over the card (eight: 8.6 and 7.4).
template <bool LEFT, bool REF, bool ROWS>
__global__ __launch_bounds__(seg_nt(ROWS)) void k_seg_k2(SegK2 A) {
    const int lane = threadIdx.x & (WAVE - 1), bq = (int)blockIdx.x / 8, xcd = (int)blockIdx.x % 8, per = (int)gridDim.x / 8;
    const bool pw = bq >= A.bat;
    const int n = pw ? A.np : A.nat;
    const int wid = (pw ? xcd * (per - A.bat) + bq - A.bat : xcd * A.bat + bq) * (seg_nt(ROWS) / WAVE) + seg_wave();
    if (!ROWS && wid >= n) return;
    const SymCls& sym = pw ? A.sp : A.sat;
    const int wq = ROWS ? min(wid, n - 1) : wid;   // (every wave reaches the barrier)
    const int NV2 = 2 * A.n2f, cls = sym.ncls ? wq : wq / NV2 + (2 * A.n2b - 1) * (wq % NV2), o0 = sym.rep(cls);
    const int NW2 = 2 * A.n2b - 1, iW = o0 % NW2, iv = o0 / NW2, m = iW - (A.n2b - 1), v = iv - A.n2f;
    const size_t ro = (size_t)(2 * A.wb) * iW + A.wb;
    const int wl = -A.wb, wh = A.wb - 1;   // the band covers the window or the mesh
    int b, e;
    sym.range(cls, b, e);
    const double2 *W0, *W1;                // the weights of p, or of a and t
    double2 tot0 = czero(), tot1 = czero();
    if constexpr (ROWS) {
        extern __shared__ double2 seg_rows[];
        double2* row = seg_rows + (size_t)(4 * A.wb) * seg_wave();
        W0 = row + A.wb;
        W1 = row + 3 * A.wb;
        if (pw) {
            tot0 = seg_row<LEFT, PCH>(A, m, lane, row);
        } else {
            if (A.at & 1) tot0 = seg_row<LEFT, ACH>(A, m, lane, row);
            if (A.at & 2) tot1 = seg_row<LEFT, TCH>(A, m, lane, row + 2 * A.wb);
        }
        __syncthreads();
        if (wid >= n) return;
    } else {
        W0 = (pw ? A.Wp : A.Wa) + ro;
        W1 = A.Wt + ro;
        if (!LEFT) {
            tot0 = A.ws[NW2 * (2 + 3 * (pw ? PCH : ACH)) + iW];
            if (!pw) tot1 = A.ws[NW2 * (2 + 3 * TCH) + iW];
        }
    }
    if (pw) {
        double2 s = czero();
        seg_term<LEFT, REF, PCH, !ROWS>(A, m, v, wl, wh, lane, [&](double2 x, int w) { s = cadd(s, cmul(x, W0[w])); });
        s = wave_sum2(s);
        if (!LEFT) s = cadd(s, cmul(seg_const<REF, PCH>(A, m, v), tot0));
        const double2 raw = cscale(s, A.T);
        for (int k = b + lane; k < e; k += WAVE) {
            const int code = sym.member(cls, k), o = code >> 2;
            const double2 x = sym_apply(code & 3, raw);
            A.Kp[o] = LEFT ? x : cadd(x, A.Lp[o]);
        }
        return;
    }
    double2 sa = czero(), st = czero(), sat = czero();   // Σ Xa Wa, Σ Xt Wt, Σ Xa Wt
    seg_term<LEFT, REF, ACH, !ROWS>(A, m, v, wl, wh, lane, [&](double2 x, int w) {
        sa = cadd(sa, cmul(x, W0[w]));
        sat = cadd(sat, cmul(x, W1[w]));
    });
    if (A.at & 2)
        seg_term<LEFT, REF, TCH, !ROWS>(A, m, v, wl, wh, lane, [&](double2 x, int w) { st = cadd(st, cmul(x, W1[w])); });
    double2 rawa = czero(), rawt = czero();
    const double2 ca = LEFT ? czero() : seg_const<REF, ACH>(A, m, v);
    if (A.at & 1) {
        sa = wave_sum2(sa);
        if (!LEFT) sa = cadd(sa, cmul(ca, tot0));
        rawa = cscale(sa, A.T);
    }
    if (A.at & 2) {
        double2 d = wave_sum2(csub(cscale(st, 2.0), sat));
        if (!LEFT)
            d = cadd(d, cmul(csub(cscale(seg_const<REF, TCH>(A, m, v), 2.0), ca), tot1));
        rawt = cscale(d, -A.T);
    }
    for (int k = b + lane; k < e; k += WAVE) {
        const int code = sym.member(cls, k), o = code >> 2;
        double2 ka;
        if (A.at & 1) {
            ka = sym_apply(code & 3, rawa);
            if (!LEFT) ka = cadd(ka, A.La[o]);
            A.Ka[o] = ka;
        } else {
            ka = A.Ka[o];
        }
        if (A.at & 2) {
            double2 kt = sym_apply(code & 3, rawt);
            if (!LEFT) kt = cadd(kt, csub(cscale(A.Lt[o], 2.0), A.La[o]));
            A.Kt[o] = cscale(cadd(kt, ka), 0.5);
        }
    }
}

// BSE_L_K2! of one channel point by point: Σ_ω Γ(Ω, ν, ω) Π0(ω) F0(Ω, ω~, ∞) over the window, Γ without F0 and the own
// channel (zero outside it).  One wave per output class, lanes over ω: all of a point's loads are in flight together,
// which for a call on its own is worth more than k_seg_k2's fewer instructions until these set the time.  p channel
// (the three channels), against k_seg_k2: SIAM boxes 33, 0.1 M points, 6.0 us (in one launch 7.0); boxes 60, 1.8 M,
// 12.5 (15.4) and 53.0 (58.8), with a reference vertex 13.7 (15.8) and 59.8 (61.2); boxes 128 with groups, 2.7 M, 16.0
// (16.4) and 62.6 (64.9), with a reference vertex 17.4 (17.2) and 70.6 (67.8); without groups, 8.4 M, 38.8 (35.2).
constexpr size_t LK2_POINTS = (size_t)2 << 20;   // the line between the two: even from there on
template <int CH>
__global__ __launch_bounds__(256) void k_point_lk2(double2* __restrict__ out, const double2* __restrict__ outa,
                                                   const double2* __restrict__ Pi0, VtxV F, int n2b, int n2f, int nWP,
                                                   int nVP, double scale, int NK, SymCls sym) {
    constexpr int SP = ChSpin<CH>::SP, FLG = FL_ALL & ~FL_F0 & ~(FL_GP << CH);
    const int wid = (int)blockIdx.x * (256 / WAVE) + seg_wave(), lane = threadIdx.x & (WAVE - 1);
    const int NW2 = 2 * n2b - 1;
    if (wid >= sym.count(NW2 * 2 * n2f)) return;
    const int o0 = sym.rep(wid), m = o0 % NW2 - (n2b - 1), v = o0 / NW2 - n2f, Wc = window(NK, m, v);
    const double2* P0 = Pi0 + (size_t)(2 * nVP) * (m + nWP - 1) + nVP;
    double2 s = czero();
    for (int w = max(-nVP, -Wc) + lane; w <= min(nVP - 1, Wc); w += WAVE)
        s = cadd(s, cmul(cmul(F.eval(m, v, w, 0, CH, SP, FLG), P0[w]), F.f0.eval(m, crossing(m, w, CH), FDGA_INF, CH, SP)));
    const double2 raw = cscale(wave_sum2(s), scale);
    int b, e;
    sym.range(wid, b, e);
    for (int k = b + lane; k < e; k += WAVE) {
        const int code = sym.member(wid, k), o = code >> 2;
        const double2 x = sym_apply(code & 3, raw);
        out[o] = CH == TCH ? cscale(cadd(x, outa[o]), 0.5) : x;
    }
}

// The SDE L-vertices of one Vertex level (src/SDE.jl:79-217), the channels at the fixed bosonic argument Ω:
//   Lpp(Ω, ν) = T U [(K1p + K2p(ν)) ΣΠpp + Σ_n K2p(n) Πpp(Ω - n - 1) + Σ_n K3p(n, ν) Πpp(Ω - n - 1)]
//   Lph(Ω, ν) = T U Σ_{r = a, t} [(K1r + K2r(ν)) ΣΠph + Σ_n K2r(n) Πph(n) + Σ_n K3r(ν, n) Πph(n)]
// One wave per class of SGpp[2] (waves [0, npp)) or of SGph[2], lanes over n.  SIAM boxes as above: 39 us (point by
// point over the window 92), with groups 17 (34).
struct SegSde {
    SegCh p, t, a;
    const double2 *Pp, *Ph, *Tp, *Th;
    double2 *Lpp, *Lph;
    double2 TU;
    int n2b, n2f, nWP, nVP;
    SymCls sp, sh;
    int npp, nph;
};
__device__ __forceinline__ double2 seg_sde_const(const SegCh& g, int m, int v) {
    double2 x = in_b(m, g.n1) ? g.K1[m + g.n1 - 1] : czero();
    if (in_b(m, g.n2b) && in_f(v, g.n2f)) x = cadd(x, g.K2[(size_t)(m + g.n2b - 1) + (size_t)(2 * g.n2b - 1) * (v + g.n2f)]);
    return x;
}
__global__ __launch_bounds__(256) void k_seg_sde(SegSde A) {
    const int wid = (int)blockIdx.x * (256 / WAVE) + seg_wave(), lane = threadIdx.x & (WAVE - 1);
    if (wid >= A.npp + A.nph) return;
    const bool pw = wid < A.npp;
    const SymCls& sym = pw ? A.sp : A.sh;
    const int cls = pw ? wid : wid - A.npp, o0 = sym.rep(cls);
    const int NW2 = 2 * A.n2b - 1, iW = o0 % NW2, iv = o0 / NW2, m = iW - (A.n2b - 1), v = iv - A.n2f;
    const size_t row = (size_t)(m + A.nWP - 1);
    const double2* Pi = (pw ? A.Pp : A.Ph) + (size_t)(2 * A.nVP) * row + A.nVP;
    const double2 tot = (pw ? A.Tp : A.Th)[3 * row + 2];
    double2 s = czero(), cst = czero();
    // Π at n (ph) or Ω - n - 1 (pp) on the mesh
    auto add = [&](double2 x, int n) { s = cadd(s, cmul(x, Pi[pw ? m - n - 1 : n])); };
    auto chan = [&](const SegCh& g) {
        cst = cadd(cst, seg_sde_const(g, m, v));
        const int l = pw ? m - A.nVP : -A.nVP, h = pw ? m + A.nVP - 1 : A.nVP - 1, NW = 2 * g.n2b - 1, N = 2 * g.n3f;
        if (in_b(m, g.n2b))
            seg_run(g.K2 + (m + g.n2b - 1) + (ptrdiff_t)NW * g.n2f, NW, max(l, -g.n2f), min(h, g.n2f - 1), lane, add);
        if (in_b(m, g.n3b) && in_f(v, g.n3f))
            seg_run(g.K3 + (ptrdiff_t)N * N * (m + g.n3b - 1) + (pw ? g.n3f + (ptrdiff_t)N * (v + g.n3f)
                                                                    : (v + g.n3f) + (ptrdiff_t)N * g.n3f),
                    pw ? 1 : N, max(l, -g.n3f), min(h, g.n3f - 1), lane, add);
    };
    if (pw) chan(A.p);
    else { chan(A.a); chan(A.t); }
    const double2 raw = cmul(cadd(wave_sum2(s), cmul(cst, tot)), A.TU);
    double2* L = pw ? A.Lpp : A.Lph;
    int b, e;
    sym.range(cls, b, e);
    for (int k = b + lane; k < e; k += WAVE) {
        const int code = sym.member(cls, k);
        L[code >> 2] = sym_apply(code & 3, raw);
    }
}

}  // namespace fdga
