// fdga_bse3.h -- BSE_L_K3! and BSE_K3! of the lattice fdPA iteration in one kernel for gfx950.
//
// Per (Ω, P) and channel r (N = Nν3, all matrices N x N at one Ω and momentum P):
//   FL = T sL Γr · (Π0 F0r)                                     (src/BSEa/BSEa_K3.jl:1-41, src/BSE_templates.jl:116-145)
//   R  = s1 [(Π - Π0) F0r + Π Γ~] + s2 Π L~ 1(ω~ in box)        (src/BSEa/BSEa_K3.jl:43-128)
//   K3 = T A · R + FL_self,  A = Fbase + K2r + K3r              (src/BSE_templates.jl:151-180)
// with t in the density component (2 t - a) and its post-processing (t + a) / 2 after both equations.
// Everything that L~, FL_self and the t combinations read belongs to the same (Ω, P), so one workgroup
// takes the left equation's result through R to the full equation without leaving the chip: F.K3 is read
// once, FL.K3 and Fbuff.K3 are written once, and neither the right operand R nor the summed left operand
// A exists in memory.
#pragma once
#include "fdga_kernels.h"

namespace fdga {

// one channel's arrays (F.K3, FL.K3 and Fbuff.K3 FP32 in the FP32 form, FP64 in the FP64 form)
struct Bse3Chan {
    const double2* G;      // Γr [ν, ω, Ω]
    const double2* F0r;    // [ω, νp, Ω]
    const double2* Gam;    // p: Γpx [ω, νp, Ω]; a, t: Γr transposed [ω, ν, Ω]
    const double2* Fbase;  // [ν, ω, Ω]
    const double2* Pi;     // Πpp or Πph
    const double2* Pi0;
    const double2* K2r;    // F.K2 [Ω, ν, P]
    const void* K3r;       // F.K3 [ν, νp, Ω, P]
    void* FL;              // FL.K3
    void* out;             // Fbuff.K3
};
struct Bse3Args {
    K3Geom g;
    double T;
    Bse3Chan p, a, t;
};

template <bool F32> struct Bse3Type { typedef double S; typedef double2 V; };
template <> struct Bse3Type<true> { typedef float S; typedef float2 V; };
template <class V>
__device__ __forceinline__ V b3_round(double2 v) { V r; r.x = v.x; r.y = v.y; return r; }
template <class V>
__device__ __forceinline__ double2 b3_wide(V v) { return cmk(v.x, v.y); }

// LDS layout of the right operand: element (k, n) at k LD + (n ^ f(k)).  The MFMA fragments read 16
// consecutive n at four consecutive k, the accumulator layout writes 16 consecutive k at columns four
// apart; the swizzle f (of the low four bits of n) and the row length spread both over all 64 banks (FP32:
// 8-byte elements, half a wave at a time; FP64: 16-byte elements, a quarter).  NT = 6 keeps the unpadded
// rows, so that two workgroups fit a CU (two-way conflicts on its reads).
template <bool F32, int NT>
struct Bse3Lds {
    static constexpr int LD = 16 * NT + ((F32 && NT % 2 == 0 && NT < 6) ? 16 : 0);
    __device__ __forceinline__ static int f(int k) { return F32 ? ((k >> 1) & 3) | (k & 8) : k & 15; }
};

// element at a uniform position plus the lane's 32-bit offset (one scalar base, one vector offset)
template <class V>
__device__ __forceinline__ V b3_ld(const V* base, unsigned lane) {
    return *reinterpret_cast<const V*>(reinterpret_cast<const char*>(base) + lane * (unsigned)sizeof(V));
}
template <class V>
__device__ __forceinline__ void b3_st(V* base, unsigned lane, V v) {
    *reinterpret_cast<V*>(reinterpret_cast<char*>(base) + lane * (unsigned)sizeof(V)) = v;
}

// A workgroup takes one (Ω, P) through channel p, or through a and then t (whose post-processing reads the
// finished a, written by the same threads).  Wave w computes the rows 16 w .. 16 w + 15 of both products, all
// 16 NT columns, so a left operand's element is needed by one wave only: Γr, Fbase (L2: they do not depend
// on P) and F.K3 go from global memory into the wave's MFMA fragments, FD steps ahead of their use, and
// the LDS holds nothing but the right operand (Π0 F0r, then R).  That leaves room for two or three
// independent workgroups per CU, whose MFMAs cover each other's operand formation, epilogues and barriers.
// At most four waves per workgroup, one per SIMD (the fifth wave of a workgroup lands on the first one's
// SIMD, and a second such workgroup then no longer fits the CU): for NT > 4 the tiles of the row tiles 4 and
// 5 are dealt out to the four waves, NE each (NT = 5: 5 tiles, two for one wave; NT = 6: 12 tiles, three each).
// EXACT: N = 16 NT (no bounds checks).
// Three waves per SIMD (168 registers) where the accumulators leave room (FP32, NT <= 4), else two.  FD = 2
// measured against 4 (the same up to 6 % slower: more registers) and 1 (N = 64: 2 % slower).  KEEP holds the
// channel's FL for its self term between the products instead of reading it back (FP64 N = 64: 2.03 -> 1.91
// ms); not where it would spill (FP32 N = 72: 2.50 -> 2.63 ms).
// Measured alone, 31 Ω x 256 P: FP32 N = 64 1.26 ms (79 TFLOP/s, matrix cores busy 56 % of the time; 4.0 GB of
// traffic beyond L2), N = 72 2.50 ms, N = 80 2.33 ms (84 TFLOP/s), N = 96 3.94 ms (86); FP64 N = 64 1.91 ms
// (52 TFLOP/s; up to 2.07 on other cards).  The separate equations took, at N = 64, 2.07 ms in FP32 (left equation
// 0.72, summed left operand 0.37, full equation 0.97) and 4.2 ms in FP64.  What is left to the matrix rate is latency: a
// workgroup's phases are separated by four barriers per channel.
template <bool F32, int NT, bool EXACT>
__global__ __launch_bounds__(64 * (NT < 4 ? NT : 4), F32 && NT <= 4 ? 3 : 2) void k_bse3(Bse3Args A) {
    typedef MfmaT<F32> MT;
    typedef typename MT::Acc Acc;
    typedef typename Bse3Type<F32>::V V;
    typedef Bse3Lds<F32, NT> LY;
    constexpr bool KEEP = !F32 || NT <= (EXACT ? 5 : 3);
    constexpr int LD = LY::LD, FD = 2, NTH = 64 * (NT < 4 ? NT : 4);
    constexpr int NE = NT == 5 ? 2 : NT == 6 ? 3 : 0;   // extra tiles of a wave (row tiles 4 and 5)
    constexpr int NX = NE > 0 ? NE : 1;
    constexpr int CS = F32 ? 4 : 1, RS = F32 ? 1 : 4;   // accumulator column in a tile: CS (lane / 16) + RS r
    static_assert(NT >= 1 && NT <= 6, "at most two row tiles are dealt out to the four waves");
    __shared__ V Bs[16 * NT * LD];
    const K3Geom g = A.g;
    int N = EXACT ? 16 * NT : g.NV();
    const int NW = g.NW(), NP = g.NP, n3f = g.n3f;
    const int lane = threadIdx.x & 63, c16 = lane & 15, q4 = lane >> 4;
    const int wave = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    if (!EXACT) {   // rows of the right operand beyond the box stay zero
        for (int e = threadIdx.x; e < (16 * NT - N) * LD; e += NTH) Bs[N * LD + e] = V{0, 0};
    }
    // the wave's extra tiles: row tile and columns (NT = 5: the wave with two turns with the workgroup)
    const int rot = (wave + (int)(blockIdx.x >> 3)) & 3;
    const int xrow = NT == 6 ? 4 + (wave >> 1) : 4;
    auto xcol = [&](int e) { return NT == 6 ? 3 * (wave & 1) + e : e ? 4 : rot; };
    const int nx = NT == 6 ? 3 : NT == 5 ? (rot == 0 ? 2 : 1) : 0;
    const int nn = N * N;
    // work items: the (Ω, P) pairs in contiguous ranges per XCD (workgroups go round-robin to the 8 XCDs),
    // momentum fastest, so that one XCD's workgroups share a few Ω and their momentum-independent operands
    // in its L2; the a/t items, twice as long, before the p items
    const int M = NW * NP, perx = (M + 7) / 8;
    for (int i = (int)(blockIdx.x / 8); i < 2 * perx; i += (int)(gridDim.x / 8)) {
        const bool pitem = i >= perx;
        const int u = (int)(blockIdx.x % 8) * perx + (pitem ? i - perx : i);
        if (u >= M) continue;
        const int iW = u / NP, P = u - iW * NP, m = iW - (g.n3b - 1);
        const size_t off = (size_t)nn * ((size_t)iW + (size_t)NW * P);
        const size_t pr = g.pidx(m, -n3f, P);
        auto channel = [&](auto tc, int s) {   // 0 p, 1 a, 2 t
            constexpr bool t = decltype(tc)::value;
            const Bse3Chan& c = s == 0 ? A.p : s == 1 ? A.a : A.t;
            const double sg = s == 1 ? 1.0 : -1.0, s2 = t ? -1.0 : 1.0;   // src/BSE_templates.jl:122-138,156-172
            const double2* G = c.G + (size_t)nn * iW;
            const double2* F0r = c.F0r + (size_t)nn * iW;
            const double2* Gam = c.Gam + (size_t)nn * iW;
            const double2* Fb = c.Fbase + (size_t)nn * iW;
            const V* K3 = static_cast<const V*>(c.K3r) + off;
            const V* K3a = static_cast<const V*>(A.a.K3r) + off;
            V* FL = static_cast<V*>(c.FL) + off;
            V* out = static_cast<V*>(c.out) + off;
            const V* FLa = static_cast<const V*>(A.a.FL) + off;
            const V* outa = static_cast<const V*>(A.a.out) + off;
            if (!EXACT) asm volatile("" : "+s"(N));
            // a lane's row of one row tile.  krow: the R row that reads FL's row, its crossing Ω - ω - 1 for p
            // (an involution of the box rows; a row whose crossing leaves the box is its own R row, without an
            // L~ term).  The 32-bit offsets are opaque to the compiler, so that addresses are formed where they
            // are used instead of being held in registers through both products.
            struct Row {
                int rowc, krow;
                bool rin, hasL;
                unsigned oK, oR, oA;   // offsets: accumulator layout at krow and at the row, left fragments
                int lw[4];             // LDS position of accumulator element r at krow
            };
            auto make_row = [&](int tile) {
                Row w;
                const int row = 16 * tile + c16;
                w.rin = EXACT || row < N;
                w.rowc = EXACT ? row : min(row, N - 1);
                const int wc = m - (w.rowc - n3f) - 1;
                w.hasL = s != 0 || in_f(wc, n3f);
                w.krow = (s == 0 && w.hasL) ? wc + n3f : w.rowc;
                w.oK = (unsigned)(w.krow + N * CS * q4);
                w.oR = (unsigned)(w.rowc + N * CS * q4);
                w.oA = (unsigned)(w.rowc + N * q4);
                asm volatile("" : "+v"(w.oK), "+v"(w.oR), "+v"(w.oA));
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    w.lw[r] = w.krow * LD + ((CS * q4 + RS * r) ^ LY::f(w.krow));
                    asm volatile("" : "+v"(w.lw[r]));
                }
                return w;
            };
            const Row w0 = make_row(wave), w1 = make_row(NE ? xrow : wave);
            int lr[4];   // LDS position of the right fragment of step st (st % 4)
#pragma unroll
            for (int q = 0; q < 4; ++q) {
                lr[q] = (4 * q + q4) * LD + (c16 ^ LY::f(4 * q + q4));
                asm volatile("" : "+v"(lr[q]));
            }
            // column 16 j + ... (accumulator layout) and k = 4 st + lane / 16 inside the box (N > 16 (NT - 1))
            auto cin = [&](int j, int r) { return EXACT || j + 1 < NT || 16 * j + CS * q4 + RS * r < N; };
            auto kin = [&](int st) { return EXACT || st < 4 * (NT - 1) || 4 * st + q4 < N; };
            // left fragments of FD steps: Γr, or Fbase with F.K3
            double2 ra[FD], xa[NE ? FD : 1];
            V rk[FD], rka[t ? FD : 1], xk[NE ? FD : 1], xka[NE && t ? FD : 1];
            auto fetchG = [&](int st) {
#pragma unroll
                for (int v = 0; v < FD; ++v) {
                    const int o = N * 4 * (st + v);
                    ra[v] = kin(st + v) ? b3_ld(G + o, w0.oA) : czero();
                    if constexpr (NE > 0) xa[v] = kin(st + v) ? b3_ld(G + o, w1.oA) : czero();
                }
            };
            auto fetchA = [&](int st) {
#pragma unroll
                for (int v = 0; v < FD; ++v) {
                    const int o = N * 4 * (st + v);
                    const bool in = kin(st + v);
                    ra[v] = in ? b3_ld(Fb + o, w0.oA) : czero();
                    rk[v] = in ? b3_ld(K3 + o, w0.oA) : V{0, 0};
                    if constexpr (t) rka[v] = in ? b3_ld(K3a + o, w0.oA) : V{0, 0};
                    if constexpr (NE > 0) {
                        xa[v] = in ? b3_ld(Fb + o, w1.oA) : czero();
                        xk[v] = in ? b3_ld(K3 + o, w1.oA) : V{0, 0};
                        if constexpr (t) xka[v] = in ? b3_ld(K3a + o, w1.oA) : V{0, 0};
                    }
                }
            };
            auto leftA = [&](int st, double2 fb, V k3, V k3a, double2 kr) {
                double2 v = b3_wide(k3);
                if constexpr (t) v = csub(cscale(v, 2.0), b3_wide(k3a));
                v = cadd(cadd(fb, v), kr);
                return kin(st) ? b3_round<V>(v) : V{0, 0};
            };
            fetchG(0);
            __syncthreads();   // the right operand's last readers are done
            auto stageB = [&](const Row& w, double2 P0, int j) {
                double2 f0[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) f0[r] = cin(j, r) ? b3_ld(F0r + N * (16 * j + RS * r), w.oK) : czero();
#pragma unroll
                for (int r = 0; r < 4; ++r)
                    if (EXACT || (w.rin && cin(j, r))) Bs[w.lw[r] + 16 * j] = b3_round<V>(cmul(P0, f0[r]));
            };
            {
                const double2 P0 = c.Pi0[pr + w0.krow];
#pragma unroll
                for (int j = 0; j < NT; ++j) stageB(w0, P0, j);
                if constexpr (NE > 0) {
                    const double2 P0x = c.Pi0[pr + w1.krow];
#pragma unroll
                    for (int e = 0; e < NE; ++e)
                        if (e < nx) stageB(w1, P0x, xcol(e));
                }
            }
            __syncthreads();
            Acc xr[NT], xi[NT], zr[NX], zi[NX];
            auto clear = [&]() {
#pragma unroll
                for (int j = 0; j < NT; ++j) xr[j] = xi[j] = Acc{0, 0, 0, 0};
#pragma unroll
                for (int e = 0; e < NE; ++e) zr[e] = zi[e] = Acc{0, 0, 0, 0};
            };
            // one 4-deep step of the product: the accumulators are transposed tiles (lane % 16 runs along the
            // rows), as in zgemm_tiles_t
            auto step = [&](V a, V ax, int st) {
                const int o = 16 * (st >> 2) * LD;
                V b[NT];
#pragma unroll
                for (int j = 0; j < NT; ++j) b[j] = Bs[lr[st & 3] + o + 16 * j];
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    xr[j] = MT::mfma(b[j].x, a.x, xr[j]);
                    xi[j] = MT::mfma(b[j].y, a.x, xi[j]);
                }
#pragma unroll
                for (int j = 0; j < NT; ++j) {
                    xr[j] = MT::mfma(b[j].y, -a.y, xr[j]);
                    xi[j] = MT::mfma(b[j].x, a.y, xi[j]);
                }
#pragma unroll
                for (int e = 0; e < NE; ++e)
                    if (NT == 6 || e < nx) {
                        const V bx = Bs[lr[st & 3] + o + 16 * xcol(e)];
                        zr[e] = MT::mfma(bx.x, ax.x, zr[e]);
                        zi[e] = MT::mfma(bx.y, ax.x, zi[e]);
                        zr[e] = MT::mfma(bx.y, -ax.y, zr[e]);
                        zi[e] = MT::mfma(bx.x, ax.y, zi[e]);
                    }
            };
            clear();
#pragma unroll
            for (int st = 0; st < 4 * NT; st += FD) {
                V a[FD], ax[FD];
#pragma unroll
                for (int v = 0; v < FD; ++v) {
                    a[v] = b3_round<V>(ra[v]);
                    ax[v] = NE ? b3_round<V>(xa[NE ? v : 0]) : a[v];
                }
                if (st + FD < 4 * NT) fetchG(st + FD);
                else fetchA(0);
#pragma unroll
                for (int v = 0; v < FD; ++v)
                    if (EXACT || st + v < 4 * (NT - 1) || 4 * (st + v) < N) step(a[v], ax[v], st + v);
            }
            __syncthreads();   // the product's reads of Π0 F0r are done
            // FL = T sL X and R = s1 [(Π - Π0) F0r + Π Γ~] + s2 T sL Π X (t: X is 2 FLt - FLa), per tile
            struct Pis { double2 d, p, l; };
            auto pis = [&](const Row& w) {
                const double2 P1 = c.Pi[pr + w.krow], P0 = c.Pi0[pr + w.krow];
                return Pis{cscale(csub(P1, P0), sg), cscale(P1, sg), cscale(P1, s2 * A.T * sg)};
            };
            V kp[KEEP ? NT : 1][4], kx[KEEP ? NX : 1][4];   // the channel's FL, for its self term
            auto epiL = [&](const Row& w, const Pis& q, int j, const Acc& ar, const Acc& ai, V* keep) {
                double2 f0[4], gm[4];
                V fa[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int o = N * (16 * j + RS * r);
                    const bool in = cin(j, r);
                    f0[r] = in ? b3_ld(F0r + o, w.oK) : czero();
                    gm[r] = in ? b3_ld(Gam + o, w.oK) : czero();
                    if constexpr (t) fa[r] = in ? b3_ld(FLa + o, w.oR) : V{0, 0};
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const double2 v = cmk((double)ar[r], (double)ai[r]);
                    const double2 vl = w.hasL ? v : czero();
                    double2 R = cmul(q.d, f0[r]), x = cscale(v, A.T * sg);
                    R = cadd(R, cmul(q.p, gm[r]));
                    R = cadd(R, cmul(q.l, vl));
                    if constexpr (t) x = cscale(cadd(x, b3_wide(fa[r])), 0.5);
                    if (EXACT || (w.rin && cin(j, r))) {
                        Bs[w.lw[r] + 16 * j] = b3_round<V>(R);
                        b3_st(FL + N * (16 * j + RS * r), w.oR, b3_round<V>(x));
                    }
                    if constexpr (KEEP) keep[r] = b3_round<V>(x);
                }
            };
            {
                const Pis q = pis(w0);
#pragma unroll
                for (int j = 0; j < NT; ++j) epiL(w0, q, j, xr[j], xi[j], kp[KEEP ? j : 0]);
                if constexpr (NE > 0) {
                    const Pis qx = pis(w1);
#pragma unroll
                    for (int e = 0; e < NE; ++e)
                        if (e < nx) epiL(w1, qx, xcol(e), zr[e], zi[e], kx[KEEP ? e : 0]);
                }
            }
            auto k2row = [&](const Row& w) {
                const size_t k2 = (size_t)(m + g.n2b - 1) +
                                  (size_t)(2 * g.n2b - 1) * ((size_t)(w.rowc - n3f + g.n2f) + (size_t)(2 * g.n2f) * P);
                double2 v = c.K2r[k2];
                if constexpr (t) v = csub(cscale(v, 2.0), A.a.K2r[k2]);
                return v;
            };
            const double2 kr = k2row(w0), krx = NE ? k2row(w1) : czero();
            __syncthreads();
            clear();
#pragma unroll
            for (int st = 0; st < 4 * NT; st += FD) {
                V a[FD], ax[FD];
#pragma unroll
                for (int v = 0; v < FD; ++v) {
                    a[v] = leftA(st + v, ra[v], rk[v], rka[t ? v : 0], kr);
                    ax[v] = NE ? leftA(st + v, xa[NE ? v : 0], xk[NE ? v : 0], xka[NE && t ? v : 0], krx) : a[v];
                }
                if (st + FD < 4 * NT) fetchA(st + FD);
#pragma unroll
                for (int v = 0; v < FD; ++v)
                    if (EXACT || st + v < 4 * (NT - 1) || 4 * (st + v) < N) step(a[v], ax[v], st + v);
            }
            auto epiK = [&](const Row& w, int j, const Acc& ar, const Acc& ai, const V* keep) {
                V l[4], la[4], oa[4];
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    const int o = N * (16 * j + RS * r);
                    const bool in = cin(j, r);
                    if constexpr (KEEP) l[r] = keep[r];
                    else l[r] = in ? b3_ld<V>(FL + o, w.oR) : V{0, 0};
                    if constexpr (t) {
                        la[r] = in ? b3_ld(FLa + o, w.oR) : V{0, 0};
                        oa[r] = in ? b3_ld(outa + o, w.oR) : V{0, 0};
                    }
                }
#pragma unroll
                for (int r = 0; r < 4; ++r) {
                    double2 self = b3_wide(l[r]);
                    if constexpr (t) self = csub(cscale(self, 2.0), b3_wide(la[r]));
                    double2 x = cadd(cscale(cmk((double)ar[r], (double)ai[r]), A.T), self);
                    if constexpr (t) x = cscale(cadd(x, b3_wide(oa[r])), 0.5);
                    if (EXACT || (w.rin && cin(j, r))) b3_st(out + N * (16 * j + RS * r), w.oR, b3_round<V>(x));
                }
            };
#pragma unroll
            for (int j = 0; j < NT; ++j) epiK(w0, j, xr[j], xi[j], kp[KEEP ? j : 0]);
#pragma unroll
            for (int e = 0; e < NE; ++e)
                if (e < nx) epiK(w1, xcol(e), zr[e], zi[e], kx[KEEP ? e : 0]);
        };
        channel(std::false_type{}, pitem ? 0 : 1);
        if (!pitem) channel(std::true_type{}, 2);
    }
}

// the largest Nν3 of the kernel: FP32 96 (72 KB of LDS, two workgroups per CU), FP64 64 (64 KB, two)
inline int bse3_max(bool f32) { return f32 ? 96 : 64; }

template <bool F32, int NT>
inline void bse3_go(const Bse3Args& a, unsigned grid, hipStream_t st) {
    if (2 * a.g.n3f == 16 * NT) k_bse3<F32, NT, true><<<grid, 64 * (NT < 4 ? NT : 4), 0, st>>>(a);
    else k_bse3<F32, NT, false><<<grid, 64 * (NT < 4 ? NT : 4), 0, st>>>(a);
}
// grid: workgroups (a multiple of 8; 0: one per work item)
template <bool F32>
inline hipError_t bse3_launch(const Bse3Args& a, size_t grid, hipStream_t st) {
    const int N = 2 * a.g.n3f;
    const size_t items = (size_t)(2 * a.g.n3b - 1) * a.g.NP, full = 16 * ((items + 7) / 8);
    const unsigned nb = (unsigned)(grid ? (grid < full ? grid : full) : full);
    switch ((N + 15) / 16) {
    case 1: bse3_go<F32, 1>(a, nb, st); break;
    case 2: bse3_go<F32, 2>(a, nb, st); break;
    case 3: bse3_go<F32, 3>(a, nb, st); break;
    case 4: bse3_go<F32, 4>(a, nb, st); break;
    case 5: if constexpr (F32) bse3_go<F32, 5>(a, nb, st); break;
    case 6: if constexpr (F32) bse3_go<F32, 6>(a, nb, st); break;
    default: return hipErrorInvalidValue;
    }
    return hipGetLastError();
}

}  // namespace fdga
