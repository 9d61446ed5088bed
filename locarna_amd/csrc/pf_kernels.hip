// gfx950 kernels of LocARNA-P (sum-product DP in FP64): inside partition
// function, and its adjoint (reverse mode), which yields the outside values
// of every arc match, the arc-match and base-match probabilities and the
// expected number of gap openings.
//
// Reference: AlignerP, src/LocARNA/aligner_p.icc: inside :148-438;
// outside :450-1139; probabilities :1150-1399.  Here the outside values come
// from the adjoint of the inside recursion: Dbar(am) = dZ/dD(am), so that
// P(am) = D(am) Dbar(am) / Z (the reference's D D' pf_scale / (Z e^{s/T}));
// the base-match probability of (i, j) is the weight of alignments with a
// match edge into (i, j) directly inside an arc match with P(am) >
// sqrt(min_am_prob), or at the top level (aligner_p.icc:1201-1399), divided
// by Z.  The unrestricted match-edge weights and the gap-opening weight give
// the gradient of log Z with respect to the score parameters.
//
// Layout per group (origin al, bl; rows al..ar-1; bound br): rows stored from
// column max(bl, min_col(i)) with stride W, as in the integer kernel.  The
// scratch of a wave holds, for the group being processed, the matrices M,
// E, F and Mbar (doubles) plus E / Ebar vectors over the columns.
//
// Cell recurrence (inside), lane l owns column j of row i:
//   E(i,j) = E(i-1,j) gA (1 - o) + M(i-1,j) gA o
//   s(i,j) = M(i-1,j-1) es(i,j) + E(i,j) + ps * sum_arcs M(p-1,q-1) D
//   F(i,j) = F(i,j-1) gB + s(i,j-1) gB o              (s(i,jlo-1) = M(i,jlo-1))
// (the reference's F gB + (M(i,j-1) - F) gB o with M = s + F; the E chain
// keeps its (1 - o) since M(i-1,j) contains E(i-1,j))
//   M(i,j) = s(i,j) + F(i,j)
// The F chain is a linear recurrence along the row, solved by a wave scan
// of (multiplier, offset) pairs; its adjoint is the mirrored suffix scan.
#include <hip/hip_runtime.h>

#include "device_layout.h"
#include "member_barrier.h"
#include "pf_layout.h"

namespace {

__device__ __forceinline__ int lane_id() { return threadIdx.x & 63; }

// DPP move of a double (both halves): lane l receives the lane CTRL names;
// lanes without a source, and rows outside ROWMASK, receive `old`
template <int CTRL, int ROWMASK>
__device__ __forceinline__ double dpp_d(double old, double v) {
    const unsigned long long o = (unsigned long long)__double_as_longlong(old);
    const unsigned long long x = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_update_dpp((int)(unsigned)o, (int)(unsigned)x, CTRL, ROWMASK, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp((int)(unsigned)(o >> 32), (int)(unsigned)(x >> 32), CTRL, ROWMASK,
                                               0xf, false);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

__device__ __forceinline__ double readlane_d(double v, int l) {
    const unsigned long long x = (unsigned long long)__double_as_longlong(v);
    const int lo = __builtin_amdgcn_readlane((int)(unsigned)x, l);
    const int hi = __builtin_amdgcn_readlane((int)(unsigned)(x >> 32), l);
    return __longlong_as_double((long long)(((unsigned long long)(unsigned)hi << 32) | (unsigned)lo));
}

// one step of the prefix composition: (a, b) after the map from the source
// lane (identity where there is none)
template <int CTRL, int ROWMASK>
__device__ __forceinline__ void affine_step(double &a, double &b) {
    const double pa = dpp_d<CTRL, ROWMASK>(1.0, a), pb = dpp_d<CTRL, ROWMASK>(0.0, b);
    b = a * pb + b;
    a = a * pa;
}

// inclusive scan of the affine maps x -> a x + b over the lanes (lane 0
// first): result (A_l, B_l) with F_l = A_l F_in + B_l.  DPP row shifts
// within rows of 16, then row broadcasts of lanes 15 and 31.
__device__ __forceinline__ void wave_scan_affine(double &a, double &b) {
    affine_step<0x111, 0xf>(a, b);  // row_shr:1
    affine_step<0x112, 0xf>(a, b);  // row_shr:2
    affine_step<0x114, 0xf>(a, b);  // row_shr:4
    affine_step<0x118, 0xf>(a, b);  // row_shr:8
    affine_step<0x142, 0xa>(a, b);  // row_bcast:15 -> rows 1, 3
    affine_step<0x143, 0xc>(a, b);  // row_bcast:31 -> rows 2, 3
}

// suffix version: x_l = g_l + c_l x_{l+1} (last lane first); returns the
// pair (C_l, G_l) with x_l = C_l x_in + G_l where x_in enters at lane 63.
// DPP row shifts to the left within rows of 16; then each row is composed
// with the rows after it (their totals read from lanes 16, 32, 48).
__device__ __forceinline__ void wave_suffix_affine(double &c, double &g) {
    affine_step<0x101, 0xf>(c, g);  // row_shl:1
    affine_step<0x102, 0xf>(c, g);  // row_shl:2
    affine_step<0x104, 0xf>(c, g);  // row_shl:4
    affine_step<0x108, 0xf>(c, g);  // row_shl:8
    const double c1 = readlane_d(c, 16), g1 = readlane_d(g, 16);
    const double c2 = readlane_d(c, 32), g2 = readlane_d(g, 32);
    const double c3 = readlane_d(c, 48), g3 = readlane_d(g, 48);
    const double s1c = c2 * c3, s1g = c2 * g3 + g2;      // rows 2..3
    const double s0c = c1 * s1c, s0g = c1 * s1g + g1;    // rows 1..3
    const int row = lane_id() >> 4;
    const double sc = row == 0 ? s0c : row == 1 ? s1c : row == 2 ? c3 : 1.0;
    const double sg = row == 0 ? s0g : row == 1 ? s1g : row == 2 ? g3 : 0.0;
    g = c * sg + g;
    c = c * sc;
}

__device__ __forceinline__ double wave_sum(double v) {
    for (int o = 32; o >= 1; o >>= 1) v += __shfl_xor(v, o);
    return v;
}

struct PfPair {
    const int *mn, *mx, *coff, *codeA, *codeB;  // LDS
    const double *egA, *egB, *es;                // LDS: exp gap scores, 8x8 exp sigma
    const int *cptr;
    const int4 *cand;
    double *Dc;     // inside D per candidate entry
    double *Dbar;   // outside dZ/dD per candidate entry
    const double *eam;  // exp(s(am)/T) per candidate entry
    double *edge_full, *edge_ref;  // per band cell
    double eo, ps;
    int n, m;
    const int *fbp, *fbk;  // LDS: fill blocks of row i (left end p, first entry)
    const int *fcand;      // int arena: fill entries (p | q<<16, j | min_col(p-1)<<16)
    double *fD;            // inside D per fill entry
    double *fDb;           // outside dZ/dD per fill entry: the fixed-column kernels' part
    double *fq;            // fragment match queries (8 doubles each)
    int nfq;
};

// Fragment match queries (A[i..j] with B[k..l]): the reverse sweep of every
// region holding the cells (i-1, k-1) and (j, l) adds M(i-1, k-1) times the
// adjoint of the summand s(j, l) (the weight of every completion from (j,
// l), the block being a summand of s that is not part of E) to the query's
// out; the block's inside is a separate fill.  P = in out ps / Z.
__device__ __forceinline__ void frag_query(const PfPair &P, int q, int &i, int &j, int &k, int &l) {
    const double *x = P.fq + 8 * q;
    i = (int)x[0];
    j = (int)x[1];
    k = (int)x[2];
    l = (int)x[3];
}

__device__ __forceinline__ int row_lo(const PfPair &P, int i, int bl) { return max(bl, P.mn[i]); }
__device__ __forceinline__ int row_hi(const PfPair &P, int i, int br) { return min(br - 1, P.mx[i]); }

struct Region {
    int al, bl, ar, br, W;
    double *M, *E, *F, *Mb;  // matrices (R x W)
    double *Ev, *Eb;         // vectors over columns bl..br-1
    __device__ __forceinline__ double *at(double *X, const PfPair &P, int i, int j) const {
        const int lo = (i == al) ? bl : row_lo(P, i, bl);
        return X + (size_t)(i - al) * W + (j - lo);
    }
    __device__ __forceinline__ bool stored(const PfPair &P, int i, int j) const {
        if (i < al || i >= ar) return false;
        const int lo = (i == al) ? bl : row_lo(P, i, bl);
        return j >= lo && j <= row_hi(P, i, br);
    }
    __device__ __forceinline__ double get(double *X, const PfPair &P, int i, int j) const {
        return stored(P, i, j) ? *at(X, P, i, j) : 0.0;
    }
};

// Orders a workgroup's accesses to its global scratch and to the pair's
// arrays.  One workgroup owns a pair, its waves run on one CU and share that
// CU's vector L1 (write-through), so a workgroup-scope fence (wait for the
// outstanding accesses) suffices; an agent-scope fence would write back and
// invalidate the L2 on every call.
__device__ __forceinline__ void scratch_sync() { __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup"); }

// Inside fill of a region (aligner_p.icc:150-312).  Stores M, E, F.
__device__ void pf_fill(const PfPair &P, const Region &R) {
    const int lane = lane_id();
    const int al = R.al, bl = R.bl, ar = R.ar, br = R.br, W = R.W;
    const double eo = P.eo, ps = P.ps;
    for (int c = lane; c < br - bl; c += 64) R.Ev[c] = 0.0;
    // row al: M(al, bl) = 1/ps, M(al, j) = eo/ps prod gB
    const int hi0 = row_hi(P, al, br);
    {
        double carry = eo / ps;
        for (int j0 = bl + 1; j0 <= hi0; j0 += 64) {
            const int j = j0 + lane;
            const bool act = j <= hi0;
            double a = act ? P.egB[j] : 1.0, b = 0.0;
            wave_scan_affine(a, b);  // prefix products
            if (act) {
                R.M[j - bl] = carry * a;
                R.E[j - bl] = 0.0;
                R.F[j - bl] = 0.0;
            }
            carry *= readlane_d(a, 63);
        }
        if (lane == 0) {
            R.M[0] = 1.0 / ps;
            R.E[0] = 0.0;
            R.F[0] = 0.0;
        }
    }
    scratch_sync();
    double colv = eo / ps;
    bool colopen = true;
    for (int i = al + 1; i < ar; ++i) {
        const int mni = P.mn[i];
        if (colopen && mni <= bl) {
            colv *= P.egA[i];
        } else {
            colopen = false;
        }
        const int lo = max(bl, mni), hi = min(br - 1, P.mx[i]);
        double *row = R.M + (size_t)(i - al) * W;
        if (colopen && lane == 0) {
            row[0] = colv;
            R.E[(size_t)(i - al) * W] = 0.0;
            R.F[(size_t)(i - al) * W] = 0.0;
        }
        const int jlo = max(bl + 1, mni);
        double Fcarry = 0.0;
        double sprev = colopen ? colv : 0.0;  // M(i, jlo-1)
        const double gA = P.egA[i];
        const int cb = P.coff[i] - mni;
        for (int j0 = jlo; j0 <= hi; j0 += 64) {
            const int j = j0 + lane;
            const bool act = j <= hi;
            double s = 0.0, gB = 1.0, e = 0.0;
            if (act) {
                const double up = R.get(R.M, P, i - 1, j), dg = R.get(R.M, P, i - 1, j - 1);
                const double ep = R.Ev[j - bl];
                e = ep * gA + (up - ep) * gA * eo;
                R.Ev[j - bl] = e;
                s = dg * P.es[P.codeA[i] * LCG_NCODES + P.codeB[j]] + e;
                const int t0 = P.cptr[cb + j], t1 = P.cptr[cb + j + 1];
                double sa = 0.0;
                for (int t = t0; t < t1; ++t) {
                    const int4 en = P.cand[t];
                    const int p = en.x & 0xffff, q = en.x >> 16;
                    if (p <= al) break;
                    if (q <= bl) continue;
                    sa += R.get(R.M, P, p - 1, q - 1) * P.Dc[t];
                }
                s += sa * ps;
                gB = P.egB[j];
            }
            // F chain: F_j = F_{j-1} gB + s_{j-1} gB o
            double sl = dpp_d<0x138, 0xf>(s, s);  // lane l-1 (lane 0: its own)
            if (lane == 0) sl = sprev;
            double a = act ? gB : 1.0, b = act ? sl * gB * eo : 0.0;
            wave_scan_affine(a, b);
            const double F = a * Fcarry + b;
            if (act) {
                row[j - lo] = s + F;
                R.E[(size_t)(i - al) * W + (j - lo)] = e;
                R.F[(size_t)(i - al) * W + (j - lo)] = F;
            }
            Fcarry = readlane_d(F, 63);
            sprev = readlane_d(s, 63);
        }
        scratch_sync();
    }
}

// Adjoint of pf_fill for a region whose Mb holds the seeds.  Accumulates
// Dbar (per candidate entry), match-edge weights into `edge` (and into
// `edge2` when given) and the gap-opening weight.  Mb is consumed.
__device__ void pf_reverse(const PfPair &P, const Region &R, bool want_dbar, double *edge, double *openings,
                           double *edge2 = nullptr) {
    const int lane = lane_id();
    const int al = R.al, bl = R.bl, ar = R.ar, br = R.br, W = R.W;
    const double eo = P.eo, ps = P.ps;
    for (int c = lane; c < br - bl; c += 64) R.Eb[c] = 0.0;
    scratch_sync();
    double open_acc = 0.0;
    for (int i = ar - 1; i > al; --i) {
        const int mni = P.mn[i];
        const int lo = max(bl, mni), hi = min(br - 1, P.mx[i]);
        const int jlo = max(bl + 1, mni);
        const double gA = P.egA[i];
        const int cb = P.coff[i] - mni;
        const bool colopen_row = (mni <= bl);  // column bl stored for this row
        // columns of the region not computed in row i end their E chain
        for (int c = lane; c < br - bl; c += 64) {
            const int j = bl + c;
            if (j < jlo || j > hi) R.Eb[c] = 0.0;
        }
        if (jlo > hi) {
            scratch_sync();
            continue;
        }
        // chunks from the right: F adjoint flows right to left
        const int nch = (hi - jlo) / 64;
        double Fb_in = 0.0;        // Fbar of the column right of the chunk
        double a_in = 0.0;         // gB of that column
        for (int ch = nch; ch >= 0; --ch) {
            const int j0 = jlo + ch * 64;
            const int j = j0 + lane;
            const bool act = j <= hi;
            const size_t idx = act ? (size_t)(i - al) * W + (j - lo) : 0;
            const double g = act ? R.Mb[idx] : 0.0;
            const double gB = act ? P.egB[j] : 1.0;
            // Fbar_j = g_j + gB(j+1) Fbar_{j+1}
            double a_next = dpp_d<0x130, 0xf>(act ? gB : 0.0, act ? gB : 0.0);  // lane l+1
            if (lane == 63 || !(j + 1 <= hi)) a_next = (lane == 63) ? a_in : 0.0;
            double c = act ? a_next : 0.0, gg = act ? g : 0.0;
            wave_suffix_affine(c, gg);
            const double Fb = c * Fb_in + gg;  // Fbar_j
            // sbar_j = g_j + Fbar_{j+1} gB(j+1) o
            double Fb_next = dpp_d<0x130, 0xf>(Fb, Fb);
            double gB_next = dpp_d<0x130, 0xf>(gB, gB);
            if (lane == 63) {
                Fb_next = Fb_in;
                gB_next = a_in;
            }
            if (!(j + 1 <= hi) && lane != 63) {
                Fb_next = 0.0;
                gB_next = 0.0;
            }
            const double sb = g + Fb_next * gB_next * eo;
            if (act && want_dbar) {
                for (int q = 0; q < P.nfq; ++q) {
                    int fi, fj, fk, fl;
                    frag_query(P, q, fi, fj, fk, fl);
                    if (fj == i && fl == j && P.fq[8 * q + 4] > 0.0 && R.stored(P, fi - 1, fk - 1))
                        atomicAdd(&P.fq[8 * q + 6], sb * *R.at(R.M, P, fi - 1, fk - 1));
                }
            }
            if (act) {
                const double F = R.F[idx];
                // F_j = F_{j-1} gB (1-o) + s_{j-1} gB o ; opening part = F_j - F_{j-1} gB
                const double Fprev = (j > jlo) ? R.F[idx - 1] : 0.0;
                open_acc += Fb * (F - Fprev * gB);
                // boundary: F_jlo uses M(i, jlo-1)
                if (j == jlo) {
                    if (colopen_row) {
                        double *mcol = R.at(R.Mb, P, i, jlo - 1);
                        *mcol += Fb * gB * eo;
                    }
                }
                // s_j = M(i-1,j-1) es + E + ps sum arcs
                const double es = P.es[P.codeA[i] * LCG_NCODES + P.codeB[j]];
                if (R.stored(P, i - 1, j - 1)) {
                    const double dg = *R.at(R.M, P, i - 1, j - 1);
                    atomicAdd(R.at(R.Mb, P, i - 1, j - 1), sb * es);
                    atomicAdd(&edge[P.coff[i] + (j - mni)], sb * dg * es);
                    if (edge2) atomicAdd(&edge2[P.coff[i] + (j - mni)], sb * dg * es);
                }
                // E_j = Eprev gA (1-o) + M(i-1,j) gA o
                const double Eb = R.Eb[j - bl] + sb;
                const double E = R.E[idx];
                const double Eprev = R.stored(P, i - 1, j) && (i - 1 > al) ? *R.at(R.E, P, i - 1, j) : 0.0;
                if (R.stored(P, i - 1, j)) atomicAdd(R.at(R.Mb, P, i - 1, j), Eb * gA * eo);
                open_acc += Eb * (E - Eprev * gA);
                R.Eb[j - bl] = Eb * gA * (1.0 - eo);
                // arcs
                const int t0 = P.cptr[cb + j], t1 = P.cptr[cb + j + 1];
                for (int t = t0; t < t1; ++t) {
                    const int4 en = P.cand[t];
                    const int p = en.x & 0xffff, q = en.x >> 16;
                    if (p <= al) break;
                    if (q <= bl) continue;
                    const double Dv = P.Dc[t];
                    if (Dv == 0.0) continue;
                    // M(p-1, q-1) outside the band reads as 0 (aligner_p.icc:150-189 zeroes
                    // every such cell the recursion can reach)
                    if (!R.stored(P, p - 1, q - 1)) continue;
                    atomicAdd(R.at(R.Mb, P, p - 1, q - 1), sb * Dv * ps);
                    if (want_dbar) atomicAdd(&P.Dbar[t], sb * (*R.at(R.M, P, p - 1, q - 1)) * ps);
                }
            }
            Fb_in = readlane_d(Fb, 0);
            a_in = readlane_d(act ? gB : 0.0, 0);
        }
        scratch_sync();
    }
    // openings of the init row al and column bl (one each per cell value)
    const int hi0 = row_hi(P, al, br);
    for (int j = bl + 1 + lane; j <= hi0; j += 64) open_acc += R.Mb[j - bl] * R.M[j - bl];
    for (int i = al + 1 + lane; i < ar; i += 64) {
        if (P.mn[i] > bl) continue;
        bool open_col = true;
        for (int k = al + 1; k <= i; ++k)
            if (P.mn[k] > bl) open_col = false;
        if (open_col) open_acc += *R.at(R.Mb, P, i, bl) * *R.at(R.M, P, i, bl);
    }
    if (openings) {
        const double tot = wave_sum(open_acc);
        if (lane == 0) atomicAdd(openings, tot);  // waves of the workgroup share it
    }
}

// ---- fixed-column group kernels (columns bl+1 .. br-1 in NC chunks of 64
// lanes, the same column on the same lane in every row; rows al+1 .. ar-1).
// Region in LDS (doubles, lcg_pf_region): [M: (ar-al) W], rows stored from
// max(bl, min_col(i)) as in the general layout; after it S, the arc sums of four
// rows (4 (br-bl)), in the forward fill and Mbar ((ar-al) W) in the adjoint.
//
// Four rows are one block, rows al+r0 .. al+r0+3 (r0 a multiple of 4).  An
// arc (p, i) spans at least three positions, so an arc term of row i reads
// (the adjoint: adds to) row p - 1 <= i - 4, outside the block: the arc
// entries of the four rows are handled together, packed on the lanes, before
// the block's rows (the adjoint: after them), and the next block's are loaded
// meanwhile.  The arc candidates of row i are the fill-list prefix p > al
// (left ends descending), located from the LDS block table.
// Bound: LDS holds 5 to 10 regions of a workgroup, so every SIMD has one to
// three waves and the latency of a row's chain (LDS, scan, store) shows; a
// row at a time cost a trip to memory and five to LDS each.  120 pairs of 150
// nt, whole kernel, 105.3 -> 61.7 ms; 48 ragged pairs of 80-250 nt 170.7 ->
// 98.5 ms; one pair of 88 nt, a wave at a time, 11.4 -> 7.0 ms.
// lane l receives lane l-1's value, lane 0 `first` (DPP wave_shr:1)
__device__ __forceinline__ double shift_up_d(double v, double first) { return dpp_d<0x138, 0xf>(first, v); }

__device__ __forceinline__ void lds_fence() { __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront"); }

// Prefix scan x_l = b_l + a_l x_{l-1} whose multipliers are the same for all
// rows of a group: the products that each step needs are computed once, so
// that a step is one move and one multiply-add.  Returns the product a_0 .. a_l.
template <int CTRL, int ROWMASK>
__device__ __forceinline__ void coef_step(double &a, double &m) {
    m = a * dpp_d<CTRL, ROWMASK>(0.0, 1.0);  // 0 where the step has no source lane
    a *= dpp_d<CTRL, ROWMASK>(1.0, a);
}
__device__ __forceinline__ double scan_coef(double a, double (&m)[6]) {
    coef_step<0x111, 0xf>(a, m[0]);
    coef_step<0x112, 0xf>(a, m[1]);
    coef_step<0x114, 0xf>(a, m[2]);
    coef_step<0x118, 0xf>(a, m[3]);
    coef_step<0x142, 0xa>(a, m[4]);
    coef_step<0x143, 0xc>(a, m[5]);
    return a;
}
__device__ __forceinline__ double scan_lin(double b, const double (&m)[6]) {
    b = fma(m[0], dpp_d<0x111, 0xf>(0.0, b), b);
    b = fma(m[1], dpp_d<0x112, 0xf>(0.0, b), b);
    b = fma(m[2], dpp_d<0x114, 0xf>(0.0, b), b);
    b = fma(m[3], dpp_d<0x118, 0xf>(0.0, b), b);
    b = fma(m[4], dpp_d<0x142, 0xa>(0.0, b), b);
    return fma(m[5], dpp_d<0x143, 0xc>(0.0, b), b);
}

// Operands of rows al+rb .. al+rb+63, one per lane: band, gap weight, symbol,
// fill entries [t0, t1); mnu, mxu: the band of the row above.
struct PfRows {
    int mn, mx, mnu, mxu, code, co, t0, t1;
    double gA;
    __device__ __forceinline__ void load(const PfPair &P, int al, int bl, int ar, int br, int rb) {
        const int r = rb + lane_id(), i = min(al + r, ar - 1), u = max(i - 1, 0);
        mn = P.mn[i];
        mx = P.mx[i];
        mnu = P.mn[u];
        mxu = P.mx[u];
        code = P.codeA[i] * LCG_NCODES;
        co = P.coff[i];
        gA = P.egA[i];
        t0 = t1 = 0;
        if (r >= 1 && al + r < ar && max(bl + 1, mn) <= min(br - 1, mx)) {
            int b = P.fbp[i];
            const int be = P.fbp[i + 1];
            t0 = P.fbk[2 * b + 1];
            while (b < be && P.fbk[2 * b] > al) ++b;
            t1 = P.fbk[2 * b + 1];
        }
    }
};
__device__ __forceinline__ int rl(int v, int l) { return __builtin_amdgcn_readlane(v, l); }

// The fill entries of a block's rows packed on the lanes, 64 PF_Q at a time:
// entry, position in the fill list (-1: none) and the base that turns the
// right-end column j into an LDS index of its row.
#define PF_Q 4
__device__ __forceinline__ int pick4(int x, int p1, int p2, int p3, int a0, int a1, int a2, int a3) {
    const int lo = x < p1 ? a0 : a1, hi = x < p3 ? a2 : a3;
    return x < p2 ? lo : hi;
}
struct PfBlock {
    int o0, o1, o2, o3, p1, p2, p3, tot;  // fill entry minus packed index, packed starts, count
    int b0, b1, b2, b3;                   // column bases of the rows
    int pq[PF_Q], jm[PF_Q], tt[PF_Q], at[PF_Q];
    double D[PF_Q];
    __device__ __forceinline__ void rows(const PfRows &T, int r0) {
        const int x = r0 & 63;
        o0 = rl(T.t0, x);
        p1 = rl(T.t1, x) - o0;
        const int s1 = rl(T.t0, x + 1), s2 = rl(T.t0, x + 2), s3 = rl(T.t0, x + 3);
        p2 = p1 + rl(T.t1, x + 1) - s1;
        p3 = p2 + rl(T.t1, x + 2) - s2;
        tot = p3 + rl(T.t1, x + 3) - s3;
        o1 = s1 - p1;
        o2 = s2 - p2;
        o3 = s3 - p3;
    }
    __device__ __forceinline__ void load(const PfPair &P, int q, int x0) {
        const int x = x0 + lane_id();
        const int t = x < tot ? x + pick4(x, p1, p2, p3, o0, o1, o2, o3) : 0;
        at[q] = pick4(x, p1, p2, p3, b0, b1, b2, b3);
        struct PJ {
            int x, y;
        };
        const PJ pj = *reinterpret_cast<const PJ *>(P.fcand + 2 * t);
        pq[q] = pj.x;
        jm[q] = pj.y;
        D[q] = P.fD[t];
        tt[q] = x < tot ? t : -1;
    }
    // the first 64 PF_Q entries
    __device__ __forceinline__ void first(const PfPair &P) {
        if (tot > 0) {
            load(P, 0, 0);
            load(P, 1, 64);
        }
        if (tot > 128) {
            load(P, 2, 128);
            load(P, 3, 192);
        }
    }
    // fn(q0) handles entries q0 and q0 + 1, of all chunks
    template <class Fn>
    __device__ __forceinline__ void each(const PfPair &P, Fn fn) {
        if (tot > 0) fn(0);
        if (tot > 128) fn(2);
        for (int x = 64 * PF_Q; x < tot; x += 64 * PF_Q) {
#pragma unroll
            for (int q = 0; q < PF_Q; ++q) load(P, q, x + 64 * q);
            fn(0);
            fn(2);
        }
    }
};

// Inside fill of a group (aligner_p.icc:150-312), values as pf_fill: M.
template <int NC>
__device__ __forceinline__ void pf_fwd_fixed(const PfPair &P, int al, int bl, int ar, int br, int W, double *base) {
    const int lane = lane_id();
    const double eo = P.eo, ps = P.ps;
    const int SR = br - bl, nrows = ar - al - 1;
    double *Mst = base, *S = base + (ar - al) * W;
    for (int c = lane; c < 4 * SR; c += 64) S[c] = 0.0;
    PfRows T;
    T.load(P, al, bl, ar, br, 0);
    PfBlock B;
    auto block = [&](int r0) __attribute__((always_inline)) {
        B.rows(T, r0);
        B.first(P);
    };
    B.b0 = -bl - 1;
    B.b1 = B.b0 + SR;
    B.b2 = B.b1 + SR;
    B.b3 = B.b2 + SR;
    double Mp[NC], Ep[NC], cf[NC][6], ac[NC], gBo[NC];
    int cBc[NC];
    const int hi0 = min(br - 1, P.mx[al]);
    {
        double carry = eo / ps;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int j = bl + 1 + 64 * c + lane;
            const bool in = j <= hi0, col = j <= br - 1;
            const double g = col ? P.egB[j] : 1.0;
            gBo[c] = g * eo;
            cBc[c] = col ? P.codeB[j] : 0;
            ac[c] = scan_coef(g, cf[c]);
            Mp[c] = in ? carry * ac[c] : 0.0;
            if (in) Mst[j - bl] = Mp[c];
            carry *= readlane_d(ac[c], 63);
            Ep[c] = 0.0;
        }
        if (lane == 0) Mst[0] = 1.0 / ps;
    }
    block(0);
    lds_fence();
    double colv = eo / ps;
    bool colopen = true;
    double Mcol_prev = 1.0 / ps;  // M(i-1, bl)
    for (int r0 = 0; r0 <= nrows; r0 += 4) {
        // arc terms ps * M(p-1, q-1) * D of the four rows, LDS atomic adds
        B.each(P, [&](int q0) __attribute__((always_inline)) {
            double v[2];
            bool ok[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int pq = B.pq[q0 + h], jm = B.jm[q0 + h];
                const int p = pq & 0xffff, q = pq >> 16, j = jm & 0xffff, mc = max(bl, jm >> 16);
                ok[h] = B.tt[q0 + h] >= 0 && q > bl && j < br && q - 1 >= mc;
                v[h] = Mst[ok[h] ? (p - 1 - al) * W + (q - 1 - mc) : 0] * B.D[q0 + h] * ps;
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (ok[h]) atomicAdd(&S[B.at[q0 + h] + (B.jm[q0 + h] & 0xffff)], v[h]);
        });
        lds_fence();
        // the rows' operands, then the next block's entries
        double sv[4][NC], es[4][NC], gAk[4];
        int mnk[4], mxk[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int x = (r0 + k) & 63;
            mnk[k] = rl(T.mn, x);
            mxk[k] = rl(T.mx, x);
            gAk[k] = readlane_d(T.gA, x);
            const int code = rl(T.code, x);
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                double *sp = S + k * SR + min(64 * c + lane, SR - 1);
                sv[k][c] = *sp;
                *sp = 0.0;
                es[k][c] = P.es[code + cBc[c]];
            }
        }
        if (r0 + 4 <= nrows) {
            if (((r0 + 4) & 63) == 0) T.load(P, al, bl, ar, br, r0 + 4);
            block(r0 + 4);
        }
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int r = r0 + k;
            if (r > nrows) break;
            if (r == 0) continue;
            const int mni = mnk[k];
            const double gA = gAk[k];
            double Mcol = 0.0;  // M(i, bl)
            if (colopen && mni <= bl) {
                colv *= gA;
                Mcol = colv;
            } else {
                colopen = false;
            }
            const int lo = max(bl, mni), hi = min(br - 1, mxk[k]), jlo = max(bl + 1, mni);
            double *row = Mst + r * W;
            if (mni <= bl && lane == 0) row[0] = Mcol;
            double Fcarry = 0.0, sprev = Mcol, dgin = Mcol_prev;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int j0 = bl + 1 + 64 * c, j = j0 + lane;
                const double up = Mp[c];
                const double last = c + 1 < NC ? readlane_d(up, 63) : 0.0;
                // a chunk without a cell of the row
                if (NC > 1 && (j0 > hi || j0 + 63 < jlo)) {
                    Mp[c] = 0.0;
                    dgin = last;
                    Fcarry = 0.0;
                    sprev = 0.0;
                    continue;
                }
                const bool act = j >= jlo && j <= hi;
                const double dg = shift_up_d(up, dgin);
                dgin = last;
                const double ep = Ep[c];
                const double e = ep * gA + (up - ep) * gA * eo;
                Ep[c] = act ? e : ep;
                const double s = act ? dg * es[k][c] + e + sv[k][c] : 0.0;
                double F = scan_lin(shift_up_d(s, sprev) * gBo[c], cf[c]);
                if (c > 0) F = fma(ac[c], Fcarry, F);
                const double Mv = s + F;
                if (act) row[j - lo] = Mv;
                Mp[c] = act ? Mv : 0.0;
                if (c + 1 < NC) {
                    Fcarry = readlane_d(F, 63);
                    sprev = readlane_d(s, 63);
                }
            }
            Mcol_prev = Mcol;
        }
        lds_fence();
    }
}

// Adjoint of pf_fwd_fixed for a group whose Mbar rows (LDS, after M) hold the
// seeds.  FULL: also Dbar (dZ/dD per fill entry) and the gap-opening weight
// (returned); edge receives the match-edge weights.  Same terms as pf_reverse.
//
// The lanes hold the columns from the right (lane l of chunk c: br-1-64c-l),
// so that the F adjoint is a prefix scan.  Blocks run from row ar-1 down.
// Once a row is done no later row reads its Mbar, so each computed cell's
// Mbar is replaced by its sbar there for the arc terms.
//
// Openings: with s = M - F, the weight sum_j Fbar_j gB_j o s_{j-1} equals
// sum_j gB_j o M(i, j-1) U_j, U_j = Mbar_j + gB_{j+1} (1-o) U_{j+1} (F_j as a
// recurrence driven by M(i, j-1), summed by parts); alike for E with U over the
// rows and the adjoint of s without its vertical part.  Only positive terms,
// and of the forward values only M is needed.
template <int NC, bool FULL>
__device__ __forceinline__ double pf_rev_fixed(const PfPair &P, int al, int bl, int ar, int br, int W, double *base,
                               double *edge, double *edge2 = nullptr) {
    const int lane = lane_id();
    const double eo = P.eo, ec = 1.0 - P.eo, ps = P.ps;
    const double *Mst = base;
    double *Mb = base + (ar - al) * W;
    const int nrows = ar - al - 1;
    double cf[NC][6], ac[NC], uf[NC][6], au[NC], gBo[NC], gBn[NC];
    double cv[NC], cd[NC], Eb[NC], Ue[NC], left[NC];
    int cBc[NC];
    // first stored column of row i of the region (row al from bl)
    auto lo_of = [&](int i) { return (i == al) ? bl : max(bl, P.mn[i]); };
    const int rs = nrows & ~3;
    PfRows T;
    T.load(P, al, bl, ar, br, rs & ~63);
#pragma unroll
    for (int c = 0; c < NC; ++c) {
        const int j = br - 1 - 64 * c - lane;
        const bool col = j > bl;
        const double gn = col && j < br - 1 ? P.egB[j + 1] : 0.0;
        gBo[c] = (col ? P.egB[j] : 0.0) * eo;
        gBn[c] = gn * eo;
        cBc[c] = col ? P.codeB[j] : 0;
        // the first lane's multiplier belongs to the chunk on the right: it
        // enters with ac / au
        ac[c] = scan_coef(gn, cf[c]);
        if (FULL) au[c] = scan_coef(gn * ec, uf[c]);
        cv[c] = cd[c] = Eb[c] = Ue[c] = 0.0;
        // M(ar-1, j-1)
        const int lo = lo_of(ar - 1), x = j - 1 - lo;
        left[c] = (nrows > 0 && x >= 0 && j - 1 <= min(br - 1, P.mx[ar - 1])) ? Mst[nrows * W + min(x, W - 1)] : 0.0;
    }
    const int lc = (br - 2 - bl) >> 6, ll = (br - 2 - bl) & 63;  // chunk and lane of column bl+1
    double colcarry = 0.0;  // contribution of row i+1 to Mbar(i, bl)
    double open_acc = 0.0;
    PfBlock B;
    auto block = [&](int r0) __attribute__((always_inline)) {
        B.rows(T, r0);
        // Mbar index of column 0 of the block's rows
        B.b0 = r0 * W - (r0 == 0 ? bl : max(bl, rl(T.mn, r0 & 63)));
        B.b1 = (r0 + 1) * W - max(bl, rl(T.mn, (r0 + 1) & 63));
        B.b2 = (r0 + 2) * W - max(bl, rl(T.mn, (r0 + 2) & 63));
        B.b3 = (r0 + 3) * W - max(bl, rl(T.mn, (r0 + 3) & 63));
        B.first(P);
    };
    block(rs);
    lds_fence();
    for (int r0 = rs; r0 >= 0; r0 -= 4) {
        // operands of the four rows (NC 3: of each row in its turn, for the registers)
        double mb[4][NC], up[4][NC], dg[4][NC], es[4][NC], gAk[4];
        int mnk[4], mxk[4], mnu[4], mxu[4], cok[4];
        auto operands = [&](int k) __attribute__((always_inline)) {
            const int x = (r0 + k) & 63, r = min(r0 + k, nrows);
            mnk[k] = rl(T.mn, x);
            mxk[k] = rl(T.mx, x);
            mnu[k] = rl(T.mnu, x);
            mxu[k] = rl(T.mxu, x);
            cok[k] = rl(T.co, x);
            gAk[k] = readlane_d(T.gA, x);
            const int code = rl(T.code, x);
            const int lo = max(bl, mnk[k]), lou = r <= 1 ? bl : max(bl, mnu[k]);
            const int hiu = min(br - 1, mxu[k]), ru = max(r - 1, 0) * W;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int j = br - 1 - 64 * c - lane;
                mb[k][c] = Mb[r * W + min(max(j - lo, 0), W - 1)];
                const double u = Mst[ru + min(max(j - lou, 0), W - 1)];
                const double d = Mst[ru + min(max(j - 1 - lou, 0), W - 1)];
                up[k][c] = j >= lou && j <= hiu ? u : 0.0;
                dg[k][c] = j - 1 >= lou && j - 1 <= hiu ? d : 0.0;
                es[k][c] = P.es[code + cBc[c]];
            }
        };
        if (NC < 3)
#pragma unroll
            for (int k = 0; k < 4; ++k) operands(k);
#pragma unroll
        for (int k = 3; k >= 0; --k) {
            const int r = r0 + k;
            if (r > nrows || r == 0) continue;
            if (NC >= 3) operands(k);
            const int mni = mnk[k];
            const int lo = max(bl, mni), hi = min(br - 1, mxk[k]), jlo = max(bl + 1, mni);
            const bool colopen = mni <= bl;
            const int lou = r == 1 ? bl : max(bl, mnu[k]), hiu = min(br - 1, mxu[k]);
            double *rowB = Mb + r * W;
            const double gA = gAk[k], gAo = gA * eo, gAc = gA * ec;
            double Fb_in = 0.0, U_in = 0.0, d_in = 0.0, colb = 0.0, cnext = 0.0;
#pragma unroll
            for (int c = 0; c < NC; ++c) {
                const int j0 = br - 1 - 64 * c, j = j0 - lane;
                const bool here = !(NC > 1 && (j0 < jlo || j0 - 63 > hi));
                const bool upst = j >= lou && j <= hiu;
                double d = 0.0;
                if (here) {
                    const bool act = j >= jlo && j <= hi;
                    const double g0 = act ? mb[k][c] + cd[c] : 0.0;
                    const double gv = act ? cv[c] : 0.0;
                    const double g = g0 + gv;
                    double Fb = scan_lin(g, cf[c]);
                    if (c > 0) Fb = fma(ac[c], Fb_in, Fb);
                    const double Fb_next = shift_up_d(Fb, Fb_in);
                    const double sp = act ? fma(Fb_next, gBn[c], g0) : 0.0;  // sbar without the vertical part
                    const double sb = sp + gv;
                    if (act) rowB[j - lo] = sb;
                    const double eb = act ? sb + Eb[c] : 0.0;
                    if (FULL) {
                        double U = scan_lin(g, uf[c]);
                        if (c > 0) U = fma(au[c], U_in, U);
                        const double ue = act ? sp + Ue[c] : 0.0;
                        // left is 0 outside the stored row, U left of its cells is not used
                        open_acc += (act ? U * left[c] : 0.0) * gBo[c] + ue * up[k][c] * gAo;
                        Ue[c] = ue * gAc;
                        if (c + 1 < NC) U_in = readlane_d(U, 63);
                    }
                    Eb[c] = eb * gAc;
                    // match: s_j uses M(i-1, j-1) es
                    const bool dgst = act && j - 1 >= lou && j - 1 <= hiu;
                    d = dgst ? sb * es[k][c] : 0.0;  // to Mbar(i-1, j-1)
                    if (dgst) {  // match-edge weight sbar M(i-1, j-1) es
                        const double w = d * dg[k][c];
                        atomicAdd(&edge[cok[k] - mni + j], w);
                        if (edge2) atomicAdd(&edge2[cok[k] - mni + j], w);
                    }
                    cv[c] = upst ? eb * gAo : 0.0;
                    if (c == lc) {
                        // s_{j-1} = M(i, bl) of column bl + 1
                        if (jlo == bl + 1 && colopen && bl + 1 <= hi) colb = readlane_d(Fb * gBo[c], ll);
                        cnext = readlane_d(d, ll);
                    }
                    if (c + 1 < NC) Fb_in = readlane_d(Fb, 63);
                } else {
                    Eb[c] = Ue[c] = cv[c] = 0.0;
                    Fb_in = U_in = 0.0;
                }
                const double dr = shift_up_d(d, d_in);
                cd[c] = upst ? dr : 0.0;
                if (c + 1 < NC) d_in = readlane_d(d, 63);
                if (FULL) left[c] = dg[k][c];
            }
            // the init column cell (i, bl): one opening per value
            if (FULL && colopen && lane == 0) open_acc += (rowB[0] + colcarry + colb) * Mst[r * W];
            colcarry = (lou == bl) ? cnext : 0.0;
        }
        lds_fence();
        // arc terms: Mbar(p-1, q-1) += sbar D ps and (FULL) Dbar += sbar
        // M(p-1, q-1) ps of the fill entry
        B.each(P, [&](int q0) __attribute__((always_inline)) {
            double sb[2], mv[2];
            int x[2];
            bool ok[2];
#pragma unroll
            for (int h = 0; h < 2; ++h) {
                const int pq = B.pq[q0 + h], jm = B.jm[q0 + h];
                const int p = pq & 0xffff, q = pq >> 16, j = jm & 0xffff, mc = max(bl, jm >> 16);
                ok[h] = B.tt[q0 + h] >= 0 && q > bl && j < br && q - 1 >= mc && B.D[q0 + h] != 0.0;
                x[h] = ok[h] ? (p - 1 - al) * W + (q - 1 - mc) : 0;
                sb[h] = Mb[ok[h] ? B.at[q0 + h] + j : 0] * ps;
                if (FULL) mv[h] = Mst[x[h]];
            }
#pragma unroll
            for (int h = 0; h < 2; ++h)
                if (ok[h]) {
                    atomicAdd(&Mb[x[h]], sb[h] * B.D[q0 + h]);
                    if (FULL) atomicAdd(&P.fDb[B.tt[q0 + h]], sb[h] * mv[h]);
                }
        });
        if (r0 >= 4) {
            if ((r0 & 63) == 0) T.load(P, al, bl, ar, br, r0 - 64);
            block(r0 - 4);
        }
        lds_fence();
    }
    // init row al: one opening per value M(al, j), j > bl
    if (FULL) {
        const int hi0 = min(br - 1, P.mx[al]);
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            const int j = br - 1 - 64 * c - lane;
            if (j > bl && j <= hi0) open_acc += (Mb[j - bl] + cv[c] + cd[c]) * Mst[j - bl];
        }
    }
    // fragment queries: the computed cells hold sbar now (lanes over queries)
    if (FULL && P.nfq > 0) {
        lds_fence();
        for (int q = lane; q < P.nfq; q += 64) {
            int fi, fj, fk, fl;
            frag_query(P, q, fi, fj, fk, fl);
            if (!(P.fq[8 * q + 4] > 0.0) || fj <= al || fj >= ar || fi - 1 < al || fk - 1 < bl) continue;
            const int clo = lo_of(fi - 1), chi = min(br - 1, P.mx[fi - 1]);
            const int jlo = max(bl + 1, P.mn[fj]), jhi = min(br - 1, P.mx[fj]);
            if (fk - 1 < clo || fk - 1 > chi || fl < jlo || fl > jhi) continue;
            const double mv = Mst[(size_t)(fi - 1 - al) * W + (fk - 1 - clo)];
            const double sbv = Mb[(size_t)(fj - al) * W + (fl - lo_of(fj))];
            atomicAdd(&P.fq[8 * q + 6], mv * sbv);
        }
    }
    return wave_sum(open_acc);
}

__device__ __forceinline__ void zero_region_bar(const Region &R, const PfPair &P) {
    const int lane = lane_id();
    const size_t total = (size_t)(R.ar - R.al) * R.W;
    for (size_t c = lane; c < total; c += 64) R.Mb[c] = 0.0;
    scratch_sync();
}

}  // namespace

// One workgroup per pair (persistent, pairs from a queue).  Inside: rows
// al = n .. 1, the groups of a row in the host's LDS rounds; narrow groups
// (columns and rows at most 128) run the fixed-column kernels on LDS
// regions, others the general kernels on per-wave global scratch.  Top
// level (wave 0, global scratch): inside, full and restricted adjoint.
// Outside: rows al = 1 .. n, each group's forward values recomputed, then
// the full adjoint (Dbar, edge weights, openings) and, if any of its arc
// matches has P(am) > sqrt(min_am_prob), the restricted one.
#define LCG_PF_SPIN_LIMIT (1 << 22)

// The group of rows g0..g1-1 whose schedule word (S[4 g + slot]) is `want`,
// -1 if none: the lanes compare 64 words at a time (a wave holds at most
// one group per round).
__device__ __forceinline__ int find_group(const int *S, int slot, int g0, int g1, int want) {
    for (int gb = g0; gb < g1; gb += 64) {
        const int g = gb + lane_id();
        const unsigned long long hit = __ballot(g < g1 && S[4 * g + slot] == want);
        if (hit) return gb + __ffsll((long long)hit) - 1;
    }
    return -1;
}

extern "C" __global__ void __launch_bounds__(512) lcg_pf_pairs(const PairDesc *__restrict__ descs,
                                                                const PfDesc *__restrict__ pdescs,
                                                                const int *__restrict__ order, int *queue,
                                                                int *arena, double *pfa, double *scratch,
                                                                const int *__restrict__ sched, int *barriers,
                                                                double *fstore, PfBatchParams bp) {
    extern __shared__ int lds[];
    __shared__ int s_pair;
    __shared__ double s_open;
    const int nwaves = blockDim.x >> 6;
    const int wave = threadIdx.x >> 6;
    const int lane = lane_id();
    const int L = bp.max_len;
    int *mn = lds, *mx = lds + (L + 1), *coff = lds + 2 * (L + 1);
    int *codeA = lds + 3 * L + 4, *codeB = lds + 4 * L + 5;
    int *fbp = lds + 5 * L + 6, *fbk = lds + 6 * L + 8;
    double *dl = reinterpret_cast<double *>(lds + ((6 * L + 8 + 2 * bp.nfblk_max + 1) & ~1));
    double *egA = dl, *egB = dl + (L + 1), *es = dl + 2 * (L + 1);
    double *pool = es + LCG_NCODES * LCG_NCODES;
    double *wscr = scratch + (size_t)(blockIdx.x * nwaves + wave) * bp.scratch_stride;
    // The first nstatic pairs of the work order have workgroups (members) of
    // their own, all resident; the groups of a row are dealt to the members,
    // which meet at a barrier after every row (arrival counter per pair,
    // bounded wait).  The other workgroups take the remaining pairs from the
    // queue, one workgroup per pair.
    const bool stat = (int)blockIdx.x < bp.dealt;
    const int *deal = sched + bp.deal + 3 * (stat ? (int)blockIdx.x : 0);
    const int K = stat ? deal[2] : 1;
    const int member = stat ? deal[1] : 0;
    const int spin_lim = bp.spin_limit ? bp.spin_limit : LCG_PF_SPIN_LIMIT;
    for (int iter = 0;; ++iter) {
        if (stat) {
            if (iter > 0) break;
            if (threadIdx.x == 0) s_pair = deal[0];
        } else if (threadIdx.x == 0) {
            s_pair = bp.nstatic + atomicAdd(queue, 1);
        }
        __syncthreads();
        const int k = s_pair;
        if (k >= bp.npairs) break;
        const int pid = order[k];
        const PairDesc d = descs[pid];
        const PfDesc f = pdescs[pid];
        const int n = d.n, m = d.m;
        for (int t = threadIdx.x; t <= n; t += blockDim.x) {
            mn[t] = arena[d.band + t];
            mx[t] = arena[d.band + n + 1 + t];
            codeA[t] = arena[d.codes + t];
            egA[t] = pfa[f.egA + t];
        }
        for (int t = threadIdx.x; t <= m; t += blockDim.x) {
            codeB[t] = arena[d.codes + n + 1 + t];
            egB[t] = pfa[f.egB + t];
        }
        for (int t = threadIdx.x; t <= n + 1; t += blockDim.x) {
            coff[t] = arena[d.band + 2 * (n + 1) + t];
            fbp[t] = arena[d.fptr + t];
        }
        for (int t = threadIdx.x; t < 2 * d.nfblk; t += blockDim.x) fbk[t] = arena[d.fblk + t];
        for (int t = threadIdx.x; t < LCG_NCODES * LCG_NCODES; t += blockDim.x) es[t] = pfa[f.es + t];
        if (member == 0) {  // the pair's accumulators (then a barrier when K > 1)
            for (int t = threadIdx.x; t < d.nam; t += blockDim.x) {
                pfa[f.Dc + t] = 0.0;
                pfa[f.Dbar + t] = 0.0;
                pfa[f.fD + t] = 0.0;
                pfa[f.fDb + t] = 0.0;
            }
            for (int t = threadIdx.x; t < d.ncells; t += blockDim.x) {
                pfa[f.edge_full + t] = 0.0;
                pfa[f.edge_ref + t] = 0.0;
            }
            if (threadIdx.x == 0) {
                pfa[f.out + 1] = 0.0;  // gap openings (members add theirs)
                pfa[f.out + 2] = 0.0;  // status: 1 if a bounded wait expired
            }
        }
        if (threadIdx.x == 0) s_open = 0.0;
        int passed = 0;  // barrier generations passed
        // all members' global writes before any member goes on
        auto pair_barrier = [&]() {
            ++passed;
            member_barrier(&barriers[k], K * passed, spin_lim, [&]() { pfa[f.out + 2] = 1.0; });
        };
        PfPair P;
        P.mn = mn;
        P.mx = mx;
        P.coff = coff;
        P.codeA = codeA;
        P.codeB = codeB;
        P.egA = egA;
        P.egB = egB;
        P.es = es;
        P.cptr = arena + d.cptr;
        P.cand = reinterpret_cast<const int4 *>(arena + d.cand);
        P.Dc = pfa + f.Dc;
        P.Dbar = pfa + f.Dbar;
        P.eam = pfa + f.eam;
        P.edge_full = pfa + f.edge_full;
        P.edge_ref = pfa + f.edge_ref;
        P.eo = pfa[f.scal + 0];
        P.ps = pfa[f.scal + 1];
        P.n = n;
        P.m = m;
        P.fbp = fbp;
        P.fbk = fbk;
        P.fcand = arena + d.fcand;
        P.fD = pfa + f.fD;
        P.fDb = pfa + f.fDb;
        P.fq = pfa + f.frag;
        P.nfq = f.nfrag;
        if (K > 1) {
            pair_barrier();
        } else {
            scratch_sync();
            __syncthreads();
        }
        const int mine = member << 16;
        const int *rows = arena + d.rows;
        const int *groups = arena + d.groups;
        const int4 *gams = reinterpret_cast<const int4 *>(arena + d.gams);
        const int *S = sched + f.sched;
        auto region = [&](int al, int bl, int ar, int br, int W) {
            Region R;
            R.al = al;
            R.bl = bl;
            R.ar = ar;
            R.br = br;
            R.W = W;
            const size_t cells = (size_t)(ar - al) * W;
            R.M = wscr;
            R.E = wscr + cells;
            R.F = wscr + 2 * cells;
            R.Mb = wscr + 3 * cells;
            R.Ev = wscr + 4 * cells;
            R.Eb = R.Ev + (br - bl);
            return R;
        };
        // stored value of (i, j) in a fixed region (row al from bl)
        auto fixed_at = [&](int al, int bl, int br, int W, int i, int j) {
            const int lo = (i == al) ? bl : max(bl, P.mn[i]);
            const int hi = min(br - 1, P.mx[i]);
            return (j >= lo && j <= hi) ? (i - al) * W + (j - lo) : -1;
        };
        // ---- inside: rows al = n .. 1
        for (int al = n; al >= 1; --al) {
            const int g0 = rows[al + 1], g1 = rows[al];
            if (g0 == g1) continue;
            const int nr = sched[f.rin + al];
            for (int rnd = 0; rnd < nr; ++rnd) {
                const int g = find_group(S, 0, g0, g1, rnd | (wave << 12) | mine);
                if (g >= 0) {
                    const int *G = groups + g * LCG_GROUP_INTS;
                    const int gal = G[0] & 0xffff, gbl = G[0] >> 16, gar = G[1] & 0xffff, gbr = G[1] >> 16;
                    const int W = G[2];
                    const int off = S[4 * g + 1];
                    if (off >= 0) {
                        double *base = pool + off;
                        const int so = sched[f.fso + g];
                        const int cells = (gar - gal) * W;
                        if (gbr - gbl - 1 <= 64)
                            pf_fwd_fixed<1>(P, gal, gbl, gar, gbr, W, base);
                        else
                            pf_fwd_fixed<2>(P, gal, gbl, gar, gbr, W, base);
                        const double *Mst = base;
                        if (so >= 0) {  // M, which the outside pass reads
                            double *Ms = fstore + 4 * (size_t)so;
                            for (int c = lane; c < cells; c += 64) Ms[c] = Mst[c];
                        }
                        for (int t = G[3] + lane; t < G[4]; t += 64) {
                            const int4 ga = gams[t];
                            const int ar = ga.x & 0xffff, br = ga.x >> 16;
                            const int x = fixed_at(gal, gbl, gbr, W, ar - 1, br - 1);
                            const double v = (x >= 0 ? Mst[x] : 0.0) * P.eam[ga.y];
                            P.Dc[ga.y] = v;
                            P.fD[ga.w] = v;
                        }
                    } else {
                        const Region R = region(gal, gbl, gar, gbr, W);
                        pf_fill(P, R);
                        for (int t = G[3] + lane; t < G[4]; t += 64) {
                            const int4 ga = gams[t];
                            const int ar = ga.x & 0xffff, br = ga.x >> 16;
                            const double v = R.get(R.M, P, ar - 1, br - 1) * P.eam[ga.y];
                            P.Dc[ga.y] = v;
                            P.fD[ga.w] = v;
                        }
                    }
                }
                __threadfence_block();
                __syncthreads();
            }
            if (K > 1) pair_barrier();
        }
        // ---- top level and its adjoint (wave 0 of member 0)
        // (the restricted base-match weights count every top-level match edge,
        // aligner_p.icc:1201-1399: the seeds are the same, so one adjoint
        // sweep gives both)
        if (wave == 0 && member == 0) {
            const int W = d.wtop;
            const size_t cells = (size_t)(n + 1) * W;
            if (n <= 192 && m <= 192 && lcg_pf_region(cells, m + 1, 1) <= bp.pool) {
                // the whole LDS pool is free while the other waves wait
                double *base = pool;
                pf_fwd_fixed<3>(P, 0, 0, n + 1, m + 1, W, base);
                const int xz = fixed_at(0, 0, m + 1, W, n, m);
                double *Mst = base;
                const double Z = xz >= 0 ? Mst[xz] : 0.0;
                if (lane == 0) pfa[f.out + 0] = Z;
                double *Mb = Mst + cells;
                for (size_t c = lane; c < cells; c += 64) Mb[c] = 0.0;
                lds_fence();
                if (lane == 0 && xz >= 0) Mb[xz] = 1.0;
                lds_fence();  // the seed before the sweep
                const double o = pf_rev_fixed<3, true>(P, 0, 0, n + 1, m + 1, W, base, P.edge_full, P.edge_ref);
                if (lane == 0) atomicAdd(&s_open, o);
            } else {
                const Region R = region(0, 0, n + 1, m + 1, W);
                pf_fill(P, R);
                const double Z = *R.at(R.M, P, n, m);
                if (lane == 0) pfa[f.out + 0] = Z;
                zero_region_bar(R, P);
                if (lane == 0) *R.at(R.Mb, P, n, m) = 1.0;
                scratch_sync();
                pf_reverse(P, R, true, P.edge_full, &s_open, P.edge_ref);
            }
        }
        if (K > 1) {
            pair_barrier();
        } else {
            scratch_sync();
            __syncthreads();
        }
        const double Z = pfa[f.out + 0];
        const double thr = pfa[f.scal + 2];
        // dZ/dD of the arc match of a gams entry, complete before its row
        auto dbar = [&](const int4 &ga) { return P.Dbar[ga.y] + P.fDb[ga.w]; };
        // ---- outside over the groups, rows al = 1 .. n
        for (int al = 1; al <= n; ++al) {
            const int g0 = rows[al + 1], g1 = rows[al];
            if (g0 == g1) continue;
            const int nr = sched[f.rout + al];
            for (int rnd = 0; rnd < nr; ++rnd) {
                const int g = find_group(S, 2, g0, g1, rnd | (wave << 12) | mine);
                if (g >= 0) {
                    const int *G = groups + g * LCG_GROUP_INTS;
                    const int gal = G[0] & 0xffff, gbl = G[0] >> 16, gar = G[1] & 0xffff, gbr = G[1] >> 16;
                    const int W = G[2];
                    const int off = S[4 * g + 3];
                    bool any = false;
                    for (int t = G[3] + lane; t < G[4]; t += 64) {
                        const int4 ga = gams[t];
                        if (P.Dc[ga.y] * dbar(ga) / Z > thr) any = true;
                    }
                    const bool sig = __ballot(any) != 0;
                    if (off >= 0) {
                        double *base = pool + off;
                        const int cells = (gar - gal) * W;
                        double *Mst = base, *Mb = Mst + cells;
                        const bool nc1 = gbr - gbl - 1 <= 64;
                        const int so = sched[f.fso + g];
                        if (so >= 0) {
                            // the inside pass's M into the region
                            const double *Ms = fstore + 4 * (size_t)so;
                            int c = lane;
                            for (; c + 7 * 64 < cells; c += 8 * 64) {
                                double v[8];
#pragma unroll
                                for (int q = 0; q < 8; ++q) v[q] = Ms[c + 64 * q];
#pragma unroll
                                for (int q = 0; q < 8; ++q) Mst[c + 64 * q] = v[q];
                            }
                            for (; c < cells; c += 64) Mst[c] = Ms[c];
                            lds_fence();
                        } else if (nc1) {
                            pf_fwd_fixed<1>(P, gal, gbl, gar, gbr, W, base);
                        } else {
                            pf_fwd_fixed<2>(P, gal, gbl, gar, gbr, W, base);
                        }
                        for (int pass = 0; pass < (sig ? 2 : 1); ++pass) {
                            for (int c = lane; c < cells; c += 64) Mb[c] = 0.0;
                            lds_fence();
                            for (int t = G[3] + lane; t < G[4]; t += 64) {
                                const int4 ga = gams[t];
                                if (pass == 1 && !(P.Dc[ga.y] * dbar(ga) / Z > thr)) continue;
                                const int ar = ga.x & 0xffff, br = ga.x >> 16;
                                const int x = fixed_at(gal, gbl, gbr, W, ar - 1, br - 1);
                                if (x >= 0) atomicAdd(&Mb[x], dbar(ga) * P.eam[ga.y]);
                            }
                            lds_fence();  // the seeds before the sweep
                            if (pass == 0) {
                                const double o = nc1 ? pf_rev_fixed<1, true>(P, gal, gbl, gar, gbr, W, base, P.edge_full)
                                                     : pf_rev_fixed<2, true>(P, gal, gbl, gar, gbr, W, base, P.edge_full);
                                if (lane == 0) atomicAdd(&s_open, o);
                            } else {
                                if (nc1)
                                    pf_rev_fixed<1, false>(P, gal, gbl, gar, gbr, W, base, P.edge_ref);
                                else
                                    pf_rev_fixed<2, false>(P, gal, gbl, gar, gbr, W, base, P.edge_ref);
                            }
                        }
                    } else {
                        const Region R = region(gal, gbl, gar, gbr, W);
                        pf_fill(P, R);
                        zero_region_bar(R, P);
                        for (int t = G[3] + lane; t < G[4]; t += 64) {
                            const int4 ga = gams[t];
                            const int ar = ga.x & 0xffff, br = ga.x >> 16;
                            if (R.stored(P, ar - 1, br - 1))
                                atomicAdd(R.at(R.Mb, P, ar - 1, br - 1), dbar(ga) * P.eam[ga.y]);
                        }
                        scratch_sync();
                        pf_reverse(P, R, true, P.edge_full, &s_open);
                        if (sig) {
                            zero_region_bar(R, P);
                            for (int t = G[3] + lane; t < G[4]; t += 64) {
                                const int4 ga = gams[t];
                                const int ar = ga.x & 0xffff, br = ga.x >> 16;
                                if (P.Dc[ga.y] * dbar(ga) / Z > thr && R.stored(P, ar - 1, br - 1))
                                    atomicAdd(R.at(R.Mb, P, ar - 1, br - 1), dbar(ga) * P.eam[ga.y]);
                            }
                            scratch_sync();
                            pf_reverse(P, R, false, P.edge_ref, nullptr);
                        }
                    }
                }
                scratch_sync();
                __syncthreads();
            }
            if (K > 1) pair_barrier();
        }
        for (int t = member * blockDim.x + threadIdx.x; t < d.nam; t += K * blockDim.x) {
            const int4 ga = gams[t];
            P.Dbar[ga.y] += P.fDb[ga.w];
        }
        // fragment queries: the inside of each block (the virtual arc match
        // (i-1, j+1; k-1, l+1), AlignerP::compute_fragment_match_prob,
        // aligner_p.icc:1440-1479), one wave per query in its global scratch
        for (int q = member * nwaves + wave; q < P.nfq; q += K * nwaves) {
            int fi, fj, fk, fl;
            frag_query(P, q, fi, fj, fk, fl);
            const int Wq = (int)P.fq[8 * q + 4];
            if (Wq <= 0) continue;
            const Region R = region(fi - 1, fk - 1, fj + 1, fl + 1, Wq);
            pf_fill(P, R);
            if (lane == 0) P.fq[8 * q + 5] = R.get(R.M, P, fj, fl);
        }
        if (threadIdx.x == 0) {
            if (K > 1)
                atomicAdd(&pfa[f.out + 1], s_open);
            else
                pfa[f.out + 1] = s_open;
        }
        __syncthreads();
    }
}

extern "C" __global__ void lcg_pf_reset_barriers(int *barriers, int n) {
    for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < n; t += gridDim.x * blockDim.x) barriers[t] = 0;
}

extern "C" __global__ void lcg_pf_reset_queue(int *queue) {
    if (threadIdx.x == 0) *queue = 0;
}

extern "C" int lcg_launch_pf(const PairDesc *descs, const PfDesc *pdescs, const int *order, int *queue, int *arena,
                             double *pfa, double *scratch, const int *sched, int *barriers, double *fstore,
                             PfBatchParams bp, int grid, int waves, size_t lds_bytes, hipStream_t stream) {
    static bool attr_set = false;
    if (!attr_set) {
        hipError_t e = hipFuncSetAttribute((const void *)lcg_pf_pairs, hipFuncAttributeMaxDynamicSharedMemorySize,
                                           160 * 1024 - 256);
        if (e != hipSuccess) return (int)e;
        attr_set = true;
    }
    hipLaunchKernelGGL(lcg_pf_reset_queue, dim3(1), dim3(64), 0, stream, queue);
    if (bp.dealt > 0)
        hipLaunchKernelGGL(lcg_pf_reset_barriers, dim3(1), dim3(256), 0, stream, barriers, bp.npairs);
    hipLaunchKernelGGL(lcg_pf_pairs, dim3(grid), dim3(waves * 64), lds_bytes, stream, descs, pdescs, order, queue,
                       arena, pfa, scratch, sched, barriers, fstore, bp);
    return (int)hipGetLastError();
}
