// Base-pair probabilities of single sequences (McCaskill's inside and
// outside algorithm) over the energy model of fold_model.h: the input step
// that mlocarna runs once per sequence (locarna_rnafold_pp ->
// RnaEnsemble, rna_ensemble.cc:141-193; mlocarna:3148-3188).
//
// Recursions (1-based, t = pair type of (i, j), 0 when (i, j) cannot pair):
//   Qb(i,j)  = H(i,j) + sum_{k,l} L(i,j,k,l) Qb(k,l) + MLC TP(t) M2(i+1,j-1)
//   Qm1(i,j) = s Qm1(i,j-1) + Qb(i,j) BR(t)
//   M2(i,j)  = sum_u Qm(i,u-1) Qm1(u,j)
//   Y(i,j)   = Qm1(i,j) + s Y(i+1,j),  Qm(i,j) = Y(i,j) + M2(i,j)
//   Z5(j)    = s Z5(j-1) + sum_k Z5(k-1) Qb(k,j) EXT(k,j),  Z = Z5(n)
// and outside, the pull form of the adjoints (b marks them; every cell is
// written once and the result does not depend on the schedule):
//   X(a,e)    = Qmb(a,e) + MLC TP Qbb(a-1,e+1)
//   Qmb(a,e)  = sum_j X(a,j) Qm1(e+1,j)
//   U(a,e)    = Qmb(a,e) + s U(a-1,e)
//   Qm1b(a,e) = sum_i X(i,e) Qm(i,a-1) + U(a,e)
//   R(a,e)    = Qm1b(a,e) + s R(a,e+1)
//   Qbb(a,e)  = Z5b(e) Z5(a-1) EXT + sum_{i,j} L(i,j,a,e) Qbb(i,j)
//               + BR (s R(a,e+1) + Qm1b(a,e))
// so that besides the interior loops one sum over the splits is left inside
// and two outside.  P = Qb Qbb / Z, P2(i,j) = Qbb(i,j) stack Qb(i+1,j-1) / Z.
// Every value of a segment of L bases is stored times sigma^-L (sigma per
// sequence, FoldDesc.log_sigma; ViennaRNA's per-nucleotide pf_scale), so
// each term carries sigma^-(bases it adds): s = sigma^-1 per unpaired base,
// sigma^-(l1 + l2 + 2) on an interior loop.  The probabilities do not depend
// on sigma; log Z = log Z5(n) + n log sigma.
//
// A loop's factor is the product of one for (l1, l2) and one for each of its
// pairs (weak or not), except for stacks and one-base bulges.  Qb is also
// stored times the inner pair's factor, so that a term of an interior loop is
// one load and one multiply-add with a factor that is the same for all cells.
#include <hip/hip_runtime.h>

#include <type_traits>

#include "fold_layout.h"
#include "member_barrier.h"

namespace {

constexpr int MAXLOOP = LCG_FOLD_MAXLOOP;

__device__ __forceinline__ int weak(int t) { return (0x72 >> t) & 1; }
__device__ __forceinline__ double readlane_d(double v, int l) {
    const long long x = __double_as_longlong(v);
    const unsigned lo = __builtin_amdgcn_readlane((int)x, l), hi = __builtin_amdgcn_readlane((int)(x >> 32), l);
    return __longlong_as_double(((long long)hi << 32) | lo);
}

struct Seq {
    const signed char *cs;  // codes in LDS, position i at cs[i]
    const int *ptab;        // pair type of (code a, code b) at a * 5 + b
    // pair type of (i, i + d), 0 if none
    __device__ __forceinline__ int pt(int i, int j) const { return ptab[cs[i] * 5 + cs[j]]; }
};

// The loop terms of a wave of NWV, one per lane: the first 64 / NWV lanes
// bulges of two bases and more, then interior loops, by loop size within each
// kind.  Wave w has every NWV-th of the 58 bulges and 435 interior loops.
struct Terms {
    int s, l1;     // unpaired bases (99: none), those of the 5' side
    double f;      // factor with two strong pairs, times sigma^-(s + 2)
};

template <int NWV>
__device__ __forceinline__ Terms wave_terms(int w, int lane, const double *tabs, double log_sigma) {
    Terms t{99, 0, 0.0};
    int l2 = 0;
    constexpr int NBU = 64 / NWV;
    if (lane < NBU) {
        const int e = w + NWV * lane;
        if (e < 2 * (MAXLOOP - 1)) {
            t.s = 2 + e / 2;
            t.l1 = (e & 1) ? t.s : 0;
        }
    } else {
        int x = w + NWV * (lane - NBU), s = 2;
        while (s <= MAXLOOP && x >= s - 1) x -= s - 1, ++s;
        if (s <= MAXLOOP) {
            t.s = s;
            t.l1 = 1 + x;
        }
    }
    if (t.s < 99) {
        l2 = t.s - t.l1;
        t.f = tabs[LCG_FOLD_TAB_LOOP + t.l1 * (MAXLOOP + 1) + l2] * exp(-(double)(t.s + 2) * log_sigma);
    }
    return t;
}

}  // namespace

// K workgroups fold a sequence, each the batches of 64 NCH cells of a
// diagonal that are its own.  The lanes of a wave are the cells of a chunk of
// 64; the waves of the workgroup split the terms of their sums (every NWV-th
// each), so that a load is 64 neighbours, many are in flight, and no lane
// waits for another; the partial sums meet in LDS, one wave per chunk adds
// them up and finishes its cells.  The interior loops are summed for the
// cells that can pair only (3 of 8 on random sequences), listed by a wave
// that has no chunk to finish.
// Bound: the chain of a diagonal, 6-10 us: of about 20,000 cycles with a clock
// in it (75 nt) the split sums take 3,500 (inside) to 6,600, the loops 5,000,
// the barrier behind them 3,500, the wave that adds up the parts and finishes
// the cells 5,000 to 6,300; with several workgroups 7 us more for the barrier
// between them.  Against a
// quarter wave per cell with gathered terms and five more sums over the
// splits: 64 sequences of 60-200 nt, span 100, 5.53 -> 2.45 ms; two of
// 700-800 nt without a limit 300 -> 26.8 ms; one of 75 nt 1.21 -> 1.10 ms.
// IN_LDS (short sequences, 8 waves): the matrices are in LDS, and both split sums
// of the outside pass have a part of their own (two barriers fewer).  One
// sequence of 20, 30, 40 and 50 nt 0.082, 0.160, 0.252 and 0.357 ms; in global
// memory with 16 waves 0.162, 0.306, 0.466 and 0.625 (the quarter wave per cell
// 0.082, 0.200, 0.375 and 0.597), in LDS with 16 waves 0.114, 0.213 and 0.319.
template <int NCH, int NWV, bool IN_LDS>
__device__ __forceinline__ void fold_seq(const FoldDesc &D, int member, const signed char *codes, const double *tabs,
                                         double *mats, double *outs, double *zout, int *counter, int *status,
                                         int polls, double *lds) {
    constexpr int NB = 64 * NCH;  // cells per batch
    constexpr int NP = IN_LDS ? 4 : 3, FT = 64 * NWV, NBU = 64 / NWV;
    const int n = D.n, W = D.W, S = IN_LDS ? n + 2 : D.S, K = NCH == 1 && !IN_LDS ? D.K : 1;
    double *part = lds + (IN_LDS ? lcg_fold_matrix_doubles(n, W) : 0);  // [sum][wave][cell]: M2 or Qmb, bulges,
                                                                        // interior loops, (NP 4) Qm1b
    double *T = part + NP * NWV * NB;      // factor table from the stacks on
    double *Z5 = T + (LCG_FOLD_TAB_HP - LCG_FOLD_TAB_STACK), *Z5b = Z5 + (n + 1);  // n + 1 each
    int *ptab = (int *)(Z5b + (n + 1));    // 25
    unsigned short *list = (unsigned short *)(ptab + 28);  // two buffers of NB: cells that can pair
    unsigned short *place = list + 2 * NB;                 // two buffers of NB: their places in the list
    int *count = (int *)(place + 2 * NB);                  // two buffers
    signed char *cs = (signed char *)(count + 2);          // n + 2
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    auto tab = [&](int x) { return T[x - LCG_FOLD_TAB_STACK]; };

    for (int x = tid; x < LCG_FOLD_TAB_HP - LCG_FOLD_TAB_STACK; x += FT) T[x] = tabs[LCG_FOLD_TAB_STACK + x];
    for (int x = tid; x < n + 2; x += FT) cs[x] = (x >= 1 && x <= n) ? codes[D.codes + x] : (signed char)4;
    if (tid < 25) {
        // canonical pairs AU, CG, GC, UA, GU, UG as types 1..6
        const int a = tid / 5, b = tid % 5;
        int t = 0;
        if (a == 0 && b == 3) t = 1;
        else if (a == 1 && b == 2) t = 2;
        else if (a == 2 && b == 1) t = 3;
        else if (a == 3 && b == 0) t = 4;
        else if (a == 2 && b == 3) t = 5;
        else if (a == 3 && b == 2) t = 6;
        ptab[tid] = t;
    }
    const Seq Q{cs, ptab};
    const Terms tm = wave_terms<NWV>(wave, lane, tabs, D.log_sigma);
    // place of a term's cell from the cell (i, d) inside and outside
    const int off_in = tm.s < 99 ? -(2 + tm.s) * S + 1 + tm.l1 : 0, off_out = -off_in;
    const double s1 = exp(-D.log_sigma), s2 = s1 * s1, s3 = s2 * s1;
    const size_t sz = (size_t)W * S;
    double *Qb = IN_LDS ? lds : mats + D.mat, *QI = Qb + sz, *QU = QI + sz, *Qm = QU + sz, *Qm1 = Qm + sz, *X = Qm1 + sz;
    double *ring = X + sz;
    double *M2 = ring, *Y = ring + 3 * (size_t)S;  // inside: 3 and 2 diagonals
    double *U = ring + 5 * (size_t)S, *R = ring + 7 * (size_t)S, *Qbb = ring + 9 * (size_t)S;  // outside: 2, 2, 4
    const size_t osz = (size_t)(n + 2) * W;
    double *P = outs + D.out, *P2 = P + osz;
    const double *hp = tabs + LCG_FOLD_TAB_HP;
    int passed = 0, buf = 0;
    if (IN_LDS)
        for (int x = tid; x < (int)lcg_fold_matrix_doubles(n, W); x += FT) lds[x] = 0.0;
    __syncthreads();

    // the cells of batch b of diagonal d that can pair, into a list buffer
    auto make_list = [&](int d, int b, int to) {
        int c = 0;
#pragma unroll
        for (int h = 0; h < NCH; ++h) {
            const int i = b * NB + 64 * h + lane + 1;
            const bool ok = d >= 4 && d < W && i + d <= n && Q.pt(i, i + d) != 0;
            const unsigned long long m = __ballot(ok);
            const int at = c + __popcll(m & ((1ull << lane) - 1));
            if (ok) {
                list[to * NB + at] = (unsigned short)(64 * h + lane);
                place[to * NB + 64 * h + lane] = (unsigned short)at;
            }
            c += __popcll(m);
        }
        if (lane == 0) count[to] = c;
    };
    // end of a diagonal: every workgroup's cells are written before any
    // workgroup reads them
    auto diagonal_done = [&]() {
        if (K > 1) {
            ++passed;
            member_barrier(counter, K * passed, polls, [&]() { atomicExch(status, 2); });
        } else {
            __threadfence_block();
            __syncthreads();
        }
    };
    // sums over the loop terms for the listed cells of batch b: term q of
    // cell i at band[off(q) + i], off by lane
    auto loops = [&](int b, int lim, const double *band_u, const double *band_i, int off) {
        const int c = count[buf];
        const unsigned long long in = __ballot(tm.s <= lim);
        const int nu = __popcll(in & ((1 << NBU) - 1)), ni = __popcll(in >> NBU);
        for (int h = 0; 64 * h < c; ++h) {
            const int x = 64 * h + lane;
            const unsigned i = b * NB + list[buf * NB + (x < c ? x : 0)] + 1;
            // terms [q0, q0 + N) of the wave with their loads in flight
            // together; those past q1 (the terms go by loop size, the limit
            // cuts a tail) load the last one's cell and count nothing
            auto terms = [&](auto nt, const double *band, int q0, int q1, double acc) {
                constexpr int N = decltype(nt)::value;
                double v[N];
#pragma unroll
                for (int u = 0; u < N; ++u)
                    v[u] = (band + __builtin_amdgcn_readlane(off, min(q0 + u, q1 - 1)))[i];
#pragma unroll
                for (int u = 0; u < N; ++u) acc = fma(v[u], q0 + u < q1 ? readlane_d(tm.f, q0 + u) : 0.0, acc);
                return acc;
            };
            double au = 0, ai = 0;
            for (int q = 0; q < nu; q += 4) au = terms(std::integral_constant<int, 4>(), band_u, q, nu, au);
            for (int q = NBU; q < NBU + ni; q += 14)
                ai = terms(std::integral_constant<int, 14>(), band_i, q, NBU + ni, ai);
            part[(NWV + wave) * NB + x] = au;
            part[(2 * NWV + wave) * NB + x] = ai;
        }
    };
    auto total = [&](int sum, int x) {
        double v = 0;
#pragma unroll
        for (int w = 0; w < NWV; ++w) v += part[(sum * NWV + w) * NB + x];
        return v;
    };

    const int nbatch = (n + NB - 1) / NB;
    // ---------------- inside
    if (wave == 0) make_list(4, member, 0);
    __syncthreads();
    for (int d = 4; d < W; ++d) {
        const double hs = D.log_sigma == 0 ? 1.0 : exp(-(double)(d + 1) * D.log_sigma);
        const double hs0 = hp[(d - 1) * 2] * hs, hs1 = hp[(d - 1) * 2 + 1] * hs;  // loaded ahead of the cells
        for (int b = member; b < nbatch && b * NB < n - d; b += K) {
            // partial sums
            double m2[NCH];
#pragma unroll
            for (int h = 0; h < NCH; ++h) m2[h] = 0;
#pragma unroll 4
            for (int a = 4 + wave; a <= d - 5; a += NWV) {
                const double *x = Qm + (size_t)a * S + b * NB + 1 + lane;
                const double *y = Qm1 + (size_t)(d - 1 - a) * S + b * NB + 1 + lane + a + 1;
#pragma unroll
                for (int h = 0; h < NCH; ++h) m2[h] += x[64 * h] * y[64 * h];
            }
#pragma unroll
            for (int h = 0; h < NCH; ++h) part[wave * NB + 64 * h + lane] = m2[h];
            loops(b, min(MAXLOOP, d - 6), QU + (size_t)d * S, QI + (size_t)d * S, off_in);
            __syncthreads();
            // finish the cells; the next batch's list
            const int nb = b + K < nbatch && (b + K) * NB < n - d ? b + K : member;
            if (wave == NWV - 1) make_list(nb == member ? d + 1 : d, nb, buf ^ 1);
            for (int h = wave; h < NCH; h += NWV - 1) {
                const int c = 64 * h + lane, i = b * NB + c + 1, j = i + d;
                if (wave == NWV - 1 || j > n) break;
                const size_t x = (size_t)d * S + i;
                const int t = Q.pt(i, j);
                const double q1p = Qm1[x - S], yp = d > 4 ? Y[(size_t)((d - 1) & 1) * S + i + 1] : 0.0;
                double qb = 0;
                if (t) {
                    const int wk = weak(t), at = place[buf * NB + c];
                    // the bulges and interior loops, stacks and one-base bulges
                    double l = total(1, at) * tab(LCG_FOLD_TAB_GU + wk) + total(2, at) * tab(LCG_FOLD_TAB_GI + wk);
                    if (d >= 6) l += tab(LCG_FOLD_TAB_STACK + t * 8 + Q.pt(i + 1, j - 1)) * s2 * Qb[x - 2 * S + 1];
                    if (d >= 7)
                        l += s3 * (tab(LCG_FOLD_TAB_BULGE1 + t * 8 + Q.pt(i + 1, j - 2)) * Qb[x - 3 * S + 1] +
                                   tab(LCG_FOLD_TAB_BULGE1 + t * 8 + Q.pt(i + 2, j - 1)) * Qb[x - 3 * S + 2]);
                    const double mq = d > 5 ? M2[(size_t)((d - 2) % 3) * S + i + 1] : 0.0;
                    qb = (wk ? hs1 : hs0) + l + mq * tab(LCG_FOLD_TAB_MLC) * tab(LCG_FOLD_TAB_TP + wk) * s2;
                    Qb[x] = qb;
                    QI[x] = qb * tab(LCG_FOLD_TAB_GI + wk);
                    QU[x] = qb * tab(LCG_FOLD_TAB_GU + wk);
                } else {
                    Qb[x] = QI[x] = QU[x] = 0.0;
                }
                const double qm1 = (d > 4 ? q1p * s1 : 0.0) + (t ? qb * tab(LCG_FOLD_TAB_BRANCH + weak(t)) : 0.0);
                const double y = qm1 + s1 * yp, m = total(0, c);
                Qm1[x] = qm1;
                Qm[x] = y + m;
                M2[(size_t)(d % 3) * S + i] = m;
                Y[(size_t)(d & 1) * S + i] = y;
                // for the exterior loop, which reads rows (from LDS any order)
                (IN_LDS ? X[x] : P[(size_t)i * W + d]) = t ? qb * tab(LCG_FOLD_TAB_EXT + weak(t)) : 0.0;
            }
            buf ^= 1;
            if (nb != member) __syncthreads();
        }
        diagonal_done();
        // a workgroup without cells on this diagonal has made no list
        if (member * NB >= n - d) {
            if (wave == 0) make_list(d + 1, member, buf);
            __syncthreads();
        }
    }

    // ---------------- exterior loop, by wave 0 of every workgroup: Z5
    // forward, pushing each Z5(k-1) over the row of pairs (k, j), then the
    // adjoints Z5b, gathered over rows.  A pair spans at least 4, so four rows
    // are taken at once.
    for (int x = tid; x <= n; x += FT) Z5[x] = Z5b[x] = 0.0;
    __syncthreads();
    auto ext = [&](int i, int d) { return IN_LDS ? X[(size_t)d * S + i] : P[(size_t)i * W + d]; };
    if (wave == 0) {
        double z = 1.0;  // Z5(k0 - 1)
        if (lane == 0) Z5[0] = 1.0;
        for (int k0 = 1; k0 <= n; k0 += 4) {
            // Z5[j] holds the pairs ending in j until j is reached
            double zk[4];
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                zk[k] = z;  // Z5(k0 + k - 1)
                if (k0 + k <= n) z = z * s1 + Z5[k0 + k];
            }
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            if (lane < 4 && k0 + lane <= n) Z5[k0 + lane] = lane == 0 ? zk[1] : lane == 1 ? zk[2] : lane == 2 ? zk[3] : z;
            for (int j0 = k0 + 4; j0 <= min(n, k0 + 3 + W - 1); j0 += 64) {
                const int j = j0 + lane;
                double f = 0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int e = j - k0 - k;
                    if (j <= n && e >= 4 && e < W && k0 + k <= n) f += zk[k] * ext(k0 + k, e);
                }
                if (j <= n) Z5[j] += f;
            }
        }
        if (lane == 0) Z5b[n] = 1.0;
        double g = 1.0;  // Z5b(m0 + 1)
        for (int m0 = n - 1; m0 >= 0; m0 -= 4) {
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
            double f[4] = {0, 0, 0, 0};
            for (int j0 = m0 + 2; j0 <= min(n, m0 + W); j0 += 64) {
                const int j = j0 + lane;
                const double zb = j <= n ? Z5b[j] : 0.0;
#pragma unroll
                for (int k = 0; k < 4; ++k) {
                    const int m = m0 - k, e = j - m - 1;  // row m + 1
                    if (m >= 0 && j <= n && e >= 4 && e < W) f[k] += zb * ext(m + 1, e);
                }
            }
#pragma unroll
            for (int o = 32; o > 0; o >>= 1)
#pragma unroll
                for (int k = 0; k < 4; ++k) f[k] += __shfl_xor(f[k], o);
            __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                if (m0 - k < 0) break;
                g = g * s1 + f[k];
                if (lane == 0) Z5b[m0 - k] = g;
            }
        }
        if (member == 0 && lane == 0) *zout = Z5[n];
    }
    // the rows of P are read before any workgroup overwrites them
    diagonal_done();
    const double Z = Z5[n];

    // ---------------- outside, probabilities
    auto has_cells = [&](int d) { return member * NB < n - d; };
    if (wave == 0) make_list(W - 1, member, buf);
    __syncthreads();
    for (int d = W - 1; d >= 4; --d) {
        for (int b = member; b < nbatch && b * NB < n - d; b += K) {
            // terms outside the sequence read cells that are never written (0): past
            // the last cell of a diagonal, which is also where an index below 1 leads
            double q1[NCH], q2[NCH];
#pragma unroll
            for (int h = 0; h < NCH; ++h) q1[h] = q2[h] = 0;
            const int a0 = b * NB + 1 + lane;
            const int top = min(W - 1, n - 1 - b * NB);  // diagonals with a cell of the batch
#pragma unroll 4
            for (int e = d + 5 + wave; e <= top; e += NWV) {
                const double *x = X + (size_t)e * S + a0, *y = Qm1 + (size_t)(e - d - 1) * S + a0 + d + 1;
#pragma unroll
                for (int h = 0; h < NCH; ++h) q1[h] += x[64 * h] * y[64 * h];
            }
            const int btop = min(W - 1 - d, b * NB + NB - 1);
#pragma unroll 4
            for (int e = 5 + wave; e <= btop; e += NWV) {
                const double *x = X + (size_t)(d + e) * S + a0 - e, *y = Qm + (size_t)(e - 1) * S + a0 - e;
#pragma unroll
                for (int h = 0; h < NCH; ++h) q2[h] += x[64 * h] * y[64 * h];
            }
            loops(b, min(MAXLOOP, W - 3 - d), QU + (size_t)d * S, QI + (size_t)d * S, off_out);
            // with three parts the sums of the splits share the first in turn
#pragma unroll
            for (int h = 0; h < NCH; ++h) part[wave * NB + 64 * h + lane] = q1[h];
            if (NP == 4)
#pragma unroll
                for (int h = 0; h < NCH; ++h) part[(3 * NWV + wave) * NB + 64 * h + lane] = q2[h];
            __syncthreads();
            double qmb = 0, lu = 0, li = 0;
            const int c = 64 * wave + lane, a = b * NB + c + 1, e = a + d;
            const bool mine = wave < NCH && e <= n;
            const int t = mine ? Q.pt(a, e) : 0;
            if (mine) qmb = total(0, c);
            if (t) {
                const int at = place[buf * NB + c];
                lu = total(1, at);
                li = total(2, at);
            }
            const int nb = b + K < nbatch && (b + K) * NB < n - d ? b + K : member;
            if (wave == NWV - 1) make_list(nb == member ? d - 1 : d, nb, buf ^ 1);
            if (NP == 3) {
                __syncthreads();
#pragma unroll
                for (int h = 0; h < NCH; ++h) part[wave * NB + 64 * h + lane] = q2[h];
                __syncthreads();
            }
            if (mine) {
                const size_t x = (size_t)d * S + a;
                const bool up = a >= 2, right = e < n;
                const double u = qmb + (up && d + 1 < W ? s1 * U[(size_t)((d + 1) & 1) * S + a - 1] : 0.0);
                const double qm1b = total(NP == 4 ? 3 : 0, c) + u;
                const double sb = right && d + 1 < W ? s1 * R[(size_t)((d + 1) & 1) * S + a] : 0.0;
                double xv = qmb;
                if (up && right && d + 2 < W) {
                    const int to = Q.pt(a - 1, e + 1);
                    if (to)
                        xv += tab(LCG_FOLD_TAB_MLC) * tab(LCG_FOLD_TAB_TP + weak(to)) * s2 *
                              Qbb[(size_t)((d + 2) & 3) * S + a - 1];
                }
                double qbb = 0, p = 0, p2 = 0;
                if (t) {
                    const int wk = weak(t);
                    double l = lu * tab(LCG_FOLD_TAB_GU + wk) + li * tab(LCG_FOLD_TAB_GI + wk);
                    if (up && right && d + 2 < W)
                        l += tab(LCG_FOLD_TAB_STACK + Q.pt(a - 1, e + 1) * 8 + t) * s2 *
                             Qbb[(size_t)((d + 2) & 3) * S + a - 1];
                    if (d + 3 < W) {
                        const double *q = Qbb + (size_t)((d + 3) & 3) * S;
                        if (up && e + 2 <= n) l += tab(LCG_FOLD_TAB_BULGE1 + Q.pt(a - 1, e + 2) * 8 + t) * s3 * q[a - 1];
                        if (a >= 3 && right) l += tab(LCG_FOLD_TAB_BULGE1 + Q.pt(a - 2, e + 1) * 8 + t) * s3 * q[a - 2];
                    }
                    qbb = Z5b[e] * Z5[a - 1] * tab(LCG_FOLD_TAB_EXT + wk) + l +
                          tab(LCG_FOLD_TAB_BRANCH + wk) * (sb + qm1b);
                    p = Qb[x] * qbb / Z;
                    if (d >= 6) {
                        const int ti = Q.pt(a + 1, e - 1);
                        if (ti) p2 = qbb * tab(LCG_FOLD_TAB_STACK + t * 8 + ti) * s2 * Qb[x - 2 * S + 1] / Z;
                    }
                    QI[x] = qbb * tab(LCG_FOLD_TAB_GI + wk);
                    QU[x] = qbb * tab(LCG_FOLD_TAB_GU + wk);
                } else {
                    QI[x] = QU[x] = 0.0;
                }
                X[x] = xv;
                U[(size_t)(d & 1) * S + a] = u;
                R[(size_t)(d & 1) * S + a] = qm1b + sb;
                Qbb[(size_t)(d & 3) * S + a] = qbb;
                P[(size_t)a * W + d] = p;
                P2[(size_t)a * W + d] = p2;
            }
            buf ^= 1;
            if (nb != member) __syncthreads();
        }
        diagonal_done();
        if (!has_cells(d)) {
            if (wave == 0) make_list(d - 1, member, buf);
            __syncthreads();
        }
    }
}

extern "C" __global__ __launch_bounds__(LCG_FOLD_THREADS) void lcg_fold_seqs(
    const FoldDesc *descs, const signed char *codes, const double *tabs, double *mats, double *outs, double *zout,
    int *counters, int *status, const int *seq_of, int polls, int nch) {
    constexpr int NWV = LCG_FOLD_THREADS / 64;
    extern __shared__ double lds[];
    const int sq = seq_of[2 * blockIdx.x], member = seq_of[2 * blockIdx.x + 1];
    const FoldDesc D = descs[sq];
    const int chunks = lcg_fold_chunks(D.n, D.K, nch);
    if (chunks == 1)
        fold_seq<1, NWV, false>(D, member, codes, tabs, mats, outs, zout + sq, counters + sq, status, polls, lds);
    else if (chunks == 2)
        fold_seq<2, NWV, false>(D, member, codes, tabs, mats, outs, zout + sq, counters + sq, status, polls, lds);
    else
        fold_seq<4, NWV, false>(D, member, codes, tabs, mats, outs, zout + sq, counters + sq, status, polls, lds);
}

// Short sequences, one workgroup each, the matrices in LDS: a diagonal has few
// terms, so half the waves (fewer partial sums to add up, shorter barriers).
extern "C" __global__ __launch_bounds__(LCG_FOLD_SHORT_THREADS) void lcg_fold_short(
    const FoldDesc *descs, const signed char *codes, const double *tabs, double *outs, double *zout,
    const int *seq_of) {
    extern __shared__ double lds[];
    const int sq = seq_of[2 * blockIdx.x];
    const FoldDesc D = descs[sq];
    fold_seq<1, LCG_FOLD_SHORT_THREADS / 64, true>(D, 0, codes, tabs, nullptr, outs, zout + sq, nullptr, nullptr, 0, lds);
}

// LDS bytes of a workgroup; nch 0: of lcg_fold_short for a band of W.
extern "C" size_t lcg_fold_lds_bytes(int nmax, int nch, int W) {
    const size_t nb = nch ? 64 * nch : 64;
    const size_t sums = nch ? 3 * (LCG_FOLD_THREADS / 64) * nb
                            : 4 * (LCG_FOLD_SHORT_THREADS / 64) * nb + lcg_fold_matrix_doubles(nmax, W);
    const size_t doubles = sums + (LCG_FOLD_TAB_HP - LCG_FOLD_TAB_STACK) + 2 * (nmax + 1);
    return doubles * sizeof(double) + 28 * sizeof(int) + 4 * nb * sizeof(unsigned short) + 2 * sizeof(int) +
           (size_t)(nmax + 2);
}

// grid workgroups: sequence and member of each in seq_of; polls: bound of the
// waits between the members of a sequence; nch 1, 2 or 4, 0: lcg_fold_short;
// lds: bytes.
extern "C" int lcg_launch_fold(const FoldDesc *descs, const signed char *codes, const double *tabs, double *mats,
                               double *outs, double *zout, int *counters, int *status, const int *seq_of, int grid,
                               int polls, int nch, size_t lds, hipStream_t stream) {
    const void *kernel = nch ? (const void *)lcg_fold_seqs : (const void *)lcg_fold_short;
    if (hipError_t e = hipFuncSetAttribute(kernel, hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds)) return (int)e;
    if (grid <= 0) return 0;
    if (nch)
        hipLaunchKernelGGL(lcg_fold_seqs, dim3(grid), dim3(LCG_FOLD_THREADS), lds, stream, descs, codes, tabs, mats, outs,
                           zout, counters, status, seq_of, polls, nch);
    else
        hipLaunchKernelGGL(lcg_fold_short, dim3(grid), dim3(LCG_FOLD_SHORT_THREADS), lds, stream, descs, codes, tabs, outs,
                           zout, seq_of);
    return (int)hipGetLastError();
}
