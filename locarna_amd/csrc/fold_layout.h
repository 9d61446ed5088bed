// Device layout of the base-pair probability step (McCaskill inside and
// outside over the energy model of fold_model.h), shared by fold.cpp and
// fold_kernels.hip.
//
// Matrices are stored by diagonals: entry (i, j), 1 <= i <= n,
// 0 <= d = j - i < W, at d * S + i, with W = min(n, max span) (a pair (i, j)
// needs j - i + 1 <= max span) and S >= n + 2, so that the cells of a diagonal
// and the cells that their sums read are neighbours.  Six such bands per
// sequence: Qb (pair (i, j) closes the segment), Qb times the inner-pair
// factor of interior loops and of bulges (in the outside pass the outside
// values of Qb times the outer-pair factors), Qm (at least one multiloop
// branch in i..j), Qm1 (exactly one branch, starting at i) and X (outside
// pass: fold_kernels.hip), and LCG_FOLD_RINGS rows of the last diagonals of
// the recursions that read only those.  Two more bands, in a separate output
// arena and stored by rows (i * W + d), hold the pair probabilities P(i, j)
// and the joint probabilities P2(i, j) of (i, j) and (i + 1, j - 1); between
// the passes the first holds Qb times its exterior-loop factor.  The matrices
// are cleared before a run; cells past the end of a diagonal stay 0.
#ifndef LOCARNA_AMD_FOLD_LAYOUT_H
#define LOCARNA_AMD_FOLD_LAYOUT_H

#include <stddef.h>

#define LCG_FOLD_MAXLOOP 30
// factor table (doubles): Boltzmann factors of the loop terms
#define LCG_FOLD_TAB_LOOP 0       // [l1 * 31 + l2], l1 + l2 >= 2, two strong pairs
#define LCG_FOLD_TAB_STACK 961    // [outer type * 8 + inner type], l1 = l2 = 0
#define LCG_FOLD_TAB_BULGE1 1025  // [outer type * 8 + inner type], l1 + l2 = 1
#define LCG_FOLD_TAB_EXT 1089     // [weak]: a pair in the exterior loop
#define LCG_FOLD_TAB_BRANCH 1091  // [weak]: a branch of a multiloop
#define LCG_FOLD_TAB_TP 1093      // [weak]: the closing pair's terminal penalty
#define LCG_FOLD_TAB_MLC 1095     // multiloop closing (closing + one branch)
#define LCG_FOLD_TAB_GI 1096      // [weak]: a weak pair of an interior loop
#define LCG_FOLD_TAB_GU 1098      // [weak]: a weak pair of a bulge
#define LCG_FOLD_TAB_HP 1100      // [L * 2 + weak]: hairpin of L unpaired bases
#define LCG_FOLD_MAX_LEN 4096     // longest sequence (Z5 and Z5b live in LDS)
#define LCG_FOLD_THREADS 1024
#define LCG_FOLD_SHORT_THREADS 512  // lcg_fold_short
#define LCG_FOLD_RINGS 16
#define LCG_FOLD_PAD 1024         // doubles past a sequence's matrices (chunks of 64 cells run past a diagonal)

#ifdef __HIPCC__
#define LCG_FOLD_HD __host__ __device__
#else
#define LCG_FOLD_HD
#endif

// Chunks of 64 cells per batch of a sequence of n bases on K workgroups: one
// with several workgroups, else as many as its diagonals have, up to nch (1, 2
// or 4: what the LDS of the launch was allocated for).
LCG_FOLD_HD inline int lcg_fold_chunks(int n, int K, int nch) {
    const int c = K > 1 || n <= 64 ? 1 : n <= 128 ? 2 : 4;
    return c < nch ? c : nch;
}

// Doubles of a sequence's matrices in LDS (lcg_fold_short): rows of n + 2, and what the lanes past
// the end of the last row read.
LCG_FOLD_HD inline size_t lcg_fold_matrix_doubles(int n, int W) {
    return ((size_t)6 * W + LCG_FOLD_RINGS) * (n + 2) + 64;
}

struct FoldDesc {
    int n;           // sequence length
    int W;           // band width
    int S;           // stride of a diagonal
    int K;           // workgroups of the sequence
    long long codes; // offset of the codes: position i at codes + i (0 A, 1 C, 2 G, 3 U, 4 other)
    long long mat;   // offset (doubles) of the six bands and the ring rows
    long long out;   // offset (doubles) of the two bands P, P2
    double log_sigma; // scale per base: values of L bases are stored times exp(-L log_sigma)
};

#endif
