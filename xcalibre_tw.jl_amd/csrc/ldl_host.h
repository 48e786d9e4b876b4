// Host LDL^T factorization for the LDL preconditioner (ldl_host.cpp).
#pragma once

#include <vector>

namespace fvh {

// L D L^T = P A P^T with P the ordering perm (position k holds row perm[k]).
// L is unit lower triangular, stored by columns without its diagonal (Lp, Li,
// Lx; rows ascending within a column), in the permuted numbering.
struct LdlHost {
    int n = 0;
    std::vector<int> perm, Lp, Li;
    std::vector<double> Lx, D;
};

// Nested-dissection ordering of a symmetric pattern from the cells' centres;
// with `bounds`, also the ranges of positions that each leaf and each
// separator occupy (range g is [bounds[g], bounds[g + 1]), in order).
void ldl_order(int n, const int *rowptr, const int *col, const double *x, const double *y, std::vector<int> &perm,
               std::vector<int> *bounds = nullptr);

// Numeric factorization; A symmetric (values read from its upper triangle).
int ldl_factor(int n, const int *rowptr, const int *col, const double *val, const std::vector<int> &perm, LdlHost &F);

// The factor as the block solves read it.  Per range of rows g the unit
// lower triangular block L_gg is replaced by its explicit inverse, so that
// the rows of a range do not wait for each other:
//   forward   r_g = x_g - L_g,before y_before,        y_g = inv(L_gg) r_g
//   backward  s_g = D_g^-1 y_g - L_after,g' z_after,  z_g = inv(L_gg)' s_g
// Work is cut into blocks of kLdlWaves waves, listed in an order in which
// every block follows the blocks whose results it reads.
// A product with the inverse rounds as the substitution does as long as the
// inverse has no growth: its entries are at most 1 where A is diagonally
// dominant, as every Laplacian of positive coefficients is.  Other matrices
// (indefinite, say) grow, and a range is cut where an entry of its inverse is
// above kLdlGrowth, down to single rows, which are substitution.
// Error of a solve against extended precision on 310 x 140 rows, whole ranges
// / cut / substitution, mean of four right-hand sides: Laplacian with 4 - 1.3
// on the diagonal 2.4e-11 / 4.4e-12 / 4.1e-12, random symmetric 2.6e-12 /
// 1.1e-12 / 1.5e-12, dominant 1.9e-16 / the same / 4.4e-16.  An apply on
// 400 x 100 takes 129 us dominant, 1,236 us with the shift (129 us uncut).
constexpr int kLdlWaves = 8;
constexpr int kLdlWhole = 64;   // rows of a range that one block takes whole ...
constexpr int kLdlLeaf = 80;    // ... and of a range without outside columns
constexpr int kLdlRange = 512;  // rows of a range (longer ones are cut)
constexpr double kLdlGrowth = 1.25;
struct LdlBlock {
    int kind;           // 0: a whole range; 1: outside rows r, r+1, ... (a row per wave); 2: inverse rows
    int r;              // first row
    int r0, rows;       // its range
    int gate[2];        // words its inputs are published with, last in the tree (-1: none)
    long long off;      // the range's packed inverse
};
struct LdlSide {
    std::vector<int> ptr, idx;  // per row (forward) or column (backward): the entries outside its range
    std::vector<double> val, inv;
    std::vector<LdlBlock> blocks;
};
struct LdlBlocks {
    LdlSide f, b;
};
// `bounds`: ranges of positions in order (ldl_order's).
void ldl_blocks(const LdlHost &F, const std::vector<int> &bounds, LdlBlocks &out);

}  // namespace fvh
