// Building-scale field step (FDM plans with 10^5-10^6 cells): the shared
// device tables and per-group buffers the host (fdm.cpp) builds and the
// kernels (fdm_kernel.hip) read. Not part of the public ABI.
//
// Layouts. A group of G envs shares one factorization; its envs are split
// into nblk blocks of Gl lanes (the last block may hold fewer envs), and every
// per-env field array is block-major, env-minor: element (cell or row x, env
// b * Gl + l) of array A sits at A[(b * rows + x) * Gl + l], so the envs of a
// block read one row as Gl adjacent doubles. The default mode's solve has
// vectors of its own, in tiles of kEnvTile envs. The solve works on the permuted
// vector of the baked factorization (SuperLU convention, complete_port/csim/
// sb_lu.c:38-63): w[i] = b[ir[i]], L w' = w, U z = w', x[t] = z[pc[t]].
#pragma once
#include <stddef.h>
#include <stdint.h>

namespace sbf {

// One triangular factor as level-ordered rows: rows[q] is the q-th row in
// level order (level l spans q in [lev[l], lev[l + 1])); its off-diagonal
// terms are (col[e], val[e]) for e in [ptr[q], ptr[q + 1]), in the order the
// reference's column sweep applies them (L: ascending column, U: descending);
// diag[q] is U's diagonal (unused for the unit L).
struct Tri {
    int nlev;
    const int* lev;
    const int* rows;
    const int* ptr;
    const int* col;
    const double* val;
    const double* diag;
};

// The default mode's form of the same two factors: dense fronts.
//
// The rows of the permuted system are grouped along the elimination tree of
// the factors' union pattern (closed under fill): whole subtrees of at most
// kLeafCols columns are one front each (the leaves), and above them chains of
// columns are merged while the merged block stays nearly dense. A front with
// columns C (w of them) and boundary B (the r later rows its columns reach)
// needs two dense operators, formed once at open from L and U:
//   F = -L_BC L_CC^-1                        [r][w]
//   K = [U_CC^-1 L_CC^-1 | -U_CC^-1 U_CB]     [w][w + r]
// A solve is then, up the tree, b' = b_C + the children's contributions and
// c = the children's contributions on B + F b' (the front's own contribution),
// and, down the tree, x_C = K [b'; x_B]: one matrix product a front and
// direction, and as many dependent steps as the tree of fronts is high (17 on
// a 205K-cell plan, against 2,288 levels of rows).
//
// Rows of W and X are in front order (leaves first, then by height), a front's
// columns contiguous from `off`. Operators are stored for
// v_mfma_f64_16x16x4: [tile of 16 rows][step of 4 columns][lane], lane l
// holding row l % 16, column l / 16 of the step; the w and the r columns of K
// are padded to whole steps separately (zeros).
constexpr int kEnvTile = 16;    // envs of a tile: the columns of one MFMA
constexpr int kLeafCols = 64;   // columns of a leaf front
constexpr int kFrontCols = 256; // columns of a front above the leaves

struct Front {
    int off, w, r;
    int brow;               // its B rows (positions in X) in FrontTab::brow, padded to a multiple of 4
    int c;                  // its contribution's first row in C
    int arow;               // its first row in FrontTab::arow (w rows, then r; fronts above the leaves)
    long long f, k;         // its operators' offsets in FrontTab::ops
};

// The unknowns are the temperatures less the env's ambient temperature (the
// right-hand side less ambient x row sum): forcing and solutions of some 10 K
// instead of 300 K keep the products' rounding a digit below the field's own,
// whatever the order of their sums.

// The contributions added to one row of a front above the leaves: rows of C,
// four at once (the zero row where there are fewer), then brow-style extras
// [xb, xe) of FrontTab::xsrc.
struct AsmRow {
    int s[4];
    int xb, xe, pad[2];
};

// One row tile of a front (16 rows from 16 * tile).
struct FrontTask {
    int front, tile;
};

// One height of the tree: its fronts' tasks up (F's row tiles, at least one a
// front above the leaves) and down (K's), and the widest front's columns.
struct FrontLevel {
    int f0, nf, k0, nk;     // tasks [f0, f0 + nf) up and [k0, k0 + nk) down
    int wmax;
};

struct FrontTab {
    int n_fronts, n_levels, n_leaf, n_c;   // n_leaf: rows of the leaves; n_c: rows of C (row n_c is zero)
    const Front* fronts;
    const int* brow;
    const AsmRow* arow;
    const int* xsrc;
    const FrontTask* tasks;
    const double* ops;
    const int* rf;          // [n] solved index t -> row of W (its right-hand side)
    const int* rx;          // [n] solved index t -> row of X (its solution)
    const int* sn_w;        // sensed entries -> row of X
    const double* rowsum;   // [n] by t: the factored system's row sums (L U 1) less capacitance and mass coupling
    const FrontLevel* levels;   // host memory (the launches read it), leaves first
};

struct Tables {
    int n, n_cvs, k, n_unsolved;
    const int* ir;          // [n] row of the permuted vector -> solved index t of its right-hand side
    const int* ipr;         // [n] solved index t -> that row (the inverse of ir)
    const int* pc;          // [n] solved index t -> row of the permuted solution
    const int* solved;      // [n] t -> cell p
    const int* unsolved;    // [n_unsolved] cells held at the ambient temperature
    const double *cap, *dir, *mcoup, *mret, *mgain;   // [n] by t
    const double *a0, *a1, *hz, *vt, *cd;             // [n] by t: exterior face areas, half widths, conductivity
    Tri L, U;
    int fast;               // dense fronts (reassociated sums) instead of every level in order
    FrontTab ft;
    // sensed rows (k): entries p in [sn_p[i], sn_p[i + 1]) weigh row sn_w[p] of the solution
    const int* sn_p;
    const int* sn_w;
    const double* sn_x;
    // applied columns, transposed per permuted row i: (column at_j[e], value at_x[e]) for
    // e in [at_p[i], at_p[i + 1]), ascending column
    const int* at_p;
    const int* at_j;
    const double* at_x;
    const double* S;        // [k][k] sensed A^-1 applied
    // default mode: R [k][n], row j the solution A^-1 applied_j of applied
    // column j by solved index t (exact-mode solves at open), so a step's
    // air-side correction A^-1 (applied q) is the combination R^T q instead of
    // a second solve; null in exact mode
    const double* R;
    // blobs with zones (full env scenarios): the zone whose heat each solved
    // cell t carries, or -1 (a zone's heat goes to its room's cells; a cell of
    // two zones' rooms takes the later zone's, as csim assigns input_q)
    const int* czone;       // [n] or null
    int nz;
};

struct Group {
    int G, Gl, nblk;
    int nt;                 // env tiles
    double* T;              // [nblk][n_cvs][Gl]
    double* M;              // [nblk][n][Gl]
    // exact mode: the forcing solve in place, [nblk][n][Gl]; default mode: the
    // right-hand side in front order, [tiles][n][kEnvTile]
    double* W1;
    double* W2;             // [nblk][n][Gl] the air-side correction (exact mode)
    double* X;              // [tiles][n][kEnvTile] the solution less the ambient temperature (default mode)
    double* Y;              // [tiles][n - n_leaf][kEnvTile] assembled right-hand sides above the leaves (default mode)
    double* C;              // [tiles][n_c + 1][kEnvTile] the fronts' contributions, then a zero row (default mode)
    double* pw;             // [G][k] air-side power, then the dense solve's result
    double* mat;            // [G][k][k] I + diag(g) S
    int* eact;              // [G] env has a nonzero air-side conductance this step
    int* bact;              // [nblk] some env of the block has (exact mode; null in the default one)
    int tiles, pad;         // the tiles that W1, X, Y and C hold (default mode)
};

// One batched step's inputs (device): input_q [G][n_cvs], ambient / h [G],
// air_g / air_T [G][k]. With q null, each cell's input_q is its zone's heat
// per cell qz [G][nz] (Tables::czone; 0 outside the rooms).
struct StepIn {
    const double* q;
    const double* amb;
    const double* h;
    const double* g;
    const double* airT;
    const double* qz;
};

// The host (g++) and the device (hipcc) compile these structs separately and
// exchange them byte for byte: both builds check the same sizes and offsets.
static_assert(sizeof(Tri) == 56 && sizeof(Front) == 40 && sizeof(AsmRow) == 32 && sizeof(FrontTab) == 104,
              "Tri / Front / FrontTab layout");
static_assert(sizeof(Tables) == 440 && offsetof(Tables, S) == 408 && offsetof(Tables, nz) == 432, "Tables layout");
static_assert(sizeof(Group) == 112 && sizeof(StepIn) == 48, "Group / StepIn layout");

}  // namespace sbf
