// The default mode's building-scale field step: dense fronts on the matrix
// cores (sbf::FrontTab), envs in tiles of kEnvTile = 16, the columns of a
// v_mfma_f64_16x16x4.
//
// Per step: forcing into W (sb_fdm.c:147-151), the solve up and down the tree
// of fronts (sb_lu.c:38-63 in another order: results agree to rounding), the
// sensed temperatures and air-side powers (sb_fdm.c:157-162), the dense solve
// (fdm_kernel.hip), then the correction R^T q, the interior mass and the field
// (sb_fdm.c:171-187). The field and the mass keep the group's own layout.
//
// MFMA operands: A lane l holds row l % 16, column l / 16 of the step (the
// operators are stored that way, one 512-byte load a step and wavefront), B
// lane l holds row l / 16 of the step, env l % 16 (a row of 16 envs is one
// 128-byte line, so rows may be gathered), D register q holds row
// l / 16 + 4 q, env l % 16.
// What bounds it: the vectors' HBM traffic at 256 envs and more, the chain of
// 2 x 17 dependent launches at a tile or two. Measured on the 205K-cell plan:
// a step of 256 envs 13.1 -> 1.9 ms, of 16 envs 10.2 -> 0.45 ms against level
// by level row solves, whose 4,577 dependent levels were the whole time.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>
#include <type_traits>

#include "fdm.h"

namespace {

typedef double d4 __attribute__((ext_vector_type(4)));
constexpr int E = sbf::kEnvTile;
static_assert(E == 16, "one MFMA column per env of a tile");

__device__ __forceinline__ d4 mfma(double a, double b, d4 c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
}

// acc[r][e] += A (row tile r) B (env tile e) over the steps [k0, k1): A from
// the operator's tiles, B through load(step, e). U steps' loads are issued
// before their products; the last U may run past k1 with zeros for A (a step
// at a time there would be a memory latency each). `before(k)`, if given, runs ahead of step k's products.
struct Nothing {
    __device__ void operator()(int) const {}
};
template <int RT, int NE, int U, class Load, class Before = Nothing>
__device__ __forceinline__ void product(const double* const (&A)[RT], int k0, int k1, Load load, d4 (&acc)[RT][NE],
                                        Before before = {}) {
    for (int k = k0; k < k1; k += U) {
        double a[RT][U], b[NE][U];
#pragma unroll
        for (int u = 0; u < U; u++) {
            const int q = min(k + u, k1 - 1);
#pragma unroll
            for (int e = 0; e < NE; e++) b[e][u] = load(q, e);
#pragma unroll
            for (int r = 0; r < RT; r++) a[r][u] = A[r][(size_t)q * 64];
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
            if (!std::is_same<Before, Nothing>::value && k + u < k1) before(k + u);
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const double x = k + u < k1 ? a[r][u] : 0.0;
#pragma unroll
                for (int e = 0; e < NE; e++) acc[r][e] = mfma(x, b[e][u], acc[r][e]);
            }
        }
    }
}

// The leaves, a wavefront per (RT row tiles of a front, NE env tiles): up
// (DOWN false) c = F b, down x = K [b; x_B]. Env tiles of one task are
// neighbouring wavefronts, so a workgroup's wavefronts share the operator.
template <bool DOWN, int RT, int NE>
__global__ __launch_bounds__(256) void leaf_kernel(sbf::FrontTab t, int task0, int ntask, int n, int nt,
                                                   const double* __restrict__ W, double* __restrict__ C,
                                                   double* __restrict__ X) {
    const int neg = (nt + NE - 1) / NE;
    const unsigned x = blockIdx.x * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int eg = (int)(x % (unsigned)neg), task = (int)(x / (unsigned)neg) * RT;
    if (task >= ntask) return;
    const int lane = threadIdx.x & 63, j = lane & 15, kk = lane >> 4;
    // RT consecutive tasks; those of another front are its own wavefront's
    // work too (a front's tiles need not start at a multiple of RT)
    for (int u = 0; u < RT;) {
        if (task + u >= ntask) break;
        const sbf::FrontTask tk = t.tasks[task0 + task + u];
        const sbf::Front f = t.fronts[tk.front];
        int m = 1;
        while (u + m < RT && task + u + m < ntask && t.tasks[task0 + task + u + m].front == tk.front) m++;
        const int kw = (f.w + 3) >> 2, ks = DOWN ? kw + ((f.r + 3) >> 2) : kw;
        const double* A[RT];
#pragma unroll
        for (int r = 0; r < RT; r++)
            A[r] = t.ops + (DOWN ? f.k : f.f) + (size_t)(tk.tile + (r < m ? r : 0)) * ks * 64 + lane;
        const double* Wb[NE];
        const double* Xb[NE];
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const size_t te = min(eg * NE + e, nt - 1);
            Wb[e] = W + (te * n + f.off) * E + j;
            Xb[e] = X + te * n * E + j;
        }
        d4 acc[RT][NE] = {};
        product<RT, NE, 4>(A, 0, kw, [&](int k, int e) { return Wb[e][min(4 * k + kk, f.w - 1) * E]; }, acc);
        if (DOWN) {
            const int* br = t.brow + f.brow + kk - 4 * kw;
            product<RT, NE, 4>(A, kw, ks, [&](int k, int e) { return Xb[e][(size_t)br[4 * k] * E]; }, acc);
        }
#pragma unroll
        for (int r = 0; r < RT; r++) {
            if (r >= m) continue;
#pragma unroll
            for (int e = 0; e < NE; e++) {
                const size_t te = eg * NE + e;
                if ((int)te >= nt) continue;
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int row = (tk.tile + r) * 16 + kk + 4 * q;
                    if (row >= (DOWN ? f.w : f.r)) continue;
                    if (DOWN) X[(te * n + f.off + row) * E + j] = acc[r][e][q];
                    else C[(te * (t.n_c + 1) + f.c + row) * E + j] = acc[r][e][q];
                }
            }
        }
        u += m;
    }
}

// The sum of the contributions to one row (FrontTab::arow) of one env.
__device__ __forceinline__ double gathered(const sbf::FrontTab& t, int row, const double* Cb) {
    const int4 s = *reinterpret_cast<const int4*>(t.arow[row].s);
    const int2 xr = *reinterpret_cast<const int2*>(&t.arow[row].xb);
    double v = (Cb[(size_t)s.x * E] + Cb[(size_t)s.y * E]) + (Cb[(size_t)s.z * E] + Cb[(size_t)s.w * E]);
    for (int q = xr.x; q < xr.y; q++) v += Cb[(size_t)t.xsrc[q] * E];
    return v;
}

// b' of the wide heights' fronts (those above the leaves with many
// workgroups), a thread per (row, env): the right-hand side and the children's
// contributions into Y.
__global__ __launch_bounds__(256) void assemble_kernel(sbf::FrontTab t, int task0, int ntask, int n, int nt,
                                                       const double* __restrict__ W, double* __restrict__ Y,
                                                       const double* __restrict__ C) {
    const int ny = n - t.n_leaf, j = threadIdx.x % E, r = threadIdx.x / E;
    const int te = (int)(blockIdx.x % (unsigned)nt), task = (int)(blockIdx.x / (unsigned)nt);
    if (task >= ntask) return;
    const sbf::FrontTask tk = t.tasks[task0 + task];   // (K's tasks: 16 of the front's columns each)
    const sbf::Front f = t.fronts[tk.front];
    const int row = tk.tile * 16 + r;
    if (row >= f.w) return;
    const double* Cb = C + (size_t)te * (t.n_c + 1) * E + j;
    Y[((size_t)te * ny + (f.off - t.n_leaf) + row) * E + j] = W[((size_t)te * n + f.off + row) * E + j]
                                                               + gathered(t, f.arow + row, Cb);
}

// Column shares of a front's product above the leaves. Every form of
// front_kernel sums the same shares in the same order, ((0 + 1) + (2 + 3)) +
// ..., so an env's result does not depend on the form its batch takes.
constexpr int kShares = 8;

// A height above the leaves, one workgroup per (RT row tiles of a front, NE
// env tiles), its KW wavefronts taking kShares / KW neighbouring shares of the
// columns each, summed in LDS. Down: x = K [b'; x_B]. Up: c = the
// children's contributions on B + F b', with b' from Y (assemble_kernel), or,
// FUSED, assembled into LDS by every workgroup of the front (its first tile's
// writes it to Y).
//
// A narrow height (one to a few fronts: the upper 13 of 16 on a 205K-cell
// plan) is a chain of memory latencies, so it runs FUSED with 8 wavefronts
// and everything that does not wait for b' loaded before it: 18 and 11 us a
// height with 4 wavefronts and 4 steps in flight, 9 and 8 so (16 envs). A wide
// height (the lowest three) assembled by every workgroup took 188 us at 256
// envs, from Y 47: there it
// is bound by the products' operand traffic: 2 x 2 tiles.
//
// The wide form with four wavefronts a SIMD: left alone, the compiler takes
// registers for three (the same two env steps 9.74 ms).
template <bool DOWN, bool FUSED, int RT, int NE, int KW, int U>
__global__ __launch_bounds__(64 * KW, KW == kShares ? 1 : 4) void front_kernel(sbf::FrontTab t, int task0, int ntask, int n, int nt,
                                                        const double* __restrict__ W, double* __restrict__ Y,
                                                        double* C, double* X) {
    static_assert(!FUSED || (RT == 1 && NE == 1 && KW == kShares), "the fused form takes single tiles and shares");
    static_assert(KW == kShares || 2 * KW == kShares, "a wavefront takes one share or a pair");
    constexpr int SH = kShares / KW;
    extern __shared__ double lds[];
    const int neg = (nt + NE - 1) / NE;
    const int eg = (int)(blockIdx.x % (unsigned)neg), task = (int)(blockIdx.x / (unsigned)neg) * RT;
    const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int j = lane & 15, kk = lane >> 4;
    const int ny = n - t.n_leaf;
    for (int u = 0; u < RT;) {
        if (task + u >= ntask) break;
        const sbf::FrontTask tk = t.tasks[task0 + task + u];
        const sbf::Front f = t.fronts[tk.front];
        int m = 1;
        while (u + m < RT && task + u + m < ntask && t.tasks[task0 + task + u + m].front == tk.front) m++;
        const int kw = (f.w + 3) >> 2, ks = DOWN ? kw + ((f.r + 3) >> 2) : kw;
        const double* A[RT];
#pragma unroll
        for (int r = 0; r < RT; r++)
            A[r] = t.ops + (DOWN ? f.k : f.f) + (size_t)(tk.tile + (r < m ? r : 0)) * ks * 64 + lane;
        const double* Yb[NE];
        const double* Xb[NE];
#pragma unroll
        for (int e = 0; e < NE; e++) {
            const size_t te = min(eg * NE + e, nt - 1);
            Yb[e] = Y + (te * ny + (f.off - t.n_leaf)) * E + j;
            Xb[e] = X + te * n * E + j;
        }
        d4 acc[RT][NE] = {};
        // partial sums: [wavefront][row tile][env tile][register][lane]
        double* red = lds;
        auto slot = [&](int w, int r, int e, int q) { return (((w * RT + r) * NE + e) * 4 + q) * 64 + lane; };
        const int rows = DOWN ? f.w : f.r;
        // the shares cut where the columns are (none for a front without rows)
        auto cut = [&](int share) { return rows > 0 ? ks * share / kShares : 0; };
        const int mid = cut(wave * SH + 1);   // the second share of a pair
        // the output's own gathered part, final before this height (up)
        double own[RT][NE] = {};
        if (!DOWN && wave < 4) {
#pragma unroll
            for (int r = 0; r < RT; r++)
#pragma unroll
                for (int e = 0; e < NE; e++) {
                    const int row = min((tk.tile + r) * 16 + kk + 4 * wave, rows - 1);
                    const size_t te = min(eg * NE + e, nt - 1);
                    if (rows > 0) own[r][e] = gathered(t, f.arow + f.w + row, C + te * (t.n_c + 1) * E + j);
                }
        }
        if (FUSED && !DOWN) {
            // b' [4 kw][E], zero past w; four rows' loads in flight a thread
            constexpr int RS = 64 * KW / E;
            const int col = tid % E;
            const double* Wb = W + ((size_t)eg * n + f.off) * E + col;
            const double* Cb = C + (size_t)eg * (t.n_c + 1) * E + col;
            double* Yw = Y + ((size_t)eg * ny + (f.off - t.n_leaf)) * E + col;
            // this wavefront's share of F, loaded meanwhile (a share has at most kFrontCols / 4 / KW steps)
            constexpr int AU = (sbf::kFrontCols / 4 + KW - 1) / KW;
            const int q0 = cut(wave), q1 = cut(wave + 1);
            double a[AU];
#pragma unroll
            for (int k = 0; k < AU; k++) a[k] = A[0][(size_t)min(q0 + k, max(q1 - 1, 0)) * 64 * (rows > 0 ? 1 : 0)];
            for (int r0 = tid / E; r0 < 4 * kw; r0 += 4 * RS) {
                int4 src[4];
                int2 more[4];
                double v[4][5];
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const sbf::AsmRow* ar = t.arow + f.arow + min(r0 + q * RS, f.w - 1);
                    src[q] = *reinterpret_cast<const int4*>(ar->s);
                    more[q] = *reinterpret_cast<const int2*>(&ar->xb);
                    v[q][4] = Wb[(size_t)min(r0 + q * RS, f.w - 1) * E];
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    v[q][0] = Cb[(size_t)src[q].x * E];
                    v[q][1] = Cb[(size_t)src[q].y * E];
                    v[q][2] = Cb[(size_t)src[q].z * E];
                    v[q][3] = Cb[(size_t)src[q].w * E];
                }
#pragma unroll
                for (int q = 0; q < 4; q++) {
                    const int row = r0 + q * RS;
                    double x = (v[q][0] + v[q][1]) + (v[q][2] + v[q][3]);
                    for (int k = more[q].x; k < more[q].y; k++) x += Cb[(size_t)t.xsrc[k] * E];
                    x += v[q][4];
                    if (row < 4 * kw) lds[row * E + col] = row < f.w ? x : 0.0;
                    if (tk.tile == 0 && row < f.w) Yw[(size_t)row * E] = x;
                }
            }
            __syncthreads();
#pragma unroll
            for (int k = 0; k < AU; k++)
                if (q0 + k < q1) acc[0][0] = mfma(a[k], lds[(4 * (q0 + k) + kk) * E + j], acc[0][0]);
            __syncthreads();
        } else {
            // one run over the wavefront's columns; at its second share the first
            // one's sums go to LDS (two env steps at 512 envs of the 205K-cell
            // building 9.36 ms; a run a share 9.55; registers for both shares 9.53)
            const int q0 = cut(wave * SH), q1 = cut(wave * SH + SH);
            auto keep = [&](int k) {
                if (SH == 1 || k != mid) return;
#pragma unroll
                for (int r = 0; r < RT; r++)
#pragma unroll
                    for (int e = 0; e < NE; e++)
#pragma unroll
                        for (int q = 0; q < 4; q++) {
                            red[slot(wave, r, e, q)] = acc[r][e][q];
                            acc[r][e][q] = 0.0;
                        }
            };
            product<RT, NE, U>(A, min(q0, kw), min(q1, kw),
                               [&](int k, int e) { return Yb[e][min(4 * k + kk, f.w - 1) * E]; }, acc, keep);
            if (DOWN) {
                const int* br = t.brow + f.brow + kk - 4 * kw;
                product<RT, NE, U>(A, max(q0, kw), max(q1, kw),
                                   [&](int k, int e) { return Xb[e][(size_t)br[4 * k] * E]; }, acc, keep);
            }
            if (SH == 2 && mid < q1) {
#pragma unroll
                for (int r = 0; r < RT; r++)
#pragma unroll
                    for (int e = 0; e < NE; e++)
#pragma unroll
                        for (int q = 0; q < 4; q++) acc[r][e][q] = red[slot(wave, r, e, q)] + acc[r][e][q];
            }
        }
#pragma unroll
        for (int r = 0; r < RT; r++)
#pragma unroll
            for (int e = 0; e < NE; e++)
#pragma unroll
                for (int q = 0; q < 4; q++) red[slot(wave, r, e, q)] = acc[r][e][q];
        __syncthreads();
        // wavefront q finishes register q of every tile
        if (wave < 4) {
#pragma unroll
            for (int r = 0; r < RT; r++) {
                const int row = (tk.tile + r) * 16 + kk + 4 * wave;
                if (r >= m || row >= rows) continue;
#pragma unroll
                for (int e = 0; e < NE; e++) {
                    const size_t te = eg * NE + e;
                    if ((int)te >= nt) continue;
                    double v = 0.0;
#pragma unroll
                    for (int w = 0; w < KW; w += KW / 4) {
                        double pair = red[slot(w, r, e, wave)];
                        if (SH == 1) pair += red[slot(w + 1, r, e, wave)];
                        v += pair;
                    }
                    if (DOWN) X[(te * n + f.off + row) * E + j] = v;
                    else C[(te * (t.n_c + 1) + f.c + row) * E + j] = v + own[r][e];
                }
            }
        }
        u += m;
        if (u < RT) __syncthreads();
    }
}

// ------------------------------------------------------------ the operators, at open

// Dense blocks of front f at dense + d0[f]: L_CC [w][w], U_CC [w][w], L_BC
// [r][w], U_CB [w][r].
struct OpsTab {
    const int* front_of;
    const int* local;
    const int* bperm;
    const long long* d0;
    double* dense;
    double* sol;            // per front at s0[f]: [w][w + r + r]: the columns of K, then those of F^T
    const long long* s0;
};

__device__ int b_index(const sbf::Front& f, const int* bperm, int i) {
    int lo = 0, hi = f.r - 1;
    while (lo < hi) {
        const int mid = (lo + hi) >> 1;
        if (bperm[f.brow + mid] < i) lo = mid + 1;
        else hi = mid;
    }
    return lo;
}

// kRowLanes lanes per scheduled row of a factor: its terms into the dense blocks
// (one lane a row: 0.8 ms for the 120 x 90 building's L).
constexpr int kRowLanes = 16;

template <bool UPPER>
__global__ void ops_scatter_kernel(sbf::Tri tri, int nrows, const sbf::Front* fronts, OpsTab o) {
    const int q = (int)((blockIdx.x * blockDim.x + threadIdx.x) / kRowLanes), l = (int)(threadIdx.x % kRowLanes);
    if (q >= nrows) return;
    const int i = tri.rows[q], fi = o.front_of[i];
    if (UPPER) {
        const sbf::Front f = fronts[fi];
        double* D = o.dense + o.d0[fi];
        const int li = o.local[i];
        if (l == 0) D[(size_t)f.w * f.w + (size_t)li * f.w + li] = tri.diag[q];
        for (int e = tri.ptr[q] + l; e < tri.ptr[q + 1]; e += kRowLanes) {
            const int c = tri.col[e];
            if (o.front_of[c] == fi) D[(size_t)f.w * f.w + (size_t)li * f.w + o.local[c]] = tri.val[e];
            else D[2 * (size_t)f.w * f.w + (size_t)f.w * f.r + (size_t)li * f.r + b_index(f, o.bperm, c)] = tri.val[e];
        }
    } else {
        for (int e = tri.ptr[q] + l; e < tri.ptr[q + 1]; e += kRowLanes) {
            const int c = tri.col[e], fc = o.front_of[c], lc = o.local[c];
            const sbf::Front f = fronts[fc];
            double* D = o.dense + o.d0[fc];
            if (fc == fi) D[(size_t)o.local[i] * f.w + lc] = tri.val[e];
            else D[2 * (size_t)f.w * f.w + (size_t)b_index(f, o.bperm, i) * f.w + lc] = tri.val[e];
        }
    }
}

// One lane per column of a front's operators: column c < w of K solves
// L U x = e_c, the next r solve U x = -U_CB, the last r (rows of F) z L = -L_BC.
// A wavefront's 64 columns are kept in LDS; a row's coefficients are the same
// for every lane (scalar loads), in four sums. What bounds it is the latency of
// a row's trips over its coefficients: 32 products a trip, and what is left
// over loaded at once. A 205K-cell plan: columns in global memory and one chain
// a row 32 ms, eight products a trip and the rest one by one 7.3 ms, 5.3 ms so.
struct OpsCol {
    double (*x)[64];
    int lane;
    // sum_q M[q * stride] x[q] over [q0, q1)
    __device__ double dot(const double* M, size_t stride, int q0, int q1) const {
        double s[4] = {0.0, 0.0, 0.0, 0.0};
        int q = q0;
        for (; q + 32 <= q1; q += 32)
#pragma unroll
            for (int u = 0; u < 32; u++) s[u & 3] = fma(M[(size_t)(q + u) * stride], x[q + u][lane], s[u & 3]);
        for (; q + 8 <= q1; q += 8)
#pragma unroll
            for (int u = 0; u < 8; u++) s[u & 3] = fma(M[(size_t)(q + u) * stride], x[q + u][lane], s[u & 3]);
        if (q < q1) {   // the loads of the rest at once too
            double m[8], y[8];
#pragma unroll
            for (int u = 0; u < 8; u++) {
                const int p = min(q + u, q1 - 1);
                m[u] = M[(size_t)p * stride];
                y[u] = x[p][lane];
            }
#pragma unroll
            for (int u = 0; u < 8; u++) s[0] = q + u < q1 ? fma(m[u], y[u], s[0]) : s[0];
        }
        return (s[0] + s[1]) + (s[2] + s[3]);
    }
};

__global__ __launch_bounds__(64) void ops_solve_kernel(const sbf::Front* fronts, OpsTab o) {
    extern __shared__ double lds[];
    const OpsCol X{reinterpret_cast<double (*)[64]>(lds), (int)threadIdx.x};
    const int fi = blockIdx.x;
    const sbf::Front f = fronts[fi];
    const int w = f.w, r = f.r, ld = w + 2 * r;
    const double* L = o.dense + o.d0[fi];
    const double* U = L + (size_t)w * w;
    const double* LB = U + (size_t)w * w;
    const double* UB = LB + (size_t)w * r;
    double* S = o.sol + o.s0[fi];
    // columns of the three kinds apart, 64 at a time, so a wavefront runs one kind
    const int nw = (w + 63) / 64, nr = (r + 63) / 64;
    for (int g = blockIdx.y; g < nw + 2 * nr; g += gridDim.y) {
        const int kind = g < nw ? 0 : g < nw + nr ? 1 : 2;
        const int c = (kind == 0 ? g : kind == 1 ? g - nw : g - nw - nr) * 64 + X.lane;
        const bool ok = c < (kind == 0 ? w : r);
        const int cc = ok ? c : 0;
        if (kind == 2) {
            for (int m = w - 1; m >= 0; m--)
                X.x[m][X.lane] = -LB[(size_t)cc * w + m] - X.dot(L + m, w, m + 1, w);
        } else {
            for (int m = 0; m < w; m++) {
                double b = kind == 0 ? (m == cc ? 1.0 : 0.0) : -UB[(size_t)m * r + cc];
                if (kind == 0) b -= X.dot(L + (size_t)m * w, 1, 0, m);
                X.x[m][X.lane] = b;
            }
            for (int m = w - 1; m >= 0; m--)
                X.x[m][X.lane] = (X.x[m][X.lane] - X.dot(U + (size_t)m * w, 1, m + 1, w)) / U[(size_t)m * w + m];
        }
        const int at = kind == 0 ? c : kind == 1 ? w + c : w + r + c;
        if (ok)
            for (int m = 0; m < w; m++) S[(size_t)m * ld + at] = X.x[m][X.lane];
    }
}

// The solutions into the operators' tiles (rows and columns past the front's are zero).
__global__ void ops_pack_kernel(const sbf::Front* fronts, int n_fronts, OpsTab o, double* ops) {
    for (int fi = blockIdx.x; fi < n_fronts; fi += gridDim.x) {
        const sbf::Front f = fronts[fi];
        const int w = f.w, r = f.r, ld = w + 2 * r, kw = (w + 3) / 4, ks = kw + (r + 3) / 4;
        const double* S = o.sol + o.s0[fi];
        const size_t nF = (size_t)((r + 15) / 16) * kw * 64, nK = (size_t)((w + 15) / 16) * ks * 64;
        for (size_t x = blockIdx.y * blockDim.x + threadIdx.x; x < nF + nK; x += gridDim.y * blockDim.x) {
            const bool up = x < nF;
            const size_t y = up ? x : x - nF;
            const int lane = (int)(y & 63), step = (int)((y >> 6) % (size_t)(up ? kw : ks));
            const int row = (int)((y >> 6) / (size_t)(up ? kw : ks)) * 16 + (lane & 15);
            int col = 4 * step + (lane >> 4);
            double v = 0.0;
            if (up) {
                if (row < r && col < w) v = S[(size_t)col * ld + w + r + row];
            } else if (row < w) {
                if (step < kw) v = col < w ? S[(size_t)row * ld + col] : 0.0;
                else if ((col -= 4 * kw) < r) v = S[(size_t)row * ld + w + col];
            }
            ops[(up ? f.f : f.k) + y] = v;
        }
    }
}

// ------------------------------------------------------------ the rest of the step

// What the env's solution is taken relative to (FrontTab).
__device__ __forceinline__ double base_of(double ambient) { return isfinite(ambient) ? ambient : 0.0; }

// Forcing (sb_fdm.c:147-151, exposure :126-140) less base x row sum: a workgroup takes 64 solved
// cells of one env tile, computes with lanes over cells (the field, the heat
// and the mass are read in the cells' order) and stores rows of 16 envs
// through LDS. Lanes past the group's envs get zeros.
__global__ __launch_bounds__(256) void front_forcing_kernel(sbf::Tables t, sbf::Group g, sbf::StepIn in) {
    __shared__ double fs[64][E + 1];
    const int te = (int)(blockIdx.x % (unsigned)g.nt), t0 = (int)(blockIdx.x / (unsigned)g.nt) * 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int n = t.n, Gl = g.Gl;
    const int tt = min(t0 + lane, n - 1);
    const int p = t.solved[tt];
    const double a0 = t.a0[tt], a1 = t.a1[tt], hz = t.hz[tt], vt = t.vt[tt], cd = t.cd[tt];
    const double cap = t.cap[tt], dir = t.dir[tt], mcoup = t.mcoup[tt], rs = t.ft.rowsum[tt];
    const int z = in.q ? -1 : t.czone[tt];
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int l = wave * 4 + q, env = te * E + l;
        double v = 0.0;
        if (env < g.G) {
            const size_t b = env / Gl, gl = env % Gl;
            const double h = in.h[env];
            double e = 0.0;
            if (a0 > 0.0) e += h * a0 / (1.0 + h * 0.5 * hz / cd);
            if (a1 > 0.0) e += h * a1 / (1.0 + h * 0.5 * vt / cd);
            double heat;
            if (in.q) heat = in.q[(size_t)env * t.n_cvs + p];
            else heat = z >= 0 ? in.qz[(size_t)env * t.nz + z] : 0.0;
            const double amb = in.amb[env], base = base_of(amb);
            v = fma(cap, g.T[(b * t.n_cvs + p) * Gl + gl] - base, heat);
            if (mcoup != 0.0) v = fma(mcoup, g.M[(b * n + tt) * Gl + gl] - base, v);
            v += fma(amb, dir + e, -base * rs);
        }
        fs[lane][l] = v;
    }
    __syncthreads();
    double* Wt = g.W1 + (size_t)te * n * E;
#pragma unroll
    for (int q = 0; q < 4; q++) {
        const int c = q * 16 + (threadIdx.x >> 4);
        if (t0 + c < n) Wt[(size_t)t.ft.rf[t0 + c] * E + (threadIdx.x & 15)] = fs[c][threadIdx.x & 15];
    }
}

// Per sensed row and env tile: the sensed temperature of the solution and the
// air-side power g (T_air - sensed) (sb_fdm.c:157-162), 32 entries at a time
// by 32 x 16 threads, summed in a fixed order.
constexpr int kSensedThreads = 512;
__global__ __launch_bounds__(kSensedThreads) void front_sensed_kernel(sbf::Tables t, sbf::Group g, sbf::StepIn in) {
    constexpr int R = kSensedThreads / E;
    __shared__ double part[R][E];
    const int te = (int)(blockIdx.x % (unsigned)g.nt), i = (int)(blockIdx.x / (unsigned)g.nt);
    const int j = threadIdx.x % E, s = threadIdx.x / E;
    const double* Xb = g.X + (size_t)te * t.n * E + j;
    const double base = base_of(in.amb[min(te * E + j, g.G - 1)]);
    double acc = 0.0;
#pragma unroll 8
    for (int p = t.sn_p[i] + s; p < t.sn_p[i + 1]; p += R) acc += t.sn_x[p] * (base + Xb[(size_t)t.ft.sn_w[p] * E]);
    part[s][j] = acc;
    __syncthreads();
    for (int h = R / 2; h > 0; h >>= 1) {
        if (s < h) part[s][j] += part[s + h][j];
        __syncthreads();
    }
    const int env = te * E + j;
    if (s == 0 && env < g.G) {
        const size_t x = (size_t)env * t.k + i;
        g.pw[x] = in.g[x] * (in.airT[x] - part[0][j]);
    }
}

// y = the forcing solve + R^T q where the air side is on (R's rows the
// solutions of the applied columns, q the dense solve's result: the same y as
// the second solve of sb_fdm.c:171-178 up to rounding), then the interior
// mass and the field (sb_fdm.c:183-187). A workgroup takes 64 solved cells of
// one env tile: 16 cells a wavefront as one MFMA tile over the k columns,
// then through LDS to lanes over cells.
__global__ __launch_bounds__(256) void front_update_kernel(sbf::Tables t, sbf::Group g, sbf::StepIn in) {
    __shared__ double ys[E][64 + 1];
    const int te = (int)(blockIdx.x % (unsigned)g.nt), t0 = (int)(blockIdx.x / (unsigned)g.nt) * 64;
    const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int j = lane & 15, kk = lane >> 4;
    const int n = t.n, k = t.k, Gl = g.Gl;
    const double* Xb = g.X + (size_t)te * n * E + j;
    const double base = base_of(in.amb[min(te * E + j, g.G - 1)]);
    double y[4];
#pragma unroll
    for (int q = 0; q < 4; q++) y[q] = Xb[(size_t)t.ft.rx[min(t0 + wave * 16 + kk + 4 * q, n - 1)] * E];
    if (t.R) {
        const int env = min(te * E + j, g.G - 1);
        const double* qv = g.pw + (size_t)env * k;
        const double* Rb = t.R + min(t0 + wave * 16 + j, n - 1);   // A: row (cell) lane % 16
        d4 acc = {};
#pragma unroll 5
        for (int c = 0; c < k; c += 4) {
            const int col = c + kk;
            const double a = col < k ? Rb[(size_t)min(col, k - 1) * n] : 0.0;
            acc = mfma(a, qv[min(col, k - 1)], acc);
        }
        const bool on = g.eact[env] != 0;
#pragma unroll
        for (int q = 0; q < 4; q++) y[q] = on ? y[q] + acc[q] : y[q];
    }
#pragma unroll
    for (int q = 0; q < 4; q++) ys[j][wave * 16 + kk + 4 * q] = base + y[q];
    __syncthreads();
    const int tt = t0 + lane;
    if (tt < n) {
        const int cell = t.solved[tt];
        const double mr = t.mret[tt], mg = t.mgain[tt];
#pragma unroll
        for (int q = 0; q < 4; q++) {
            const int l = wave * 4 + q, env = te * E + l;
            if (env >= g.G) break;
            const size_t b = env / Gl, gl = env % Gl, mi = (b * n + tt) * Gl + gl;
            const double v = ys[l][lane];
            g.M[mi] = g.M[mi] * mr + mg * v;
            g.T[(b * t.n_cvs + cell) * Gl + gl] = v;
        }
    }
    const size_t tu = (size_t)g.nblk * t.n_unsolved * Gl;
    for (size_t x = (size_t)blockIdx.x * 256 + threadIdx.x; x < tu; x += (size_t)gridDim.x * 256) {
        const size_t bu = x / Gl;
        const int u = (int)(bu % t.n_unsolved);
        const size_t b = bu / t.n_unsolved;
        const int env = (int)(b * Gl + x % Gl);
        if (env < g.G) g.T[(b * t.n_cvs + t.unsolved[u]) * Gl + x % Gl] = in.amb[env];
    }
}

size_t front_lds(bool fused, int rt, int ne, int kw, int wmax) {
    const size_t red = (size_t)kw * rt * ne * 256, b = fused ? (size_t)((wmax + 3) / 4 * 4) * E : 0;
    return sizeof(double) * std::max(red, b);
}

// Workgroups (2 x 2 tiles) below which a height counts as narrow: with fewer
// than two workgroups a CU the matrix cores idle and the chain of latencies is
// what the height costs.
constexpr unsigned kWideGroups = 512;

template <bool DOWN>
void launch_level(const sbf::Tables& t, const sbf::Group& g, int h, hipStream_t s) {
    const sbf::FrontLevel& L = t.ft.levels[h];
    const int t0 = DOWN ? L.k0 : L.f0, m = DOWN ? L.nk : L.nf;
    if (m == 0) return;
    const unsigned nt = (unsigned)g.nt;
    if (h == 0) {
        if (nt > 1) {
            const unsigned waves = (unsigned)((m + 1) / 2) * ((nt + 1) / 2);
            hipLaunchKernelGGL((leaf_kernel<DOWN, 2, 2>), dim3((waves + 3) / 4), dim3(256), 0, s, t.ft, t0, m, t.n,
                               g.nt, g.W1, g.C, g.X);
        } else {
            const unsigned waves = (unsigned)((m + 1) / 2);
            hipLaunchKernelGGL((leaf_kernel<DOWN, 2, 1>), dim3((waves + 3) / 4), dim3(256), 0, s, t.ft, t0, m, t.n,
                               g.nt, g.W1, g.C, g.X);
        }
        return;
    }
    const unsigned wide = (unsigned)((m + 1) / 2) * ((nt + 1) / 2);
    if (nt > 1 && wide >= kWideGroups) {
        if (!DOWN)
            hipLaunchKernelGGL(assemble_kernel, dim3((unsigned)L.nk * nt), dim3(256), 0, s, t.ft, L.k0, L.nk, t.n, g.nt,
                               g.W1, g.Y, g.C);
        hipLaunchKernelGGL((front_kernel<DOWN, false, 2, 2, 4, 4>), dim3(wide), dim3(256),
                           front_lds(false, 2, 2, 4, L.wmax), s, t.ft, t0, m, t.n, g.nt, g.W1, g.Y, g.C, g.X);
    } else {
        hipLaunchKernelGGL((front_kernel<DOWN, !DOWN, 1, 1, 8, 8>), dim3((unsigned)m * nt), dim3(512),
                           front_lds(!DOWN, 1, 1, 8, L.wmax), s, t.ft, t0, m, t.n, g.nt, g.W1, g.Y, g.C, g.X);
    }
}

}  // namespace

extern "C" int sbf_launch_dense(const sbf::Tables* t, const sbf::Group* g, const sbf::StepIn* in, hipStream_t s);

namespace {

void launch_solve(const sbf::Tables& t, const sbf::Group& g, hipStream_t s) {
    for (int h = 0; h < t.ft.n_levels; h++) launch_level<false>(t, g, h, s);
    for (int h = t.ft.n_levels; h-- > 0;) launch_level<true>(t, g, h, s);
}

int launch_pass(const sbf::Tables* t, const sbf::Group* g, const sbf::StepIn* in, hipStream_t s) {
    const unsigned tiles = (unsigned)((t->n + 63) / 64) * (unsigned)g->nt;
    hipLaunchKernelGGL(front_forcing_kernel, dim3(tiles), dim3(256), 0, s, *t, *g, *in);
    launch_solve(*t, *g, s);
    if (t->k > 0) {
        hipLaunchKernelGGL(front_sensed_kernel, dim3((unsigned)t->k * (unsigned)g->nt), dim3(kSensedThreads), 0, s,
                           *t, *g, *in);
        if (int e = sbf_launch_dense(t, g, in, s)) return e;
    }
    hipLaunchKernelGGL(front_update_kernel, dim3(tiles), dim3(256), 0, s, *t, *g, *in);
    return (int)hipGetLastError();
}

}  // namespace

// One batched step of a group in the default mode, in passes over the env
// tiles that the vectors hold: a pass is a group of its own envs, its arrays
// and inputs from its first env on (an env's result does not depend on its pass).
extern "C" int sbf_launch_front_step(const sbf::Tables* t, const sbf::Group* group, const sbf::StepIn* in,
                                     hipStream_t s) {
    const size_t k = t->k, Gl = group->Gl;
    for (int e0 = 0; e0 < group->G; e0 += group->tiles * E) {   // (a multiple of Gl)
        sbf::Group p = *group;
        p.G = std::min(group->G - e0, group->tiles * E);
        p.nblk = (p.G + p.Gl - 1) / p.Gl;
        p.nt = (p.G + E - 1) / E;
        p.T += e0 / Gl * t->n_cvs * Gl;
        p.M += e0 / Gl * t->n * Gl;
        p.pw += e0 * k;
        p.mat += e0 * k * k;
        p.eact += e0;
        sbf::StepIn q = *in;
        if (q.q) q.q += (size_t)e0 * t->n_cvs;
        if (q.qz) q.qz += (size_t)e0 * t->nz;
        if (q.g) q.g += e0 * k;
        if (q.airT) q.airT += e0 * k;
        q.amb += e0;
        q.h += e0;
        if (int e = launch_pass(t, &p, &q, s)) return e;
    }
    return 0;
}

// Worst error of a solve whose solution is all ones: the largest |x - 1| over
// the rows, as the bits of a double that is not negative (a NaN's lie above).
namespace {

__global__ void check_fill_kernel(sbf::Tables t, double* W, unsigned long long* worst) {
    const size_t x = (size_t)blockIdx.x * 256 + threadIdx.x;
    const int tt = (int)(x / E);
    if (x == 0) *worst = 0;
    if (tt < t.n) W[(size_t)t.ft.rf[tt] * E + x % E] = (t.ft.rowsum[tt] + t.mcoup[tt]) + t.cap[tt];
}

__global__ void check_max_kernel(int n, const double* X, unsigned long long* worst) {
    const int row = (int)(blockIdx.x * 256 + threadIdx.x);
    if (row < n) atomicMax(worst, (unsigned long long)__double_as_longlong(fabs(X[(size_t)row * E] - 1.0)));
}

}  // namespace

extern "C" int sbf_launch_front_check(const sbf::Tables* t, const sbf::Group* group, unsigned long long* worst) {
    sbf::Group g = *group;
    g.nt = 1;
    hipLaunchKernelGGL(check_fill_kernel, dim3((unsigned)(((size_t)t->n * E + 255) / 256)), dim3(256), 0, nullptr, *t,
                       g.W1, worst);
    launch_solve(*t, g, nullptr);
    hipLaunchKernelGGL(check_max_kernel, dim3((unsigned)((t->n + 255) / 256)), dim3(256), 0, nullptr, t->n, g.X, worst);
    return (int)hipGetLastError();
}

// The fronts' operators from the factors (rows scheduled in L and U: nl, nu;
// the first leaf_fronts fronts are the leaves),
// on the null stream; front_of, local, bperm: FrontPlan's, on the device;
// d0, s0: per front the offsets of its dense blocks and solutions.
extern "C" int sbf_launch_front_ops(const sbf::Tables* t, int nl, int nu, int leaf_fronts, const int* front_of, const int* local,
                                    const int* bperm, const long long* d0, const long long* s0, double* dense,
                                    double* sol, double* ops) {
    const OpsTab o{front_of, local, bperm, d0, dense, sol, s0};
    const sbf::Front* fr = t->ft.fronts;
    const int nf = t->ft.n_fronts;
    constexpr int rows = 256 / kRowLanes;   // a workgroup's
    if (nl > 0)
        hipLaunchKernelGGL((ops_scatter_kernel<false>), dim3((nl + rows - 1) / rows), dim3(256), 0, nullptr, t->L, nl,
                           fr, o);
    hipLaunchKernelGGL((ops_scatter_kernel<true>), dim3((nu + rows - 1) / rows), dim3(256), 0, nullptr, t->U, nu, fr, o);
    int wmax = 1;
    for (int h = 0; h < t->ft.n_levels; h++) wmax = std::max(wmax, t->ft.levels[h].wmax);
    const size_t lds = sizeof(double) * 64 * (size_t)wmax;
    if (lds > 64 * 1024) {
        const hipError_t e = hipFuncSetAttribute((const void*)ops_solve_kernel,
                                                 hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
        if (e != hipSuccess) return (int)e;
    }
    // leaves (the fronts before the first one above them) have at most 64 columns
    const int leaves = t->ft.n_levels > 1 ? leaf_fronts : nf;
    const size_t small = sizeof(double) * 64 * (size_t)sbf::kLeafCols;
    hipLaunchKernelGGL(ops_solve_kernel, dim3(leaves, 3), dim3(64), small, nullptr, fr, o);
    if (nf > leaves) {
        OpsTab up = o;
        up.d0 += leaves;
        up.s0 += leaves;
        hipLaunchKernelGGL(ops_solve_kernel, dim3(nf - leaves, 16), dim3(64), lds, nullptr, fr + leaves, up);
    }
    hipLaunchKernelGGL(ops_pack_kernel, dim3(nf, 4), dim3(256), 0, nullptr, fr, nf, o, ops);
    return (int)hipGetLastError();
}
