// Multigrid V-cycle kernels: one fused kernel per level on the way down
// (red-black pre-smoothing from a zero guess + residual + restriction),
// one on the way up (prolongation + red-black post-smoothing), and one
// single-workgroup kernel for all levels of at most TAIL_MAX points.
//
// Every kernel stages its operands (b, x, the operator) for a tile plus the
// halo its passes need in LDS with one unrolled load phase, then runs the
// colour passes out of LDS: a sweep reads each coefficient once from HBM
// and pays one memory latency instead of one per pass.  On the 9-point
// coarse levels the red-black passes treat couplings between cells of the
// same colour (the diagonal ones) Jacobi-wise: new values are staged in
// registers and written after a barrier, which keeps the update independent
// of thread order and the cycle symmetric (post-smoothing runs the colours
// in reverse order).
#include "sg_internal.hpp"
#include "sg_mg_common.hpp"
#include "sg_reduce.hpp"

namespace sg {

namespace {

constexpr int NTB = 256;

constexpr int TAIL_MAX = 1024;   // levels with at most this many points run in the tail kernel
// threads of the tail, a 2x2 block of its first level each: 256 for up to 256
// blocks, as on a level of 32 x 32 -- one wavefront per SIMD, so that a
// thread's couplings, weights and vectors fit its registers in FP64 too -- and
// 512 for the longer or odd levels, none of which has more blocks; those have
// half the registers each, and what does not fit stands in LDS (TailArgs)
constexpr int TAIL_NT = 256, TAIL_NT_MAX = 512;
constexpr int MAX_TAIL = 10;
constexpr size_t TAIL_LDS_MAX = 150 * 1024;  // of the tail levels' operators, vectors and weights

struct Slots {
    double* part;
    int max_blocks;
};

__device__ inline bool in_dom(const Dims& D, int i, int j) { return i >= 0 && j >= 0 && i < D.ni && j < D.nj; }

// ---------------------------------------------------------------------------
// 9-point coarse levels that are not in the tail: the operator is read from
// global memory (through the caches) and only b, x live in LDS, which keeps
// occupancy high.  Couplings between cells of one colour (the diagonals) are
// taken Jacobi-wise: a colour pass computes into registers and writes after
// a barrier.

// A 9-point row's couplings (d, west, east, south, north, NE, SW, NW, SE),
// loaded ahead of the passes that use them
template <typename T>
struct Row9 {
    T d, w, e, s, n, ne, sw, nw, se;
};
template <typename T>
__device__ __forceinline__ Row9<T> load_row9(const OpV<T>& A, size_t p, size_t ld) {
    Row9<T> r;
    r.d = A.diag[p];
    r.w = A.cE[p - 1];
    r.e = A.cE[p];
    r.s = A.cN[p - ld];
    r.n = A.cN[p];
    if (A.cNE) {
        r.ne = A.cNE[p];
        r.sw = A.cNE[p - ld - 1];
        r.nw = A.cNW[p];
        r.se = A.cNW[p - ld + 1];
    } else {
        r.ne = r.sw = r.nw = r.se = T(0);
    }
    return r;
}
// coupled_sum over a loaded row (same terms, same order)
template <typename T, typename XF>
__device__ __forceinline__ T row9_sum(const Row9<T>& r, bool nine, XF X) {
    T s = r.w * X(-1, 0) + r.e * X(1, 0) + r.s * X(0, -1) + r.n * X(0, 1);
    if (nine) s += r.ne * X(1, 1) + r.sw * X(-1, -1) + r.nw * X(-1, 1) + r.se * X(1, -1);
    return s;
}

// down: x = S(0; b) (red from zero, then black), r = b - A x, bc = P^T r.
// With tiles of at most NTB cells every coupling and restriction weight the
// passes read is loaded before the first barrier (a few cells per thread):
// the passes then wait on LDS only, which matters on the small levels, where
// a kernel is a chain of memory latencies.
template <typename T, int TW, int TH>
__global__ void __launch_bounds__(NTB) k_down9(Dims F, OpV<T> A, const T* __restrict__ b, T* __restrict__ xo,
                                               Dims C, Prol<T> P, T* __restrict__ bc, const int* on) {
    if (on && !*on) return;
    constexpr int RW = TW + 5, RH = TH + 5;  // local (li,lj) <-> cell (i0+li-3, j0+lj-3)
    constexpr int NL = (RW * RH + NTB - 1) / NTB;
    __shared__ T sb[RH][RW];
    __shared__ T sx[RH][RW];
    int tx, ty;
    xcd_tile(tx, ty);
    const int i0 = tx * TW, j0 = ty * TH;
    const int tid = threadIdx.x;
    const size_t ld = F.ld;
#pragma unroll
    for (int m = 0; m < NL; ++m) {
        const int k = tid + m * NTB;
        if (k >= RW * RH) continue;
        const int li = k % RW, lj = k / RW;
        const int gi = i0 + li - 3, gj = j0 + lj - 3;
        T bv = T(0), xv = T(0);
        if (in_dom(F, gi, gj)) {
            const size_t p = F.off(gi, gj);
            bv = b[p];
            if (((gi + gj) & 1) == 0) {
                const T d = A.diag[p];
                xv = d > T(0) ? bv / d : T(0);
            }
        }
        sb[lj][li] = bv;
        sx[lj][li] = xv;
    }
    constexpr bool PRE = TW * TH <= NTB;
    const bool nine = A.cNE != nullptr;
    constexpr int PR = (RW - 1) / 2;
    constexpr int NBK = (PR * (RH - 2) + NTB - 1) / NTB;
    constexpr int NRS = ((TW + 1) * (TH + 1) + NTB - 1) / NTB;
    // black cell n of this thread: local (li, lj), or li < 0
    auto black_cell = [&](int n, int& li, int& lj) {
        const int k = tid + n * NTB;
        li = -1;
        lj = 0;
        if (k >= PR * (RH - 2)) return;
        lj = k / PR + 1;
        const int l = 2 * (k % PR) + 1 + (lj & 1);
        if (l >= RW - 1 || !in_dom(F, i0 + l - 3, j0 + lj - 3)) return;
        li = l;
    };
    Row9<T> rbk[PRE ? NBK : 1], rrs[PRE ? NRS : 1];
    T rw[9];
    if constexpr (PRE) {
#pragma unroll
        for (int n = 0; n < NBK; ++n) {
            int li, lj;
            black_cell(n, li, lj);
            if (li >= 0) rbk[n] = load_row9(A, F.off(i0 + li - 3, j0 + lj - 3), ld);
        }
#pragma unroll
        for (int m = 0; m < NRS; ++m) {
            const int k = tid + m * NTB;
            const int li = k % (TW + 1) + 2, lj = k / (TW + 1) + 2;
            if (k < (TW + 1) * (TH + 1) && in_dom(F, i0 + li - 3, j0 + lj - 3))
                rrs[m] = load_row9(A, F.off(i0 + li - 3, j0 + lj - 3), ld);
        }
        const int I = i0 / 2 + tid % (TW / 2), J = j0 / 2 + tid / (TW / 2);
        if (tid < (TW / 2) * (TH / 2) && I < C.ni && J < C.nj) {
            T* const* w = P.w;
            const size_t c = C.off(I, J), cw = C.off(I - 1, J), cs = C.off(I, J - 1), csw = C.off(I - 1, J - 1);
            rw[0] = w[W_INJ][c];
            rw[1] = w[W_XW][c];
            rw[2] = w[W_XE][cw];
            rw[3] = w[W_YS][c];
            rw[4] = w[W_YN][cs];
            rw[5] = w[W_SW][c];
            rw[6] = w[W_SE][cw];
            rw[7] = w[W_NW][cs];
            rw[8] = w[W_NE][csw];
        }
    }
    __syncthreads();
    // black on [-2,TW+1) x [-2,TH+1); local parity: black <=> (li + lj) odd
    {
        T nv[NBK];
        int pos[NBK];
#pragma unroll
        for (int n = 0; n < NBK; ++n) {
            int li, lj;
            black_cell(n, li, lj);
            pos[n] = -1;
            nv[n] = T(0);
            if (li < 0) continue;
            const Row9<T> R = PRE ? rbk[n] : load_row9(A, F.off(i0 + li - 3, j0 + lj - 3), ld);
            auto X = [&](int di, int dj) { return sx[lj + dj][li + di]; };
            nv[n] = R.d > T(0) ? (sb[lj][li] + row9_sum(R, nine, X)) / R.d : T(0);
            pos[n] = lj * RW + li;
        }
        __syncthreads();
#pragma unroll
        for (int n = 0; n < NBK; ++n)
            if (pos[n] >= 0) (&sx[0][0])[pos[n]] = nv[n];
    }
    __syncthreads();
    // residual on [-1,TW) x [-1,TH), in place over b (each cell reads only
    // its own b)
#pragma unroll
    for (int m = 0; m < NRS; ++m) {
        const int k = tid + m * NTB;
        if (k >= (TW + 1) * (TH + 1)) continue;
        const int li = k % (TW + 1) + 2, lj = k / (TW + 1) + 2;
        const int gi = i0 + li - 3, gj = j0 + lj - 3;
        T r = T(0);
        if (in_dom(F, gi, gj)) {
            const Row9<T> R = PRE ? rrs[m] : load_row9(A, F.off(gi, gj), ld);
            auto X = [&](int di, int dj) { return sx[lj + dj][li + di]; };
            r = sb[lj][li] - R.d * sx[lj][li] + row9_sum(R, nine, X);
        }
        sb[lj][li] = r;
    }
    __syncthreads();
    for (int k = tid; k < (TW / 2) * (TH / 2); k += NTB) {
        const int I = i0 / 2 + k % (TW / 2), J = j0 / 2 + k / (TW / 2);
        if (I < C.ni && J < C.nj) {
            const int li = 2 * I - i0 + 3, lj = 2 * J - j0 + 3;
            auto R = [&](int a, int bb) { return sb[lj + bb][li + a]; };
            if constexpr (PRE) {
                // restrict_point with the weights loaded above (same terms, same order)
                T s = rw[0] * R(0, 0);
                s += rw[1] * R(1, 0) + rw[2] * R(-1, 0);
                s += rw[3] * R(0, 1) + rw[4] * R(0, -1);
                s += rw[5] * R(1, 1) + rw[6] * R(-1, 1) + rw[7] * R(1, -1) + rw[8] * R(-1, -1);
                bc[C.off(I, J)] = s;
            } else {
                bc[C.off(I, J)] = restrict_point<T>(C, P, I, J, R);
            }
        }
    }
    for (int k = tid; k < TW * TH; k += NTB) {
        const int li = k % TW + 3, lj = k / TW + 3;
        const int gi = i0 + li - 3, gj = j0 + lj - 3;
        if (in_dom(F, gi, gj)) xo[F.off(gi, gj)] = sx[lj][li];
    }
}

// up: x = xin + P e, then black and red passes; writes xo
template <typename T, int TW, int TH>
__global__ void __launch_bounds__(NTB) k_up9(Dims F, OpV<T> A, const T* __restrict__ b, const T* __restrict__ xin,
                                             Dims C, Prol<T> P, const T* __restrict__ e, T* __restrict__ xo,
                                             const int* on) {
    if (on && !*on) return;
    constexpr int RW = TW + 4, RH = TH + 4;  // local (li,lj) <-> cell (i0+li-2, j0+lj-2)
    __shared__ T sb[RH][RW];
    __shared__ T sx[RH][RW];
    int tx, ty;
    xcd_tile(tx, ty);
    const int i0 = tx * TW, j0 = ty * TH;
    const int tid = threadIdx.x;
    const size_t ld = F.ld;
    {
        constexpr int BW = RW / 2, BH = RH / 2;
        constexpr int NL2 = (BW * BH + NTB - 1) / NTB;
        const int Ib = i0 / 2 - 1, Jb = j0 / 2 - 1;
#pragma unroll
        for (int m = 0; m < NL2; ++m) {
            const int k = tid + m * NTB;
            if (k >= BW * BH) continue;
            const int a = k % BW, c = k / BW;
            const int I = Ib + a, J = Jb + c;
            T xv[2][2] = {{T(0), T(0)}, {T(0), T(0)}}, bv[2][2] = {{T(0), T(0)}, {T(0), T(0)}};
            if (I >= 0 && J >= 0 && I < C.ni && J < C.nj) {
                const size_t cc = C.off(I, J);
                T* const* w = P.w;
                const T e00 = e[cc], e10 = e[cc + 1], e01 = e[cc + C.ld], e11 = e[cc + C.ld + 1];
                const T pe[2][2] = {
                    {w[W_INJ][cc] * e00, w[W_XW][cc] * e00 + w[W_XE][cc] * e10},
                    {w[W_YS][cc] * e00 + w[W_YN][cc] * e01,
                     w[W_SW][cc] * e00 + w[W_SE][cc] * e10 + w[W_NW][cc] * e01 + w[W_NE][cc] * e11}};
#pragma unroll
                for (int dj = 0; dj < 2; ++dj)
#pragma unroll
                    for (int di = 0; di < 2; ++di) {
                        const int gi = 2 * I + di, gj = 2 * J + dj;
                        if (gi < F.ni && gj < F.nj) {
                            const size_t p = F.off(gi, gj);
                            bv[dj][di] = b[p];
                            xv[dj][di] = xin[p] + pe[dj][di];
                        }
                    }
            }
#pragma unroll
            for (int dj = 0; dj < 2; ++dj)
#pragma unroll
                for (int di = 0; di < 2; ++di) {
                    sb[2 * c + dj][2 * a + di] = bv[dj][di];
                    sx[2 * c + dj][2 * a + di] = xv[dj][di];
                }
        }
    }
    // with tiles of at most NTB cells, the couplings of the black cells and
    // of the red tile cell of this thread are loaded before the first barrier
    constexpr bool PRE = TW * TH <= NTB;
    const bool nine = A.cNE != nullptr;
    constexpr int PR = (RW - 2) / 2;
    constexpr int NBK = (PR * (RH - 2) + NTB - 1) / NTB;
    auto black_cell = [&](int m, int& li, int& lj) {
        const int k = tid + m * NTB;
        li = -1;
        lj = 0;
        if (k >= PR * (RH - 2)) return;
        lj = k / PR + 1;
        const int l = 2 * (k % PR) + 1 + (lj & 1);
        if (l >= RW - 1 || !in_dom(F, i0 + l - 2, j0 + lj - 2)) return;
        li = l;
    };
    Row9<T> rbk[PRE ? NBK : 1], rred;
    if constexpr (PRE) {
#pragma unroll
        for (int m = 0; m < NBK; ++m) {
            int li, lj;
            black_cell(m, li, lj);
            if (li >= 0) rbk[m] = load_row9(A, F.off(i0 + li - 2, j0 + lj - 2), ld);
        }
        const int gi = i0 + tid % TW, gj = j0 + tid / TW;
        if (tid < TW * TH && in_dom(F, gi, gj) && ((gi + gj) & 1) == 0) rred = load_row9(A, F.off(gi, gj), ld);
    }
    __syncthreads();
    // black on [-1,TW+1) x [-1,TH+1), staged (Jacobi among black cells)
    {
        T nv[NBK];
        int pos[NBK];
#pragma unroll
        for (int m = 0; m < NBK; ++m) {
            int li, lj;
            black_cell(m, li, lj);
            pos[m] = -1;
            nv[m] = T(0);
            if (li < 0) continue;
            const Row9<T> R = PRE ? rbk[m] : load_row9(A, F.off(i0 + li - 2, j0 + lj - 2), ld);
            auto X = [&](int di, int dj) { return sx[lj + dj][li + di]; };
            nv[m] = R.d > T(0) ? (sb[lj][li] + row9_sum(R, nine, X)) / R.d : T(0);
            pos[m] = lj * RW + li;
        }
        __syncthreads();
#pragma unroll
        for (int m = 0; m < NBK; ++m)
            if (pos[m] >= 0) (&sx[0][0])[pos[m]] = nv[m];
    }
    __syncthreads();
    // red on the tile, written straight out (reads only sx)
    for (int k = tid; k < TW * TH; k += NTB) {
        const int li = k % TW + 2, lj = k / TW + 2;
        const int gi = i0 + li - 2, gj = j0 + lj - 2;
        if (!in_dom(F, gi, gj)) continue;
        const size_t p = F.off(gi, gj);
        T v = sx[lj][li];
        if (((gi + gj) & 1) == 0) {
            const Row9<T> R = PRE ? rred : load_row9(A, p, ld);
            auto X = [&](int di, int dj) { return sx[lj + dj][li + di]; };
            v = R.d > T(0) ? (sb[lj][li] + row9_sum(R, nine, X)) / R.d : T(0);
        }
        xo[p] = v;
    }
}

// ---------------------------------------------------------------------------
// Fine (5-point) level at full size: many tiles hide the memory latency, so
// the operator is read straight from global memory (through the caches)
// rather than staged, which keeps LDS small and occupancy high.
constexpr int GW = 64, GH = 16;  // fine-level tile

// down on the fine level: x = S(0; b) (red from zero, then black), r = b - A
// x, bc = P^T r.  As in the up-sweep, each thread holds the couplings of its
// pairs of tile cells in registers for all three passes; cells of the halo
// read theirs from memory.  SEMI: level 1 coarsens in y only (coarse (I,J)
// on fine (I,2J)).
template <typename T, typename TB, int TW, int TH, bool SEMI>
__global__ void __launch_bounds__(NTB) k_down5(Dims F, OpV<T> A, const TB* __restrict__ b, T* __restrict__ xo,
                                               Dims C, Prol<T> P, T* __restrict__ bc, const int* on) {
    if (on && !*on) return;
    constexpr int RW = TW + 5, RH = TH + 5;  // local (li,lj) <-> cell (i0+li-3, j0+lj-3)
    constexpr int PPR = TW / 2;
    constexpr int PPT = PPR * TH / NTB;
    static_assert(PPR * TH % NTB == 0, "tile pairs must divide among the threads");
    constexpr int NL = (RW * RH + NTB - 1) / NTB;
    __shared__ T sb[RH][RW];
    __shared__ T sx[RH][RW];
    int tx, ty;
    xcd_tile(tx, ty);
    const int i0 = tx * TW, j0 = ty * TH;
    const int tid = threadIdx.x;
    const size_t ld = F.ld;
    T* sxf = &sx[0][0];
    T* sbf = &sb[0][0];
    auto in_tile = [&](int li, int lj) { return li >= 3 && li < TW + 3 && lj >= 3 && lj < TH + 3; };
    auto coef = [&](size_t p, T (&c)[5]) {
        c[0] = A.diag[p];
        c[1] = A.cE[p - 1];
        c[2] = A.cE[p];
        c[3] = A.cN[p - ld];
        c[4] = A.cN[p];
    };
    auto gs = [&](const T (&c)[5], int pos) {
        const T s = c[1] * sxf[pos - 1] + c[2] * sxf[pos + 1] + c[3] * sxf[pos - RW] + c[4] * sxf[pos + RW];
        return c[0] > T(0) ? (sbf[pos] + s) / c[0] : T(0);
    };
    // b; red from a zero guess on the halo (the tile's red cells below)
#pragma unroll
    for (int m = 0; m < NL; ++m) {
        const int k = tid + m * NTB;
        if (k >= RW * RH) continue;
        const int li = k % RW, lj = k / RW;
        const int gi = i0 + li - 3, gj = j0 + lj - 3;
        T bv = T(0), xv = T(0);
        if (in_dom(F, gi, gj)) {
            const size_t p = F.off(gi, gj);
            bv = (T)b[p];
            if (((gi + gj) & 1) == 0 && !in_tile(li, lj)) {
                const T d = A.diag[p];
                xv = d > T(0) ? bv / d : T(0);
            }
        }
        sb[lj][li] = bv;
        sx[lj][li] = xv;
    }
    // every operand the passes below read from memory is loaded here, before
    // the first barrier: the ring cells' couplings and the restriction
    // weights of the thread's coarse point, beside the pairs' couplings
    constexpr int HW = RW - 2, HH = RH - 2;  // the black ring: li, lj in [1, RW-1) x [1, RH-1) off the tile
    constexpr int NBR = 3 * HW + 3 * TH;     // rows 1, 2, TH+3; columns 1, 2, TW+3 of rows 3..TH+2
    static_assert(NBR <= NTB && TW + 1 + TH <= NTB, "one ring cell per thread");
    int bpos = -1;  // this thread's black ring cell (LDS position), -1 if none
    T bcf[5] = {T(0), T(0), T(0), T(0), T(0)};
    if (tid < NBR) {
        int li, lj;
        if (tid < 3 * HW) {
            li = 1 + tid % HW;
            lj = tid < 2 * HW ? 1 + tid / HW : TH + 3;
        } else {
            const int k2 = tid - 3 * HW;
            li = k2 < 2 * TH ? 1 + k2 % 2 : TW + 3;
            lj = k2 < 2 * TH ? 3 + k2 / 2 : 3 + (k2 - 2 * TH);
        }
        const int gi = i0 + li - 3, gj = j0 + lj - 3;
        if (((li + lj) & 1) != 0 && in_dom(F, gi, gj)) {
            coef(F.off(gi, gj), bcf);
            bpos = lj * RW + li;
        }
    }
    int rpos = -1;  // this thread's residual ring cell: row -1 (columns -1..TW-1), column -1 (rows 0..TH-1)
    bool rin = false;
    T rcf[5] = {T(0), T(0), T(0), T(0), T(0)};
    if (tid < TW + 1 + TH) {
        const int li = tid <= TW ? tid + 2 : 2;
        const int lj = tid <= TW ? 2 : tid - TW + 2;
        const int gi = i0 + li - 3, gj = j0 + lj - 3;
        rpos = lj * RW + li;
        rin = in_dom(F, gi, gj);
        if (rin) coef(F.off(gi, gj), rcf);
    }
    static_assert(SEMI || (TW / 2) * (TH / 2) == NTB, "one coarse point per thread");
    T rw[9];
    int rI = -1, rJ = 0;
    if (!SEMI) {
        const int I = i0 / 2 + tid % (TW / 2), J = j0 / 2 + tid / (TW / 2);
        if (I < C.ni && J < C.nj) {
            T* const* w = P.w;
            const size_t c = C.off(I, J), cw = C.off(I - 1, J), cs = C.off(I, J - 1), csw = C.off(I - 1, J - 1);
            rw[0] = w[W_INJ][c];
            rw[1] = w[W_XW][c];
            rw[2] = w[W_XE][cw];
            rw[3] = w[W_YS][c];
            rw[4] = w[W_YN][cs];
            rw[5] = w[W_SW][c];
            rw[6] = w[W_SE][cw];
            rw[7] = w[W_NW][cs];
            rw[8] = w[W_NE][csw];
            rI = I;
            rJ = J;
        }
    }
    // couplings of the thread's pairs: [0] black, [1] red
    T cf[PPT][2][5];
    int cl[PPT][2];
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
        const int k = tid + u * NTB;
        const int lj = k / PPR + 3;
        const int l0 = 2 * (k % PPR) + 3;
        // black <=> (li + lj) odd (i0, j0 even; local offset 3 on both axes)
        const int lb = l0 + (lj & 1), lr = l0 + ((lj + 1) & 1);
        const int ll[2] = {lb, lr};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int gi = i0 + ll[h] - 3, gj = j0 + lj - 3;
            cl[u][h] = -1;
#pragma unroll
            for (int t = 0; t < 5; ++t) cf[u][h][t] = T(0);
            if (!in_dom(F, gi, gj)) continue;
            coef(F.off(gi, gj), cf[u][h]);
            cl[u][h] = lj * RW + ll[h];
        }
    }
    __syncthreads();
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
        const int pos = cl[u][1];
        if (pos >= 0) sxf[pos] = cf[u][1][0] > T(0) ? sbf[pos] / cf[u][1][0] : T(0);
    }
    __syncthreads();
    // black on [-2,TW+1) x [-2,TH+1): the tile's from registers, the halo's
    // from memory (in place: black couples only to red)
#pragma unroll
    for (int u = 0; u < PPT; ++u)
        if (cl[u][0] >= 0) sxf[cl[u][0]] = gs(cf[u][0], cl[u][0]);
    if (bpos >= 0) sxf[bpos] = gs(bcf, bpos);
    __syncthreads();
    // residual on [-1,TW) x [-1,TH), in place over b (each cell reads only
    // its own b)
    auto resid = [&](const T (&c)[5], int pos) {
        return sbf[pos] - c[0] * sxf[pos] +
               (c[1] * sxf[pos - 1] + c[2] * sxf[pos + 1] + c[3] * sxf[pos - RW] + c[4] * sxf[pos + RW]);
    };
    T rt[PPT][2];
#pragma unroll
    for (int u = 0; u < PPT; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h) rt[u][h] = cl[u][h] >= 0 ? resid(cf[u][h], cl[u][h]) : T(0);
    if (rpos >= 0) sbf[rpos] = rin ? resid(rcf, rpos) : T(0);
#pragma unroll
    for (int u = 0; u < PPT; ++u)
#pragma unroll
        for (int h = 0; h < 2; ++h)
            if (cl[u][h] >= 0) sbf[cl[u][h]] = rt[u][h];
    __syncthreads();
    if (SEMI) {
        // P^T r over the fine column: (I,2J) injected, (I,2J+1) by YS(I,J),
        // (I,2J-1) by YN(I,J-1)
        for (int k = tid; k < TW * (TH / 2); k += NTB) {
            const int I = i0 + k % TW, J = j0 / 2 + k / TW;
            if (I < C.ni && J < C.nj) {
                const int li = I - i0 + 3, lj = 2 * J - j0 + 3;
                const size_t cc = C.off(I, J);
                bc[cc] = P.w[W_INJ][cc] * sb[lj][li] + P.w[W_YS][cc] * sb[lj + 1][li] +
                         P.w[W_YN][cc - C.ld] * sb[lj - 1][li];
            }
        }
    } else if (rI >= 0) {
        // restrict_point with the weights loaded above (same terms, same order)
        const int li = 2 * rI - i0 + 3, lj = 2 * rJ - j0 + 3;
        auto R = [&](int a, int bb) { return sb[lj + bb][li + a]; };
        T s = rw[0] * R(0, 0);
        s += rw[1] * R(1, 0) + rw[2] * R(-1, 0);
        s += rw[3] * R(0, 1) + rw[4] * R(0, -1);
        s += rw[5] * R(1, 1) + rw[6] * R(-1, 1) + rw[7] * R(1, -1) + rw[8] * R(-1, -1);
        bc[C.off(rI, rJ)] = s;
    }
    for (int k = tid; k < TW * TH; k += NTB) {
        const int li = k % TW + 3, lj = k / TW + 3;
        const int gi = i0 + li - 3, gj = j0 + lj - 3;
        if (in_dom(F, gi, gj)) xo[F.off(gi, gj)] = sx[lj][li];
    }
}

// up on the fine level: x = xin + P e, black then red, z = x, dots.  The
// tile's cells are taken in pairs (2m, 2m+1) of a row -- one black, one red
// -- and each thread loads the couplings of its pairs once into registers:
// the black pass uses the black cell's, the red pass the red cell's, so no
// coefficient is read from memory twice.  The one-cell black ring around the
// tile is smoothed from global reads.  b stays in LDS in FP64 for the dots.
// SEMI: level 1 coarsens in y only.
template <typename T, typename V, int TW, int TH, bool SEMI>
__global__ void __launch_bounds__(NTB) k_up5(Dims F, OpV<T> A, const V* __restrict__ b,
                                             const T* __restrict__ xin, Dims C, Prol<T> P, const T* __restrict__ e,
                                             V* __restrict__ z, const V* __restrict__ q, Slots Sl,
                                             const int* on) {
    if (on && !*on) return;
    constexpr int RW = TW + 4, RH = TH + 4;  // local (li,lj) <-> cell (i0+li-2, j0+lj-2)
    constexpr int PPR = TW / 2;              // pairs per row
    constexpr int PPT = PPR * TH / NTB;      // pairs per thread
    static_assert(PPR * TH % NTB == 0, "tile pairs must divide among the threads");
    __shared__ double sb[RH][RW];
    __shared__ T sx[RH][RW];
    int tx, ty;
    xcd_tile(tx, ty);
    const int i0 = tx * TW, j0 = ty * TH;
    const int tid = threadIdx.x;
    const size_t ld = F.ld;
    // b and x + P e per 2x2 block of cells sharing one coarse parent (the
    // region starts on an even cell, so blocks align with coarse cells); with
    // SEMI per 1x2 block (fine (I,2J) and (I,2J+1) of coarse (I,J))
    if (SEMI) {
        constexpr int BW = RW, BH = RH / 2;
        constexpr int NL2 = (BW * BH + NTB - 1) / NTB;
        const int Ib = i0 - 2, Jb = j0 / 2 - 1;
#pragma unroll
        for (int m = 0; m < NL2; ++m) {
            const int k = tid + m * NTB;
            if (k >= BW * BH) continue;
            const int a = k % BW, cr = k / BW;
            const int I = Ib + a, J = Jb + cr;
            T xv[2] = {T(0), T(0)};
            double bv[2] = {0.0, 0.0};
            if (I >= 0 && J >= 0 && I < C.ni && J < C.nj) {
                const size_t cc = C.off(I, J);
                T* const* w = P.w;
                const T e00 = e[cc], e01 = e[cc + C.ld];
                const T pe[2] = {w[W_INJ][cc] * e00, w[W_YS][cc] * e00 + w[W_YN][cc] * e01};
#pragma unroll
                for (int dj = 0; dj < 2; ++dj) {
                    const int gj = 2 * J + dj;
                    if (gj < F.nj) {
                        const size_t p = F.off(I, gj);
                        bv[dj] = (double)b[p];
                        xv[dj] = xin[p] + pe[dj];
                    }
                }
            }
#pragma unroll
            for (int dj = 0; dj < 2; ++dj) {
                sb[2 * cr + dj][a] = bv[dj];
                sx[2 * cr + dj][a] = xv[dj];
            }
        }
    } else {
        constexpr int BW = RW / 2, BH = RH / 2;
        constexpr int NL2 = (BW * BH + NTB - 1) / NTB;
        const int Ib = i0 / 2 - 1, Jb = j0 / 2 - 1;
#pragma unroll
        for (int m = 0; m < NL2; ++m) {
            const int k = tid + m * NTB;
            if (k >= BW * BH) continue;
            const int a = k % BW, c = k / BW;
            const int I = Ib + a, J = Jb + c;
            T xv[2][2] = {{T(0), T(0)}, {T(0), T(0)}};
            double bv[2][2] = {{0.0, 0.0}, {0.0, 0.0}};
            if (I >= 0 && J >= 0 && I < C.ni && J < C.nj) {
                const size_t cc = C.off(I, J);
                T* const* w = P.w;
                const T e00 = e[cc], e10 = e[cc + 1], e01 = e[cc + C.ld], e11 = e[cc + C.ld + 1];
                const T pe[2][2] = {
                    {w[W_INJ][cc] * e00, w[W_XW][cc] * e00 + w[W_XE][cc] * e10},
                    {w[W_YS][cc] * e00 + w[W_YN][cc] * e01,
                     w[W_SW][cc] * e00 + w[W_SE][cc] * e10 + w[W_NW][cc] * e01 + w[W_NE][cc] * e11}};
#pragma unroll
                for (int dj = 0; dj < 2; ++dj)
#pragma unroll
                    for (int di = 0; di < 2; ++di) {
                        const int gi = 2 * I + di, gj = 2 * J + dj;
                        if (gi < F.ni && gj < F.nj) {
                            const size_t p = F.off(gi, gj);
                            bv[dj][di] = (double)b[p];
                            xv[dj][di] = xin[p] + pe[dj][di];
                        }
                    }
            }
#pragma unroll
            for (int dj = 0; dj < 2; ++dj)
#pragma unroll
                for (int di = 0; di < 2; ++di) {
                    sb[2 * c + dj][2 * a + di] = bv[dj][di];
                    sx[2 * c + dj][2 * a + di] = xv[dj][di];
                }
        }
    }
    // couplings of the thread's pairs: [0] the black cell, [1] the red one
    // (d, west, east, south, north)
    T cf[PPT][2][5];
    int cl[PPT][2];  // LDS position (lj * RW + li), -1 outside the domain
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
        const int k = tid + u * NTB;
        const int lj = k / PPR + 2;
        const int l0 = 2 * (k % PPR) + 2;
        const int lb = l0 + ((lj + 1) & 1), lr = l0 + (lj & 1);  // black <=> (li + lj) odd
        const int ll[2] = {lb, lr};
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int gi = i0 + ll[h] - 2, gj = j0 + lj - 2;
            cl[u][h] = -1;
#pragma unroll
            for (int t = 0; t < 5; ++t) cf[u][h][t] = T(0);
            if (!in_dom(F, gi, gj)) continue;
            const size_t p = F.off(gi, gj);
            cf[u][h][0] = A.diag[p];
            cf[u][h][1] = A.cE[p - 1];
            cf[u][h][2] = A.cE[p];
            cf[u][h][3] = A.cN[p - ld];
            cf[u][h][4] = A.cN[p];
            cl[u][h] = lj * RW + ll[h];
        }
    }
    __syncthreads();
    T* sxf = &sx[0][0];
    const double* sbf = &sb[0][0];
    auto gs = [&](const T (&c)[5], int pos) {
        const T s = c[1] * sxf[pos - 1] + c[2] * sxf[pos + 1] + c[3] * sxf[pos - RW] + c[4] * sxf[pos + RW];
        return c[0] > T(0) ? ((T)sbf[pos] + s) / c[0] : T(0);
    };
    // black: the tile's black cells from registers, the ring from memory (in
    // place: black couples only to red)
#pragma unroll
    for (int u = 0; u < PPT; ++u)
        if (cl[u][0] >= 0) sxf[cl[u][0]] = gs(cf[u][0], cl[u][0]);
    {
        // ring cells: rows -1 and TH (columns -1..TW), columns -1 and TW (rows 0..TH-1)
        constexpr int NRING = 2 * (TW + 2) + 2 * TH;
        for (int k = tid; k < NRING; k += NTB) {
            int li, lj;
            if (k < TW + 2) {
                li = k + 1;
                lj = 1;
            } else if (k < 2 * (TW + 2)) {
                li = k - (TW + 2) + 1;
                lj = TH + 2;
            } else {
                const int r = k - 2 * (TW + 2);
                li = (r & 1) ? TW + 2 : 1;
                lj = r / 2 + 2;
            }
            if (((li + lj) & 1) == 0) continue;  // red
            const int gi = i0 + li - 2, gj = j0 + lj - 2;
            if (!in_dom(F, gi, gj)) continue;
            const size_t p = F.off(gi, gj);
            const T c[5] = {A.diag[p], A.cE[p - 1], A.cE[p], A.cN[p - ld], A.cN[p]};
            sxf[lj * RW + li] = gs(c, lj * RW + li);
        }
    }
    __syncthreads();
    // red from registers; z = x, dots (b, z), (z, q)
    double v0 = 0.0, v1 = 0.0;
#pragma unroll
    for (int u = 0; u < PPT; ++u) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
            const int pos = cl[u][h];
            if (pos < 0) continue;
            const T v = h ? gs(cf[u][1], pos) : sxf[pos];
            const int li = pos % RW, lj = pos / RW;
            const size_t p = F.off(i0 + li - 2, j0 + lj - 2);
            const V zs = (V)v;
            const double zv = (double)zs;
            z[p] = zs;
            v0 += sbf[pos] * zv;
            v1 += zv * (double)q[p];
        }
    }
    double vv[2] = {v0, v1};
    block_partials<2, NTB>(vv, Sl.part, Sl.max_blocks);
}

// the fine-level kernels with the level-1 coarsening chosen at run time
template <typename T, typename TB>
void launch_down5(bool semi, hipStream_t s, Dims F, OpV<T> A, const TB* b, T* xo, Dims C, Prol<T> P, T* bc,
                  const int* on) {
    const dim3 g((F.ni + GW - 1) / GW, (F.nj + GH - 1) / GH);
    if (semi)
        hipLaunchKernelGGL((k_down5<T, TB, GW, GH, true>), g, dim3(NTB), 0, s, F, A, b, xo, C, P, bc, on);
    else
        hipLaunchKernelGGL((k_down5<T, TB, GW, GH, false>), g, dim3(NTB), 0, s, F, A, b, xo, C, P, bc, on);
}

template <typename T, typename V>
void launch_up5(bool semi, hipStream_t s, Dims F, OpV<T> A, const V* b, const T* xin, Dims C, Prol<T> P,
                const T* e, V* z, const V* q, Slots S, const int* on) {
    const dim3 g((F.ni + GW - 1) / GW, (F.nj + GH - 1) / GH);
    if (semi)
        hipLaunchKernelGGL((k_up5<T, V, GW, GH, true>), g, dim3(NTB), 0, s, F, A, b, xin, C, P, e, z, q, S, on);
    else
        hipLaunchKernelGGL((k_up5<T, V, GW, GH, false>), g, dim3(NTB), 0, s, F, A, b, xin, C, P, e, z, q, S, on);
}

// ---------------------------------------------------------------------------
// tail: levels lt..nlev-1 in one workgroup.
//
// Nothing here is bound by bytes or operations: a V-cycle of these levels is a
// chain of some twenty passes, each waiting for the neighbours' values of the
// one before, so a pass costs an LDS round trip, its arithmetic's latency and a
// barrier.  The split keeps that chain short:
//   level 0 (lt)   a thread owns a 2x2 block of cells, its couplings and
//                  values in registers; LDS carries only what neighbours read.
//                  The block is one point of level 1,
//   level 1        which the same thread owns: the restricted residual and the
//                  prolongation's weights never leave its registers;
//   levels 2..     small enough for one wavefront as a rule, which then runs
//                  them without barriers while the others wait at one.
// A colour pass reads the other colour from one array and writes its own to
// another, so one barrier ends it.  Sums keep one order of terms and cells,
// which is the level's and not that of the threads.  At 32 x 32 points, 4 inner
// iterations, FP64 / FP32: 42.1 / 39.7 us; with a thread per cell, every level in
// LDS and sixteen wavefronts at each barrier, 59.9 / 55.4 us.  At 31 x 33, whose
// 272 blocks take 512 threads: 61.9 / 52.4 us against 78.0 / 71.5 (82.4 / 59.9 with
// all weights in registers, of which the compiler spilled 210 / 8).
enum { TA_D = 0, TA_E, TA_N, TA_NE, TA_NW, TA_X, TA_B, TA_R, TA_COUNT };

template <typename T>
struct TailLevel {
    Dims d;   // global layout
    Dims cd;  // LDS layout of a level >= 2
    int base;  // LDS offset (elements) of such a level's TA_COUNT arrays
    int wbase; // LDS offset of its 9 prolongation-weight arrays (next level's cd)
    int sh;    // thread k of a pass takes cell (k & (2^sh - 1), k >> sh), 2^sh >= ni
    OpV<T> A;
    Prol<T> P;  // to the next level
    T* x;       // global x of the level (written back for the first tail level)
    const T* b; // global b (read for the first tail level)
};

template <typename T>
struct TailArgs {
    int n;  // number of tail levels (the last is the coarsest)
    TailLevel<T> L[MAX_TAIL];
    const double* inv;  // dense inverse of the coarsest operator (FP64 in both precisions)
    const int* on; // the PCG's convergence flag (the cycle runs while *on), or null
    int krylov;    // inner flexible-CG iterations on the first tail level (0: one V-cycle)
    int ld0, x0, x1;  // level 0's arrays XA, XB: element (i, j) at (j + 1) * ld0 + i + 1
    int ld1, y0, y1;  // level 1's arrays YA, YB, likewise
    int lin;          // three level 0 vectors in linear order (inner iterations)
    int n1;           // points of level 1, the threads with a block
    // TAIL_NT_MAX threads: weights in LDS, nine planes each, of the restriction to
    // level 2 and (tail_staged) of the restriction from a block and the
    // prolongation to it
    int w2, rw1, pw1;
};

// whether TAIL_NT_MAX threads keep the weights between the first two levels in LDS:
// at most 114 KB with them on any level that fits the budget, 88 KB in FP32 without
template <typename T>
constexpr bool tail_staged = sizeof(T) == 8;

// offset of cell (i,j) in the LDS arrays of a level >= 2 (compact layout)
__device__ inline int toff(const Dims& D, int i, int j) { return (j + 2) * D.ld + i; }

template <typename T>
__device__ inline T* tarr(T* lds, const TailLevel<T>& L, int k) {
    return lds + L.base + (size_t)k * L.cd.alloc_elems();
}

// ends a pass of the threads that run levels >= 2: the whole workgroup, or one
// wavefront, whose LDS accesses are in order and only must not be moved
template <bool WAVE>
__device__ __forceinline__ void tail_sync() {
    if (WAVE) {
        __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
        __builtin_amdgcn_wave_barrier();
    } else {
        __syncthreads();
    }
}
// threads that run them
template <bool WAVE>
__device__ __forceinline__ int tail_threads() {
    return WAVE ? 64 : (int)blockDim.x;
}

// One colour pass on a level >= 2, double-buffered: the cells of colour `col`
// get (b + sum of couplings * src) / d, the others keep src; every cell is
// written to dst, so one barrier ends the pass (same-colour diagonal couplings
// read src, i.e. Jacobi-wise).  zero_start: src = 0.
template <bool WAVE, typename T>
__device__ void tail_pass(T* lds, const TailLevel<T>& L, const T* src, T* dst, int col, bool zero_start) {
    const Dims& D = L.cd;
    const int ld = D.ld;
    const T* d = tarr(lds, L, TA_D);
    const T* e = tarr(lds, L, TA_E);
    const T* nn = tarr(lds, L, TA_N);
    const T* ne = tarr(lds, L, TA_NE);
    const T* nw = tarr(lds, L, TA_NW);
    const T* b = tarr(lds, L, TA_B);
    const int mask = (1 << L.sh) - 1;
    for (int k = threadIdx.x; k < (D.nj << L.sh); k += tail_threads<WAVE>()) {
        const int i = k & mask, j = k >> L.sh;
        if (i >= D.ni) continue;
        const int p = toff(D, i, j);
        T v = zero_start ? T(0) : src[p];
        if (((i + j) & 1) == col) {
            const T dd = d[p];
            if (zero_start) {
                v = dd > T(0) ? b[p] / dd : T(0);
            } else {
                const T s = e[p - 1] * src[p - 1] + e[p] * src[p + 1] + nn[p - ld] * src[p - ld] +
                            nn[p] * src[p + ld] + ne[p] * src[p + ld + 1] + ne[p - ld - 1] * src[p - ld - 1] +
                            nw[p] * src[p + ld - 1] + nw[p - ld + 1] * src[p - ld + 1];
                v = dd > T(0) ? (b[p] + s) / dd : T(0);
            }
        }
        dst[p] = v;
    }
    tail_sync<WAVE>();
}

// dense solve on the coarsest level in FP64 (in both precisions): four threads
// per row of the inverse in LDS, B(q) and X(row) the level's values.  Run by
// the first wavefront.
template <typename BF, typename XF>
__device__ __forceinline__ void tail_dense(const double* inv, int n, BF B, XF X) {
    const int row = threadIdx.x >> 2, quarter = threadIdx.x & 3;
    double s = 0.0;
    if (row < n)
        for (int q = quarter; q < n; q += 4) s += inv[row * n + q] * (double)B(q);
    s += __shfl_xor(s, 1, 64);
    s += __shfl_xor(s, 2, 64);
    if (row < n && quarter == 0) X(row, s);
}

// V-cycle on the levels 2.. from level 2's TA_B to its TA_R (a.n > 2).  On
// every level the smoothed x ends in TA_R; TA_X holds the first pass and then
// the residual that is restricted.
template <bool WAVE, typename T>
__device__ void tail_lower(T* lds, const TailArgs<T>& a, const double* inv) {
    const int NTH = tail_threads<WAVE>();
    const int tid = threadIdx.x;
    const int last = a.n - 1;
    for (int l = 2; l < last; ++l) {
        const TailLevel<T>& L = a.L[l];
        const TailLevel<T>& Cl = a.L[l + 1];
        const Dims& D = L.cd;
        const int ld = D.ld;
        T* r = tarr(lds, L, TA_X);
        T* x = tarr(lds, L, TA_R);
        const T* b = tarr(lds, L, TA_B);
        tail_pass<WAVE, T>(lds, L, nullptr, r, 0, true);
        tail_pass<WAVE, T>(lds, L, r, x, 1, false);
        const T* d = tarr(lds, L, TA_D);
        const T* e = tarr(lds, L, TA_E);
        const T* nn = tarr(lds, L, TA_N);
        const T* ne = tarr(lds, L, TA_NE);
        const T* nw = tarr(lds, L, TA_NW);
        const int mask = (1 << L.sh) - 1;
        for (int k = tid; k < (D.nj << L.sh); k += NTH) {
            const int i = k & mask;
            if (i >= D.ni) continue;
            const int p = toff(D, i, k >> L.sh);
            const T s = e[p - 1] * x[p - 1] + e[p] * x[p + 1] + nn[p - ld] * x[p - ld] + nn[p] * x[p + ld] +
                        ne[p] * x[p + ld + 1] + ne[p - ld - 1] * x[p - ld - 1] + nw[p] * x[p + ld - 1] +
                        nw[p - ld + 1] * x[p - ld + 1];
            r[p] = b[p] - d[p] * x[p] + s;
        }
        tail_sync<WAVE>();
        T* bc = tarr(lds, Cl, TA_B);
        const Dims& Cd = Cl.cd;
        const int ws = (int)Cd.alloc_elems(), cld = Cd.ld;
        const T* w0 = lds + L.wbase;
        const int cmask = (1 << Cl.sh) - 1;
        for (int k = tid; k < (Cd.nj << Cl.sh); k += NTH) {
            const int I = k & cmask, J = k >> Cl.sh;
            if (I >= Cd.ni) continue;
            const int c = toff(Cd, I, J), f = toff(D, 2 * I, 2 * J);
            const T* w = w0 + c;
            T s = w[W_INJ * ws] * r[f];
            s += w[W_XW * ws] * r[f + 1] + w[W_XE * ws - 1] * r[f - 1];
            s += w[W_YS * ws] * r[f + ld] + w[W_YN * ws - cld] * r[f - ld];
            s += w[W_SW * ws] * r[f + ld + 1] + w[W_SE * ws - 1] * r[f + ld - 1] + w[W_NW * ws - cld] * r[f - ld + 1] +
                 w[W_NE * ws - cld - 1] * r[f - ld - 1];
            bc[c] = s;
        }
        tail_sync<WAVE>();
    }
    {
        const TailLevel<T>& L = a.L[last];
        const Dims& D = L.cd;
        const T* b = tarr(lds, L, TA_B);
        T* x = tarr(lds, L, TA_R);
        if (tid < 64)
            tail_dense(inv, D.ni * D.nj, [&](int q) { return b[D.off(q % D.ni, q / D.ni)]; },
                       [&](int q, double v) { x[D.off(q % D.ni, q / D.ni)] = (T)v; });
        tail_sync<WAVE>();
    }
    for (int l = last - 1; l >= 2; --l) {
        const TailLevel<T>& L = a.L[l];
        const TailLevel<T>& Cl = a.L[l + 1];
        const Dims& D = L.cd;
        const Dims& Cd = Cl.cd;
        const int ws = (int)Cd.alloc_elems(), cld = Cd.ld;
        const T* w0 = lds + L.wbase;
        const T* ec = tarr(lds, Cl, TA_R);
        T* xa = tarr(lds, L, TA_X);
        T* xb = tarr(lds, L, TA_R);
        const int mask = (1 << L.sh) - 1;
        for (int k = tid; k < (D.nj << L.sh); k += NTH) {
            const int i = k & mask, j = k >> L.sh;
            if (i >= D.ni) continue;
            const int c = toff(Cd, i >> 1, j >> 1);
            const T* w = w0 + c;
            const int pi = i & 1, pj = j & 1;
            T v;
            if (!pi && !pj) v = w[W_INJ * ws] * ec[c];
            else if (pi && !pj) v = w[W_XW * ws] * ec[c] + w[W_XE * ws] * ec[c + 1];
            else if (!pi && pj) v = w[W_YS * ws] * ec[c] + w[W_YN * ws] * ec[c + cld];
            else v = w[W_SW * ws] * ec[c] + w[W_SE * ws] * ec[c + 1] + w[W_NW * ws] * ec[c + cld] +
                     w[W_NE * ws] * ec[c + cld + 1];
            xb[toff(D, i, j)] += v;
        }
        tail_sync<WAVE>();
        tail_pass<WAVE, T>(lds, L, xb, xa, 1, false);
        tail_pass<WAVE, T>(lds, L, xa, xb, 0, false);
    }
}

// A row's couplings in registers (all zero for a point outside the level)
template <typename T>
__device__ __forceinline__ Row9<T> tail_row(const TailLevel<T>& L, int i, int j) {
    if (i < L.d.ni && j < L.d.nj) return load_row9(L.A, L.d.off(i, j), L.d.ld);
    return Row9<T>{};
}
// sums of couplings * neighbours, one order everywhere; axis_sum where the
// diagonal neighbours are zero
template <typename T>
__device__ __forceinline__ T axis_sum(const Row9<T>& r, T w, T e, T s, T n) {
    return r.w * w + r.e * e + r.s * s + r.n * n;
}
template <typename T>
__device__ __forceinline__ T full_sum(const Row9<T>& r, T w, T e, T s, T n, T ne, T sw, T nw, T se) {
    return r.w * w + r.e * e + r.s * s + r.n * n + r.ne * ne + r.sw * sw + r.nw * nw + r.se * se;
}
// Gauss-Seidel value of a row from its right-hand side and that sum
template <typename T>
__device__ __forceinline__ T relaxed(const Row9<T>& r, T b, T s) {
    return r.d > T(0) ? (b + s) / r.d : T(0);
}
// x + v with v rounded first (a correction is one value whatever its number of terms)
template <typename T>
__device__ __forceinline__ T corrected(T x, T v) {
#pragma clang fp contract(off)
    return x + v;
}

// The restriction's weights of coarse point (I, J), in restrict_point's order,
// and the prolongation's to the 2x2 cells of that point
template <typename T>
__device__ __forceinline__ void restrict_weights(const Dims& C, const Prol<T>& P, int I, int J, T (&rw)[9]) {
    T* const* w = P.w;
    const size_t c = C.off(I, J), cw = C.off(I - 1, J), cs = C.off(I, J - 1), csw = C.off(I - 1, J - 1);
    rw[0] = w[W_INJ][c];
    rw[1] = w[W_XW][c];
    rw[2] = w[W_XE][cw];
    rw[3] = w[W_YS][c];
    rw[4] = w[W_YN][cs];
    rw[5] = w[W_SW][c];
    rw[6] = w[W_SE][cw];
    rw[7] = w[W_NW][cs];
    rw[8] = w[W_NE][csw];
}

// Sums over the cells of level 0 in their linear order, returned to every
// thread: F(t, v) gives cell t's terms; 64 cells reduce as a wavefront's
// butterfly, the groups of 64 add up in order.  (The order is the level's, not
// the threads' that own its blocks.)  part is not reused before another barrier.
constexpr int TAIL_GROUPS = TAIL_MAX / 64;
template <int NT, int NV, typename CellF>
__device__ __forceinline__ void tail_allreduce(CellF F, double (&sum)[NV], double (*part)[NV]) {
    double v[TAIL_MAX / NT][NV];
#pragma unroll
    for (int g = 0; g < TAIL_MAX / NT; ++g) F((int)threadIdx.x + g * NT, v[g]);
#pragma unroll
    for (int k = 0; k < NV; ++k)
#pragma unroll
        for (int m = 32; m >= 1; m >>= 1)
#pragma unroll
            for (int g = 0; g < TAIL_MAX / NT; ++g) v[g][k] += __shfl_xor(v[g][k], m, 64);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int g = 0; g < TAIL_MAX / NT; ++g)
#pragma unroll
            for (int k = 0; k < NV; ++k) part[(threadIdx.x >> 6) + g * (NT / 64)][k] = v[g][k];
    __syncthreads();
#pragma unroll
    for (int k = 0; k < NV; ++k) {
        double s = 0.0;
#pragma unroll
        for (int w = 0; w < TAIL_GROUPS; ++w) s += part[w][k];
        sum[k] = s;
    }
}

// A thread's part of the levels
template <typename T>
struct TailOwn {
    // level 0: cells 0 (2I,2J), 1 (2I+1,2J), 2 (2I,2J+1), 3 (2I+1,2J+1); 0 and 3 are red
    Row9<T> r[4];
    int p;     // LDS offset of cell 0
    bool own;  // the thread has a block, and point (I, J) of level 1
    // level 1
    Row9<T> r1;
    int p1;
    bool red1;
    T rw[9], pw[9];  // restriction from the block and prolongation to it
    T pw1[4];        // its prolongation from level 2: from point e2, the one east of it, north, north-east
    int par1, e2;    // parity bits (x, y) of the point
    // level 2
    Row9<T> r2;
    int c2, f2;  // LDS offset of the thread's point (-1: none), and of the level 1 point on it
    bool red2;
    T rw2[9];
};

// cells around a block: south row, west and east columns, north row
template <typename T>
struct Ring12 {
    T s0, s1, s2, s3, w0, w1, e0, e1, n0, n1, n2, n3;
};
template <typename T>
__device__ __forceinline__ Ring12<T> ring(const T* x, int ld) {
    return Ring12<T>{x[-ld - 1], x[-ld],    x[-ld + 1],    x[-ld + 2], x[-1],         x[ld - 1],
                     x[2],       x[ld + 2], x[2 * ld - 1], x[2 * ld],  x[2 * ld + 1], x[2 * ld + 2]};
}
// sum of couplings * x over the neighbours of each cell of the block
template <typename T>
__device__ __forceinline__ void block_sums(const TailOwn<T>& O, const Ring12<T>& g, const T (&x)[4], T (&s)[4]) {
    s[0] = full_sum(O.r[0], g.w0, x[1], g.s1, x[2], x[3], g.s0, g.w1, g.s2);
    s[1] = full_sum(O.r[1], x[0], g.e0, g.s2, x[3], g.e1, g.s1, x[2], g.s3);
    s[2] = full_sum(O.r[2], g.w1, x[3], x[0], g.n1, g.n2, g.w0, g.n0, x[1]);
    s[3] = full_sum(O.r[3], x[2], g.e1, x[1], g.n2, g.n3, x[0], g.n1, g.e0);
}
// the sum over a point's eight neighbours in an array
template <typename T>
__device__ __forceinline__ T point_sum(const Row9<T>& r, const T* x, int ld) {
    return full_sum(r, x[-1], x[1], x[-ld], x[ld], x[ld + 1], x[-ld - 1], x[ld - 1], x[1 - ld]);
}

// Level 2 and the dense solve below it on one wavefront, a point a lane (a.n =
// 4): from the right-hand side b2 to the level's TA_R
template <typename T>
__device__ __forceinline__ void tail_level2(T* lds, const TailArgs<T>& a, const TailOwn<T>& O, const double* inv,
                                            T b2) {
    const TailLevel<T>& L = a.L[2];
    const TailLevel<T>& C = a.L[3];
    const Dims& D = L.cd;
    const Dims& Dc = C.cd;
    const int ld = D.ld;
    const bool own = O.c2 >= 0;
    const int c2 = own ? O.c2 : 0;
    T* xa = tarr(lds, L, TA_X) + c2;
    T* xb = tarr(lds, L, TA_R) + c2;
    T* ec = tarr(lds, C, TA_R);
    T x2 = T(0);
    if (O.red2) x2 = relaxed(O.r2, b2, T(0));
    if (own) xa[0] = x2;
    tail_sync<true>();
    if (own && !O.red2) {
        x2 = relaxed(O.r2, b2, axis_sum(O.r2, xa[-1], xa[1], xa[-ld], xa[ld]));
        xa[0] = x2;
    }
    tail_sync<true>();
    if (own) xb[0] = b2 - O.r2.d * x2 + point_sum(O.r2, xa, ld);
    tail_sync<true>();
    const int ws = (int)Dc.alloc_elems(), cld = Dc.ld;
    const int k3 = threadIdx.x;
    if (k3 < Dc.ni * Dc.nj) {
        const int I = k3 % Dc.ni, J = k3 / Dc.ni;
        const T* r = tarr(lds, L, TA_R) + toff(D, 2 * I, 2 * J);
        const T* w = lds + L.wbase + toff(Dc, I, J);
        T s = w[W_INJ * ws] * r[0];
        s += w[W_XW * ws] * r[1] + w[W_XE * ws - 1] * r[-1];
        s += w[W_YS * ws] * r[ld] + w[W_YN * ws - cld] * r[-ld];
        s += w[W_SW * ws] * r[ld + 1] + w[W_SE * ws - 1] * r[ld - 1] + w[W_NW * ws - cld] * r[1 - ld] +
             w[W_NE * ws - cld - 1] * r[-ld - 1];
        tarr(lds, C, TA_B)[toff(Dc, I, J)] = s;
    }
    tail_sync<true>();
    const T* b3 = tarr(lds, C, TA_B);
    tail_dense(inv, Dc.ni * Dc.nj, [&](int q) { return b3[toff(Dc, q % Dc.ni, q / Dc.ni)]; },
               [&](int q, double v) { ec[toff(Dc, q % Dc.ni, q / Dc.ni)] = (T)v; });
    tail_sync<true>();
    if (own) {
        const int i = threadIdx.x % D.ni, j = threadIdx.x / D.ni;
        const int c = toff(Dc, i >> 1, j >> 1);
        const T* w = lds + L.wbase + c;
        const T* e = ec + c;
        const int pi = i & 1, pj = j & 1;
        T v;
        if (!pi && !pj) v = w[W_INJ * ws] * e[0];
        else if (pi && !pj) v = w[W_XW * ws] * e[0] + w[W_XE * ws] * e[1];
        else if (!pi && pj) v = w[W_YS * ws] * e[0] + w[W_YN * ws] * e[cld];
        else v = w[W_SW * ws] * e[0] + w[W_SE * ws] * e[1] + w[W_NW * ws] * e[cld] + w[W_NE * ws] * e[cld + 1];
        x2 = corrected(x2, v);
        xa[0] = x2;
    }
    tail_sync<true>();
    T dne = T(0), dsw = T(0), dnw = T(0), dse = T(0);
    if (own) {
        dne = xa[ld + 1];
        dsw = xa[-ld - 1];
        dnw = xa[ld - 1];
        dse = xa[1 - ld];
        if (!O.red2) {
            x2 = relaxed(O.r2, b2, full_sum(O.r2, xa[-1], xa[1], xa[-ld], xa[ld], dne, dsw, dnw, dse));
            xb[0] = x2;
        }
    }
    tail_sync<true>();
    if (own && O.red2)
        xb[0] = relaxed(O.r2, b2, full_sum(O.r2, xb[-1], xb[1], xb[-ld], xb[ld], dne, dsw, dnw, dse));
    tail_sync<true>();
}

// One V-cycle over the tail levels: b -> x on the thread's block.  lower: how
// the levels 2.. run (TAIL_LOWER_*).
enum { TAIL_LOWER_ALL = 0, TAIL_LOWER_WAVE, TAIL_LOWER_OWN };
template <int NT, typename T>
__device__ __forceinline__ void tail_vcycle(T* lds, const TailArgs<T>& a, const TailOwn<T>& O, const double* inv,
                                            int lower, const T (&b)[4], T (&x)[4]) {
    constexpr bool MANY = NT > TAIL_NT, STAGED = MANY && tail_staged<T>;
    const int tid = threadIdx.x;
    T* XA = lds + a.x0;
    T* XB = lds + a.x1;
    T* YA = lds + a.y0;
    T* YB = lds + a.y1;
    const int ld = a.ld0, ld1 = a.ld1;
    T* xa = XA + O.p;
    T* xb = XB + O.p;
    if (!MANY && a.n == 1) {
        // the first tail level is the coarsest
        const Dims& D = a.L[0].d;
        if (O.own) {
            xa[0] = b[0];
            xa[1] = b[1];
            xa[ld] = b[2];
            xa[ld + 1] = b[3];
        }
        __syncthreads();
        auto at = [&](int q) { return (q / D.ni + 1) * ld + q % D.ni + 1; };
        if (tid < 64)
            tail_dense(inv, D.ni * D.nj, [&](int q) { return XA[at(q)]; }, [&](int q, double v) { XB[at(q)] = (T)v; });
        __syncthreads();
        if (O.own) {
            x[0] = xb[0];
            x[1] = xb[1];
            x[2] = xb[ld];
            x[3] = xb[ld + 1];
        }
        return;
    }
    // level 0 down: red from zero, black, residual
    x[0] = relaxed(O.r[0], b[0], T(0));
    x[3] = relaxed(O.r[3], b[3], T(0));
    if (O.own) {
        xa[0] = x[0];
        xa[ld + 1] = x[3];
    }
    __syncthreads();
    if (O.own) {
        // the black cells were zero, so only red neighbours count
        x[1] = relaxed(O.r[1], b[1], axis_sum(O.r[1], x[0], xa[2], xa[1 - ld], x[3]));
        x[2] = relaxed(O.r[2], b[2], axis_sum(O.r[2], xa[ld - 1], x[3], x[0], xa[2 * ld]));
        xa[1] = x[1];
        xa[ld] = x[2];
    }
    __syncthreads();
    T r[4] = {T(0), T(0), T(0), T(0)};
    if (O.own) {
        T s[4];
        block_sums(O, ring(xa, ld), x, s);
#pragma unroll
        for (int k = 0; k < 4; ++k) r[k] = b[k] - O.r[k].d * x[k] + s[k];
        xb[0] = r[0];
        xb[1] = r[1];
        xb[ld] = r[2];
        xb[ld + 1] = r[3];
    }
    __syncthreads();
    // level 1: its right-hand side, then the same
    T b1 = T(0), x1 = T(0);
    T* ya = YA + O.p1;
    T* yb = YB + O.p1;
    if (O.own) {
        T w[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = STAGED ? lds[a.rw1 + k * a.n1 + tid] : O.rw[k];
        b1 = w[0] * r[0];
        b1 += w[1] * r[1] + w[2] * xb[-1];
        b1 += w[3] * r[2] + w[4] * xb[-ld];
        b1 += w[5] * r[3] + w[6] * xb[ld - 1] + w[7] * xb[1 - ld] + w[8] * xb[-ld - 1];
    }
    if (!MANY && a.n == 2) {
        const Dims& D = a.L[1].d;
        if (O.own) ya[0] = b1;
        __syncthreads();
        auto at = [&](int q) { return (q / D.ni + 1) * ld1 + q % D.ni + 1; };
        if (tid < 64)
            tail_dense(inv, D.ni * D.nj, [&](int q) { return YA[at(q)]; }, [&](int q, double v) { YB[at(q)] = (T)v; });
        __syncthreads();
    } else {
        if (O.red1) x1 = relaxed(O.r1, b1, T(0));
        if (O.own) ya[0] = x1;
        __syncthreads();
        if (O.own && !O.red1) {
            x1 = relaxed(O.r1, b1, axis_sum(O.r1, ya[-1], ya[1], ya[-ld1], ya[ld1]));
            ya[0] = x1;
        }
        __syncthreads();
        if (O.own) yb[0] = b1 - O.r1.d * x1 + point_sum(O.r1, ya, ld1);
        __syncthreads();
        // levels 2..
        const TailLevel<T>& L2 = a.L[2];
        T b2 = T(0);
        if (O.c2 >= 0) {
            const T* f = YB + O.f2;
            const int n2 = L2.d.ni * L2.d.nj;
            T w[9];
#pragma unroll
            for (int k = 0; k < 9; ++k) w[k] = MANY ? lds[a.w2 + k * n2 + tid] : O.rw2[k];
            b2 = w[0] * f[0];
            b2 += w[1] * f[1] + w[2] * f[-1];
            b2 += w[3] * f[ld1] + w[4] * f[-ld1];
            b2 += w[5] * f[ld1 + 1] + w[6] * f[ld1 - 1] + w[7] * f[1 - ld1] + w[8] * f[-ld1 - 1];
            if (lower != TAIL_LOWER_OWN) tarr(lds, L2, TA_B)[O.c2] = b2;
        }
        if (lower == TAIL_LOWER_OWN) {
            if (tid < 64) tail_level2(lds, a, O, inv, b2);
            __syncthreads();
        } else if (lower == TAIL_LOWER_WAVE) {
            if (tid < 64) {
                tail_sync<true>();
                tail_lower<true, T>(lds, a, inv);
            }
            __syncthreads();
        } else {
            __syncthreads();
            tail_lower<false, T>(lds, a, inv);
        }
        // level 1 up: correction, black, red
        if (O.own) {
            const T* e = tarr(lds, L2, TA_R) + O.e2;
            const int l2 = L2.cd.ld;
            T v;
            if (O.par1 == 0) v = O.pw1[0] * e[0];
            else if (O.par1 == 1) v = fma(O.pw1[0], e[0], O.pw1[1] * e[1]);
            else if (O.par1 == 2) v = fma(O.pw1[0], e[0], O.pw1[2] * e[l2]);
            else v = fma(O.pw1[3], e[l2 + 1], fma(O.pw1[2], e[l2], fma(O.pw1[0], e[0], O.pw1[1] * e[1])));
            x1 = corrected(x1, v);
            ya[0] = x1;
        }
        __syncthreads();
        T dne = T(0), dsw = T(0), dnw = T(0), dse = T(0);
        if (O.own) {
            dne = ya[ld1 + 1];
            dsw = ya[-ld1 - 1];
            dnw = ya[ld1 - 1];
            dse = ya[1 - ld1];
            if (!O.red1) {
                x1 = relaxed(O.r1, b1, full_sum(O.r1, ya[-1], ya[1], ya[-ld1], ya[ld1], dne, dsw, dnw, dse));
                yb[0] = x1;
            }
        }
        __syncthreads();
        // a red point's row of yb holds black cells only; its own place there is not read by others yet
        if (O.red1)
            yb[0] = relaxed(O.r1, b1, full_sum(O.r1, yb[-1], yb[1], yb[-ld1], yb[ld1], dne, dsw, dnw, dse));
        __syncthreads();
    }
    // level 0 up: correction, black, red
    if (O.own) {
        const T e00 = yb[0], e10 = yb[1], e01 = yb[ld1], e11 = yb[ld1 + 1];
        T w[9];
#pragma unroll
        for (int k = 0; k < 9; ++k) w[k] = STAGED ? lds[a.pw1 + k * a.n1 + tid] : O.pw[k];
        x[0] = corrected(x[0], w[0] * e00);
        x[1] = corrected(x[1], w[1] * e00 + w[2] * e10);
        x[2] = corrected(x[2], w[3] * e00 + w[4] * e01);
        x[3] = corrected(x[3], w[5] * e00 + w[6] * e10 + w[7] * e01 + w[8] * e11);
        xa[0] = x[0];
        xa[1] = x[1];
        xa[ld] = x[2];
        xa[ld + 1] = x[3];
    }
    __syncthreads();
    Ring12<T> g{};
    T r0 = T(0), r3 = T(0);
    if (O.own) {
        g = ring(xa, ld);
        r0 = x[0];
        r3 = x[3];
        const T x1n = relaxed(O.r[1], b[1], full_sum(O.r[1], x[0], g.e0, g.s2, x[3], g.e1, g.s1, x[2], g.s3));
        const T x2n = relaxed(O.r[2], b[2], full_sum(O.r[2], g.w1, x[3], x[0], g.n1, g.n2, g.w0, g.n0, x[1]));
        x[1] = x1n;
        x[2] = x2n;
        xb[1] = x1n;
        xb[ld] = x2n;
    }
    __syncthreads();
    if (O.own) {
        x[0] = relaxed(O.r[0], b[0], full_sum(O.r[0], xb[-1], x[1], xb[-ld], x[2], r3, g.s0, g.w1, g.s2));
        x[3] = relaxed(O.r[3], b[3], full_sum(O.r[3], x[2], xb[ld + 2], x[1], xb[2 * ld + 1], g.n3, r0, g.n1, g.e0));
    }
}

// The tail: one V-cycle over levels lt..nlev-1, or -- with a.krylov > 0 --
// that many iterations of flexible CG on level lt preconditioned by the
// V-cycle (x0 = 0; each direction A-orthogonal to the previous one).  The
// coarse levels of a bubbly flow carry slow modes (the pressure of each
// bubble against the liquid around it) that one V-cycle resolves poorly;
// the inner iterations remove them at the cost of a few V-cycles of the
// smallest levels, all inside one workgroup.
template <typename T, int NT>
__global__ void __launch_bounds__(NT) k_tail(TailArgs<T> a, int lds_elems) {
    extern __shared__ __align__(16) unsigned char smem_raw[];
    __shared__ double inv[COARSEST_MAX * COARSEST_MAX];
    __shared__ double part_b[TAIL_GROUPS][2];
    __shared__ double part_a[TAIL_GROUPS][2];
    T* lds = reinterpret_cast<T*>(smem_raw);
    // more than 256 blocks are as many points on level 1 and more than 64 on
    // level 2: there is a level 2, and the whole workgroup runs it
    constexpr bool MANY = NT > TAIL_NT, STAGED = MANY && tail_staged<T>;
    const int tid = threadIdx.x;
    const int live = a.on ? *a.on : 1;
    // everything the passes read from memory, asked for before the flag is looked at
    const TailLevel<T>& L0 = a.L[0];
    const Dims& D0 = L0.d;
    const int ci = (D0.ni + 1) / 2, cj = (D0.nj + 1) / 2;
    const int I = tid % ci, J = tid / ci;
    TailOwn<T> O{};
    O.own = J < cj;
    O.p = O.own ? (2 * J + 1) * a.ld0 + 2 * I + 1 : 0;
    O.p1 = O.own ? (J + 1) * a.ld1 + I + 1 : 0;
    O.c2 = O.f2 = -1;
    T b[4] = {T(0), T(0), T(0), T(0)};
    if (O.own) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = 2 * I + (k & 1), j = 2 * J + (k >> 1);
            O.r[k] = tail_row(L0, i, j);
            if (i < D0.ni && j < D0.nj) b[k] = L0.b[D0.off(i, j)];
        }
        if (!STAGED && a.n > 1) {
            const Dims& D1 = a.L[1].d;
            restrict_weights(D1, L0.P, I, J, O.rw);
#pragma unroll
            for (int k = 0; k < 9; ++k) O.pw[k] = L0.P.w[k][D1.off(I, J)];
        }
        if (a.n > 2) {
            O.r1 = tail_row(a.L[1], I, J);
            O.red1 = ((I + J) & 1) == 0;
            const Dims& D2 = a.L[2].d;
            T* const* w = a.L[1].P.w;
            const size_t c = D2.off(I >> 1, J >> 1);
            const int pi = I & 1, pj = J & 1;
            O.par1 = pi | pj << 1;
            O.e2 = toff(a.L[2].cd, I >> 1, J >> 1);
            O.pw1[0] = w[pi ? (pj ? W_SW : W_XW) : (pj ? W_YS : W_INJ)][c];
            O.pw1[1] = pi ? w[pj ? W_SE : W_XE][c] : T(0);
            O.pw1[2] = pj ? w[pi ? W_NW : W_YN][c] : T(0);
            O.pw1[3] = pi && pj ? w[W_NE][c] : T(0);
        }
    }
    // levels 2.. on one wavefront where they are no larger, level 2 from
    // registers where the coarsest comes right below it
    int lower = TAIL_LOWER_ALL;
    if (a.n > 2) {
        const Dims& D2 = a.L[2].d;
        const int n2 = D2.ni * D2.nj;
        if (!MANY && n2 <= 64) lower = a.n == 4 ? TAIL_LOWER_OWN : TAIL_LOWER_WAVE;
        const int I2 = tid % D2.ni, J2 = tid / D2.ni;
        if (J2 < D2.nj) {
            if (!MANY) restrict_weights(D2, a.L[1].P, I2, J2, O.rw2);
            O.c2 = toff(a.L[2].cd, I2, J2);
            O.f2 = (2 * J2 + 1) * a.ld1 + 2 * I2 + 1;
            O.red2 = ((I2 + J2) & 1) == 0;
            if (lower == TAIL_LOWER_OWN) O.r2 = tail_row(a.L[2], I2, J2);
        }
    }
    if (!live) return;
    for (int k = tid; k < lds_elems; k += NT) lds[k] = T(0);
    {
        const Dims& Dc = a.L[a.n - 1].d;
        const int nc = Dc.ni * Dc.nj;
        for (int k = tid; k < nc * nc; k += NT) inv[k] = a.inv[k];
    }
    __syncthreads();
    if (STAGED && O.own) {
        const Dims& D1 = a.L[1].d;
        T w[9];
        restrict_weights(D1, L0.P, I, J, w);
#pragma unroll
        for (int k = 0; k < 9; ++k) {
            lds[a.rw1 + k * a.n1 + tid] = w[k];
            lds[a.pw1 + k * a.n1 + tid] = L0.P.w[k][D1.off(I, J)];
        }
    }
    if (MANY && O.c2 >= 0) {
        const Dims& D2 = a.L[2].d;
        T w[9];
        restrict_weights(D2, a.L[1].P, tid % D2.ni, tid / D2.ni, w);
#pragma unroll
        for (int k = 0; k < 9; ++k) lds[a.w2 + k * D2.ni * D2.nj + tid] = w[k];
    }
    // operators and weights of the levels 2..
    for (int l = 2; l < a.n; ++l) {
        const TailLevel<T>& L = a.L[l];
        const int n = L.d.ni * L.d.nj;
        if (lower != TAIL_LOWER_OWN)
            for (int k = tid; k < n; k += NT) {
                const int i = k % L.d.ni, j = k / L.d.ni;
                const size_t g = L.d.off(i, j), c = L.cd.off(i, j);
                tarr(lds, L, TA_D)[c] = L.A.diag[g];
                tarr(lds, L, TA_E)[c] = L.A.cE[g];
                tarr(lds, L, TA_N)[c] = L.A.cN[g];
                tarr(lds, L, TA_NE)[c] = L.A.cNE[g];
                tarr(lds, L, TA_NW)[c] = L.A.cNW[g];
            }
        if (l + 1 < a.n) {
            const TailLevel<T>& Cl = a.L[l + 1];
            const int nc = Cl.d.ni * Cl.d.nj;
            for (int k = tid; k < nc; k += NT) {
                const int ic = k % Cl.d.ni, jc = k / Cl.d.ni;
                const size_t g = Cl.d.off(ic, jc), c = Cl.cd.off(ic, jc);
#pragma unroll
                for (int m = 0; m < 9; ++m) lds[L.wbase + (size_t)m * Cl.cd.alloc_elems() + c] = L.P.w[m][g];
            }
        }
    }
    __syncthreads();
    T x[4] = {T(0), T(0), T(0), T(0)};
    if (a.krylov <= 0) {
        tail_vcycle<NT>(lds, a, O, inv, lower, b, x);
    } else {
        // b holds the inner residual; the level's vectors z, q, p and b go to
        // LDS in linear order for the dots
        const int n = D0.ni * D0.nj;
        T *zl = lds + a.lin, *ql = zl + TAIL_MAX, *bl = ql + TAIL_MAX;
        auto store = [&](T* to, const T (&v)[4]) {
            if (!O.own) return;
            const int i = 2 * I, j = 2 * J;
            T* at = to + j * D0.ni + i;
            at[0] = v[0];
            if (i + 1 < D0.ni) at[1] = v[1];
            if (j + 1 < D0.nj) {
                at[D0.ni] = v[2];
                if (i + 1 < D0.ni) at[D0.ni + 1] = v[3];
            }
        };
        T p[4] = {T(0), T(0), T(0), T(0)}, q[4] = {T(0), T(0), T(0), T(0)}, z[4];
        T* xa = lds + a.x0 + O.p;
        double pq_prev = 0.0, rr0 = 0.0;
        for (int it = 0; it < a.krylov; ++it) {
#pragma unroll
            for (int k = 0; k < 4; ++k) z[k] = T(0);
            store(bl, b);
            tail_vcycle<NT>(lds, a, O, inv, lower, b, z);
            store(zl, z);
            __syncthreads();
            double v[2];
            tail_allreduce<NT, 2>(
                [&](int t, double (&w)[2]) {
                    const T zp = t < n ? zl[t] : T(0), qv = t < n ? ql[t] : T(0);
                    const double rp = t < n ? (double)bl[t] : 0.0;
                    w[0] = (double)zp * (double)qv;
                    w[1] = rp * rp;
                },
                v, part_b);
            // every thread holds the same sums, so the exits below are uniform:
            // stop once the inner residual has fallen 1e4 (further iterations
            // would work on rounding noise, in FP32 above all)
            if (it == 0) rr0 = v[1];
            else if (!(v[1] > 1e-8 * rr0)) break;
            const T beta = (it > 0 && pq_prev > 0.0) ? (T)(-v[0] / pq_prev) : T(0);
#pragma unroll
            for (int k = 0; k < 4; ++k) p[k] = z[k] + beta * p[k];
            if (O.own) {
                xa[0] = p[0];
                xa[1] = p[1];
                xa[a.ld0] = p[2];
                xa[a.ld0 + 1] = p[3];
            }
            store(zl, p);
            __syncthreads();
            if (O.own) {
                T s[4];
                block_sums(O, ring(xa, a.ld0), p, s);
#pragma unroll
                for (int k = 0; k < 4; ++k) q[k] = O.r[k].d * p[k] - s[k];
            }
            store(ql, q);
            __syncthreads();
            double v2[2];
            tail_allreduce<NT, 2>(
                [&](int t, double (&w)[2]) {
                    const T pp = t < n ? zl[t] : T(0), qv = t < n ? ql[t] : T(0);
                    const double rp = t < n ? (double)bl[t] : 0.0;
                    w[0] = (double)pp * rp;
                    w[1] = (double)pp * (double)qv;
                },
                v2, part_a);
            const double al = v2[0] / v2[1];
            if (!(v2[1] > 0.0) || !(fabs(al) < 1e30)) break;
            const T alpha = (T)al;
            pq_prev = v2[1];
#pragma unroll
            for (int k = 0; k < 4; ++k) {
                x[k] += alpha * p[k];
                b[k] -= alpha * q[k];
            }
        }
    }
    if (O.own) {
#pragma unroll
        for (int k = 0; k < 4; ++k) {
            const int i = 2 * I + (k & 1), j = 2 * J + (k >> 1);
            if (i < D0.ni && j < D0.nj) L0.x[D0.off(i, j)] = x[k];
        }
    }
}

// coarsest-only hierarchy (grids of at most COARSEST_MAX cells): the dense
// FP64 solve
template <typename TB, typename TZ>
__global__ void __launch_bounds__(256) k_direct(Dims C, const double* __restrict__ inv, const TB* __restrict__ b,
                                                TZ* __restrict__ x, const int* on) {
    if (on && !*on) return;
    const int n = C.ni * C.nj;
    const int r = threadIdx.x;
    if (r >= n) return;
    double s = 0.0;
    for (int q = 0; q < n; ++q) s += inv[(size_t)r * n + q] * (double)b[C.off(q % C.ni, q / C.ni)];
    x[C.off(r % C.ni, r / C.ni)] = (TZ)s;
}

template <typename T>
struct Acc;
template <>
struct Acc<double> {
    static const Op<double>& op(const Level& L) { return L.A; }
    static const Prol<double>& pr(const Level& L) { return L.P; }
    static const LevelVecs<double>& vec(const Level& L) { return L.v; }
};
template <>
struct Acc<float> {
    static const Op<float>& op(const Level& L) { return L.Af; }
    static const Prol<float>& pr(const Level& L) { return L.Pf; }
    static const LevelVecs<float>& vec(const Level& L) { return L.vf; }
};

inline dim3 tiles(const Dims& d, int tw, int th) { return dim3((d.ni + tw - 1) / tw, (d.nj + th - 1) / th); }

// 64x16 tiles on coarse levels of 2048^2 and more, 32x8 below: the latency
// of a tile's passes is hidden only with several tiles per CU
inline bool big(const Dims& d) { return (size_t)d.ni * d.nj >= (size_t)2048 * 2048; }

inline Dims compact(const Dims& d) {
    Dims c = d;
    c.ld = d.ni + 1;
    return c;
}

// The tail's levels and their LDS: level 0 two arrays with a ring of zeros,
// level 1 two, the levels below it their operators, vectors and weights.  A
// tail is refused by the size of all its levels' operators, vectors and
// weights, whatever of that sits in registers.
template <typename T>
int tail_layout(Ctx* c, int lt, const int* on, TailArgs<T>& ta, size_t& lds) {
    const int nl = c->nlev;
    ta.n = nl - lt;
    if (ta.n > MAX_TAIL) {
        set_error("multigrid: too many tail levels");
        return SG_ERR_STATE;
    }
    ta.krylov = c->prm.mg_coarse_krylov;
    ta.inv = c->coarse_inv;
    ta.on = on;
    const Dims &d0 = c->lev[lt].d;
    const int ci = (d0.ni + 1) / 2, cj = (d0.nj + 1) / 2;
    int off = 0;
    auto take = [&](int n) {
        const int at = off;
        off += n;
        return at;
    };
    ta.ld0 = 2 * ci + 2;
    ta.x0 = take(ta.ld0 * (2 * cj + 2));
    ta.x1 = take(ta.ld0 * (2 * cj + 2));
    ta.ld1 = ci + 2;
    ta.y0 = take(ta.ld1 * (cj + 2));
    ta.y1 = take(ta.ld1 * (cj + 2));
    ta.lin = take(ta.krylov > 0 ? 3 * TAIL_MAX : 0);
    ta.n1 = ci * cj;
    const bool many = ta.n1 > TAIL_NT;
    ta.w2 = take(many ? 9 * c->lev[lt + 2].d.ni * c->lev[lt + 2].d.nj : 0);
    ta.rw1 = take(many && tail_staged<T> ? 9 * ta.n1 : 0);
    ta.pw1 = take(many && tail_staged<T> ? 9 * ta.n1 : 0);
    size_t all = ta.krylov > 0 ? compact(d0).alloc_elems() : 0;
    for (int k = 0; k < ta.n; ++k) {
        const Level& L = c->lev[lt + k];
        TailLevel<T>& t = ta.L[k];
        t.d = L.d;
        t.cd = compact(L.d);
        t.sh = 0;
        while ((1 << t.sh) < L.d.ni) ++t.sh;
        t.A = opv(Acc<T>::op(L));
        t.P = Acc<T>::pr(L);
        t.x = Acc<T>::vec(L).x;
        t.b = Acc<T>::vec(L).b;
        const int next = k + 1 < ta.n ? 9 * (int)compact(c->lev[lt + k + 1].d).alloc_elems() : 0;
        if (k >= 2) {
            t.base = take(TA_COUNT * (int)t.cd.alloc_elems());
            t.wbase = take(next);
        }
        all += 8 * t.cd.alloc_elems() + next;
    }
    const size_t nc = (size_t)c->lev[nl - 1].d.ni * c->lev[nl - 1].d.nj;
    if (all * sizeof(T) + nc * nc * sizeof(double) > TAIL_LDS_MAX) {
        set_error("multigrid: tail levels exceed the LDS budget");
        return SG_ERR_STATE;
    }
    lds = (size_t)off;
    return SG_OK;
}

// z = M^{-1} r ; fine-level dots (r,z), (z,q) go to the partials slot S;
// V = type of the PCG vectors r, z, q; every kernel returns at once while
// *on == 0 (a converged PCG)
template <typename T, typename V>
int vcycle(Ctx* c, const V* r, V* z, const V* q, Slots S, int* dots_done, const int* on) {
    hipStream_t s = c->stream;
    const int nl = c->nlev;
    *dots_done = 0;
    if (nl == 1) {
        const Level& L = c->lev[0];
        hipLaunchKernelGGL((k_direct<V, V>), dim3(1), dim3(256), 0, s, L.d, (const double*)c->coarse_inv, r, z, on);
        SG_HIP(hipGetLastError());
        return SG_OK;
    }
    *dots_done = 1;
    int lt = 1;  // first level of the tail
    while (lt < nl - 1 && (size_t)c->lev[lt].d.ni * c->lev[lt].d.nj > (size_t)TAIL_MAX) ++lt;
    // down
    for (int l = 0; l < lt; ++l) {
        const Level& L = c->lev[l];
        const Level& Cl = c->lev[l + 1];
        if (l == 0)
            launch_down5<T, V>(c->semi0 != 0, s, L.d, opv(Acc<T>::op(L)), r, Acc<T>::vec(L).x, Cl.d, Acc<T>::pr(L),
                               Acc<T>::vec(Cl).b, on);
        else if (big(L.d))
            hipLaunchKernelGGL((k_down9<T, 64, 16>), tiles(L.d, 64, 16), dim3(NTB), 0, s, L.d, opv(Acc<T>::op(L)),
                               (const T*)Acc<T>::vec(L).b, Acc<T>::vec(L).x, Cl.d, Acc<T>::pr(L),
                               Acc<T>::vec(Cl).b, on);
        else
            hipLaunchKernelGGL((k_down9<T, 32, 8>), tiles(L.d, 32, 8), dim3(NTB), 0, s, L.d, opv(Acc<T>::op(L)),
                               (const T*)Acc<T>::vec(L).b, Acc<T>::vec(L).x, Cl.d, Acc<T>::pr(L),
                               Acc<T>::vec(Cl).b, on);
    }
    // tail
    TailArgs<T> ta{};
    size_t tail_lds = 0;
    int rc = tail_layout<T>(c, lt, on, ta, tail_lds);
    if (rc) return rc;
    if (ta.n1 <= TAIL_NT)
        hipLaunchKernelGGL((k_tail<T, TAIL_NT>), dim3(1), dim3(TAIL_NT), tail_lds * sizeof(T), s, ta, (int)tail_lds);
    else
        hipLaunchKernelGGL((k_tail<T, TAIL_NT_MAX>), dim3(1), dim3(TAIL_NT_MAX), tail_lds * sizeof(T), s, ta,
                           (int)tail_lds);
    // up: level l reads x_l from the down pass and e_{l+1}; writes its own
    // correction into r_l (its solution for the level above)
    for (int l = lt - 1; l >= 0; --l) {
        const Level& L = c->lev[l];
        const Level& Cl = c->lev[l + 1];
        const T* e = (l + 1 == lt) ? Acc<T>::vec(Cl).x : Acc<T>::vec(Cl).r;
        if (l == 0)
            launch_up5<T, V>(c->semi0 != 0, s, L.d, opv(Acc<T>::op(L)), r, (const T*)Acc<T>::vec(L).x, Cl.d,
                             Acc<T>::pr(L), e, z, q, S, on);
        else if (big(L.d))
            hipLaunchKernelGGL((k_up9<T, 64, 16>), tiles(L.d, 64, 16), dim3(NTB), 0, s, L.d, opv(Acc<T>::op(L)),
                               (const T*)Acc<T>::vec(L).b, (const T*)Acc<T>::vec(L).x, Cl.d, Acc<T>::pr(L), e,
                               Acc<T>::vec(L).r, on);
        else
            hipLaunchKernelGGL((k_up9<T, 32, 8>), tiles(L.d, 32, 8), dim3(NTB), 0, s, L.d, opv(Acc<T>::op(L)),
                               (const T*)Acc<T>::vec(L).b, (const T*)Acc<T>::vec(L).x, Cl.d, Acc<T>::pr(L), e,
                               Acc<T>::vec(L).r, on);
    }
    SG_HIP(hipGetLastError());
    return SG_OK;
}

}  // namespace

int mg_vcycle_dots(Ctx* c, double* partials, int max_blocks, int* dots_done) {
    Slots S{partials, max_blocks};
    if (c->prm.precision == SG_PREC_MIXED)
        return vcycle<float, float>(c, c->rf, c->zf, c->qf, S, dots_done, &c->sc->active);
    return vcycle<double, double>(c, c->r, c->z, c->q, S, dots_done, &c->sc->active);
}

namespace {
__global__ void __launch_bounds__(256) k_copy(size_t n, const double* __restrict__ a, double* __restrict__ b) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i < n) b[i] = a[i];
}
}  // namespace

// One launch of a fine-level kernel on the current data (measurement):
// 1 = down-sweep, 2 = up-sweep, 3 = plain copy of the level-0 padded vector.
int mg_launch_fine(Ctx* c, int which) {
    hipStream_t s = c->stream;
    const Level& L = c->lev[0];
    if (c->nlev < 2) return SG_ERR_STATE;
    const Level& Cl = c->lev[1];
    Slots S{c->red.partials + (size_t)7 * NRED * c->red.max_blocks, c->red.max_blocks};
    const bool mixed = c->prm.precision == SG_PREC_MIXED;
    if (which == 1) {
        if (mixed)
            launch_down5<float, float>(c->semi0 != 0, s, L.d, opv(L.Af), (const float*)c->rf, L.vf.x, Cl.d, L.Pf,
                                       Cl.vf.b, nullptr);
        else
            launch_down5<double, double>(c->semi0 != 0, s, L.d, opv(L.A), (const double*)c->r, L.v.x, Cl.d, L.P,
                                         Cl.v.b, nullptr);
    } else if (which == 2) {
        // the coarse correction sits in x when level 1 is the tail's first level, else in r
        const bool tail1 = c->nlev == 2 || (size_t)Cl.d.ni * Cl.d.nj <= (size_t)TAIL_MAX;
        if (mixed)
            launch_up5<float, float>(c->semi0 != 0, s, L.d, opv(L.Af), (const float*)c->rf, (const float*)L.vf.x,
                                     Cl.d, L.Pf, (const float*)(tail1 ? Cl.vf.x : Cl.vf.r), c->zf,
                                     (const float*)c->qf, S, nullptr);
        else
            launch_up5<double, double>(c->semi0 != 0, s, L.d, opv(L.A), (const double*)c->r, (const double*)L.v.x,
                                       Cl.d, L.P, (const double*)(tail1 ? Cl.v.x : Cl.v.r), c->z,
                                       (const double*)c->q, S, nullptr);
    } else if (which == 3) {
        const size_t n = L.d.alloc_elems();
        hipLaunchKernelGGL(k_copy, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, s, n, (const double*)L.v.b,
                           L.v.r);
    } else {
        return SG_ERR_ARG;
    }
    SG_HIP(hipGetLastError());
    return SG_OK;
}

int mg_partial_blocks(Ctx* c) {
    const dim3 t = tiles(c->lev[0].d, GW, GH);
    return (int)(t.x * t.y);
}

}  // namespace sg
