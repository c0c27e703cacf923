// FP64 natural-gradient solves on the GPU, one workgroup per system (batched
// over blockIdx.x), every loop bounded.
//
//  - lu_solve_c128: (A) x = b by LU with partial pivoting, singular when
//    |pivot|^2 < 1e-10 on columns 0..P-2 -- the rule of QGTL's
//    lu_decomposition / solve_linear_system
//    (src/quantum_geometric/core/matrix_operations.c:60-160) that
//    compute_regularized_natural_gradient relies on
//    (src/quantum_geometric/core/quantum_geometric_gradient.c:2887-2964).
//  - herm_eig_c128: parallel cyclic Jacobi (round-robin pairs) for Hermitian
//    matrices: eigenvalues ascending and eigenvectors, for the pseudo-inverse
//    fallback (:2733-2884).
//  - herm_extremes_c128: the eigenvalues a condition number needs, without vectors.
//  - cholesky_f64: (A + lambda I) x = b for real SPD A, the exact yardstick.
//  - pcg_f64: preconditioned CG from x0 = 0 to ||r||/||b|| <= tol with
//    M^-1 = diag(d) + U U^T (U = 0 gives Jacobi-PCG with d = 1/diag(A)),
//    QGTL's CG (src/quantum_geometric/hybrid/classical_optimization_engine.c:543-610)
//    with a preconditioner.
#include "qgtl_hip_common.h"

namespace {

constexpr int kT = 1024;

__device__ __forceinline__ double2 cmul(double2 a, double2 b) {
    return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}

__device__ __forceinline__ double2 cdiv(double2 a, double2 b) {
    const double d = b.x * b.x + b.y * b.y;
    return make_double2((a.x * b.x + a.y * b.y) / d, (a.y * b.x - a.x * b.y) / d);
}

// One lane of a double moved by a DPP pattern (two 32-bit DPP moves).
template <int CTRL>
__device__ __forceinline__ double dpp_f64(double v) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const int lo = __builtin_amdgcn_update_dpp(0, (int)(unsigned)b, CTRL, 0xf, 0xf, false);
    const int hi = __builtin_amdgcn_update_dpp(0, (int)(unsigned)(b >> 32), CTRL, 0xf, 0xf, false);
    return __builtin_bit_cast(double, ((unsigned long long)(unsigned)hi << 32) | (unsigned)lo);
}

__device__ __forceinline__ double readlane_f64(double v, int lane) {
    const unsigned long long b = __builtin_bit_cast(unsigned long long, v);
    const unsigned lo = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)b, lane);
    const unsigned hi = (unsigned)__builtin_amdgcn_readlane((int)(unsigned)(b >> 32), lane);
    return __builtin_bit_cast(double, ((unsigned long long)hi << 32) | lo);
}

// Sum over the 64 lanes of a wave, identical in every lane and independent of timing:
// pairs, quads (quad_perm), half rows and rows of 16 (row_half_mirror, row_mirror) by DPP,
// each step adding two equal-shaped partial sums so every lane of a row holds the same bits;
// then the four row sums (lanes 0, 16, 32, 48) in the order (r0 + r1) + (r2 + r3).
__device__ __forceinline__ double wave_sum_f64(double v) {
    v += dpp_f64<0xB1>(v);                            // quad_perm [1,0,3,2]
    v += dpp_f64<0x4E>(v);                            // quad_perm [2,3,0,1]
    v += dpp_f64<0x141>(v);                           // row_half_mirror
    v += dpp_f64<0x140>(v);                           // row_mirror
    return (readlane_f64(v, 0) + readlane_f64(v, 16)) + (readlane_f64(v, 32) + readlane_f64(v, 48));
}

// Largest of the 64 lanes, in every lane (no NaN among them).
__device__ __forceinline__ double wave_max_f64(double v) {
    v = fmax(v, dpp_f64<0xB1>(v));
    v = fmax(v, dpp_f64<0x4E>(v));
    v = fmax(v, dpp_f64<0x141>(v));
    v = fmax(v, dpp_f64<0x140>(v));
    return fmax(fmax(readlane_f64(v, 0), readlane_f64(v, 16)), fmax(readlane_f64(v, 32), readlane_f64(v, 48)));
}

// Block-wide sum in a fixed order (deterministic).
__device__ double block_sum(double v, double *red) {
    red[threadIdx.x] = v;
    __syncthreads();
    for (int h = kT / 2; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    const double s = red[0];
    __syncthreads();
    return s;
}

// ---------------------------------------------------------------- LU (complex)
__global__ __launch_bounds__(kT) void lu_solve_c128_kernel(double2 *Aall, const double2 *ball, double2 *xall,
                                                           int *pivall, int P, int *status) {
    double2 *A = Aall + (size_t)blockIdx.x * P * P;
    const double2 *b = ball + (size_t)blockIdx.x * P;
    double2 *x = xall + (size_t)blockIdx.x * P;
    int *piv = pivall + (size_t)blockIdx.x * P;
    __shared__ double red_v[kT];
    __shared__ int red_i[kT];
    __shared__ int s_fail;
    for (int i = threadIdx.x; i < P; i += kT) piv[i] = i;
    if (threadIdx.x == 0) s_fail = 0;
    __syncthreads();
    for (int i = 0; i < P - 1; i++) {
        // pivot: max |a_ji|^2 over j >= i, first index on ties
        double best = -1.0;
        int bi = i;
        for (int j = i + threadIdx.x; j < P; j += kT) {
            const double2 a = A[(size_t)j * P + i];
            const double v = a.x * a.x + a.y * a.y;
            if (v > best) { best = v; bi = j; }
        }
        red_v[threadIdx.x] = best;
        red_i[threadIdx.x] = bi;
        __syncthreads();
        for (int h = kT / 2; h > 0; h >>= 1) {
            if ((int)threadIdx.x < h) {
                const double o = red_v[threadIdx.x + h];
                const int oi = red_i[threadIdx.x + h];
                if (o > red_v[threadIdx.x] || (o == red_v[threadIdx.x] && oi < red_i[threadIdx.x])) {
                    red_v[threadIdx.x] = o;
                    red_i[threadIdx.x] = oi;
                }
            }
            __syncthreads();
        }
        const double mx = red_v[0];
        const int p = red_i[0];
        __syncthreads();
        if (mx < 1e-10) {
            if (threadIdx.x == 0) s_fail = 1;
            break;
        }
        if (p != i) {
            for (int k = threadIdx.x; k < P; k += kT) {
                const double2 t = A[(size_t)i * P + k];
                A[(size_t)i * P + k] = A[(size_t)p * P + k];
                A[(size_t)p * P + k] = t;
            }
            if (threadIdx.x == 0) { const int t = piv[i]; piv[i] = piv[p]; piv[p] = t; }
        }
        __syncthreads();
        const double2 d = A[(size_t)i * P + i];
        for (int j = i + 1 + threadIdx.x; j < P; j += kT) A[(size_t)j * P + i] = cdiv(A[(size_t)j * P + i], d);
        __syncthreads();
        const int m = P - i - 1;
        for (int e = threadIdx.x; e < m * m; e += kT) {
            const int j = i + 1 + e / m, k = i + 1 + e % m;
            const double2 l = A[(size_t)j * P + i], u = A[(size_t)i * P + k];
            double2 a = A[(size_t)j * P + k];
            const double2 lu = cmul(l, u);
            a.x -= lu.x;
            a.y -= lu.y;
            A[(size_t)j * P + k] = a;
        }
        __syncthreads();
    }
    if (s_fail) {
        if (threadIdx.x == 0) status[blockIdx.x] = -1;
        return;
    }
    // forward (unit lower) and back substitution by one wave through LDS
    __shared__ double2 sx[1024];
    if (threadIdx.x < 64) {
        const int lane = threadIdx.x;
        for (int i = lane; i < P; i += 64) sx[i] = b[piv[i]];
        qgtl::wave_sync();
        for (int i = 0; i < P; i++) {
            double sr = 0.0, si = 0.0;
            for (int j = lane; j < i; j += 64) {
                const double2 t = cmul(A[(size_t)i * P + j], sx[j]);
                sr += t.x;
                si += t.y;
            }
            for (int o = 32; o > 0; o >>= 1) { sr += __shfl_xor(sr, o, 64); si += __shfl_xor(si, o, 64); }
            if (lane == 0) sx[i] = make_double2(sx[i].x - sr, sx[i].y - si);
            qgtl::wave_sync();
        }
        for (int i = P - 1; i >= 0; i--) {
            double sr = 0.0, si = 0.0;
            for (int j = i + 1 + lane; j < P; j += 64) {
                const double2 t = cmul(A[(size_t)i * P + j], sx[j]);
                sr += t.x;
                si += t.y;
            }
            for (int o = 32; o > 0; o >>= 1) { sr += __shfl_xor(sr, o, 64); si += __shfl_xor(si, o, 64); }
            if (lane == 0) sx[i] = cdiv(make_double2(sx[i].x - sr, sx[i].y - si), A[(size_t)i * P + i]);
            qgtl::wave_sync();
        }
        for (int i = lane; i < P; i += 64) x[i] = sx[i];
        if (lane == 0) status[blockIdx.x] = 0;
    }
}

// The same for P <= 128 with the matrix in registers: wave w holds columns w + 16 s, its lane l
// rows l + 64 c.  Rows stay where they are; pos is the position each has in the permuted order
// (kept by every wave), so the pivots, ties included, are those of the kernel above.  The wave of
// column i finds its pivot and the multipliers without leaving the wave and hands
// them on through LDS; the others take the pivot row's element of a column from the lane
// that holds it.  One barrier a step: the wave of column i + 1 updates that column first and
// finds its pivot while the others update theirs.  b is one more column, of the last wave.  U goes
// to LDS by columns for the back substitution of one wave.  What bounds it: the latency of that
// chain (LDS, the maximum over a wave, a complex division).
// P = 96: 162 us; 274 us with rows split over waves (two barriers a step, the multipliers formed
// by two waves while the others wait), 434 us in global memory.
template <int COLS, int ROWS>
__global__ __launch_bounds__(kT) void lu_solve_regs_kernel(const double2 *Aall, const double2 *ball, double2 *xall,
                                                           int P, int *status) {
    constexpr int N = 64 * ROWS;
    static_assert(16 * COLS == N, "square");
    __shared__ double2 mul[2][N], yp[N], upk[N * (N + 1) / 2];
    __shared__ int spiv[2];                  // pivot row | its position << 8, or -1: singular
    const double2 *A = Aall + (size_t)blockIdx.x * P * P, *b = ball + (size_t)blockIdx.x * P;
    double2 *x = xall + (size_t)blockIdx.x * P;
    const int t = threadIdx.x, lane = t & 63, wave = qgtl::uniform(t >> 6);
    double2 a[COLS][ROWS], y[ROWS];
    int pos[ROWS];
#pragma unroll
    for (int c = 0; c < ROWS; c++) {
        const int i = lane + 64 * c;
        pos[c] = i;
        y[c] = (wave == 15 && i < P) ? b[i] : make_double2(0.0, 0.0);
#pragma unroll
        for (int s = 0; s < COLS; s++) {
            const int j = wave + 16 * s;
            a[s][c] = (i < P && j < P) ? A[(size_t)i * P + j] : make_double2(0.0, 0.0);
        }
    }
    // row pr's element of a column, for every lane
    auto of_row = [](const double2 (&v)[ROWS], int pr) __attribute__((always_inline)) -> double2 {
        const bool up = ROWS > 1 && pr >= 64;
        return make_double2(readlane_f64(up ? v[ROWS - 1].x : v[0].x, pr & 63),
                            readlane_f64(up ? v[ROWS - 1].y : v[0].y, pr & 63));
    };
    auto column = [&](int j, double2 (&v)[ROWS]) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < ROWS; c++) {
            v[c] = a[0][c];
#pragma unroll
            for (int s = 1; s < COLS; s++) {
                const bool here = s == j >> 4;
                v[c].x = here ? a[s][c].x : v[c].x;
                v[c].y = here ? a[s][c].y : v[c].y;
            }
        }
    };
    // column i (this wave's, v): pivot and multipliers
    auto factor = [&](int i, const double2 (&v)[ROWS]) __attribute__((always_inline)) {
        // max |a_ji|^2 over the rows at positions >= i, the first position on ties
        double best = -1.0;
        int brow = 0, bpos = 0;
#pragma unroll
        for (int c = 0; c < ROWS; c++) {
            const int row = lane + 64 * c;
            const double m = v[c].x * v[c].x + v[c].y * v[c].y;
            if (row < P && pos[c] >= i && (m > best || (m == best && pos[c] < bpos))) { best = m; brow = row; bpos = pos[c]; }
        }
        const double mx = wave_max_f64(best);
        unsigned long long cand = __ballot(best == mx);
        int pr = 0, pp = P;
        while (cand) {
            const int src = __ffsll((long long)cand) - 1;
            cand &= cand - 1;
            const int q = __builtin_amdgcn_readlane(bpos, src);
            if (q < pp) { pp = q; pr = __builtin_amdgcn_readlane(brow, src); }
        }
        const double2 d = of_row(v, pr);
#pragma unroll
        for (int c = 0; c < ROWS; c++) mul[i & 1][lane + 64 * c] = cdiv(v[c], d);
        if (lane == 0) spiv[i & 1] = mx < 1e-10 ? -1 : pr | pp << 8;
    };
    // v -= l u on the rows below the pivot
    auto eliminate = [&](double2 (&v)[ROWS], const double2 (&l)[ROWS], double2 u, int i) __attribute__((always_inline)) {
#pragma unroll
        for (int c = 0; c < ROWS; c++)
            if (pos[c] > i) {
                v[c].x = fma(l[c].y, u.y, fma(-l[c].x, u.x, v[c].x));
                v[c].y = fma(-l[c].y, u.x, fma(-l[c].x, u.y, v[c].y));
            }
    };
    if (wave == 0 && P > 1) factor(0, a[0]);
    for (int i = 0; i < P - 1; i++) {
        __syncthreads();
        const int piv = qgtl::uniform(spiv[i & 1]);
        if (piv < 0) {                       // the same for every wave
            if (t == 0) status[blockIdx.x] = -1;
            return;
        }
        const int pr = piv & 255, pp = piv >> 8;
        double2 l[ROWS];
#pragma unroll
        for (int c = 0; c < ROWS; c++) {
            const int row = lane + 64 * c;
            l[c] = mul[i & 1][row];
            if (row == pr) pos[c] = i;
            else if (pos[c] == i) pos[c] = pp;
        }
        if (wave == ((i + 1) & 15)) {
            __builtin_amdgcn_s_setprio(3);                   // the chain the others wait for
            double2 v[ROWS];
            column(i + 1, v);
            eliminate(v, l, of_row(v, pr), i);               // a copy: the loop below does the column itself
            if (i + 1 < P - 1) factor(i + 1, v);
            __builtin_amdgcn_s_setprio(0);
        }
#pragma unroll
        for (int s = 0; s < COLS; s++) {
            const int j = wave + 16 * s;
            if (j > i && j < P) eliminate(a[s], l, of_row(a[s], pr), i);
        }
        if (wave == 15) eliminate(y, l, of_row(y, pr), i);
    }
    // U by columns, b in the permuted order
#pragma unroll
    for (int c = 0; c < ROWS; c++) {
        if (lane + 64 * c >= P) continue;
        if (wave == 15) yp[pos[c]] = y[c];
#pragma unroll
        for (int s = 0; s < COLS; s++) {
            const int j = wave + 16 * s;
            if (j < P && pos[c] <= j) upk[j * (j + 1) / 2 + pos[c]] = a[s][c];
        }
    }
    __syncthreads();
    if (wave != 0) return;
#pragma unroll
    for (int c = 0; c < ROWS; c++) y[c] = yp[lane + 64 * c];
    double2 un[ROWS];
    auto fetch = [&](int i, double2 (&u)[ROWS]) -> double2 {
#pragma unroll
        for (int c = 0; c < ROWS; c++) {
            const int j = lane + 64 * c;
            u[c] = upk[i * (i + 1) / 2 + (j < i ? j : i)];
        }
        return upk[i * (i + 1) / 2 + i];
    };
    double2 dn = fetch(P - 1, un);
    for (int i = P - 1; i >= 0; i--) {
        double2 u[ROWS];
        const double2 d = dn;
#pragma unroll
        for (int c = 0; c < ROWS; c++) u[c] = un[c];
        if (i > 0) dn = fetch(i - 1, un);
        const double2 xi = cdiv(of_row(y, i), d);
#pragma unroll
        for (int c = 0; c < ROWS; c++) {
            const int j = lane + 64 * c;
            const double2 v = cmul(u[c], xi);
            if (j < i) { y[c].x -= v.x; y[c].y -= v.y; }
            if (j == i) y[c] = xi;
        }
    }
#pragma unroll
    for (int c = 0; c < ROWS; c++)
        if (lane + 64 * c < P) x[lane + 64 * c] = y[c];
    if (lane == 0) status[blockIdx.x] = 0;
}

// ------------------------------------------------------- Hermitian Jacobi
// A (in/out, destroyed), V (out, columns = eigenvectors), ev (out, ascending).
__global__ __launch_bounds__(kT) void herm_eig_c128_kernel(double2 *Aall, double2 *Vall, double *evall, int P,
                                                           int max_sweeps, int *sweeps_out) {
    double2 *A = Aall + (size_t)blockIdx.x * P * P;
    double2 *V = Vall + (size_t)blockIdx.x * P * P;
    double *ev = evall + (size_t)blockIdx.x * P;
    __shared__ double red[kT];
    __shared__ int pair_p[512], pair_q[512];
    __shared__ double rot[512][6];   // c, s, er, ei, active
    const int M = (P + 1) & ~1;      // even count; index P is a dummy when P is odd
    for (int e = threadIdx.x; e < P * P; e += kT) V[e] = make_double2((e / P) == (e % P) ? 1.0 : 0.0, 0.0);
    double fro = 0.0;
    for (int e = threadIdx.x; e < P * P; e += kT) fro += A[e].x * A[e].x + A[e].y * A[e].y;
    fro = sqrt(block_sum(fro, red));
    int sweep = 0;
    for (; sweep < max_sweeps; sweep++) {
        double off = 0.0;
        for (int e = threadIdx.x; e < P * P; e += kT)
            if (e / P != e % P) off += A[e].x * A[e].x + A[e].y * A[e].y;
        off = sqrt(block_sum(off, red));
        if (off <= 1e-15 * (fro > 0.0 ? fro : 1.0)) break;
        for (int step = 0; step < M - 1; step++) {
            // round-robin: position 0 fixed, others rotate
            for (int k = threadIdx.x; k < M / 2; k += kT) {
                int a = (k == 0) ? 0 : 1 + (k - 1 + step) % (M - 1);
                int bidx = 1 + (M - 2 - k + step) % (M - 1);
                int p = a < bidx ? a : bidx, q = a < bidx ? bidx : a;
                pair_p[k] = p;
                pair_q[k] = q;
                double c = 1.0, s = 0.0, er = 1.0, ei = 0.0, act = 0.0;
                if (q < P) {
                    const double2 apq = A[(size_t)p * P + q];
                    const double mag = sqrt(apq.x * apq.x + apq.y * apq.y);
                    if (mag > 0.0) {
                        er = apq.x / mag;
                        ei = apq.y / mag;
                        const double tau = (A[(size_t)q * P + q].x - A[(size_t)p * P + p].x) / (2.0 * mag);
                        const double t = (tau >= 0 ? 1.0 : -1.0) / (fabs(tau) + sqrt(1.0 + tau * tau));
                        c = 1.0 / sqrt(1.0 + t * t);
                        s = t * c;
                        act = 1.0;
                    }
                }
                rot[k][0] = c; rot[k][1] = s; rot[k][2] = er; rot[k][3] = ei; rot[k][4] = act;
            }
            __syncthreads();
            // columns: A <- A J, V <- V J with J = [[c, s], [-s conj(e), c conj(e)]]
            for (int e = threadIdx.x; e < P * (M / 2); e += kT) {
                const int k = e / P, r = e % P;
                if (rot[k][4] == 0.0) continue;
                const int p = pair_p[k], q = pair_q[k];
                const double c = rot[k][0], s = rot[k][1], er = rot[k][2], ei = rot[k][3];
                const double2 jqp = make_double2(-s * er, s * ei), jqq = make_double2(c * er, -c * ei);
                double2 *Ar = A + (size_t)r * P;
                const double2 ap = Ar[p], aq = Ar[q];
                const double2 t1 = cmul(aq, jqp), t2 = cmul(aq, jqq);
                Ar[p] = make_double2(c * ap.x + t1.x, c * ap.y + t1.y);
                Ar[q] = make_double2(s * ap.x + t2.x, s * ap.y + t2.y);
                double2 *Vr = V + (size_t)r * P;
                const double2 vp = Vr[p], vq = Vr[q];
                const double2 u1 = cmul(vq, jqp), u2 = cmul(vq, jqq);
                Vr[p] = make_double2(c * vp.x + u1.x, c * vp.y + u1.y);
                Vr[q] = make_double2(s * vp.x + u2.x, s * vp.y + u2.y);
            }
            __syncthreads();
            // rows: A <- J^H A
            for (int e = threadIdx.x; e < P * (M / 2); e += kT) {
                const int k = e / P, col = e % P;
                if (rot[k][4] == 0.0) continue;
                const int p = pair_p[k], q = pair_q[k];
                const double c = rot[k][0], s = rot[k][1], er = rot[k][2], ei = rot[k][3];
                const double2 cjqp = make_double2(-s * er, -s * ei), cjqq = make_double2(c * er, c * ei);
                const double2 pk = A[(size_t)p * P + col], qk = A[(size_t)q * P + col];
                const double2 t1 = cmul(cjqp, qk), t2 = cmul(cjqq, qk);
                A[(size_t)p * P + col] = make_double2(c * pk.x + t1.x, c * pk.y + t1.y);
                A[(size_t)q * P + col] = make_double2(s * pk.x + t2.x, s * pk.y + t2.y);
            }
            __syncthreads();
            for (int k = threadIdx.x; k < M / 2; k += kT) {
                if (rot[k][4] == 0.0) continue;
                const int p = pair_p[k], q = pair_q[k];
                A[(size_t)p * P + q] = make_double2(0.0, 0.0);
                A[(size_t)q * P + p] = make_double2(0.0, 0.0);
                A[(size_t)p * P + p].y = 0.0;
                A[(size_t)q * P + q].y = 0.0;
            }
            __syncthreads();
        }
    }
    // eigenvalues ascending (rank by value, index breaks ties), permute V's columns
    for (int i = threadIdx.x; i < P; i += kT) {
        const double vi = A[(size_t)i * P + i].x;
        int rank = 0;
        for (int j = 0; j < P; j++) {
            const double vj = A[(size_t)j * P + j].x;
            rank += (vj < vi) || (vj == vi && j < i);
        }
        ev[rank] = vi;
        red[i] = rank;   // P <= kT
    }
    __syncthreads();
    // copy V into A (scratch) then scatter columns
    for (int e = threadIdx.x; e < P * P; e += kT) A[e] = V[e];
    __syncthreads();
    for (int e = threadIdx.x; e < P * P; e += kT) {
        const int r = e / P, c = e % P;
        V[(size_t)r * P + (int)red[c]] = A[e];
    }
    if (threadIdx.x == 0 && sweeps_out) sweeps_out[blockIdx.x] = sweep;
}

// ------------------------------------------------------------- Cholesky (real)
// Blocked right-looking factorisation of A + lambda I, one workgroup per
// system, NB columns a step: the diagonal block by one wave (a row per lane, in
// registers), the rows below it one per thread from LDS, the trailing update on
// v_mfma_f64_16x16x4_f64 (16 x 16 tiles of the lower triangle, the panel in
// LDS).  b is carried as one more row, so the forward substitution comes with
// the factorisation; the back substitution runs block by block on L.  What
// bounds it: the serial chain of the diagonal blocks (square root, reciprocal
// and a row of multiply-adds per column), the first of which nothing hides; the
// others run beside the trailing updates.  P = 192: 140 us (263 us without that
// overlap and with the panel rows reading the diagonal block by columns), from 1220 us with a
// rank-1 update of the whole trailing matrix per column in global memory and
// one reduction over a wave per row of the substitutions.
//
// NB = 32 while the panel fits LDS beside the rest (P <= 512), 16 above: one workgroup of eight
// waves a CU (the register rows of 32 doubles take 232 VGPRs).  Small systems, of which a batch
// has many, take narrower blocks and fewer waves, so that a short column is not padded to 32 and
// several workgroups share a CU: 1024 systems of P = 8 14 us, of P = 33 32 us (82 and 169 us with NB = 32).
typedef double f64x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ double readlane_f64(double v, int lane);

// Factor of the diagonal block in dg (by rows; the lower triangle is read) by one
// wave, a row per lane in registers: dg receives it by columns (dg[j][i] = l_ij,
// i > j), inv the reciprocals of its diagonal.  Returns nonzero when a pivot is
// not positive.
template <int NB>
__device__ __forceinline__ int factor_diag(double (*dg)[NB + 2], double *inv, int lane) {
    const int row = lane < NB ? lane : NB - 1;       // lanes past the block repeat its last row
    double a[NB];
#pragma unroll
    for (int c = 0; c < NB; c++) a[c] = dg[row][c];
    int bad = 0;
#pragma unroll
    for (int j = 0; j < NB; j++) {
        const double d = readlane_f64(a[j], j);
        bad |= !(d > 0.0);
        // 1 / l_jj from one reciprocal square root and two Newton steps
        double r = __builtin_amdgcn_rsq(d);
        if (d < __builtin_inf()) {                   // an infinite pivot keeps its reciprocal, 0
            r = fma(r * 0.5, fma(-d * r, r, 1.0), r);
            r = fma(r * 0.5, fma(-d * r, r, 1.0), r);
        }
        const double l = a[j] * r;
        a[j] = l;
        if (lane == 0) inv[j] = r;
#pragma unroll
        for (int k = j + 1; k < NB; k++) a[k] = fma(-l, readlane_f64(l, k), a[k]);
    }
    if (lane < NB)
#pragma unroll
        for (int c = 0; c < NB; c++) dg[c][lane] = a[c];
    return bad;
}

template <int NB, int ROWS, int CT>
__global__ __launch_bounds__(CT) void cholesky_f64_kernel(double *Lall, const double *ball, double *xall, int P,
                                                          double lambda, int *status) {
    constexpr int LD = ROWS + 1;                     // odd: the transposing writes hit all banks
    constexpr int kOwn = NB == 32 ? 3 : 1;           // 16 x 16 tiles of a diagonal block
    __shared__ double lp[NB * LD];                   // panel, column c of row i at c * LD + i
    __shared__ __attribute__((aligned(16))) double dgs[2][NB][NB + 2];
    __shared__ double y[ROWS + NB], invs[2][NB];
    __shared__ int s_fail;
    double *L = Lall + (size_t)blockIdx.x * P * P;   // holds A on entry (row-major, symmetric)
    const double *b = ball + (size_t)blockIdx.x * P;
    double *x = xall + (size_t)blockIdx.x * P;
    const int t = threadIdx.x, lane = t & 63;
    const int w = __builtin_amdgcn_readfirstlane(t >> 6);
    if (t == 0) s_fail = 0;
    for (int i = t; i < P; i += CT) {
        y[i] = b[i];
        L[(size_t)i * P + i] += lambda;
    }
    __syncthreads();
    for (int e = t; e < NB * NB; e += CT) {
        const int r = e / NB, c = e % NB;
        dgs[0][r][c] = (r < P && c <= r) ? L[(size_t)r * P + c] : (r == c ? 1.0 : 0.0);
    }
    __syncthreads();
    if (w == 0 && factor_diag<NB>(dgs[0], invs[0], lane) && lane == 0) s_fail = 1;
    int cur = 0;
    for (int kb = 0; kb < P; kb += NB, cur ^= 1) {
        double (*dg)[NB + 2] = dgs[cur];
        const double *inv = invs[cur];
        const int nb = min(NB, P - kb);
        const int m = P - kb - nb + 1;               // rows below the block and the row of b
        const int m16 = (m + 15) / 16 * 16;
#pragma unroll 4
        for (int e = t; e < m16 * NB; e += CT) {
            const int r = e / NB, c = e % NB;
            const bool in = c < nb && r < m - 1;
            double v = L[in ? (size_t)(kb + nb + r) * P + kb + c : (size_t)0];
            if (!in) v = (c < nb && r == m - 1) ? y[kb + c] : 0.0;
            lp[c * LD + r] = v;
        }
        __syncthreads();
        if (s_fail) break;                           // uniform
        for (int r = t; r < m; r += CT) {
            double v[NB];
#pragma unroll
            for (int c = 0; c < NB; c++) v[c] = lp[c * LD + r];
#pragma unroll
            for (int j = 0; j < NB; j++) {
                v[j] *= inv[j];
                if (((j + 1) & 1) && j + 1 < NB) v[j + 1] = fma(-v[j], dg[j][j + 1], v[j + 1]);
#pragma unroll
                for (int k = (j + 2) & ~1; k < NB; k += 2) {
                    const double2 q = *reinterpret_cast<const double2 *>(&dg[j][k]);
                    v[k] = fma(-v[j], q.x, v[k]);
                    v[k + 1] = fma(-v[j], q.y, v[k + 1]);
                }
                // a few columns' reads in flight at a time: all of them hoisted would spill
                if (j % 4 == 3) __builtin_amdgcn_sched_barrier(0);
            }
#pragma unroll
            for (int c = 0; c < NB; c++) lp[c * LD + r] = v[c];
        }
        __syncthreads();
        // trailing tiles (ti >= tj) of 16 x 16, one wave each: C -= L21 L21^T.  Lane l holds
        // A[l % 16][k0 + l / 16], B alike, and D[4 e + l / 16][l % 16] in register e.  Wave 0
        // takes the tiles of the next diagonal block and factors it while the other waves
        // update the rest, so its serial chain overlaps their work.
        const int nt = m16 / 16, base = kb + nb;
        const int nn = min(NB, P - base);            // the next block's size (<= 0: none)
        auto tile = [&](int u, bool next) {
            int ti = 0, tj = u;
            while (tj > ti) { ti++; tj -= ti; }
            const int col = tj * 16 + (lane & 15);
            f64x4 acc = {0.0, 0.0, 0.0, 0.0};
            double c[4];
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = ti * 16 + 4 * e + (lane >> 4);
                const bool in = col < m - 1 && r < m - 1;
                c[e] = L[in ? (size_t)(base + r) * P + base + col : (size_t)0];
                if (!in && col < m - 1 && r == m - 1) c[e] = y[base + col];
            }
#pragma unroll
            for (int k0 = 0; k0 < NB; k0 += 4) {
                const double av = lp[(k0 + (lane >> 4)) * LD + ti * 16 + (lane & 15)];
                const double bv = lp[(k0 + (lane >> 4)) * LD + tj * 16 + (lane & 15)];
                acc = __builtin_amdgcn_mfma_f64_16x16x4f64(av, bv, acc, 0, 0, 0);
            }
#pragma unroll
            for (int e = 0; e < 4; e++) {
                const int r = ti * 16 + 4 * e + (lane >> 4);
                if (col >= m - 1) continue;
                if (r == m - 1) y[base + col] = c[e] - acc[e];
                else if (r < m - 1 && next && col <= r) dgs[cur ^ 1][r][col] = c[e] - acc[e];
                else if (r < m - 1 && !next) L[(size_t)(base + r) * P + base + col] = c[e] - acc[e];
            }
        };
        if (w == 0) {
            if (NB >= 16 && nn > 0) {                            // NB = 4: P <= 4, one block
                for (int e = lane; e < NB * NB; e += 64)         // identity past a short last block
                    if (e / NB >= nn) dgs[cur ^ 1][e / NB][e % NB] = e / NB == e % NB ? 1.0 : 0.0;
                for (int u = 0; u < kOwn && u < nt * (nt + 1) / 2; u++) tile(u, true);
                qgtl::wave_sync();                   // the lanes' tile elements are read by rows
                if (factor_diag<NB>(dgs[cur ^ 1], invs[cur ^ 1], lane) && lane == 0) s_fail = 1;
            }
        } else {
            for (int u = kOwn + w - 1; u < nt * (nt + 1) / 2; u += CT / 64 - 1) tile(u, false);
            // the factor's columns, for the back substitution (the diagonal inverted; b's row: y)
            for (int e = t - 64; e < NB * NB; e += CT - 64) {
                const int r = e / NB, c = e % NB;
                if (c <= r && r < nb) L[(size_t)(kb + r) * P + kb + c] = c == r ? inv[r] : dg[c][r];
            }
            for (int e = t - 64; e < m * NB; e += CT - 64) {
                const int r = e / NB, c = e % NB;
                if (c >= nb) continue;
                if (r < m - 1) L[(size_t)(kb + nb + r) * P + kb + c] = lp[c * LD + r];
                else y[kb + c] = lp[c * LD + r];
            }
        }
        __syncthreads();
    }
    if (s_fail) {
        if (t == 0) status[blockIdx.x] = -1;
        return;
    }
    // L^T x = y, blocks from the last: the block by one wave (lane i: unknown i), then its
    // columns taken out of the unknowns above; the next block's rows are fetched meanwhile
    double row[NB];
    auto fetch = [&](int kb) {
#pragma unroll
        for (int j = 0; j < NB; j++) {
            const bool in = kb >= 0 && kb + j < P && lane <= j;
            row[j] = L[in ? (size_t)(kb + j) * P + kb + lane : (size_t)0];
            if (!in) row[j] = 0.0;
        }
    };
    const int kl = (P - 1) / NB * NB;
    if (w == 0) fetch(kl);
    for (int kb = kl; kb >= 0; kb -= NB) {
        const int nb = min(NB, P - kb);
        double lc[NB];
        if (w == 0) {
            double v = lane < nb ? y[kb + lane] : 0.0;
#pragma unroll
            for (int j = NB - 1; j >= 0; j--) {
                const double xj = readlane_f64(v, j) * readlane_f64(row[j], j);   // 0 past the block
                if (lane == j) v = xj;
                else if (lane < j) v = fma(-row[j], xj, v);
            }
            if (lane < nb) {
                y[kb + lane] = v;
                x[kb + lane] = v;
            }
            fetch(kb - NB);
        } else if (t - 64 < kb) {
#pragma unroll
            for (int j = 0; j < NB; j++) lc[j] = L[(size_t)(kb + min(j, nb - 1)) * P + t - 64];
        }
        __syncthreads();
        if (w != 0) {
            if (t - 64 < kb) {
                double s = y[t - 64];
#pragma unroll
                for (int j = 0; j < NB; j++) s = fma(-lc[j], j < nb ? y[kb + j] : 0.0, s);
                y[t - 64] = s;
            }
            for (int i = t - 64 + CT - 64; i < kb; i += CT - 64) {
                double s = y[i];
#pragma unroll 4
                for (int j = 0; j < nb; j++) s = fma(-L[(size_t)(kb + j) * P + i], y[kb + j], s);
                y[i] = s;
            }
        }
        __syncthreads();
    }
    if (t == 0) status[blockIdx.x] = 0;
}

// ------------------------------------------------------------------- PCG
// A symmetric (row-major, so A[j][i] = A[i][j] gives coalesced column reads).

// PCG A-column cache: each thread keeps kPcgRegs of its matrix-vector columns in registers
// and the next kPcgLds in LDS; the rest (P above about 170) come from global memory.
constexpr int kPcgRegs = 18;
constexpr int kPcgLds = 14;
// U (P x r) is copied to LDS when P * r fits.
constexpr int kPcgUCache = 2048;

// W block sums with one barrier: wave sums into wp[wave][c], barrier, every thread adds the
// 16 wave sums in wave order.  wp must not be rewritten before the next barrier, so callers
// alternate between two buffers.
template <int W>
__device__ __forceinline__ void block_sums(double (&v)[W], double (*wp)[8]) {
    static_assert(W >= 1 && W <= 2, "one or two sums per call");
#pragma unroll
    for (int c = 0; c < W; c++) v[c] = wave_sum_f64(v[c]);
    if ((threadIdx.x & 63) == 0)
#pragma unroll
        for (int c = 0; c < W; c++) wp[threadIdx.x >> 6][c] = v[c];
    __syncthreads();
    double t[W];
#pragma unroll
    for (int c = 0; c < W; c++) t[c] = 0.0;
#pragma unroll
    for (int w = 0; w < kT / 64; w++)
#pragma unroll
        for (int c = 0; c < W; c++) t[c] += wp[w][c];
#pragma unroll
    for (int c = 0; c < W; c++) v[c] = t[c];
}

// PCG with M^-1 = diag(d) + U U^T (d = NULL: identity diagonal; U = NULL: no low-rank part),
// one workgroup per system, three barriers per iteration (four with a low-rank part).  Matrix-vector product: thread t
// takes row t % P and the column segment t / P (kT / P segments), its A entries cached in
// registers and LDS at the start; the segments are added in a fixed order, and p^T A p comes
// from the same partial sums (sum over threads of p_row * partial) with no extra pass.  One
// more reduction gives |r|^2, r^T D r and w = U^T r together, so z = D r + U w and
// r^T z = r^T D r + |w|^2.
__global__ __launch_bounds__(kT) void pcg_f64_kernel(const double *Aall, const double *ball, double *xall, int P,
                                                     double lambda, const double *dall, const double *Uall, int r,
                                                     double tol, int maxit, int *iters, double *relres) {
    const double *A = Aall + (size_t)blockIdx.x * P * P;
    const double *b = ball + (size_t)blockIdx.x * P;
    double *x = xall + (size_t)blockIdx.x * P;
    const double *d = dall ? dall + (size_t)blockIdx.x * P : nullptr;
    const double *U = Uall ? Uall + (size_t)blockIdx.x * P * r : nullptr;
    __shared__ double sp[1024], seg_sum[kT], wbuf[2][kT / 64][8], tot[72], sd[1024];
    __shared__ double sa[kPcgLds * kT], su[kPcgUCache];
    const int i = threadIdx.x;
    const bool own = i < P;
    const int rk = (U && r > 0) ? r : 0;
    const int seg = kT / P;
    const int row = i % P, sg = i / P;
    const int seg_len = (P + seg - 1) / seg;
    const int j0 = min(P, sg * seg_len);
    const int len = sg < seg ? min(P, j0 + seg_len) - j0 : 0;
    double areg[kPcgRegs];
#pragma unroll
    for (int k = 0; k < kPcgRegs; k++) areg[k] = (k < len) ? A[(size_t)(j0 + k) * P + row] : 0.0;
    for (int k = kPcgRegs; k < min(len, kPcgRegs + kPcgLds); k++)
        sa[(k - kPcgRegs) * kT + i] = A[(size_t)(j0 + k) * P + row];
    const bool u_lds = rk > 0 && P * rk <= kPcgUCache;
    if (u_lds)
        for (int e = i; e < P * rk; e += kT) su[(e % rk) * P + e / rk] = U[e];
    const double di = own ? (d ? d[i] : 1.0) : 0.0;
    if (own) sd[i] = di;
    __syncthreads();
    auto uval = [&](int c) -> double { return u_lds ? su[c * P + i] : U[(size_t)i * rk + c]; };
    int ph = 0;
    double xi = 0.0, ri = own ? b[i] : 0.0;
    // Reduction of r: returns |r|^2, sets z = D r + U (U^T r) and rz = r^T z.
    auto reduce_r = [&](double &z, double &rz) -> double {
        double rr;
        z = di * ri;
        if (rk == 0) {
            double v[2] = {ri * ri, di * ri * ri};
            block_sums<2>(v, wbuf[ph]);
            ph ^= 1;
            rr = v[0];
            rz = v[1];
        } else {
            // the 2 + rk dot products r.r, r.(D r), (U^T r)_c share the waves: wave c % 16 takes
            // value c as a lane-strided sum over r in LDS and a wave sum.  sp is free here: the
            // matrix-vector reads of p ended at the previous barrier.
            const int lane = i & 63, wv = i >> 6;
            if (own) sp[i] = ri;
            __syncthreads();
            for (int c = wv; c < 2 + rk; c += kT / 64) {
                double acc = 0.0;
                for (int k = lane; k < P; k += 64) {
                    const double rv = sp[k];
                    const double f = (c == 0) ? rv
                                   : (c == 1) ? sd[k] * rv
                                   : (u_lds ? su[(c - 2) * P + k] : U[(size_t)k * rk + c - 2]);
                    acc += f * rv;
                }
                acc = wave_sum_f64(acc);
                if (lane == 0) tot[c] = acc;
            }
            __syncthreads();
            rr = tot[0];
            rz = tot[1];
            for (int c = 0; c < rk; c++) {
                const double wc = tot[2 + c];
                if (own) z += uval(c) * wc;
                rz += wc * wc;
            }
        }
        if (!own) z = 0.0;
        return rr;
    };
    double zi, rz;
    const double bn = sqrt(reduce_r(zi, rz));
    if (bn == 0.0) {
        if (own) x[i] = 0.0;
        if (i == 0) { iters[blockIdx.x] = 0; relres[blockIdx.x] = 0.0; }
        return;
    }
    double pi = zi;
    int it = 0;
    double rel = 1.0;
    for (; it < maxit; it++) {
        if (own) sp[i] = pi;
        __syncthreads();
        double partial = 0.0;
#pragma unroll
        for (int k = 0; k < kPcgRegs; k++)
            if (k < len) partial += areg[k] * sp[j0 + k];
        for (int k = kPcgRegs; k < min(len, kPcgRegs + kPcgLds); k++) partial += sa[(k - kPcgRegs) * kT + i] * sp[j0 + k];
        for (int k = kPcgRegs + kPcgLds; k < len; k++) partial += A[(size_t)(j0 + k) * P + row] * sp[j0 + k];
        seg_sum[i] = partial;
        // p^T (A + lambda I) p = sum over threads of p_row * partial, plus lambda |p|^2
        double v[1] = {(len > 0 ? partial * sp[row] : 0.0) + (own ? lambda * pi * pi : 0.0)};
        block_sums<1>(v, wbuf[ph]);                   // its barrier also publishes seg_sum
        ph ^= 1;
        double api = 0.0;
        if (own) {
            for (int q = 0; q < seg; q++) api += seg_sum[q * P + i];
            api += lambda * pi;
        }
        const double alpha = rz / v[0];
        xi += alpha * pi;
        ri -= alpha * api;
        double rz_new;
        rel = sqrt(reduce_r(zi, rz_new)) / bn;
        if (rel <= tol) { it++; break; }
        const double beta = rz_new / rz;
        rz = rz_new;
        pi = zi + beta * pi;
    }
    if (own) x[i] = xi;
    if (i == 0) { iters[blockIdx.x] = it; relres[blockIdx.x] = rel; }
}

// ------------------------------------------- extreme Hermitian eigenvalues
// The eigenvalues a condition number needs -- the smallest, the largest and
// the two next to zero -- of a Hermitian matrix (its upper triangle), without
// eigenvectors: Householder reduction to a real tridiagonal, then
// multisection on the Sturm counts, 128 points at a time for each of the four.
//
// One workgroup per component (a set of indices that the matrix couples to no other, adjacent in A):
// a small component beside a large one keeps its own accuracy and its own bounds.
// P <= 128: the matrix in registers (below); beyond, thread t owns column t % n
// and rows t / n (mod nseg) in W (global, in L2).  A step of the reduction applies the previous
// step's rank-2 update and forms the next matrix-vector product, with three
// barriers.  What bounds it: the latency of those steps.  P = 96: 335 us; 412 with rows split over
// waves (their vectors broadcast from LDS row by row), 667 with the threads' columns crossing the waves, and
// 29.5 ms by the cyclic Jacobi iteration, which still gives the eigenvectors elsewhere (8 to 10
// sweeps of P - 1 steps, each two passes over A and one over V in global memory).
// Indices whose row is zero off the diagonal are set aside first: their
// diagonal entries are exact eigenvalues (a parameter without effect leaves a
// zero row, and its exact zero is no part of the condition number).
// number of eigenvalues of the tridiagonal (d, e2 = squared off-diagonals) below x
__device__ __forceinline__ int sturm_count(const double *d, const double *e2, int n, double x, double pivmin) {
    int c = 0;
    double q = 1.0, prev = 0.0;
    for (int i = 0; i < n; i++) {
        double r = __builtin_amdgcn_rcp(q);
        const double e = fma(-q, r, 1.0);                    // |e| < 2^-23: third order leaves 2^-69
        r = fma(r, fma(e, e, e), r);
        q = (d[i] - x) - prev * r;
        if (fabs(q) < pivmin) q = -pivmin;
        c += q < 0.0;
        prev = e2[i];
    }
    return c;
}

// The four extremes of the tridiagonal (d, e2) of order n, into the threads that searched them, and a
// bound of its eigenvalues' sizes, which every thread receives; near: the smallest size of an
// eigenvalue, zero when one is within 1e-30 of the bound of zero.
__device__ __forceinline__ void tridiagonal_extremes(const double *sd, const double *se2, int n, double (*swv)[6],
                                                     int *cnt, double &lo_all, double &hi_all, double &pos_all,
                                                     double &neg_all, double &near, double &bd) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // Gershgorin bound
    bd = 0.0;
    if (t < n)
        bd = fabs(sd[t]) + (t > 0 ? sqrt(se2[t - 1]) : 0.0) + (t + 1 < n ? sqrt(se2[t]) : 0.0);
    if (!(bd < __builtin_inf())) bd = __builtin_inf();       // NaN too: the caller sees the bound
    for (int o = 32; o > 0; o >>= 1) bd = fmax(bd, __shfl_xor(bd, o, 64));
    if (lane == 0) swv[wave][0] = bd;
    __syncthreads();
    bd = 0.0;
    for (int w = 0; w < kT / 64; w++) bd = fmax(bd, swv[w][0]);
    const double B = bd * (1.0 + 1e-10), tiny = 1e-30 * bd, pivmin = 1e-40 * bd;
    // 128 points for each of the four, by the first eight waves: two waves a SIMD, whose issue then keeps
    // pace with the recurrence's latency (n = 96: the kernel takes 335 us; with all sixteen, 256 points and 9 rounds, 359)
    const int grp = t >> 7, m = t & 127;
    const int cz = bd > 0.0 && grp < 4 ? sturm_count(sd, se2, n, (t & 1) ? tiny : -tiny, pivmin) : 0;
    const int n_neg = __shfl(cz, 0, 64), n_pos = __shfl(cz, 1, 64);   // below -tiny, below +tiny
    const int idx = grp == 0 ? 0 : grp == 1 ? n - 1 : grp == 2 ? n_pos : n_neg - 1;
    const bool want = bd > 0.0 && grp < 4 && idx >= 0 && idx < n;
    double lo = grp == 2 ? 0.0 : -B, hi = grp == 3 ? 0.0 : B;
    for (int round = 0; round < 11; round++) {
        const double h = (hi - lo) * (1.0 / 129.0);
        int c = 0;
        if (want) c = sturm_count(sd, se2, n, lo + h * (m + 1), pivmin) <= idx;
        const int below = __popcll(__ballot(c != 0));
        if (lane == 0) cnt[wave] = below;
        __syncthreads();
        const int k = cnt[2 * grp] + cnt[2 * grp + 1];       // (grp < 8: within cnt)
        const double nl = k == 0 ? lo : lo + h * k, nh = k == 128 ? hi : lo + h * (k + 1);
        lo = nl;
        hi = nh;
        __syncthreads();
    }
    const double v = bd > 0.0 ? 0.5 * (lo + hi) : 0.0;
    if (grp == 0 && (want || bd == 0.0)) lo_all = fmin(lo_all, v);
    if (grp == 1 && (want || bd == 0.0)) hi_all = fmax(hi_all, v);
    if (grp == 2 && want) pos_all = fmin(pos_all, v);
    if (grp == 3 && want) neg_all = fmax(neg_all, v);
    if (grp >= 2 && want) near = fmin(near, fabs(v));
    if (t < 128 && (n_pos != n_neg || !(bd > 0.0))) near = 0.0;
}

__device__ __forceinline__ void write_extremes(double lo_all, double hi_all, double pos_all, double neg_all,
                                               double near, double bd, double (*swv)[6], double *out) {
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    for (int o = 32; o > 0; o >>= 1) {
        lo_all = fmin(lo_all, __shfl_xor(lo_all, o, 64));
        hi_all = fmax(hi_all, __shfl_xor(hi_all, o, 64));
        pos_all = fmin(pos_all, __shfl_xor(pos_all, o, 64));
        neg_all = fmax(neg_all, __shfl_xor(neg_all, o, 64));
        near = fmin(near, __shfl_xor(near, o, 64));
    }
    __syncthreads();
    if (lane == 0) {
        swv[wave][0] = lo_all; swv[wave][1] = hi_all; swv[wave][2] = pos_all; swv[wave][3] = neg_all;
        swv[wave][4] = near;
    }
    __syncthreads();
    if (t == 0) {
        for (int w = 1; w < kT / 64; w++) {
            lo_all = fmin(lo_all, swv[w][0]);
            hi_all = fmax(hi_all, swv[w][1]);
            pos_all = fmin(pos_all, swv[w][2]);
            neg_all = fmax(neg_all, swv[w][3]);
            near = fmin(near, swv[w][4]);
        }
        out[0] = lo_all; out[1] = hi_all; out[2] = pos_all; out[3] = neg_all;
        out[4] = near; out[5] = bd;
    }
}

// Householder vector of column k from x (x[i], i > k): u = x + (x_{k+1} / |x_{k+1}|) |x| e_{k+1}.  tail: the
// sum of |x_i|^2 over i > k + 1; x0 in: x_{k+1}, out: u_{k+1}.  Returns tau = 2 / |u|^2 (0: nothing to do).
__device__ __forceinline__ double householder(double tail, double2 &u0, double &e2) {
    const double x0 = u0.x * u0.x + u0.y * u0.y;
    e2 = x0;
    if (!(tail > 0.0)) return 0.0;
    e2 = tail + x0;
    const double s = sqrt(e2), m = sqrt(x0);
    const double tau = 1.0 / (s * (s + m));
    if (m > 0.0) { u0.x += u0.x * (s / m); u0.y += u0.y * (s / m); }
    else u0.x = s;
    return tau;
}

// The component of this workgroup in A (rows of ld): its first entry, its order in P.
__device__ __forceinline__ const double2 *component(const double2 *A, int ld, const int2 *comps, int &P) {
    P = ld;
    if (!comps) return A;
    const int2 c = comps[blockIdx.x];
    P = qgtl::uniform(c.y);
    return A + (size_t)qgtl::uniform(c.x) * (ld + 1);
}

// out, six values a component: smallest, largest, smallest positive (+inf: none), largest negative
// (-inf: none) eigenvalue; the smallest size of an eigenvalue that the reduction found (indices set
// aside left out; +inf: none) and a bound of the reduced part's eigenvalues, of which it is a
// few P eps uncertain
__global__ __launch_bounds__(kT) void herm_extremes_kernel(const double2 *__restrict__ Aall, int ld,
                                                           const int2 *__restrict__ comps, double2 *Wall,
                                                           double *outs) {
    int P;
    const double2 *A = component(Aall, ld, comps, P);
    double2 *W = Wall + (A - Aall) / (ld + 1) * (size_t)ld;   // n^2 of ld n: apart for all components
    double *out = outs + 6 * blockIdx.x;
    __shared__ double2 su[kT], sq[kT], sx[kT], part[kT];
    __shared__ double sd[kT], se2[kT], swv[kT / 64][6];
    __shared__ int map[kT];
    __shared__ unsigned long long bal[kT / 64];
    __shared__ int cnt[kT / 64];
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    // isolated indices
    bool iso = false;
    double isov = 0.0;
    if (t < P) {
        iso = true;
        for (int i = 0; i < P; i++) {
            if (i == t) continue;
            const double2 a = i < t ? A[(size_t)i * ld + t] : A[(size_t)t * ld + i];
            if (a.x != 0.0 || a.y != 0.0) iso = false;
        }
        isov = A[(size_t)t * ld + t].x;
    }
    const bool live = t < P && !iso;
    const unsigned long long b = __ballot(live);
    if (lane == 0) bal[wave] = b;
    su[t] = sq[t] = make_double2(0.0, 0.0);
    __syncthreads();
    int rank = 0, n = 0;
    for (int w = 0; w < kT / 64; w++) {
        const int c = __popcll(bal[w]);
        if (w < wave) rank += c;
        n += c;
    }
    rank += __popcll(b & ((1ull << lane) - 1ull));
    if (live) map[rank] = t;
    __syncthreads();
    const double inf = __builtin_inf();
    double lo_all = iso ? isov : inf, hi_all = iso ? isov : -inf;
    double pos_all = iso && isov > 0.0 ? isov : inf, neg_all = iso && isov < 0.0 ? isov : -inf;
    double near = inf, bd = 0.0;
    if (n > 0) {                                             // n >= 2: an index is live with another
        const int nseg = kT / n, seg = t / n, j = t % n;
        const int rows = (n + nseg - 1) / nseg;
        const int oj = map[j];
        auto entry = [&](int i) -> double2 {
            const int oi = map[i];
            if (oi <= oj) { double2 v = A[(size_t)oi * ld + oj]; if (oi == oj) v.y = 0.0; return v; }
            const double2 v = A[(size_t)oj * ld + oi];
            return make_double2(v.x, -v.y);
        };
        if (seg < nseg)
            for (int i = seg; i < n; i += nseg) W[(size_t)i * n + j] = entry(i);
        // x_i of column k for this thread's rows (it owns column k): the entry with the pending update
        auto pend = [&](double2 v, int i, double2 uk, double2 qk) -> double2 {
            const double2 ui = su[i], qi = sq[i];
            v.x -= ui.x * qk.x + ui.y * qk.y + qi.x * uk.x + qi.y * uk.y;
            v.y -= ui.y * qk.x - ui.x * qk.y + qi.y * uk.x - qi.x * uk.y;
            return v;
        };
        for (int k = 0; k < n; k++) {
            const double2 uj = su[j], qj = sq[j];
            if (j == k && seg < nseg)
                for (int r = 0; r < rows; r++) {
                    const int i = seg + nseg * r;
                    if (i >= k && i < n) sx[i] = pend(W[(size_t)i * n + j], i, uj, qj);
                }
            __syncthreads();
            if (t == 0) sd[k] = sx[k].x;
            if (k == n - 1) break;
            double tail = 0.0;
            for (int i = k + 2 + lane; i < n; i += 64) tail += sx[i].x * sx[i].x + sx[i].y * sx[i].y;
            tail = wave_sum_f64(tail);
            double2 u0 = sx[k + 1];
            double e2;
            const double tau = householder(tail, u0, e2);
            if (t == 0) se2[k] = e2;
            double pr = 0.0, pi = 0.0;
            if (j > k && seg < nseg) {
                auto one = [&](double2 v, int i) -> double2 {
                    v = pend(v, i, uj, qj);
                    const double2 ui = i == k + 1 ? u0 : sx[i];
                    pr += v.x * ui.x + v.y * ui.y;           // conj(a_ij) u_i
                    pi += v.x * ui.y - v.y * ui.x;
                    return v;
                };
                for (int r = 0; r < rows; r++) {
                    const int i = seg + nseg * r;
                    if (i > k && i < n) W[(size_t)i * n + j] = one(W[(size_t)i * n + j], i);
                }
            }
            part[t] = make_double2(pr, pi);
            __syncthreads();
            // p = tau A u; K = tau / 2 u^H p; q = p - K u (every wave forms u^H p for itself)
            double up = 0.0;
            for (int i = k + 1 + lane; i < n; i += 64) {
                double2 s = part[i];
                for (int g = 1; g < nseg; g++) { s.x += part[g * n + i].x; s.y += part[g * n + i].y; }
                const double2 ui = i == k + 1 ? u0 : sx[i];
                up += ui.x * s.x + ui.y * s.y;
            }
            up = wave_sum_f64(up);
            if (t < n) {
                double2 ut = make_double2(0.0, 0.0), qt = make_double2(0.0, 0.0);
                if (t > k && tau > 0.0) {
                    double2 s = part[t];
                    for (int g = 1; g < nseg; g++) { s.x += part[g * n + t].x; s.y += part[g * n + t].y; }
                    ut = t == k + 1 ? u0 : sx[t];
                    const double kk = tau * (0.5 * tau * up);      // tau^2 alone overflows below 1e-77
                    qt = make_double2(tau * s.x - kk * ut.x, tau * s.y - kk * ut.y);
                }
                su[t] = ut;
                sq[t] = qt;
            }
            __syncthreads();
        }
        __syncthreads();
        tridiagonal_extremes(sd, se2, n, swv, cnt, lo_all, hi_all, pos_all, neg_all, near, bd);
    }
    write_extremes(lo_all, hi_all, pos_all, neg_all, near, bd, swv, out);
}

// The same for P <= 16 COLS = 64 ROWS with the matrix in registers: wave w holds columns w + 16 s,
// its lane l rows l + 64 c.  A step: the wave of column k brings it up to date and forms the
// Householder vector by itself while the others apply the previous step's rank-2 update; then
// every wave adds its columns to p = A u, and two waves add up the sixteen parts.
template <int COLS, int ROWS>
__global__ __launch_bounds__(kT) void herm_extremes_regs_kernel(const double2 *__restrict__ Aall, int ld,
                                                                const int2 *__restrict__ comps, double *outs) {
    constexpr int N = 64 * ROWS;
    int P;
    const double2 *A = component(Aall, ld, comps, P);
    double *out = outs + 6 * blockIdx.x;
    static_assert(16 * COLS == N, "square");
    __shared__ double2 su[N], sq[N], part[16][N];
    __shared__ double sd[N], se2[N], swv[kT / 64][6], sup[kT / 64], stau;
    __shared__ int map[N], live[N], cnt[kT / 64];
    const int t = threadIdx.x, lane = t & 63, wave = qgtl::uniform(t >> 6);
    auto entry = [&](int oi, int oj) __attribute__((always_inline)) -> double2 {   // the upper triangle's
        if (oi <= oj) { double2 v = A[(size_t)oi * ld + oj]; if (oi == oj) v.y = 0.0; return v; }
        const double2 v = A[(size_t)oj * ld + oi];
        return make_double2(v.x, -v.y);
    };
    double2 a[COLS][ROWS];
#pragma unroll
    for (int s = 0; s < COLS; s++) {
        const int j = wave + 16 * s;
        bool any = false;
#pragma unroll
        for (int c = 0; c < ROWS; c++) {
            const int i = lane + 64 * c;
            a[s][c] = (i < P && j < P) ? entry(i, j) : make_double2(0.0, 0.0);
            any = any || (i != j && (a[s][c].x != 0.0 || a[s][c].y != 0.0));
        }
        const bool col = __ballot(any) != 0;
        if (lane == 0) live[j] = col;
    }
    __syncthreads();
    // live indices in order, counted by every wave
    int n = 0;
#pragma unroll
    for (int c = 0; c < ROWS; c++) {
        const bool l = live[lane + 64 * c] != 0;
        const unsigned long long b = __ballot(l);
        if (wave == 0 && l) map[n + __popcll(b & ((1ull << lane) - 1ull))] = lane + 64 * c;
        n += __popcll(b);
    }
    n = qgtl::uniform(n);
    __syncthreads();
    if (n < P && n > 0) {                                    // close up the isolated indices
#pragma unroll
        for (int s = 0; s < COLS; s++)
#pragma unroll
            for (int c = 0; c < ROWS; c++) {
                const int i = lane + 64 * c, j = wave + 16 * s;
                a[s][c] = (i < n && j < n) ? entry(map[i], map[j]) : make_double2(0.0, 0.0);
            }
    }
    double2 u[ROWS], q[ROWS];                                // the pending update, this lane's rows
#pragma unroll
    for (int c = 0; c < ROWS; c++) u[c] = q[c] = make_double2(0.0, 0.0);
    auto lane_of = [](double2 v, int l) __attribute__((always_inline)) -> double2 {
        return make_double2(readlane_f64(v.x, l), readlane_f64(v.y, l));
    };
    auto at = [&](const double2 (&v)[ROWS], int i) __attribute__((always_inline)) -> double2 {   // row i
        const bool up = ROWS > 1 && i >= 64;
        return lane_of(make_double2(up ? v[ROWS - 1].x : v[0].x, up ? v[ROWS - 1].y : v[0].y), i & 63);
    };
    // v - u_i conj(q_j) - q_i conj(u_j)
    auto pend = [&](double2 v, double2 ui, double2 qi, double2 uj, double2 qj) __attribute__((always_inline)) -> double2 {
        v.x = fma(-ui.x, qj.x, fma(-ui.y, qj.y, fma(-qi.x, uj.x, fma(-qi.y, uj.y, v.x))));
        v.y = fma(-ui.y, qj.x, fma(ui.x, qj.y, fma(-qi.y, uj.x, fma(qi.x, uj.y, v.y))));
        return v;
    };
    for (int k = 0; k < n; k++) {
        if (wave == (k & 15)) {
            __builtin_amdgcn_s_setprio(3);                   // the chain the others wait for
            const double2 uk = at(u, k), qk = at(q, k);
            double2 v[ROWS];
            double tail = 0.0;
#pragma unroll
            for (int c = 0; c < ROWS; c++) {
                v[c] = a[0][c];
#pragma unroll
                for (int s = 1; s < COLS; s++) {
                    const bool here = s == k >> 4;
                    v[c].x = here ? a[s][c].x : v[c].x;
                    v[c].y = here ? a[s][c].y : v[c].y;
                }
                v[c] = pend(v[c], u[c], q[c], uk, qk);
                const int i = lane + 64 * c;
                if (i > k + 1 && i < n) tail += v[c].x * v[c].x + v[c].y * v[c].y;
            }
            const double dk = at(v, k).x;
            if (lane == 0) sd[k] = dk;
            if (k < n - 1) {
                tail = wave_sum_f64(tail);
                double2 u0 = at(v, k + 1);
                double e2;
                const double tau = householder(tail, u0, e2);
                if (lane == 0) { se2[k] = e2; stau = tau; }
#pragma unroll
                for (int c = 0; c < ROWS; c++) {
                    const int i = lane + 64 * c;
                    double2 w = i == k + 1 ? u0 : v[c];
                    if (i <= k || i >= n || !(tau > 0.0)) w = make_double2(0.0, 0.0);
                    su[i] = w;
                }
            }
            __builtin_amdgcn_s_setprio(0);
        }
        if (k == n - 1) break;
#pragma unroll
        for (int s = 0; s < COLS; s++) {
            const int j = wave + 16 * s;
            if (j > k && j < n) {                            // the same for the wave
                const double2 uj = lane_of(u[s >> 2], j & 63), qj = lane_of(q[s >> 2], j & 63);
#pragma unroll
                for (int c = 0; c < ROWS; c++) a[s][c] = pend(a[s][c], u[c], q[c], uj, qj);
            }
        }
        __syncthreads();
        const double tau = stau;
        double2 p[ROWS];
#pragma unroll
        for (int c = 0; c < ROWS; c++) {
            u[c] = su[lane + 64 * c];
            p[c] = make_double2(0.0, 0.0);
        }
#pragma unroll
        for (int s = 0; s < COLS; s++) {
            const int j = wave + 16 * s;
            if (j > k && j < n) {
                const double2 uj = lane_of(u[s >> 2], j & 63);
#pragma unroll
                for (int c = 0; c < ROWS; c++) {
                    const double2 v = a[s][c];
                    p[c].x = fma(v.x, uj.x, fma(-v.y, uj.y, p[c].x));
                    p[c].y = fma(v.x, uj.y, fma(v.y, uj.x, p[c].y));
                }
            }
        }
        // p = tau A u; K = tau / 2 u^H p; q = p - K u
        double up = 0.0;
#pragma unroll
        for (int c = 0; c < ROWS; c++) {
            part[wave][lane + 64 * c] = p[c];
            up += u[c].x * p[c].x + u[c].y * p[c].y;         // u is zero outside k + 1 .. n - 1
        }
        up = wave_sum_f64(up);
        if (lane == 0) sup[wave] = up;
        __syncthreads();
        if (wave < ROWS) {
            double2 s = part[0][t];
            up = sup[0];
#pragma unroll 5
            for (int w = 1; w < 16; w++) {
                s.x += part[w][t].x;
                s.y += part[w][t].y;
                up += sup[w];
            }
            const double2 ut = su[t];
            const double kk = tau * (0.5 * tau * up);      // tau^2 alone overflows below 1e-77
            const bool in = t > k && t < n;
            sq[t] = make_double2(in ? tau * s.x - kk * ut.x : 0.0, in ? tau * s.y - kk * ut.y : 0.0);
        }
        __syncthreads();
#pragma unroll
        for (int c = 0; c < ROWS; c++) q[c] = sq[lane + 64 * c];
    }
    __syncthreads();
    const double inf = __builtin_inf();
    const bool iso = t < P && !live[t < N ? t : 0];
    const double isov = iso ? A[(size_t)t * ld + t].x : 0.0;
    double lo_all = iso ? isov : inf, hi_all = iso ? isov : -inf;
    double pos_all = iso && isov > 0.0 ? isov : inf, neg_all = iso && isov < 0.0 ? isov : -inf;
    double near = inf, bd = 0.0;
    if (n > 0) tridiagonal_extremes(sd, se2, n, swv, cnt, lo_all, hi_all, pos_all, neg_all, near, bd);
    write_extremes(lo_all, hi_all, pos_all, neg_all, near, bd, swv, out);
}

// B = M^H M for the singular values of a general complex matrix
__global__ void gram_small_c128_kernel(const double2 *M, double2 *B, int P) {
    for (int e = blockIdx.x * blockDim.x + threadIdx.x; e < P * P; e += gridDim.x * blockDim.x) {
        const int i = e / P, j = e % P;
        double sr = 0.0, si = 0.0;
        for (int k = 0; k < P; k++) {
            const double2 a = M[(size_t)k * P + i], c = M[(size_t)k * P + j];
            sr += a.x * c.x + a.y * c.y;
            si += a.x * c.y - a.y * c.x;
        }
        B[e] = make_double2(sr, si);
    }
}

// x = V diag(1/ev_i for |ev_i| > cutoff, else 0) V^H g   (one workgroup)
__global__ __launch_bounds__(kT) void pinv_apply_c128_kernel(const double2 *V, const double *ev, const double2 *g,
                                                             double2 *x, int P, double cutoff) {
    __shared__ double2 t[1024];
    for (int i = threadIdx.x; i < P; i += kT) {
        double sr = 0.0, si = 0.0;
        for (int k = 0; k < P; k++) {
            const double2 v = V[(size_t)k * P + i], gk = g[k];
            sr += v.x * gk.x + v.y * gk.y;       // conj(v) g
            si += v.x * gk.y - v.y * gk.x;
        }
        const double e = ev[i];
        t[i] = (fabs(e) > cutoff) ? make_double2(sr / e, si / e) : make_double2(0.0, 0.0);
    }
    __syncthreads();
    for (int k = threadIdx.x; k < P; k += kT) {
        double sr = 0.0, si = 0.0;
        for (int i = 0; i < P; i++) {
            const double2 p = cmul(V[(size_t)k * P + i], t[i]);
            sr += p.x;
            si += p.y;
        }
        x[k] = make_double2(sr, si);
    }
}

// ---- device-resident natural-gradient step ----
// A[k][l] = Re Q[s(k)][s(l)] + lambda delta_kl (Q: P x P complex in D-slot order),
// D[k] = A[k][k], g[k] = eg[1 + s(k)]: parameter order from slot order.
__global__ void ng_assemble_kernel(const double *__restrict__ Q, const int *__restrict__ slot, int P, double lambda,
                                   const double *__restrict__ eg, double *A, double *D, double *g) {
    const size_t total = (size_t)P * P;
    for (size_t idx = blockIdx.x * (size_t)blockDim.x + threadIdx.x; idx < total; idx += (size_t)gridDim.x * blockDim.x) {
        const int k = (int)(idx / P), l = (int)(idx % P);
        double v = Q[2 * ((size_t)slot[k] * P + slot[l])];
        if (k == l) {
            v += lambda;
            D[k] = v;
            g[k] = eg[1 + slot[k]];
        }
        A[idx] = v;
    }
}

// learned-preconditioner features: sin theta, cos theta, log D, field
__global__ void pc_features_kernel(const double *__restrict__ theta, const double *__restrict__ D, double field,
                                   int P, float *x) {
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k <= P; k += gridDim.x * blockDim.x) {
        if (k == P) {
            x[3 * P] = (float)field;
        } else {
            x[k] = (float)sin(theta[k]);
            x[P + k] = (float)cos(theta[k]);
            x[2 * P + k] = (float)log(D[k]);
        }
    }
}

// network output y (P (1 + r)) -> d = e^s / D, U = u / sqrt(P D)
__global__ void pc_transform_kernel(const float *__restrict__ y, const double *__restrict__ D, int P, int r,
                                    double *d, double *U) {
    const int st = 1 + r;
    const double us = 1.0 / sqrt((double)P);
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < P; k += gridDim.x * blockDim.x) {
        d[k] = exp((double)y[(size_t)k * st]) / D[k];
        const double sd = us / sqrt(D[k]);
        for (int j = 0; j < r; j++) U[(size_t)k * r + j] = (double)y[(size_t)k * st + 1 + j] * sd;
    }
}

__global__ void reciprocal_kernel(const double *__restrict__ D, int P, double *d) {
    for (int k = blockIdx.x * blockDim.x + threadIdx.x; k < P; k += gridDim.x * blockDim.x) d[k] = 1.0 / D[k];
}

}  // namespace

extern "C" {

int qgtl_hip_ng_assemble(const double *Q, const int *slot, int P, double lambda, const double *eg, double *A,
                         double *D, double *g) {
    const size_t total = (size_t)P * P;
    unsigned grid = (unsigned)((total + 255) / 256);
    if (grid > 4096) grid = 4096;
    hipLaunchKernelGGL(ng_assemble_kernel, dim3(grid), dim3(256), 0, qgtl::stream(), Q, slot, P, lambda, eg, A, D, g);
    QGTL_LAUNCH_CHECK("ng_assemble");
    return 0;
}

int qgtl_hip_pc_features(const double *theta, const double *D, double field, int P, float *x) {
    hipLaunchKernelGGL(pc_features_kernel, dim3((unsigned)((P + 256) / 256)), dim3(256), 0, qgtl::stream(), theta, D,
                       field, P, x);
    QGTL_LAUNCH_CHECK("pc_features");
    return 0;
}

int qgtl_hip_pc_transform(const float *y, const double *D, int P, int r, double *d, double *U) {
    hipLaunchKernelGGL(pc_transform_kernel, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, qgtl::stream(), y, D, P,
                       r, d, U);
    QGTL_LAUNCH_CHECK("pc_transform");
    return 0;
}

int qgtl_hip_reciprocal(const double *D, int P, double *d) {
    hipLaunchKernelGGL(reciprocal_kernel, dim3((unsigned)((P + 255) / 256)), dim3(256), 0, qgtl::stream(), D, P, d);
    QGTL_LAUNCH_CHECK("reciprocal");
    return 0;
}

int qgtl_hip_pinv_apply_c128(const void *V, const double *ev, const void *g, void *x, int P, double cutoff) {
    if (P > 1024) return qgtl::set_error_msg(-118, "pinv: P > 1024");
    hipLaunchKernelGGL(pinv_apply_c128_kernel, dim3(1), dim3(kT), 0, qgtl::stream(), (const double2 *)V, ev,
                       (const double2 *)g, (double2 *)x, P, cutoff);
    QGTL_LAUNCH_CHECK("pinv_apply_c128");
    return 0;
}

int qgtl_hip_lu_solve_c128(void *A, const void *b, void *x, int *piv, int P, int batch, int *status) {
    if (P <= 64)
        hipLaunchKernelGGL((lu_solve_regs_kernel<4, 1>), dim3(batch), dim3(kT), 0, qgtl::stream(), (const double2 *)A,
                           (const double2 *)b, (double2 *)x, P, status);
    else if (P <= 128)
        hipLaunchKernelGGL((lu_solve_regs_kernel<8, 2>), dim3(batch), dim3(kT), 0, qgtl::stream(), (const double2 *)A,
                           (const double2 *)b, (double2 *)x, P, status);
    else
        hipLaunchKernelGGL(lu_solve_c128_kernel, dim3(batch), dim3(kT), 0, qgtl::stream(), (double2 *)A,
                           (const double2 *)b, (double2 *)x, piv, P, status);
    QGTL_LAUNCH_CHECK("lu_solve_c128");
    return 0;
}

int qgtl_hip_herm_eig_c128(void *A, void *V, double *ev, int P, int batch, int max_sweeps, int *sweeps) {
    if (P > 1024) return qgtl::set_error_msg(-118, "herm_eig: P > 1024");
    hipLaunchKernelGGL(herm_eig_c128_kernel, dim3(batch), dim3(kT), 0, qgtl::stream(), (double2 *)A, (double2 *)V,
                       ev, P, max_sweeps, sweeps);
    QGTL_LAUNCH_CHECK("herm_eig_c128");
    return 0;
}

int qgtl_hip_herm_extremes_c128(const void *A, void *W, int P, const int *comps, int ncomps, int largest,
                                double *out) {
    if (P < 1 || P > kT || ncomps < 1 || ncomps > P || largest < 1 || largest > P || (!comps && largest != P))
        return qgtl::set_error_msg(-118, "herm_extremes: needs 1 <= P <= 1024 and components of 1 .. P indices");
    const dim3 grid((unsigned)(comps ? ncomps : 1));
    const int2 *c = (const int2 *)comps;
    if (largest <= 64)
        hipLaunchKernelGGL((herm_extremes_regs_kernel<4, 1>), grid, dim3(kT), 0, qgtl::stream(), (const double2 *)A, P, c,
                           out);
    else if (largest <= 128)
        hipLaunchKernelGGL((herm_extremes_regs_kernel<8, 2>), grid, dim3(kT), 0, qgtl::stream(), (const double2 *)A, P, c,
                           out);
    else
        hipLaunchKernelGGL(herm_extremes_kernel, grid, dim3(kT), 0, qgtl::stream(), (const double2 *)A, P, c,
                           (double2 *)W, out);
    QGTL_LAUNCH_CHECK("herm_extremes_c128");
    return 0;
}

int qgtl_hip_cholesky_solve_f64(double *A, const double *b, double *x, int P, int batch, double lambda, int *status) {
    if (P < 1 || P > 1024) return qgtl::set_error_msg(-118, "cholesky: needs 1 <= P <= 1024");
#define QGTL_CHOL(NB, ROWS, CT)                                                                                   \
    hipLaunchKernelGGL((cholesky_f64_kernel<NB, ROWS, CT>), dim3(batch), dim3(CT), 0, qgtl::stream(), A, b, x, P, lambda, \
                       status)
    // ROWS >= round16(P - NB + 1).  Device time of one system, this line / the next one's form: P = 4 7 / 12 us,
    // P = 32 20 / 25, P = 64 34 / 49
    if (P <= 4) QGTL_CHOL(4, 16, 128);
    else if (P <= 32) QGTL_CHOL(16, 32, 128);
    else if (P <= 64) QGTL_CHOL(16, 64, 256);
    else if (P <= 256) QGTL_CHOL(32, 240, 512);      // P = 192: 145 us, 147 with the next line's panel
    else if (P <= 512) QGTL_CHOL(32, 496, 512);
    else QGTL_CHOL(16, 1024, 512);
#undef QGTL_CHOL
    QGTL_LAUNCH_CHECK("cholesky_f64");
    return 0;
}

int qgtl_hip_pcg_f64(const double *A, const double *b, double *x, int P, int batch, double lambda, const double *d,
                     const double *U, int r, double tol, int maxit, int *iters, double *relres) {
    if (P > 1024 || r > 64) return qgtl::set_error_msg(-118, "pcg: P > 1024 or rank > 64");
    hipLaunchKernelGGL(pcg_f64_kernel, dim3(batch), dim3(kT), 0, qgtl::stream(), A, b, x, P, lambda, d, U, r, tol,
                       maxit, iters, relres);
    QGTL_LAUNCH_CHECK("pcg_f64");
    return 0;
}

int qgtl_hip_gram_small_c128(const void *M, void *B, int P) {
    const unsigned grid = (unsigned)((P * P + 255) / 256);
    hipLaunchKernelGGL(gram_small_c128_kernel, dim3(grid), dim3(256), 0, qgtl::stream(), (const double2 *)M,
                       (double2 *)B, P);
    QGTL_LAUNCH_CHECK("gram_small_c128");
    return 0;
}

}  // extern "C"
