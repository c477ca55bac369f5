// Discrete adjoint (reverse mode) and tangent (forward mode) of the FP64
// WENO5 + TVD-RK3 advection step and of the WENO5-RK3 reinitialization with
// its subcell fix, on one grid.
//
// Every fused stage maps its input field fs (and the previous RK level fn)
// to out_i = c_s (fs_i - step_i) + e_s fn_i (c_s, e_s = 1, 0 / 1/4, 3/4 /
// 2/3, 1/3), where step_i depends on fs along the three 7-point lines through
// i (clamped at the box) and on per-point parameters: the velocity for the
// advection; the mask, subcell distances and pseudo-time step of the
// reinitialization.  The Jacobian kernels differentiate the forward formulas
// exactly, the WENO weights included, with every branch (upwind side,
// sign-change test, Godunov selection, frozen points) the one the forward pass
// took: the uniform correction and the Godunov step by one sweep back through
// their operations (jp_q_grad, godunov_grad), the nonuniform stencil at the
// interface points on dual numbers (vls_dual.hpp).  They store, per point, the 21
// derivatives of out_i along its three lines (rows a*7+k, a = x,y,z, k =
// offset+3), for the adjoint times lam_i; the parameter derivatives go to
// their gradients at once in the adjoint and to memory in the tangent.  The
// adjoint sweep gathers the transposed stencil (deterministic: each output
// point sums its own contributions in a fixed order); the tangent sweep
// applies it.
//
// The subcell distances of the reinitialization depend on its initial field
// F0 through the root of the quintic through six values (six_distance,
// boundary_location.cu:53-80): d(root)/dy_k = -l_k(root)/p'(root) with l_k the
// Lagrange basis (implicit function theorem); roots clamped to the cell end
// do not move; the quadratic-ENO branch is differentiated on dual numbers.
#include <algorithm>

#include "vls_dual.hpp"
#include "vls_tile.hpp"

namespace vls {

__device__ __forceinline__ double stage_c(int stage) { return stage == 0 ? 1.0 : (stage == 1 ? 0.25 : 2.0 / 3.0); }

// index of the point at `off` from (r,c,p) along axis a, clamped
__device__ __forceinline__ idx_t shifted(const Box& b, int r, int c, int p, int a, int off)
{
    if (a == 0) c = clampi(c + off, b.cols - 1);
    else if (a == 1) r = clampi(r + off, b.rows - 1);
    else p = clampi(p + off, b.pges - 1);
    return lin(b, r, c, p);
}

__device__ __forceinline__ void point_coords(const Box& b, idx_t i, int& r, int& c, int& p) { coords_of(b, i, r, c, p); }

// ---------------------------------------------------------------------------
// advection stage Jacobian, a wave per axis over 64 points.  Tangent (lam
// null): J (21 rows of n) and U[a] = d out_i / d u_a,i.  Adjoint: J times
// lam_i, and U[a] += d out_i / d u_a,i lam_i (the velocity gradient).
// ---------------------------------------------------------------------------
// Derivatives of the uniform WENO5 derivatives of a line.  The correction Q
// depends on four second differences; the seven line values enter through the
// second differences D_j = p_j - 2 p_{j+1} + p_{j+2} and the central part
// C = p_1 - p_5 + 8 (p_4 - p_2), whose derivatives are constants (line_row).
//
// Q(d[i0], d[i1], d2, d[i3]) of the back (0, 1, 3) or fore (4, 3, 1) side and its
// four derivatives.  The value is jp_q's operation by operation; the derivatives
// come from one sweep back through it (names with b: dQ / d that value), ~50
// operations where four duals carried through jp_q took ~170: the bulk Jacobian,
// bound by its FP64 issue, 24.2 -> 17.5 us at 64^3 (with godunov_grad below), the
// advection one 16.4 -> 15.4.
struct JpGrad {
    double v, d[4];
};
__device__ __forceinline__ JpGrad jp_q_grad(const JPcd<double>& m, bool fore, double e)
{
    const double k = 3.0 / 13.0;
    const double a = fore ? m.d[4] : m.d[0], b = fore ? m.d[3] : m.d[1], c = m.d[2], d = fore ? m.d[1] : m.d[3];
    const double t0 = a - b, t1 = b - c, t2 = c - d;
    const double y0 = fma(-3.0, b, a), y1 = b + c, y2 = fma(3.0, c, -d);
    const double k0 = k * y0, k1 = k * y1, k2 = k * y2;
    const double s0 = fma(t0, t0, fma(k0, y0, e)), s1 = fma(t1, t1, fma(k1, y1, e)), s2 = fma(t2, t2, fma(k2, y2, e));
    const double a0 = s0 * s0, a1 = s1 * s1, a2 = s2 * s2;
    const double w0 = a1 * a2, w1 = 6.0 * (a0 * a2), w2 = 3.0 * (a0 * a1);
    const double W = (w0 + w1) + w2, tA = t0 - t1, tB = t1 - t2, c2 = fma(2.0, w2, -W);
    const RecipT<double> rW = recip(W);
    JpGrad q;
    q.v = quot(fma(4.0 * w0, tA, c2 * tB), rW);
    // Q = (4 w0 tA + (2 w2 - W) tB) / W with W = w0 + w1 + w2
    const double w1b = -(q.v + tB) * rW.y, w0b = fma(4.0 * tA, rW.y, w1b), w2b = fma(2.0 * tB, rW.y, w1b);
    const double tAb = 4.0 * w0 * rW.y, tBb = c2 * rW.y;
    // a_k = s_k^2, with the factor 2 s_k of ds_k and the 2 of dt_k, dy_k: 4 s_k
    const double g0 = 4.0 * s0 * fma(6.0 * a2, w1b, 3.0 * a1 * w2b);
    const double g1 = 4.0 * s1 * fma(a2, w0b, 3.0 * a0 * w2b);
    const double g2 = 4.0 * s2 * fma(a1, w0b, 6.0 * a0 * w1b);
    const double t0b = fma(g0, t0, tAb), t1b = fma(g1, t1, tBb - tAb), t2b = fma(g2, t2, -tBb);
    const double y0b = g0 * k0, y1b = g1 * k1, y2b = g2 * k2;
    q.d[0] = t0b + y0b;
    q.d[1] = fma(-3.0, y0b, (t1b - t0b) + y1b);
    q.d[2] = fma(3.0, y2b, (t2b - t1b) + y1b);
    q.d[3] = -(t2b + y2b);
    return q;
}
// row k of sc * C + sum_j ed[j] D_j
__device__ __forceinline__ double line_row(int k, double sc, const double ed[5])
{
    const double c = k == 1 ? 1.0 : (k == 5 ? -1.0 : (k == 4 ? 8.0 : (k == 2 ? -8.0 : 0.0)));
    double w = c * sc;
    if (k < 5) w += ed[k];
    if (k >= 1 && k < 6) w -= 2.0 * ed[k - 1];
    if (k >= 2) w += ed[k - 2];
    return w;
}

struct Grad3 {
    double* g[3];
};

__global__ void __launch_bounds__(192) ka_advect_jac(double* __restrict__ J, Grad3 U, const double* __restrict__ lam,
                                                     const double* __restrict__ fs, const double* __restrict__ vx,
                                                     const double* __restrict__ vy, const double* __restrict__ vz,
                                                     double dt, Box b, Inv inv, int stage)
{
    const idx_t n = (idx_t)b.rows * b.cols * b.pges;
    const int a = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const idx_t i = (idx_t)blockIdx.x * 64 + (threadIdx.x & 63);
    if (i >= n) return;
    int r, c, p;
    point_coords(b, i, r, c, p);
    const double cs = stage_c(stage);
    const double vel = (a == 0 ? vx : (a == 1 ? vy : vz))[i];
    double v[7];
    line7(fs, r, c, p, a, b, v);
    // the term of axis a: coef(u_a) * D_a (upwind_axis), D = (C -+ Q) k
    const JPd jp = inv.jd[a];
    const JPcd<double> m = jp_centre(v);
    const bool fore = vel < 0;
    const JpGrad q = jp_q_grad(m, fore, jp.e);
    const double d = (fore ? m.c + q.v : m.c - q.v) * jp.k;
    const double li = lam ? lam[i] : 1.0;
    // out = c (fs - dt * sum_a t_a) + e fn
    const double w0 = -cs * dt * (fore ? vel : dmax(0.0, vel)) * jp.k, sq = fore ? w0 : -w0;
    const double ed[5] = {fore ? 0.0 : sq * q.d[0], sq * (fore ? q.d[3] : q.d[1]), sq * q.d[2],
                          sq * (fore ? q.d[1] : q.d[3]), fore ? sq * q.d[0] : 0.0};
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        double w = line_row(k, w0, ed);
        if (a == 0 && k == 3) w += cs;
        J[(size_t)(a * 7 + k) * n + i] = w * li;
    }
    const double ju = (vel < 0 || vel > 0) ? -cs * dt * d : 0.0;
    U.g[a][i] = lam ? U.g[a][i] + ju * li : ju;
}

// ---------------------------------------------------------------------------
// reinitialization stage Jacobian (re_step.cu:283-393 as the fused stage
// kernels evaluate it) in two launches.  The first takes the points without
// subcell distances on the uniform WENO5 (spacing distances, the bulk time
// step, no parameter derivatives) and appends those next to a sign change of
// fs to `extra`, which the forward evaluates on the nonuniform form too; the
// second takes the listed points and those.  Parameter derivatives of a
// listed point, d out / d (xpr, xpl, ypf, ypb, zpu, zpd, dt), 7 rows of cap in
// list order: tangent (lam null) JP, adjoint JP += derivative times lam_i.
//
// In both launches a block takes 64 points with one wave per axis; the values
// of the three axes' pairs meet in LDS for the Godunov step, and each wave
// writes its axis's rows.  In the second the 9 inputs of an axis (7 line
// values, r1, l1) are three groups (blockIdx.y), so that the duals of the
// nonuniform form stay in registers.  (With one lane per point the duals of 9
// inputs and 3 axes spilled 2.9 KB a lane, and a list of a few thousand points
// filled a few dozen CUs.  Measured on MI355X at 64^3:
// 68 + 172 us -> 17.5 + 22 us; the first is bound by its FP64 arithmetic, the
// second by the dependent chain of the nonuniform form.)
// ---------------------------------------------------------------------------
// the Godunov step's derivatives with respect to this axis's pair (d[0] fore,
// d[1] back) and dt (d[2]) from the six values of the pairs: the selections of
// godunov_axis and the square root of godunov_step; dt < 0: frozen, step 0
struct GodunovGrad {
    double d[3];
};
__device__ __forceinline__ GodunovGrad godunov_grad(const double (&val6)[3][2][64], int lane, int a, bool inside,
                                                    double dt)
{
    GodunovGrad r = {};
    if (!(dt >= 0)) return r;
    double g = 0.0;
#pragma unroll
    for (int k = 0; k < 3; ++k) {
        const double m = godunov_axis(inside, val6[k][1][lane], val6[k][0][lane]);
        g = k == 0 ? m : g + m;
    }
    const double s = sqrt(g), h = s > 0 ? 0.5 / s : 0.0, sd = inside ? -dt : dt;
    const double fo = val6[a][0][lane], bk = val6[a][1][lane];
    const bool back = (0.0 < bk) != inside;
    const double m = back ? bk : 0.0;
    const bool fore = (m < -fo) != inside;
    const double dn = 2.0 * (fore ? -fo : m) * h * sd;  // of the selected extremum
    r.d[0] = fore ? -dn : 0.0;
    r.d[1] = !fore && back ? dn : 0.0;
    r.d[2] = inside ? -(s - 1.0) : s - 1.0;
    return r;
}

__global__ void __launch_bounds__(192)
ka_reinit_jac_bulk(double* __restrict__ J, const double* __restrict__ lam, const double* __restrict__ fs,
                   const uint8_t* __restrict__ flags, Box b, Inv inv, int stage, int* __restrict__ extra,
                   int* __restrict__ extra_count, int seq)
{
    __shared__ double val6[3][2][64];
    __shared__ unsigned long long crossing[3];
    const idx_t n = (idx_t)b.rows * b.cols * b.pges;
    const int lane = (int)(threadIdx.x & 63), a = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const idx_t i = (idx_t)blockIdx.x * 64 + lane;
    if (blockIdx.x == 0 && threadIdx.x == 0) extra_count[(seq + 1) & 1] = 0;
    const uint8_t fl = i < n ? flags[i] : (uint8_t)FLAG_SUBCELL;
    const bool mine = !(fl & FLAG_SUBCELL);
    JpGrad qf = {}, qb = {};
    double fo = 0.0, bk = 0.0;
    const JPd jp = inv.jd[a];
    bool cross = false;
    if (mine) {
        int r, c, p;
        point_coords(b, i, r, c, p);
        double v[7];
        line7(fs, r, c, p, a, b, v);
        cross = sign_change3(v);
        const JPcd<double> cd = jp_centre(v);
        qb = jp_q_grad(cd, false, jp.e);
        qf = jp_q_grad(cd, true, jp.e);
        bk = (cd.c - qb.v) * jp.k;
        fo = (cd.c + qf.v) * jp.k;
    }
    val6[a][0][lane] = fo;
    val6[a][1][lane] = bk;
    const unsigned long long m = __ballot(cross);
    if (lane == 0) crossing[a] = m;
    __syncthreads();
    const bool any = ((crossing[0] | crossing[1] | crossing[2]) >> lane) & 1;
    if (a == 0) wave_append(any, (int)i, extra, &extra_count[seq & 1]);
    if (!mine || any) return;
    const GodunovGrad g = godunov_grad(val6, lane, a, (fl & FLAG_MASK) != 0, inv.dt_bulk);
    const double cs = stage_c(stage), li = lam ? lam[i] : 1.0;
    const double wf = -cs * g.d[0] * jp.k, wb = -cs * g.d[1] * jp.k;
    const double ed[5] = {-wb * qb.d[0], wf * qf.d[3] - wb * qb.d[1], wf * qf.d[2] - wb * qb.d[2],
                          wf * qf.d[1] - wb * qb.d[3], wf * qf.d[0]};
#pragma unroll
    for (int k = 0; k < 7; ++k) {
        double w = line_row(k, wf + wb, ed);
        if (k == 3 && a == 0) w += cs;
        J[(size_t)(a * 7 + k) * n + i] = w * li;
    }
}

// axis pair (fore, back) with reinit_axis's branch, on duals that carry the
// derivatives with respect to M of its 9 inputs, the 7 line values (0..6), r1
// and l1 (7, 8): inputs first .. first + M - 1
template <int M>
__device__ __forceinline__ void reinit_axis_dual(Dual<M>& fo, Dual<M>& bk, const double v[7], double r1, double l1,
                                                 double ds, JPd jp, int first)
{
    Dual<M> q[9];
#pragma unroll
    for (int k = 0; k < 9; ++k) {
        q[k] = Dual<M>(k < 7 ? v[k] : (k == 7 ? r1 : l1));
#pragma unroll
        for (int m = 0; m < M; ++m) q[k].d[m] = (k == first + m) ? 1.0 : 0.0;
    }
    if (v[2] * v[3] < 0 || v[3] * v[4] < 0) {
        const PairT<Dual<M>> pr = weno_nonuniform_pair_inl(q[0], q[1], q[2], q[3], q[4], q[5], q[6], q[7], q[8], ds,
                                                           Dual<M>(0.0), Dual<M>(0.0));
        fo = pr.fore;
        bk = pr.back;
    } else {
        weno5_pair(fo, bk, q, jp);
    }
}

constexpr int kJacGroup = 3;  // inputs per block of the listed points' launch

__global__ void __launch_bounds__(192) ka_reinit_jac_list(double* __restrict__ J, double* __restrict__ JP,
                                                          const double* __restrict__ lam,
                                                          const double* __restrict__ fs,
                                                          const uint8_t* __restrict__ flags, IList il, Box b, Inv inv,
                                                          int stage, const int* __restrict__ extra,
                                                          const int* __restrict__ extra_count, int seq)
{
    __shared__ double val6[3][2][64];
    const idx_t n = (idx_t)b.rows * b.cols * b.pges;
    const int lane = (int)(threadIdx.x & 63), a = __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6));
    const int first = (int)blockIdx.y * kJacGroup;
    const int listed = *il.count, total = listed + extra_count[seq & 1];
    const double ds = a == 0 ? b.dx : (a == 1 ? b.dy : b.dz);
    const double cs = stage_c(stage);
    for (int j0 = (int)blockIdx.x * 64; j0 < total; j0 += (int)gridDim.x * 64) {
        const int j = j0 + lane;
        const bool in = j < total, list = j < listed;
        const idx_t i = in ? (list ? (idx_t)il.idx[j] : (idx_t)extra[j - listed]) : 0;
        const uint8_t fl = flags[i];
        const double dt = list ? il.dt[j] : inv.dt_bulk;
        Dual<kJacGroup> fo(0.0), bk(0.0);
        if (in && dt >= 0) {
            int r, c, p;
            point_coords(b, i, r, c, p);
            double v[7], r1 = ds, l1 = ds;
            line7(fs, r, c, p, a, b, v);
            if (list) {
                r1 = il.dist[(size_t)(2 * a) * il.cap + j];
                l1 = il.dist[(size_t)(2 * a + 1) * il.cap + j];
            }
            reinit_axis_dual(fo, bk, v, r1, l1, ds, inv.jd[a], first);
        }
        val6[a][0][lane] = fo.v;
        val6[a][1][lane] = bk.v;
        __syncthreads();
        if (in) {
            const GodunovGrad g = godunov_grad(val6, lane, a, (fl & FLAG_MASK) != 0, dt);
            const double li = lam ? lam[i] : 1.0;
#pragma unroll
            for (int m = 0; m < kJacGroup; ++m) {
                const int k = first + m;
                double w = -cs * (g.d[0] * fo.d[m] + g.d[1] * bk.d[m]);
                if (k == 3 && a == 0) w += cs;
                w *= li;
                if (k < 7) {
                    J[(size_t)(a * 7 + k) * n + i] = w;
                } else if (list) {
                    double* o = JP + (size_t)(2 * a + k - 7) * il.cap + j;
                    *o = lam ? *o + w : w;
                }
            }
            if (list && a == 0 && first == 0) {
                double* o = JP + (size_t)6 * il.cap + j;
                const double w = -cs * g.d[2] * li;
                *o = lam ? *o + w : w;
            }
        }
        __syncthreads();  // val6 is read before the next points' values come in
    }
}

// ---------------------------------------------------------------------------
// sweeps
// ---------------------------------------------------------------------------
// adjoint: out[j] = sum over (i, a, k) with clamp(i + (k-3) e_a) = j of
// P[a*7+k][i] (the Jacobian's rows times lam_i), plus ca*A[j] + cb*B[j] (A, B may
// be null).  Every (a, k) has the point i = j - (k-3) e_a if that is in the box;
// these 21 loads are issued together.  A point on a face of the box also
// takes the rows of the points whose taps were clamped to it.  out may be A
// or B.  Reads 21 rows once: 44 MB at 64^3 in 8.9 us
// (4.9 TB/s; 20 us with the loads one after another near a face, which every
// wave of 64 rows touches).
__global__ void __launch_bounds__(256) ka_transpose(double* out, const double* __restrict__ P, Box b, double ca,
                                                    const double* A, double cb, const double* B)
{
    const idx_t n = (idx_t)b.rows * b.cols * b.pges;
    const idx_t j = (idx_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (j >= n) return;
    int r, c, p;
    point_coords(b, j, r, c, p);
    const double va = A ? A[j] : 0.0, vb = B ? B[j] : 0.0;
    const idx_t st[3] = {(idx_t)b.rows, 1, (idx_t)b.rows * b.cols};
    const int pos[3] = {c, r, p}, len[3] = {b.cols, b.rows, b.pges};
    double w[21], acc = 0.0;
#pragma unroll
    for (int e = 0; e < 21; ++e) {
        const int a = e / 7, o = e % 7 - 3, ia = pos[a] - o;
        const bool in = ia >= 0 && ia < len[a];
        w[e] = P[(size_t)e * n + (in ? j - o * st[a] : j)];
        if (!in) w[e] = 0.0;
    }
#pragma unroll
    for (int e = 0; e < 21; ++e) acc += w[e];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        // the taps beyond the face: offset -o of the points 0 .. o-1, and mirrored
        if (pos[a] == 0)
            for (int o = 1; o <= 3; ++o)
                for (int ia = 0; ia < o; ++ia) acc += P[(size_t)(a * 7 + 3 - o) * n + (j + ia * st[a])];
        if (pos[a] == len[a] - 1)
            for (int o = 1; o <= 3; ++o)
                for (int ia = 0; ia < o; ++ia) acc += P[(size_t)(a * 7 + 3 + o) * n + (j - ia * st[a])];
    }
    out[j] = (ca * va + cb * vb) + acc;
}

// tangent: out[i] = sum_{a,k} J[a*7+k][i] x[clamp(i + (k-3) e_a)]
__global__ void __launch_bounds__(256) ka_apply(double* __restrict__ out, const double* __restrict__ J,
                                                const double* __restrict__ x, Box b)
{
    const idx_t n = (idx_t)b.rows * b.cols * b.pges;
    const idx_t i = (idx_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    int r, c, p;
    point_coords(b, i, r, c, p);
    double acc = 0.0;
#pragma unroll 1
    for (int a = 0; a < 3; ++a)
        for (int k = 0; k < 7; ++k) acc += J[(size_t)(a * 7 + k) * n + i] * x[shifted(b, r, c, p, a, k - 3)];
    out[i] = acc;
}

__global__ void ka_fill(double* __restrict__ y, double v, idx_t n)
{
    const idx_t i = (idx_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) y[i] = v;
}

// y = alpha*x + beta*y (beta == 0 overwrites)
__global__ void ka_axpby(double* __restrict__ y, const double* __restrict__ x, double alpha, double beta, idx_t n)
{
    const idx_t i = (idx_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    y[i] = alpha * x[i] + (beta == 0.0 ? 0.0 : beta * y[i]);
}

// out[i] += sum_a JU[a][i] * udot_a[i]   (velocity tangent)
__global__ void ka_velocity_tangent(double* __restrict__ out, const double* __restrict__ JU,
                                    const double* __restrict__ ux, const double* __restrict__ uy,
                                    const double* __restrict__ uz, idx_t n)
{
    const idx_t i = (idx_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    out[i] += JU[i] * ux[i] + JU[(size_t)n + i] * uy[i] + JU[(size_t)2 * n + i] * uz[i];
}

// reinitialization parameters, list order (7 rows of cap):
// out[idx[j]] += sum_e JP[e][j] Pdot[e][j]
__global__ void ka_param_tangent(double* __restrict__ out, const double* __restrict__ JP,
                                 const double* __restrict__ Pdot, IList il)
{
    const int cnt = *il.count;
    for (int j = (int)(blockIdx.x * blockDim.x + threadIdx.x); j < cnt; j += (int)(gridDim.x * blockDim.x)) {
        double s = 0.0;
        for (int e = 0; e < 7; ++e) s += JP[(size_t)e * il.cap + j] * Pdot[(size_t)e * il.cap + j];
        out[il.idx[j]] += s;
    }
}

// ---------------------------------------------------------------------------
// subcell distances as functions of F0
// ---------------------------------------------------------------------------
// eno_quadratic_distance (boundary_location.cu:6-20) on duals
template <int N>
__device__ __forceinline__ Dual<N> eno_quadratic_distance_d(Dual<N> v1, Dual<N> v0, Dual<N> v2, Dual<N> v3, double ds)
{
#pragma clang fp contract(off)
    const double eps = 10e-10;
    const Dual<N> p2l = v2 - 2.0 * v0 + v1;
    const Dual<N> p2r = v3 - 2.0 * v2 + v0;
    // min_mod on values, derivative of the chosen argument
    Dual<N> p2;
    if (p2l.v * p2r.v < 0) p2 = Dual<N>(0.0);
    else p2 = (fabs(p2l.v) < fabs(p2r.v)) ? p2l : p2r;
    if (p2.v > eps || p2.v < -eps) {
        const Dual<N> disc = sq(0.5 * p2 - v0 - v2) - 4. * v0 * v2;
        return ds * (0.5 + (v0 - v2 - ksign(v0.v - v2.v) * sqrt(disc)) / p2);
    }
    return ds * v0 / (v0 - v2);
}

// d(distance)/d(y_0..y_5) of six_distance(y_0..y_5, s); returns false when the
// distance does not move (no crossing or a root clamped to the cell end)
__device__ bool six_distance_grad(const double y[6], double s, double g[6])
{
    for (int k = 0; k < 6; ++k) g[k] = 0.0;
    if (y[1] * y[2] < 0 || y[3] * y[4] < 0) {
        Dual<4> q[4];
        for (int k = 0; k < 4; ++k) q[k] = ad::dvar<4>(y[k + 1], k);
        const Dual<4> d = eno_quadratic_distance_d(q[0], q[1], q[2], q[3], s);
        for (int k = 0; k < 4; ++k) g[k + 1] = d.d[k];
        return true;
    }
    const double xx[6] = {0.0, s, 2 * s, 3 * s, 4 * s, 5 * s};
    double coef[6];
    poly5_interp(xx, y, coef);
    const double x = zeroin_poly5(coef, 2 * s, 3 * s, 3e-16);
    if (!(x > 2 * s && x < 3 * s)) return false;
    // p'(x) from the monomial coefficients, Lagrange basis at x
    double dp = 0.0, pw = 1.0;
    for (int m = 1; m <= 5; ++m) {
        dp += m * coef[m] * pw;
        pw *= x;
    }
    if (dp == 0.0) return false;
    for (int k = 0; k < 6; ++k) {
        double l = 1.0;
        for (int m = 0; m < 6; ++m)
            if (m != k) l *= (x - xx[m]) / (xx[k] - xx[m]);
        g[k] = -l / dp;
    }
    return true;
}

// the six distances of a listed point i as functions of F0: for each of the
// 12 (axis, side) pairs, the six F0 indices and derivatives
__device__ void dist_grads(const double* __restrict__ F0, const Box& b, idx_t i, int a, int side, idx_t idx[6],
                           double g[6], bool& moves)
{
    int r, c, p;
    point_coords(b, i, r, c, p);
    double v[7];
    line7(F0, r, c, p, a, b, v);
    const double sp[3] = {b.dx, b.dy, b.dz};
    moves = false;
    if (side == 0) {  // r-side: crossing (i, i+1), stencil i-2..i+3
        const idx_t nb = shifted(b, r, c, p, a, 1);
        if (!(v[3] * F0[nb] < 0)) return;
        for (int k = 0; k < 6; ++k) idx[k] = shifted(b, r, c, p, a, k - 2);
        const double y[6] = {v[1], v[2], v[3], v[4], v[5], v[6]};
        moves = six_distance_grad(y, sp[a], g);
    } else {  // l-side: ds - distance of the crossing (i-1, i), stencil i-3..i+2
        const idx_t nb = shifted(b, r, c, p, a, -1);
        if (!(F0[nb] * v[3] < 0)) return;
        for (int k = 0; k < 6; ++k) idx[k] = shifted(b, r, c, p, a, k - 3);
        const double y[6] = {v[0], v[1], v[2], v[3], v[4], v[5]};
        moves = six_distance_grad(y, sp[a], g);
        for (int k = 0; k < 6; ++k) g[k] = -g[k];
    }
}

// which of the six distances the time step 0.3*min_dist follows (min6's order)
__device__ __forceinline__ int argmin6(const double d[6])
{
    // min6 = dmin(dmin(xr, xl), dmin(dmin(yr, yl), dmin(zr, zl))) with d = {xr, xl, yr, yl, zr, zl}
    auto pick = [](int a, int b2, const double* e) { return (e[a] < e[b2]) ? a : b2; };
    const int x = pick(0, 1, d), y = pick(2, 3, d), z = pick(4, 5, d);
    const int yz = pick(y, z, d);
    return pick(x, yz, d);
}

// adjoint of the distances: lam_F0[stencil] += d(dist)/dF0 * lam_dist, where
// lam_dist[2a+side] = lamP[2a+side] + (argmin == 2a+side) * 0.3 * lamP[6]
__global__ void __launch_bounds__(256) ka_dist_adjoint(double* __restrict__ lamF0, const double* __restrict__ F0,
                                                       const double* __restrict__ lamP, IList il, Box b)
{
    const int cnt = *il.count;
    for (int j = (int)(blockIdx.x * blockDim.x + threadIdx.x); j < cnt; j += (int)(gridDim.x * blockDim.x)) {
        const idx_t i = il.idx[j];
        double d[6];
        for (int e = 0; e < 6; ++e) d[e] = il.dist[(size_t)e * il.cap + j];
        const bool frozen_pt = !(il.dt[j] >= 0);
        const int am = argmin6(d);
        for (int e = 0; e < 6; ++e) {
            double lam = lamP[(size_t)e * il.cap + j];
            if (!frozen_pt && e == am) lam += 0.3 * lamP[(size_t)6 * il.cap + j];
            if (lam == 0.0) continue;
            idx_t idx[6];
            double g[6];
            bool moves;
            dist_grads(F0, b, i, e >> 1, e & 1, idx, g, moves);
            if (!moves) continue;
            for (int k = 0; k < 6; ++k) atomicAdd(&lamF0[idx[k]], g[k] * lam);
        }
    }
}

// tangent of the parameters: Pdot[e][j] for the distances and the time step
__global__ void __launch_bounds__(256) ka_dist_tangent(double* __restrict__ Pdot, const double* __restrict__ F0,
                                                       const double* __restrict__ F0dot, IList il, Box b)
{
    const int cnt = *il.count;
    for (int j = (int)(blockIdx.x * blockDim.x + threadIdx.x); j < cnt; j += (int)(gridDim.x * blockDim.x)) {
        const idx_t i = il.idx[j];
        double d[6], dd[6];
        for (int e = 0; e < 6; ++e) {
            d[e] = il.dist[(size_t)e * il.cap + j];
            idx_t idx[6];
            double g[6];
            bool moves;
            dist_grads(F0, b, i, e >> 1, e & 1, idx, g, moves);
            double s = 0.0;
            if (moves)
                for (int k = 0; k < 6; ++k) s += g[k] * F0dot[idx[k]];
            dd[e] = s;
            Pdot[(size_t)e * il.cap + j] = s;
        }
        Pdot[(size_t)6 * il.cap + j] = (il.dt[j] >= 0) ? 0.3 * dd[argmin6(d)] : 0.0;
    }
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
static inline dim3 grid1(int64_t n) { return dim3((unsigned)((n + 255) / 256)); }
static inline Box abox(const Geom& g) { return Box{g.rows, g.cols, g.pges, g.dx, g.dy, g.dz}; }
static inline Inv ainv(const Geom& g)
{
    const double m = std::min(std::min(g.dx, g.dx), std::min(std::min(g.dy, g.dy), std::min(g.dz, g.dz)));
    Inv v{{1.0 / g.dx, 1.0 / g.dy, 1.0 / g.dz}, 0.3 * m, {}, {}};
    set_jp(v.jd, v.jf, g.dx, g.dy, g.dz);
    return v;
}
static inline IList alist(const ListView& lv) { return IList{lv.idx, lv.count, lv.dist, lv.dt, lv.cap}; }

hipError_t launch_adj_advect_jac(double* J, double* ux, double* uy, double* uz, const double* lam, const double* fs,
                                 const double* vx, const double* vy, const double* vz, double dt, const Geom& g,
                                 int stage, hipStream_t s)
{
    ka_advect_jac<<<dim3((unsigned)((g.n() + 63) / 64)), 192, 0, s>>>(J, Grad3{{ux, uy, uz}}, lam, fs, vx, vy, vz, dt,
                                                                     abox(g), ainv(g), stage);
    return hipGetLastError();
}

hipError_t launch_adj_reinit_jac(double* J, double* JP, const double* lam, const double* fs, const uint8_t* flags,
                                 const ListView& lv, const Geom& g, int stage, int* extra, int* extra_count, int seq,
                                 hipStream_t s)
{
    ka_reinit_jac_bulk<<<dim3((unsigned)((g.n() + 63) / 64)), 192, 0, s>>>(J, lam, fs, flags, abox(g), ainv(g), stage,
                                                                         extra, extra_count, seq);
    ka_reinit_jac_list<<<dim3(512, 9 / kJacGroup), 192, 0, s>>>(J, JP, lam, fs, flags, alist(lv), abox(g), ainv(g),
                                                               stage, extra, extra_count, seq);
    return hipGetLastError();
}

hipError_t launch_adj_transpose(double* out, const double* P, const Geom& g, double ca, const double* A, double cb,
                                const double* B, hipStream_t s)
{
    ka_transpose<<<grid1(g.n()), 256, 0, s>>>(out, P, abox(g), ca, A, cb, B);
    return hipGetLastError();
}

hipError_t launch_adj_apply(double* out, const double* J, const double* x, const Geom& g, hipStream_t s)
{
    ka_apply<<<grid1(g.n()), 256, 0, s>>>(out, J, x, abox(g));
    return hipGetLastError();
}

hipError_t launch_adj_axpby(double* y, const double* x, double alpha, double beta, int64_t n, hipStream_t s)
{
    ka_axpby<<<grid1(n), 256, 0, s>>>(y, x, alpha, beta, (idx_t)n);
    return hipGetLastError();
}

hipError_t launch_adj_fill(double* y, double v, int64_t n, hipStream_t s)
{
    ka_fill<<<grid1(n), 256, 0, s>>>(y, v, (idx_t)n);
    return hipGetLastError();
}

hipError_t launch_adj_velocity_tangent(double* out, const double* JU, const double* ux, const double* uy,
                                       const double* uz, int64_t n, hipStream_t s)
{
    ka_velocity_tangent<<<grid1(n), 256, 0, s>>>(out, JU, ux, uy, uz, (idx_t)n);
    return hipGetLastError();
}

hipError_t launch_adj_param_tangent(double* out, const double* JP, const double* Pdot, const ListView& lv,
                                    hipStream_t s)
{
    ka_param_tangent<<<256, 256, 0, s>>>(out, JP, Pdot, alist(lv));
    return hipGetLastError();
}

hipError_t launch_adj_dist(double* lamF0, const double* F0, const double* lamP, const ListView& lv, const Geom& g,
                           hipStream_t s)
{
    ka_dist_adjoint<<<256, 256, 0, s>>>(lamF0, F0, lamP, alist(lv), abox(g));
    return hipGetLastError();
}

hipError_t launch_tan_dist(double* Pdot, const double* F0, const double* F0dot, const ListView& lv, const Geom& g,
                           hipStream_t s)
{
    ka_dist_tangent<<<256, 256, 0, s>>>(Pdot, F0, F0dot, alist(lv), abox(g));
    return hipGetLastError();
}

}  // namespace vls
