// Device pieces shared by the single-grid kernels (vls_kernels.hip) and the
// batched kernels (vls_batch.hip): launch geometry, RK combinations, interface
// lists, plane tiles, axis-lane grouping and compensated block reductions.
#pragma once
#include "vls_device.hpp"
#include "vls_kernels.hpp"

namespace vls {

// ---------------------------------------------------------------------------
// launch geometry helpers
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool point_of_thread(const Box& b, int& r, int& c, int& p)
{
    r = blockIdx.x * blockDim.x + threadIdx.x;
    c = blockIdx.y * blockDim.y + threadIdx.y;
    p = blockIdx.z;
    return r < b.rows && c < b.cols;
}

__device__ __forceinline__ idx_t lin(const Box& b, int r, int c, int p)
{
    return (idx_t)p * b.rows * b.cols + (idx_t)c * b.rows + r;
}

// Division of an index within a page (below 2^26) by the box's rows: a product
// and a shift
struct RowDiv {
    unsigned m;
    int s;
};
inline RowDiv row_div(int rows)
{
    int l = 0;
    while ((1ll << l) < rows) ++l;
    return RowDiv{(unsigned)(((1ull << (26 + l)) + (unsigned)rows - 1) / (unsigned)rows), 26 + l};
}

// A point kernel's threads over pages (blockIdx.y): 256 consecutive points of the
// page in memory order, whatever the rows (64 x 4 tiles leave a quarter of the
// lanes of a 96-row box idle), or, TILES, 64 x 4 tiles, whose four columns share
// their x-taps
struct PagePoint {
    int r, c, p;
    unsigned in;  // index within the page
    bool valid;
};
// the point of thread t of this block
template <bool TILES = false>
__device__ __forceinline__ PagePoint page_point(const Box& b, RowDiv d, int t)
{
    PagePoint q;
    q.p = (int)blockIdx.y;
    if constexpr (TILES) {
        const int ntr = (b.rows + 63) >> 6, cb = (int)blockIdx.x / ntr;
        q.r = ((int)blockIdx.x - cb * ntr) * 64 + (t & 63);
        q.c = cb * 4 + (t >> 6);
        q.valid = q.r < b.rows && q.c < b.cols;
        if (!q.valid) q.r = q.c = 0;
        q.in = (unsigned)(q.c * b.rows + q.r);
    } else {
        q.in = blockIdx.x * 256u + (unsigned)t;
        q.valid = q.in < (unsigned)b.rows * (unsigned)b.cols;
        if (!q.valid) q.in = 0;
        q.c = (int)(((unsigned long long)q.in * d.m) >> d.s);
        q.r = (int)q.in - q.c * b.rows;
    }
    return q;
}
template <bool TILES = false>
inline dim3 page_grid(int rows, int cols, int pges)
{
    return TILES ? dim3((unsigned)((rows + 63) / 64) * (unsigned)((cols + 3) / 4), (unsigned)pges)
                 : dim3((unsigned)(((int64_t)rows * cols + 255) / 256), (unsigned)pges);
}
// whether a page's 64 x 4 tiles hold at most `percent` of its points beyond them
inline bool tiles_fit(int rows, int cols, int percent)
{
    return (int64_t)((rows + 63) / 64) * ((cols + 3) / 4) * 256 * 100 <= (int64_t)rows * cols * (100 + percent);
}

// The long evaluations of a point kernel (the nonuniform stencil, the quintic
// root or interpolation), which a few points of a block need on one or two
// axes: `need` is this thread's set of them (bit k < 6).  The block lists them in
// LDS (job, 256 per bit in use) and its threads take one each, body(t, k) for
// bit k of thread t, so that a wave runs the long code once per 64 evaluations.
// Where a lane does its own three axes, a wave runs it three times, however few of
// its lanes need it, and every wave near the interface does.  Every thread of the
// block calls this; the caller synchronizes before it reads what body left in LDS.
template <class Body>
__device__ __forceinline__ void axis_jobs(unsigned need, unsigned short* job, int* count, Body body)
{
    if (threadIdx.x == 0) *count = 0;
    __syncthreads();
    if (need != 0) {
        int at = atomicAdd(count, __popc(need));
        for (; need != 0; need &= need - 1)
            job[at++] = (unsigned short)((__ffs((int)need) - 1) << 8 | (int)threadIdx.x);
    }
    __syncthreads();
    const int total = *count;
    for (int j = (int)threadIdx.x; j < total; j += 256) body((int)(job[j] & 255), (int)(job[j] >> 8));
}

// The six distances of a block's P candidate points (setDistance's second pass),
// dist[k][point] with k = 2 axis + side: a thread per point and axis tests the two
// sides (detect returns them as bits 0, 1 and presets their distances), the
// block lists the crossings, and its threads locate one each.  Most points cross
// on one or two of their six sides: with a lane per point a wave ran the root
// finder, ~1000 dependent operations, for all six in turn: 38 us at 64^3 and
// 40 at 113x97x81, 12 now (64 points a block, so that 10^4 candidates reach most
// CUs); 176 and 97 for the 6 10^5 candidates of a batch (256 points, one atomic
// for their list slots).
template <int P, class Detect, class Locate>
__device__ __forceinline__ void crossing_jobs(double (*dist)[P], unsigned short* job, int* count, Detect detect,
                                              Locate locate)
{
    __syncthreads();  // the last points' distances are read
    if (threadIdx.x == 0) *count = 0;
    __syncthreads();
    for (int e = (int)threadIdx.x; e < 3 * P; e += 256) {
        const int point = e % P, axis = __builtin_amdgcn_readfirstlane(e / P);  // P is a multiple of the wave
        unsigned need = detect(point, axis);
        if (need != 0) {
            int at = atomicAdd(count, __popc(need));
            for (; need != 0; need &= need - 1)
                job[at++] = (unsigned short)(point << 3 | (2 * axis + __ffs((int)need) - 1));
        }
    }
    __syncthreads();
    const int total = *count;
    for (int j = (int)threadIdx.x; j < total; j += 256)
        dist[job[j] & 7][job[j] >> 3] = locate((int)(job[j] >> 3), (int)(job[j] & 7));
    __syncthreads();
}

// 1/dx, 1/dy, 1/dz and the pseudo-time step of a point without subcell
// distances, 0.3*min(dx,dx,dy,dy,dz,dz) (setDistance.m:17-21 with every
// distance equal to the spacing), computed once on the host
struct Inv {
    double i[3];
    double dt_bulk;
    JPd jd[3];  // per-axis constants of the WENO5 form (set_jp)
    JPf jf[3];
};

// the per-axis constants of the WENO5 helpers for FP64 and FP32 fields
__device__ __forceinline__ JPd axis_arg(const Inv& v, int a, double) { return v.jd[a]; }
__device__ __forceinline__ JPf axis_arg(const Inv& v, int a, float) { return v.jf[a]; }

// RK combinations in the order the MATLAB wrappers evaluate them
// (+SD/@SDF3/WENO5RK3Reinitialization.m:20-37), without fused multiply-adds.
__device__ __forceinline__ double rk_combine(int stage, double fs, double step, double fn)
{
#pragma clang fp contract(off)
    const double t = fs - step;
    if (stage == 0) return t;
    if (stage == 1) return 3. / 4. * fn + 1. / 4. * t;
    return 1. / 3. * fn + 2. / 3. * t;
}

__device__ __forceinline__ float rk_combine(int stage, float fs, float step, float fn)
{
    const float t = fs - step;
    if (stage == 0) return t;
    if (stage == 1) return fmaf(0.75f, fn, 0.25f * t);
    return fmaf(1.f / 3.f, fn, (2.f / 3.f) * t);
}

// the interface test of re_step.cu:260-267 at the middle node of v[2..4]:
// a sign change between it and either neighbour, the reference's product test
__device__ __forceinline__ bool sign_change3(const double v[7]) { return (v[2] * v[3] < 0) | (v[3] * v[4] < 0); }

// append `take` lanes' values to list[*count ...] with one atomic per wave
__device__ __forceinline__ void wave_append(bool take, int value, int* __restrict__ list, int* __restrict__ count)
{
    const unsigned long long m = __ballot(take);
    if (m == 0) return;
    const int lane = (int)__lane_id();
    const int leader = __ffsll((long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(count, __popcll(m));
    base = __shfl(base, leader, 64);
    if (take) list[base + __popcll(m & ((1ull << lane) - 1ull))] = value;
}

// Block-aggregated list append: the lanes of a block collect their entries
// in LDS and the block moves them to the list with one global atomic per
// flush.  A wave-aggregated append costs one global atomic per wave, and
// when many waves append, those atomics serialize on the one counter.  Every
// thread of the block calls push() the same number of times and flush() once
// at the end; both contain block barriers.
template <int CAP>
struct BlockList {
    int* buf;    // LDS, CAP entries
    int* count;  // LDS
    int* base;   // LDS
    __device__ __forceinline__ void init()
    {
        if (threadIdx.x == 0) *count = 0;
        __syncthreads();
    }
    __device__ __forceinline__ void flush(int* __restrict__ list, int* __restrict__ list_count)
    {
        __syncthreads();
        const int n = *count;  // the same in every thread after the barrier
        if (n > 0) {
            if (threadIdx.x == 0) *base = atomicAdd(list_count, n);
            __syncthreads();
            const int b = *base;
            for (int i = (int)threadIdx.x; i < n; i += (int)blockDim.x) list[b + i] = buf[i];
            __syncthreads();
            if (threadIdx.x == 0) *count = 0;
            __syncthreads();
        }
    }
    __device__ __forceinline__ void push(bool take, int value, int* __restrict__ list, int* __restrict__ list_count)
    {
        __syncthreads();  // the previous push's entries are in, so *count is final
        if (*count > CAP - (int)blockDim.x) flush(list, list_count);
        const unsigned long long m = __ballot(take);
        if (m == 0) return;
        const int lane = (int)__lane_id();
        const int leader = __ffsll((long long)m) - 1;
        int off = 0;
        if (lane == leader) off = atomicAdd(count, __popcll(m));
        off = __shfl(off, leader, 64);
        if (take) buf[off + __popcll(m & ((1ull << lane) - 1ull))] = value;
    }
};

// Block-aggregated slot assignment: every thread of the block calls it; the
// taking lanes get consecutive slots of the list counted by *count, with one
// global atomic for the whole block (lds_cnt, lds_base: two LDS ints).
__device__ __forceinline__ int block_slot(bool take, int* __restrict__ count, int* lds_cnt, int* lds_base)
{
    __syncthreads();  // the previous call's readers of *lds_base are done
    if (threadIdx.x == 0) *lds_cnt = 0;
    __syncthreads();
    const unsigned long long m = __ballot(take);
    const int lane = (int)__lane_id();
    int off = 0;
    if (m != 0) {
        const int leader = __ffsll((long long)m) - 1;
        if (lane == leader) off = atomicAdd(lds_cnt, __popcll(m));
        off = __shfl(off, leader, 64) + __popcll(m & ((1ull << lane) - 1ull));
    }
    __syncthreads();
    if (threadIdx.x == 0) *lds_base = (*lds_cnt > 0) ? atomicAdd(count, *lds_cnt) : 0;
    __syncthreads();
    return take ? *lds_base + off : -1;
}

// as wave_append, returning each taking lane's slot (-1 for the others)
__device__ __forceinline__ int wave_append_slot(bool take, int* __restrict__ count)
{
    const unsigned long long m = __ballot(take);
    if (m == 0) return -1;
    const int lane = (int)__lane_id();
    const int leader = __ffsll((long long)m) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(count, __popcll(m));
    base = __shfl(base, leader, 64);
    return take ? base + __popcll(m & ((1ull << lane) - 1ull)) : -1;
}

struct Dists {
    double r[3], l[3];
};

// an interface list in the form the stage kernels read: indices and, in list
// order, the six distances (row k of `dist` is xpr,xpl,ypf,ypb,zpu,zpd for
// k = 0..5, rows `cap` apart) and the pseudo-time step 0.3*min_dist, or -1 for
// a frozen point
struct IList {
    const int* idx;
    const int* count;
    const double* dist;
    const double* dt;
    int cap;
};

__device__ __forceinline__ bool frozen(const Dists& q, double dx)
{
    const double eps = 1e-6 * dx;
    return q.r[0] < eps || q.l[0] < eps || q.r[1] < eps || q.l[1] < eps || q.r[2] < eps || q.l[2] < eps;
}

__device__ __forceinline__ double min6(const Dists& q)
{
    return dmin(dmin(q.r[0], q.l[0]), dmin(dmin(q.r[1], q.l[1]), dmin(q.r[2], q.l[2])));
}

// Interface schemes of the fused stage kernels (IFACE_WENO, IFACE_CUBIC of
// vls_kernels.hpp): the WENO5 path's nonuniform WENO (re_step.cu:79-243,
// shared_utilities.cup:49-278) or the WENO-RK3 variants' cubic ENO
// (weno_rk3_reinitialization.cu:149-247, wenork3_extend.cu:88-190).  Away from
// the interface both use the same uniform WENO5, so the bulk of a stage is
// shared.

// the upwind combination of extend_step.cu:121-123 (enork2_extend.cu:262-264,
// wenork3_extend.cu:490-492), summed left to right, times dt
__device__ __forceinline__ double upwind_sum(const double fo[3], const double bk[3], double vx, double vy, double vz,
                                             double dt)
{
#pragma clang fp contract(off)
    return (dmin(0.0, vx) * fo[0] + dmax(0.0, vx) * bk[0] + dmin(0.0, vy) * fo[1] + dmax(0.0, vy) * bk[1] +
            dmin(0.0, vz) * fo[2] + dmax(0.0, vz) * bk[2]) *
           dt;
}

// ENO-RK2 extension step at a point (enork2_extend.cu:213-266; no frozen
// test) with the interface values of each axis given (hf, hb: fore and back;
// each is used only where that side's distance differs from ds)
__device__ __forceinline__ double enork2_residual(const double* __restrict__ f, int r, int c, int p, const Box& b,
                                                  const Dists& q, const double hf[3], const double hb[3], double vx,
                                                  double vy, double vz, double dt)
{
    const double sp[3] = {b.dx, b.dy, b.dz};
    double fo[3], bk[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        double v[7];
        line7(f, r, c, p, a, b, v);
        eno2_field_pair(fo[a], bk[a], v, q.r[a], q.l[a], sp[a], (q.r[a] != sp[a]) ? hf[a] : 0.0,
                        (q.l[a] != sp[a]) ? hb[a] : 0.0);
    }
    return upwind_sum(fo, bk, vx, vy, vz, dt);
}

// per-axis pair with the sign-change interface test in the cubic-ENO scheme
__device__ __forceinline__ void reinit_axis_cubic(double& fore, double& back, const double v[7], double r1,
                                                  double l1, double ds, JPd jp)
{
    wenork3_pair(fore, back, v, r1, l1, ds, jp, v[2] * v[3] < 0 || v[3] * v[4] < 0, 0.0, 0.0);
}

// per-axis derivative pair with the sign-change interface test (re_step.cu:248-269);
// Q: the quotients of the nonuniform faces
template <int Q>
__device__ __forceinline__ void reinit_axis(double& fore, double& back, const double v[7], double r1, double l1,
                                            double ds, JPd jp)
{
    if (v[2] * v[3] < 0 || v[3] * v[4] < 0) {
        const Pair q = weno_nonuniform_pair_inl<Q>(v[0], v[1], v[2], v[3], v[4], v[5], v[6], r1, l1, ds, 0.0, 0.0);
        fore = q.fore;
        back = q.back;
    } else {
        weno5_pair(fore, back, v, jp);
    }
}

// (row, col, page) of element ind of a grid; 32-bit division (a grid holds
// fewer than 2^31 points: interface lists store int indices)
__device__ __forceinline__ void coords_of(const Box& b, idx_t ind, int& r, int& c, int& p)
{
    const unsigned u = (unsigned)ind, rows = (unsigned)b.rows, plane = rows * (unsigned)b.cols;
    const unsigned pp = u / plane, rem = u - pp * plane, cc = rem / rows;
    p = (int)pp;
    c = (int)cc;
    r = (int)(rem - cc * rows);
}

// the crossings of a point on one axis: bit 0 with the +1 neighbour, bit 1 with
// the -1 neighbour (the locators' own tests)
template <typename T>
__device__ __forceinline__ unsigned crossing_sides(const T* __restrict__ f, const Box& b, idx_t ind, int a)
{
    int r, c, p;
    coords_of(b, ind, r, c, p);
    const int pos = a == 0 ? c : (a == 1 ? r : p);
    const int last = (a == 0 ? b.cols : (a == 1 ? b.rows : b.pges)) - 1;
    const idx_t stride = a == 0 ? (idx_t)b.rows : (a == 1 ? (idx_t)1 : (idx_t)b.rows * b.cols);
    const double f0 = (double)f[ind], fu = (double)f[ind + (idx_t)(clampi(pos + 1, last) - pos) * stride],
                 fd = (double)f[ind + (idx_t)(clampi(pos - 1, last) - pos) * stride];
    return (f0 * fu < 0 ? 1u : 0u) | (fd * f0 < 0 ? 2u : 0u);
}

// The distance from a point to its crossing on side k = 2 axis + (0: with the +1
// neighbour, 1: with the -1 neighbour).  The r-side distance is the locator at
// the point; the l-side one is ds minus the locator of the -1 neighbour's
// crossing, evaluated here from that neighbour's stencil (the point's own line
// shifted by one, clamped the same way), so it is the value
// k_boundary_location stores from the neighbour's thread.
template <int ORDER, typename T>
__device__ __forceinline__ double crossing_distance(const T* __restrict__ f, const Box& b, idx_t ind, int k, double ds)
{
    int r, c, p;
    coords_of(b, ind, r, c, p);
    const int a = k >> 1;
    const int pos = a == 0 ? c : (a == 1 ? r : p);
    const int last = (a == 0 ? b.cols : (a == 1 ? b.rows : b.pges)) - 1;
    const idx_t stride = a == 0 ? (idx_t)b.rows : (a == 1 ? (idx_t)1 : (idx_t)b.rows * b.cols);
    const int at = pos - (k & 1);  // the lower point of the crossing pair
    double v[6];                   // the line at offsets -2..+3 around it, clamped
#pragma unroll
    for (int s = -2; s <= 3; ++s) v[s + 2] = (double)f[ind + (idx_t)(clampi(at + s, last) - pos) * stride];
    const double dist = (ORDER == 2)   ? eno_quadratic_distance(v[1], v[2], v[3], v[4], ds)
                        : (ORDER == 3) ? cubic_distance(v[1], v[2], v[3], v[4], ds)
                                       : six_distance(v[0], v[1], v[2], v[3], v[4], v[5], ds);
    return (k & 1) ? ds - dist : dist;
}

__device__ __forceinline__ void load_dists(Dists& q, const Dist6c& d, idx_t ind)
{
#pragma unroll
    for (int a = 0; a < 3; ++a) { q.r[a] = d.r[a][ind]; q.l[a] = d.l[a][ind]; }
}

// ---------------------------------------------------------------------------
// plane tiles: a block covers 64 x 4 (rows x cols) points of one page.  The
// page's values with a 3-point halo in rows and cols are staged in LDS once
// (clamped there), so the x- and y-taps of the WENO stencil are LDS reads at
// constant offsets; the z-taps are global loads at a wave-uniform page offset.
// ---------------------------------------------------------------------------
constexpr int HALO = 3;

// tile shapes: R rows x 256/R cols of one page (R = 64: a wave is one column
// of 64 rows; R = 32: a wave is two columns of 32 rows, for boxes whose
// rows are a multiple of 32 but not of 64), staged with a 3-point halo
template <int R>
struct Shape {
    static constexpr int TR = R, TC = 256 / R, LR = R + 2 * HALO, LC = TC + 2 * HALO, N = LR * LC;
};

struct Tile {
    int r0, c0, p;  // tile origin (row, col) and page
    int r, c;       // this thread's point
    bool valid;
    int base;       // LDS index of this thread's point
    idx_t page;     // element offset of page p in the box (uniform)
    unsigned in;    // element offset of the point in its page, c * rows + r
};

// A page of a field as a buffer resource: a uniform base in scalar registers, to
// which a buffer load or store adds the lane's 32-bit byte offset itself.
// (With global loads the compiler kept 64-bit lane offsets and added them to
// the page's base in a vector instruction per load.)
struct Page {
    __amdgpu_buffer_rsrc_t r;
};
template <typename T>
__device__ __forceinline__ Page page_of(T* field, idx_t page)
{
    return Page{__builtin_amdgcn_make_buffer_rsrc((void*)(field + page), 0, 0xffffffffu, 0x00027000)};
}
// element `off` of the page; NT: non-temporal, for a stream read once per
// launch (the velocity of the extension and advection stages), so that its
// lines do not push the staged tiles' halos out of L2 (measured: extension
// stage at 256^3 FP32 103-107 -> 98-100 us)
template <typename T, bool NT = false>
__device__ __forceinline__ T ldb(const Page& q, unsigned off)
{
    constexpr int aux = NT ? 2 : 0;
    const int o = (int)(off * (unsigned)sizeof(T));
    if constexpr (sizeof(T) == 8) return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(q.r, o, 0, aux));
    else if constexpr (sizeof(T) == 4)
        return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(q.r, o, 0, aux));
    else return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b8(q.r, o, 0, aux));
}
template <typename T>
__device__ __forceinline__ void stb(const Page& q, unsigned off, T v)
{
    const int o = (int)(off * (unsigned)sizeof(T));
    typedef unsigned U2 __attribute__((ext_vector_type(2)));
    if constexpr (sizeof(T) == 8) __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, v), q.r, o, 0, 0);
    else __builtin_amdgcn_raw_buffer_store_b32(__builtin_bit_cast(unsigned, v), q.r, o, 0, 0);
}

// element `off` of a page: the uniform 64-bit page base plus a 32-bit byte
// offset per lane, so a load or store is one instruction with a scalar base
// (offsets reach 7 pages of doubles: pages hold fewer than 2^26 points,
// vls_sdf3_create and vls_batch_create refuse larger ones)
template <typename T>
__device__ __forceinline__ T ldp(const T* __restrict__ base, unsigned off)
{
    return *(const T*)((const char*)base + off * (unsigned)sizeof(T));
}
template <typename T>
__device__ __forceinline__ void stp(T* __restrict__ base, unsigned off, T v)
{
    *(T*)((char*)base + off * (unsigned)sizeof(T)) = v;
}

// Blocks are dispatched round-robin over the 8 XCDs (block i to XCD i % 8),
// each with its own L2.  Give every XCD a contiguous range of tiles instead,
// so neighbouring tiles share their halos in one L2.  XCD x runs one block
// more than the others while x < nblk % 8; its range starts behind the longer
// ranges before it.  (With the ranges only for counts that are a multiple of
// 8, odd-sized boxes and most batches ran without them.  Measured on MI355X:
// extension stage of a 150x131x120 FP32 box at 4 pages a block 28.9 -> 22.2 us,
// surface redistance of it 13.5 -> 12.0 ms; eight FP64 grids of 48..96, 20
// iterations of the WENO-RK3 and ENO-RK2 calls, 11.0 -> 10.4 ms.)
__device__ __forceinline__ int xcd_remap(int blk, int nblk)
{
    const int x = blk & 7, rem = nblk & 7;
    return x * (nblk >> 3) + (x < rem ? x : rem) + (blk >> 3);
}

// tiles per column and per row of a page
template <int R>
__host__ __device__ inline int tiles_per_col(int rows) { return (rows + R - 1) / R; }
template <int R>
__host__ __device__ inline int tiles_per_row(int cols) { return (cols + Shape<R>::TC - 1) / Shape<R>::TC; }

// tile number `blk` of the box (rows fastest, then cols, then pages)
template <int R>
__device__ __forceinline__ Tile tile_at(const Box& b, int blk)
{
    using S = Shape<R>;
    const int ntr = tiles_per_col<R>(b.rows), ntc = tiles_per_row<R>(b.cols);
    Tile t;
    const int rb = blk % ntr;
    const int q = blk / ntr;
    const int cb = q % ntc;
    t.p = q / ntc;
    t.r0 = rb * S::TR;
    t.c0 = cb * S::TC;
    const int ty = (int)(threadIdx.x % S::TR), tx = (int)(threadIdx.x / S::TR);
    t.r = t.r0 + ty;
    t.c = t.c0 + tx;
    t.valid = t.r < b.rows && t.c < b.cols;
    t.base = (tx + HALO) * S::LR + ty + HALO;
    t.page = (idx_t)t.p * b.rows * b.cols;
    t.in = (unsigned)t.c * (unsigned)b.rows + (unsigned)t.r;
    return t;
}

// the tiles a block of a persistent launch visits: XCD x (= blockIdx.x % 8,
// the hardware's round-robin) takes the contiguous range
// [x*chunk, (x+1)*chunk) and its blocks stride through it
struct TileRange {
    int first, end, step;
};

__device__ __forceinline__ TileRange tile_range(int ntiles)
{
    TileRange r;
    const int nb = (int)gridDim.x;
    if ((nb & 7) == 0) {
        const int x = (int)(blockIdx.x & 7), j = (int)(blockIdx.x >> 3), per = nb >> 3;
        const int chunk = (ntiles + 7) >> 3;
        r.first = x * chunk + j;
        r.end = min(ntiles, (x + 1) * chunk);
        r.step = per;
    } else {
        r.first = (int)blockIdx.x;
        r.end = ntiles;
        r.step = nb;
    }
    return r;
}

// A staged tile: one page's values of a tile with its clamped 3-point halo
// in lds[Shape<R>::N], column-major (LR rows per column).  The loads go to
// registers first (zstep_load) and store_tile writes them to LDS, so a
// kernel issues every other load of its points in between and waits for
// memory once.  Each thread loads one row of the first TR staged rows in
// every TC-th staged column (the column offsets are wave-uniform for R = 64),
// and threads below 6*LC one element of the last 6 staged rows.
template <int R, typename T>
struct TileRegs {
    static constexpr int NK = (Shape<R>::LC + Shape<R>::TC - 1) / Shape<R>::TC;
    T m[NK];
    T s;
};

template <int R>
__device__ __forceinline__ int tile_tx()
{
    const int tx = (int)threadIdx.x / R;
    return (R % 64 == 0) ? __builtin_amdgcn_readfirstlane(tx) : tx;
}

template <int R, typename T>
__device__ __forceinline__ void store_tile(T* lds, const TileRegs<R, T>& g)
{
    using S = Shape<R>;
    const int ty = (int)threadIdx.x % R, tx = tile_tx<R>();
#pragma unroll
    for (int k = 0; k < TileRegs<R, T>::NK; ++k) {
        const int lc = tx + S::TC * k;
        if (lc < S::LC) lds[lc * S::LR + ty] = g.m[k];
    }
    const int e = (int)threadIdx.x;
    if (e < 2 * HALO * S::LC) lds[(e / (2 * HALO)) * S::LR + S::TR + e % (2 * HALO)] = g.s;
}

template <typename T>
__device__ __forceinline__ void tile_line_y(const T* lds, int base, T v[7])
{
#pragma unroll
    for (int k = 0; k < 7; ++k) v[k] = lds[base + k - 3];
}

template <int R, typename T>
__device__ __forceinline__ void tile_line_x(const T* lds, int base, T v[7])
{
#pragma unroll
    for (int k = 0; k < 7; ++k) v[k] = lds[base + (k - 3) * Shape<R>::LR];
}

// Interface work is spread over three lanes per point, one per axis (21
// points per wave64, lane 63 idle): the per-axis chains are long (the
// nonuniform WENO divides ~30 times) and the lists short, so this triples the
// parallelism.  The axis results meet in the group's first lane, which adds
// them in the reference's x, y, z order.
struct AxisLane {
    int point;  // index into the point list, or -1
    int axis;   // 0 x, 1 y, 2 z
    int base;   // lane of the group's x member
};

// the lane's group in sweep j0 of block blk (of a 256-thread launch)
__device__ __forceinline__ AxisLane axis_lane(int j0, int blk)
{
    const int lane = (int)(threadIdx.x & 63);
    const int wave = blk * 4 + (int)(threadIdx.x >> 6);
    AxisLane a;
    a.axis = lane % 3;
    a.base = lane - a.axis;
    a.point = (lane < 63) ? j0 + wave * 21 + lane / 3 : -1;
    return a;
}
__device__ __forceinline__ AxisLane axis_lane(int j0) { return axis_lane(j0, (int)blockIdx.x); }

// stride, in points, between the groups nblk blocks visit per sweep
__device__ __forceinline__ int axis_lane_stride(int nblk) { return nblk * 4 * 21; }
__device__ __forceinline__ int axis_lane_stride() { return axis_lane_stride((int)gridDim.x); }

// per-axis pair with the distance interface test (shared_utilities.cup:256-278)
__device__ __forceinline__ void extend_axis(double& fore, double& back, const double v[7], double r1, double l1,
                                            double ds, JPd jp, double h_fore, double h_back)
{
    if (r1 < ds || l1 < ds) {
        const Pair q = weno_nonuniform_pair(v, r1, l1, ds, h_fore, h_back);
        fore = q.fore;
        back = q.back;
    } else {
        weno5_pair(fore, back, v, jp);
    }
}

// Neumaier accumulator
struct KSum {
    double s, c;
    __device__ __forceinline__ void add(double x)
    {
        const double t = s + x;
        c += (fabs(s) >= fabs(x)) ? ((s - t) + x) : ((x - t) + s);
        s = t;
    }
    __device__ __forceinline__ void merge(const KSum& o)
    {
        add(o.s);
        c += o.c;
    }
};

__device__ __forceinline__ double shfl_xor_d(double v, int m)
{
    return __shfl_xor(v, m, 64);
}

__device__ __forceinline__ void wave_reduce(KSum& k)
{
#pragma unroll
    for (int m = 32; m >= 1; m >>= 1) {
        KSum o;
        o.s = shfl_xor_d(k.s, m);
        o.c = shfl_xor_d(k.c, m);
        k.merge(o);
    }
}

// block of 256 threads -> thread 0 holds the merged (s,c) of each quantity
template <int NQ>
__device__ __forceinline__ void block_reduce(KSum (&k)[NQ])
{
    __shared__ double lds[NQ][2][4];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
    for (int q = 0; q < NQ; ++q) {
        wave_reduce(k[q]);
        if (lane == 0) { lds[q][0][wave] = k[q].s; lds[q][1][wave] = k[q].c; }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            KSum t{0.0, 0.0};
            for (int w = 0; w < 4; ++w) { KSum o{lds[q][0][w], lds[q][1][w]}; t.merge(o); }
            k[q] = t;
        }
    }
}

template <int NQ>
__device__ __forceinline__ void block_reduce_store(KSum (&k)[NQ], double* __restrict__ partial)
{
    block_reduce<NQ>(k);
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < NQ; ++q) {
            partial[(size_t)blockIdx.x * 2 * NQ + 2 * q] = k[q].s;
            partial[(size_t)blockIdx.x * 2 * NQ + 2 * q + 1] = k[q].c;
        }
}


// the five middle values of the three lines through a point (x, y, z; clamped):
// uniform page bases, one 32-bit offset per value
__device__ __forceinline__ void line5s(const double* __restrict__ f, const Box& b, const PagePoint& q,
                                       double v[3][5])
{
    const idx_t plane = (idx_t)b.rows * b.cols;
    const double* fp = f + (idx_t)q.p * plane;
    const double v0 = ldp(fp, q.in);
#pragma unroll
    for (int s = -2; s <= 2; ++s) {
        if (s == 0) {
            v[0][2] = v[1][2] = v[2][2] = v0;
            continue;
        }
        v[0][s + 2] = ldp(fp, (unsigned)(clampi(q.c + s, b.cols - 1) * b.rows + q.r));
        v[1][s + 2] = ldp(fp, (unsigned)(q.c * b.rows + clampi(q.r + s, b.rows - 1)));
        v[2][s + 2] = ldp(f + (idx_t)clampi(q.p + s, b.pges - 1) * plane, q.in);
    }
}

// ---------------------------------------------------------------------------
// per-point bodies of the fused stage kernels.  The single-grid kernels and
// the batched kernels call the same functions, with the field pointers of one
// grid (offset into the packed fields for a batch), so a grid gives the same
// result bit for bit either way.
// ---------------------------------------------------------------------------

// Waves per SIMD the fused stage kernels are compiled for (128 VGPRs): the
// FP64 bulk z-march fits them, and so do the interface lanes (the nonuniform
// WENO, inlined).  The FP32 bulk needs 92 VGPRs, but at 5 waves (96) the
// interface lanes spill 100 bytes: the batch of 96 FP32 grids of 32..96 runs
// 58.9 ms a step with 5 waves and 56.6 ms with 4, 256^3 is equal.
constexpr int kStageWaves = 4;
// The advection stages have no interface lanes.  Left to itself the compiler aims
// at 8 waves a SIMD (51 VGPRs in FP32, 80 in FP64) and puts a page's chains one
// behind the other, which small boxes wait for.  Measured on MI355X without -> at 6
// waves: 60 stages of 4 grids of 32^3 FP32 449 -> 426 us, of 8 odd grids 578 -> 498,
// FP64 795 -> 758; a stage of 160^3 FP32 23.7 -> 22.3, 200^3 FP64 86.8 -> 85.4.
// 5 waves lose 2-6% of small FP64 stages, 7 spill in FP64 (926 for the odd grids).
constexpr int kAdvectWaves = 6;

// ---------------------------------------------------------------------------
// z-marching walk (single grid): a block takes one tile column (TR rows x TC
// cols of every page) over pages [p0, p1).  The z-taps of a point are a
// register window over pages p-3..p+3 that shifts by one page per step, so a
// step loads one new z-value per point; the tile and the point's other inputs
// of page p+1 are loaded while page p is evaluated (two LDS buffers, one
// barrier per page).  In-page offsets are computed once per block; moving to
// the next page only moves the (scalar) page base.
// ---------------------------------------------------------------------------
template <int R>
struct ZCol {
    unsigned m[TileRegs<R, double>::NK];  // in-page offsets of the tile-row loads
    unsigned s;                           // in-page offset of the strip load
    unsigned in;                          // the point's in-page offset (0 outside the box)
    int base;                             // the point's LDS index
    bool valid;                           // the point is in the box
};

template <int R>
__device__ __forceinline__ ZCol<R> zcol(const Box& b, int r0, int c0)
{
    using S = Shape<R>;
    ZCol<R> z;
    const int ty = (int)threadIdx.x % R, tx = tile_tx<R>();
    const unsigned rows = (unsigned)b.rows;
    const unsigned row = (unsigned)clampi(r0 - HALO + ty, b.rows - 1);
#pragma unroll
    for (int k = 0; k < TileRegs<R, double>::NK; ++k) {
        const int lc = tx + S::TC * k;
        z.m[k] = (lc < S::LC) ? (unsigned)clampi(c0 - HALO + lc, b.cols - 1) * rows + row : 0u;
    }
    const int e = (int)threadIdx.x;
    z.s = (e < 2 * HALO * S::LC) ? (unsigned)clampi(c0 - HALO + e / (2 * HALO), b.cols - 1) * rows +
                                       (unsigned)clampi(r0 - HALO + S::TR + e % (2 * HALO), b.rows - 1)
                                 : 0u;
    const int r = r0 + ty, c = c0 + tx;
    z.valid = r < b.rows && c < b.cols;
    z.in = z.valid ? (unsigned)c * rows + (unsigned)r : 0u;
    z.base = (tx + HALO) * S::LR + ty + HALO;
    return z;
}

// the loads of one page: the staged tile, the point's velocity, start value
// and flags, and the z-value the window takes in at this page.  The loaded
// values are kept as loaded; nothing is computed from them until the page is
// evaluated, so the loads of page p+1 stay in flight while page p is (an
// operation on them here would make the compiler wait for every load first).
template <int R, typename T, bool VEL>
struct ZStep {
    TileRegs<R, T> reg;
    T vel[VEL ? 3 : 1];
    T fn, w;  // fn: the start value (at stage 0 the point's own value, unused)
    uint8_t fl;  // the point's flags as loaded
    // the point's flags, FLAG_SUBCELL for a lane outside the box (never written)
    __device__ __forceinline__ uint8_t flags(const ZCol<R>& zc) const { return zc.valid ? fl : (uint8_t)FLAG_SUBCELL; }
};

// Every load is issued by every lane on every path: the lanes without a tile
// element to stage load element 0 of the page (their offsets are 0), and the
// march always loads a next page (the last page again at its end).  The
// compiler's wait counts then do not depend on the path taken, so a page's
// evaluation never waits for the loads of the page after it.  FL: the point
// flags are loaded (else 0).
template <int R, typename T, bool VEL, bool FL>
__device__ __forceinline__ void zstep_load(ZStep<R, T, VEL>& s, const ZCol<R>& zc, int p, const Box& b, idx_t plane,
                                           const T* __restrict__ fs, const T* __restrict__ fn,
                                           const T* __restrict__ vx, const T* __restrict__ vy,
                                           const T* __restrict__ vz, const uint8_t* __restrict__ flags, int stage)
{
    const idx_t po = (idx_t)p * plane;
    const Page fp = page_of(fs, po);
#pragma unroll
    for (int k = 0; k < TileRegs<R, T>::NK; ++k) s.reg.m[k] = ldb<T>(fp, zc.m[k]);
    s.reg.s = ldb<T>(fp, zc.s);
    s.w = ldb<T>(page_of(fs, (idx_t)min(p + 3, b.pges - 1) * plane), zc.in);
    if (VEL) {
        s.vel[0] = ldb<T, true>(page_of(vx, po), zc.in);
        s.vel[1] = ldb<T, true>(page_of(vy, po), zc.in);
        s.vel[2] = ldb<T, true>(page_of(vz, po), zc.in);
    }
    // at stage 0 (no start value) the point's own value is read and not used
    // (rk_combine does not read fn at stage 0)
    s.fn = ldb<T>(page_of(stage != 0 ? fn : fs, po), zc.in);
    if (FL) s.fl = ldb<uint8_t>(page_of(flags, po), zc.in);
    else s.fl = 0;
}

template <typename T>
__device__ __forceinline__ void window_shift(T w[7], T in)
{
#pragma unroll
    for (int k = 0; k < 6; ++k) w[k] = w[k + 1];
    w[6] = in;
}

// body(lds, zc, w, step, p) evaluates page p: x- and y-taps from lds, z-taps w;
// start(w) is called once before it with the values of pages p0-3 .. p0+2
template <int R, typename T, bool VEL, bool FL, class Start, class Body>
__device__ __forceinline__ void zmarch(T* lds0, T* lds1, const Box& b, int r0, int c0, int p0, int p1,
                                       const T* __restrict__ fs, const T* __restrict__ fn,
                                       const T* __restrict__ vx, const T* __restrict__ vy,
                                       const T* __restrict__ vz, const uint8_t* __restrict__ flags, int stage,
                                       Start start, Body body)
{
    if (p0 >= p1) return;
    const ZCol<R> zc = zcol<R>(b, r0, c0);
    const idx_t plane = (idx_t)b.rows * b.cols;
    // the window of page p0 - 1 (pages p0-4 .. p0+2, clamped); its first
    // value leaves the window before any page reads it, so it is not loaded
    T w[7];
    w[0] = T(0);
#pragma unroll
    for (int k = 1; k < 7; ++k) w[k] = ldp(fs + (idx_t)clampi(p0 - 4 + k, b.pges - 1) * plane, zc.in);
    ZStep<R, T, VEL> sa, sb;
    zstep_load<R, T, VEL, FL>(sa, zc, p0, b, plane, fs, fn, vx, vy, vz, flags, stage);
    start(w + 1);
    for (int p = p0;;) {
        window_shift(w, sa.w);
        store_tile<R>(lds0, sa.reg);
        __syncthreads();
        zstep_load<R, T, VEL, FL>(sb, zc, min(p + 1, p1 - 1), b, plane, fs, fn, vx, vy, vz, flags, stage);
        body(lds0, zc, w, sa, p);
        if (++p >= p1) break;
        window_shift(w, sb.w);
        store_tile<R>(lds1, sb.reg);
        __syncthreads();
        zstep_load<R, T, VEL, FL>(sa, zc, min(p + 1, p1 - 1), b, plane, fs, fn, vx, vy, vz, flags, stage);
        body(lds1, zc, w, sb, p);
        if (++p >= p1) break;
    }
}

// Division of a number below 2^31 by d: a product and a shift
struct IntDiv {
    unsigned m;
    int s, d;
};
inline IntDiv int_div(int d)
{
    int l = 0;
    while ((1ll << l) < d) ++l;
    return IntDiv{(unsigned)(((1ull << (31 + l)) + (unsigned)d - 1) / (unsigned)d), 31 + l, d};
}
__host__ __device__ __forceinline__ int quotient(int n, IntDiv d)
{
    return (int)(((unsigned long long)(unsigned)n * d.m) >> d.s);
}

// The shares of a z-march launch: tile columns (nct of them, ntr to a column of
// the page) and nch chunks of `len` pages, one more in `rem` of them, spread
// evenly: an XCD takes a contiguous range of chunks (the longer ones first made
// the first XCDs last, 1% at 200^3).  Computed on the host: a block's first
// loads wait for its share, and four divisions there (two of them of 64 bits)
// were 360 instructions.  Advection stage, one page a block: 48^3 FP32 4.26 ->
// 3.63 us, FP64 5.24 -> 4.61; 96^3 FP32 at 4 pages 8.9 -> 8.0, its extension
// stage 12.05 -> 11.1.
struct ZShare {
    IntDiv nct, ntr, nch;
    int len, rem;
};
template <int R>
inline ZShare zmarch_shares(int rows, int cols, int pges, int depth)
{
    // equal chunks of at most `depth` pages (a last chunk of a page or two would
    // pay a whole block's start-up)
    const int ntr = tiles_per_col<R>(rows), nch = (pges + depth - 1) / depth;
    return ZShare{int_div(ntr * tiles_per_row<R>(cols)), int_div(ntr), int_div(nch), pges / nch, pges % nch};
}
// the share of block blk of the launch's nblk = zmarch_blocks(...): tile column
// (r0, c0) and pages [p0, p1).  Consecutive blocks of one XCD take neighbouring
// columns, which share their halos in its L2.
template <int R>
__device__ __forceinline__ void zmarch_share(const ZShare& z, int blk, int nblk, int& r0, int& c0, int& p0, int& p1)
{
    const int gi = xcd_remap(blk, nblk);
    const int ch = quotient(gi, z.nct), ct = gi - ch * z.nct.d;
    const int cb = quotient(ct, z.ntr);
    r0 = (ct - cb * z.ntr.d) * R;
    c0 = cb * Shape<R>::TC;
    // rem is 0 at one page a chunk, so nch * rem stays below 65535^2 / 4
    p0 = ch * z.len + quotient(ch * z.rem, z.nch);
    p1 = (ch + 1) * z.len + quotient((ch + 1) * z.rem, z.nch);
}

// blocks of a z-march launch with `depth` pages per block
template <int R>
__host__ __device__ inline int zmarch_blocks(int rows, int cols, int pges, int depth)
{
    return tiles_per_col<R>(rows) * tiles_per_row<R>(cols) * ((pges + depth - 1) / depth);
}

// Whether the reinitialization bulk defers a point next to a sign change of
// the stage field to the interface path.  The reference evaluates such a
// point with its nonuniform WENO at full spacings (re_step.cu:248-269: the
// point has no subcell distance), which is the uniform WENO5 up to rounding
// (the oracle tests hold the two within 1e-14 relative); FP64 defers so the
// results stay the reference's bit for bit, FP32 evaluates them in its bulk.
template <typename T>
constexpr bool defers_crossings()
{
    return sizeof(T) == sizeof(double);
}

// WENO5-RK3 reinitialization stage at a bulk point: x- and y-taps from the
// staged tile (lds, the point at index base), z-taps z[0..6] (z[3] the point),
// the start value fn and flags fl.  Returns the new value; where the bulk
// defers crossings (FP64), cross is set for a point next to a sign change of
// the stage field (its block evaluates it after the march), else it stays false.
// zf: the z-faces the march's previous page left (zface_start at its start)
template <int R, typename T>
__device__ __forceinline__ T reinit_value(const T* lds, int base, const T z[7], T fn, uint8_t fl, const Inv& invs,
                                          int stage, bool& cross, ZFace<T>& zf)
{
    cross = false;
    T fo[3], bk[3];
#pragma unroll
    for (int a = 0; a < 2; ++a) {
        T v[7];
        if (a == 0) tile_line_x<R>(lds, base, v);
        else tile_line_y(lds, base, v);
        if constexpr (defers_crossings<T>()) cross |= sign_change3(v);
        weno5_pair(fo[a], bk[a], v, axis_arg(invs, a, T()));
    }
    if constexpr (defers_crossings<T>()) {
        bool cz;
        weno5_pair_z(fo[2], bk[2], cz, z, zf, axis_arg(invs, 2, T()));
        cross |= cz;
    } else {
        weno5_pair_z(fo[2], bk[2], z, zf, axis_arg(invs, 2, T()));
    }
    const T step = godunov_step((fl & FLAG_MASK) != 0, fo[0], bk[0], fo[1], bk[1], fo[2], bk[2], (T)invs.dt_bulk);
    return rk_combine(stage, z[3], step, fn);
}

// A block of an FP64 reinitialization stage lists in LDS the bulk points of its
// tile that take the nonuniform stencil (defers_crossings), as page << 8 | thread,
// and evaluates them after its march.  The list holds every point of this many
// pages, which bounds the pages of such a block.
constexpr int kDeferPages = 16;
template <typename T>
constexpr int reinit_depth(int depth)
{
    return defers_crossings<T>() && depth > kDeferPages ? kDeferPages : depth;
}
// the parts that items of at most `depth` pages are split into for it
template <typename T>
__host__ __device__ constexpr int reinit_parts(int depth)
{
    return defers_crossings<T>() ? (depth + kDeferPages - 1) / kDeferPages : 1;
}

// the interface lanes' quotients: an FP32 field's differences over distances of
// at least 1e-6 of a spacing have finite products
template <typename T>
constexpr int lane_quot()
{
    return sizeof(T) == 8 ? QUOT_WIDE : QUOT_FAST;
}

// one lane (point, axis) of the reinitialization interface pass
struct ReinitLane {
    double m = 0.0;   // this axis's Godunov term
    double dt = 0.0;  // pseudo-time step; < 0: frozen point
    idx_t gind = 0;   // where the point's result goes
    bool inside = false;
};

// the point (r, c, p); slot: its position in the interface list, or -1 for a
// deferred bulk point (spacing distances, bulk time step); ind: its index in
// the grid (fs, flags of that grid); gind: its index in the output fields
template <typename T, int SCHEME = IFACE_WENO>
__device__ __forceinline__ ReinitLane reinit_iface_lane(const T* __restrict__ fs, const uint8_t* __restrict__ flags,
                                                        const Box& b, const Inv& inv, const IList& il, int slot, int r,
                                                        int c, int p, idx_t ind, idx_t gind, int a)
{
    const double sp[3] = {b.dx, b.dy, b.dz};
    ReinitLane q;
    q.gind = gind;
    q.dt = inv.dt_bulk;
    q.inside = (flags[ind] & FLAG_MASK) != 0;
    double r1 = sp[a], l1 = sp[a];
    if (slot >= 0) {
        q.dt = il.dt[slot];
        r1 = il.dist[(size_t)(2 * a) * il.cap + slot];
        l1 = il.dist[(size_t)(2 * a + 1) * il.cap + slot];
    }
    if (q.dt >= 0) {
        double v[7], fo, bk;
        line7_lane(fs, r, c, p, a, b, v);
        if constexpr (SCHEME == IFACE_CUBIC) reinit_axis_cubic(fo, bk, v, r1, l1, sp[a], inv.jd[a]);
        else reinit_axis<lane_quot<T>()>(fo, bk, v, r1, l1, sp[a], inv.jd[a]);
        q.m = godunov_axis(q.inside, bk, fo);
    }
    return q;
}

// the group's x lane adds the three axis terms in x, y, z order and writes
// the RK combination (every lane of the wave must call this)
template <typename T>
__device__ __forceinline__ void reinit_iface_finish(T* __restrict__ out, const T* __restrict__ fs,
                                                    const T* __restrict__ fn, const ReinitLane& q,
                                                    const AxisLane& al, bool active, int stage)
{
    const double my = __shfl(q.m, al.base + 1, 64), mz = __shfl(q.m, al.base + 2, 64);
    if (active && al.axis == 0) {
        double step = 0.0;  // frozen point (dt < 0)
        if (q.dt >= 0) {
            // godunov_step: (sqrt((mx + my) + mz) - 1) * dt, negated inside
            const double s1 = (sqrt((q.m + my) + mz) - 1) * q.dt;
            step = q.inside ? -s1 : s1;
        }
        out[q.gind] = (T)rk_combine(stage, (double)fs[q.gind], step, (stage == 0) ? 0.0 : (double)fn[q.gind]);
    }
}

// upwind WENO5 rate of the extension and advection stages at a bulk point
// (x- and y-taps from the staged tile, z-taps z[0..6]) and the RK
// combination with the stage's time step: acc * scale is the step.
// zd: the second differences along z that the march's previous page left
// (zdiff_start at its start)
template <int R, typename T>
__device__ __forceinline__ T upwind_value(const T* lds, int base, const T z[7], const T vel[3], T fn, T scale,
                                          const Inv& inv, int stage, ZDiff<T>& zd)
{
    T acc = 0;
    T v[7];
    tile_line_x<R>(lds, base, v);
    acc = upwind_axis(acc, vel[0], v, axis_arg(inv, 0, T()));
    tile_line_y(lds, base, v);
    acc = upwind_axis(acc, vel[1], v, axis_arg(inv, 1, T()));
    acc = upwind_axis_z(acc, vel[2], z, zd, axis_arg(inv, 2, T()));
    return rk_combine(stage, z[3], acc * scale, fn);
}

// one lane (point, axis) of the extension interface pass
struct ExtendLane {
    double t = 0.0;    // this axis's term coef * derivative
    double dt = -1.0;  // pseudo-time step; < 0: frozen point
    idx_t gind = 0;
};

// slot: position in the list (lcp, lv, il.dist, il.dt rows); ind: index in
// the grid of cs; gind: index in the output fields
template <typename T, int SCHEME = IFACE_WENO>
__device__ __forceinline__ ExtendLane extend_iface_lane(const T* __restrict__ cs, const Box& b, const Inv& inv,
                                                        const IList& il, const double* __restrict__ lcp,
                                                        const double* __restrict__ lv, int slot, idx_t ind,
                                                        idx_t gind, int a)
{
    const double sp[3] = {b.dx, b.dy, b.dz};
    ExtendLane q;
    q.gind = gind;
    q.dt = il.dt[slot];
    if (q.dt >= 0) {
        int r, c, p;
        coords_of(b, ind, r, c, p);
        double v[7];
        line7_lane(cs, r, c, p, a, b, v);
        const double vel = lv[(size_t)a * il.cap + slot];
        const double r1 = il.dist[(size_t)(2 * a) * il.cap + slot];
        const double l1 = il.dist[(size_t)(2 * a + 1) * il.cap + slot];
        if (r1 < sp[a] || l1 < sp[a]) {
            const bool fore = vel < 0;
            const double hf = lcp[(size_t)(2 * a) * il.cap + slot], hb = lcp[(size_t)(2 * a + 1) * il.cap + slot];
            double dv;
            if constexpr (SCHEME == IFACE_CUBIC) {
                double x[7], h[7], df, db;
                cubic_stencil(x, h, v, r1, l1, sp[a], hf, hb);
                eno_cubic_pair(df, db, x, h);
                dv = fore ? df : db;
            } else {
                dv = weno_nonuniform_one_inl<lane_quot<T>()>(v[0], v[1], v[2], v[3], v[4], v[5], v[6], r1, l1, sp[a], hf, hb, !fore);
            }
            q.t = 0.0 + (fore ? vel : dmax(0.0, vel)) * dv;
        } else {
            q.t = upwind_axis(0.0, vel, v, inv.jd[a]);
        }
    }
    return q;
}

template <typename T>
__device__ __forceinline__ void extend_iface_finish(T* __restrict__ out, const T* __restrict__ cs,
                                                    const T* __restrict__ cn, const ExtendLane& q,
                                                    const AxisLane& al, bool active, int stage)
{
    const double ty = __shfl(q.t, al.base + 1, 64), tz = __shfl(q.t, al.base + 2, 64);
    if (active && al.axis == 0) {
        const double step = (q.dt >= 0) ? ((q.t + ty) + tz) * q.dt : 0.0;
        out[q.gind] = (T)rk_combine(stage, (double)cs[q.gind], step, (stage == 0) ? 0.0 : (double)cn[q.gind]);
    }
}

}  // namespace vls
