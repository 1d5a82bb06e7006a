// Compat mode: ImmerseFlow::ADsolver and ImmerseFlow::PPESolver as the
// reference codes them (src/include/ADSolver.cu:268-395,
// src/include/PPESolver.cu:13-71,137-205), quirks included, on gfx950.
// These reproduce the reference's own output files (results/uc.dat, vc.dat,
// p.dat); the performance path is physics mode (kernels.hip).
//
// Layout: the reference's unpadded nx*ny arrays (idx = i + j*nx); uf is
// (nx-1)*(ny-2), vf is (nx-2)*(ny-1).
#include <cmath>
#include <cstring>
#include <vector>

#include "compat.h"
#include "io.h"

namespace iff {

__device__ __forceinline__ double blk_sum(double v)
{
    __shared__ double s[4];
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
    if ((threadIdx.x & 63) == 0) s[threadIdx.x >> 6] = v;
    __syncthreads();
    const double r = (s[0] + s[1]) + (s[2] + s[3]);
    __syncthreads();
    return r;
}

// initializeKernel, preSim.cu:53-97 (vortex IC, p = 0), and the iBlank stub
// of iBlankComputeKernel, preSim.cu:110-136 (1.0 everywhere).
__global__ void kc_init(int nx, int ny, const double *xc, const double *yc, double *u,
                        double *v, double *p, double *iblank)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= nx * ny) return;
    const int i = id % nx, j = id / nx;
    const double r = sqrt(pow(xc[i] - 0.5, 2.0) + pow(yc[j] - 0.5, 2.0));
    const double r0 = 0.1;
    u[id] = 1.0 - 0.25 * (yc[j] - 0.5) * exp((1.0 - pow(r / r0, 2.0)) / 2.0);
    v[id] = 0.25 * (xc[i] - 0.5) * exp((1.0 - pow(r / r0, 2.0)) / 2.0);
    p[id] = 0.0;
    iblank[id] = 1.0;
}

// Compute_velf, ADSolver.cu:162-189.  Under the reference launch (one
// grid-stride pass per thread) the vf loop runs only for ids in
// [(nx-1)(ny-2), (nx-2)(ny-1)), which is empty unless nx > ny.
__global__ void kc_velf(int nx, int ny, const double *dx, const double *dy, const double *u,
                        const double *v, double *uf, double *vf)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    const int nuf = (nx - 1) * (ny - 2), nvf = (nx - 2) * (ny - 1);
    if (id < nuf) {
        const int i = id % (nx - 1), j = id / (nx - 1);
        const int idc = j * nx + i;
        uf[id] = 1.0 / (dx[i] + dx[i + 1]) * (u[idc + nx + 1] * dx[i] + u[idc + nx] * dx[i + 1]);
    } else if (id < nvf) {
        const int i = id % (nx - 2), j = id / (nx - 2);
        const int idc = j * nx + i;
        vf[id] = 1.0 / (dy[j + 1] + dy[j]) * (v[idc + nx + 1] * dy[j] + v[idc + 1] * dy[j + 1]);
    }
}

// set_velocity_BC, ADSolver.cu:191-217.  Edge ghosts read interior cells
// only.  The reference's corner cells race with the edge writes; this
// kernel fixes the outcome of a sequential sweep over id: corner (0,0)
// takes the pre-call ghost (0,1), the other corners take freshly written
// edge ghosts.  Each corner is written by the thread that owns the edge
// ghost it depends on, so no cell is read by one thread while another
// writes it.
__global__ void kc_bc(int nx, int ny, double *q, double qbc)
{
    const int k = blockIdx.x * blockDim.x + threadIdx.x;
    const double two = qbc * 2.0;
    if (k < ny - 2) {  // west and east edges, j = 1 + k
        const int j = 1 + k;
        const int w = j * nx, e = nx - 1 + j * nx;
        const double old_w = q[w];
        const double nw = -q[w + 1] + two;
        const double ne = -q[e - 1] + two;
        q[w] = nw;
        q[e] = ne;
        if (j == 1) q[0] = -old_w + two;                               // (0,0)
        if (j == ny - 2) q[(ny - 1) * nx] = -nw + two;                 // (0,ny-1)
        if (j == ny - 2) q[nx - 1 + (ny - 1) * nx] = -ne + two;        // (nx-1,ny-1)
    } else if (k < (ny - 2) + (nx - 2)) {  // south and north edges, i = 1 + k'
        const int i = 1 + (k - (ny - 2));
        const double ns = -q[i + nx] + two;
        q[i] = ns;
        q[i + (ny - 1) * nx] = -q[i + (ny - 2) * nx] + two;
        if (i == nx - 2) q[nx - 1] = -ns + two;                        // (nx-1,0)
    }
}

// ADSource, ADSolver.cu:46-79, for u and v.
__global__ void kc_source(int nx, int ny, const double *dx, const double *dy, double dt,
                          const double *u, const double *v, const double *uf, const double *vf,
                          double *sx, double *sy)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= nx * ny) return;
    const int i = id % nx, j = id / nx;
    double su = 0.0, sv = 0.0;
    if (i > 0 && i < nx - 1 && j > 0 && j < ny - 1) {
        const double dx_i = dx[i], dx_ip1 = dx[i + 1], dx_im1 = dx[i - 1];
        const double dy_j = dy[j], dy_jp1 = dy[j + 1], dy_jm1 = dy[j - 1];
        const double ufe = uf[i + (j - 1) * (nx - 1)], ufw = uf[i - 1 + (j - 1) * (nx - 1)];
        const double vfn = vf[i - 1 + j * (nx - 2)], vfs = vf[i - 1 + (j - 1) * (nx - 2)];
        su = (u[id] - (dt / dx_i) * 0.5 * (((1 / (dx_i + dx_ip1)) * (u[id + 1] * dx_i + u[id] * dx_ip1) * ufe)
                                           - ((1 / (dx_i + dx_im1)) * (u[id] * dx_im1 + u[id - 1] * dx_i) * ufw)))
             - (dt / dy_j) * 0.5 * (((1 / (dy_j + dy_jp1)) * (u[id + nx] * dy_j + u[id] * dy_jp1) * vfn)
                                    - ((1 / (dy_j + dy_jm1)) * (u[id] * dy_jm1 + u[id - nx] * dy_j) * vfs));
        sv = (v[id] - (dt / dx_i) * 0.5 * (((1 / (dx_i + dx_ip1)) * (v[id + 1] * dx_i + v[id] * dx_ip1) * ufe)
                                           - ((1 / (dx_i + dx_im1)) * (v[id] * dx_im1 + v[id - 1] * dx_i) * ufw)))
             - (dt / dy_j) * 0.5 * (((1 / (dy_j + dy_jp1)) * (v[id + nx] * dy_j + v[id] * dy_jp1) * vfn)
                                    - ((1 / (dy_j + dy_jm1)) * (v[id] * dy_jm1 + v[id - nx] * dy_j) * vfs));
    }
    sx[id] = su;
    sy[id] = sv;
}

// ADusolver_kernel + ADvsolver_kernel, ADSolver.cu:81-120: interior only;
// coefficients per axis (calculateADCoefficients, :34-39).  w != 1: the
// w_AD relaxation written and commented out at :95,:116.
__global__ void kc_sweep(int nx, int ny, const double *xp, const double *xm, const double *px,
                         const double *yp, const double *ym, const double *py,
                         const double *iblank, const double *sx, const double *sy,
                         const double *u, const double *v, double *un, double *vn, double w)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= nx * ny) return;
    const int i = id % nx, j = id / nx;
    if (i > 0 && i < nx - 1 && j > 0 && j < ny - 1) {
        const double ap = px[i] + py[j];
        double t = sx[id] + xp[i] * u[id + 1] + xm[i] * u[id - 1] + yp[j] * u[id + nx] + ym[j] * u[id - nx];
        double qu = iblank[id] * t / ap;
        t = sy[id] + xp[i] * v[id + 1] + xm[i] * v[id - 1] + yp[j] * v[id + nx] + ym[j] * v[id - nx];
        double qv = iblank[id] * t / ap;
        if (w != 1.0) {
            qu = (1.0 - w) * u[id] + w * qu;
            qv = (1.0 - w) * v[id] + w * qv;
        }
        un[id] = qu;
        vn[id] = qv;
    }
}

// Reduction, preSim.cu:376-445, in the reference's summation order: pass 1
// is reduce6<256> (:22-50) over n values with CUDAQuery's grid of
// ceil(n/256) blocks (:190-193): thread tid of block b starts at
// i = b*512 + tid and adds val(i) + val(i+256) (val(i) alone when i+256 >= n)
// per grid-stride step of grid_size = 512 * blocks; the block then folds its
// 256 sums pairwise, s[t] += s[t+h] for h = 128 .. 1 (warpReduce's lockstep
// reads leave the same s[0]).  Pass 2 is the same over the block sums with
// one block (grid_size 512).
template <typename F>
__device__ __forceinline__ double reduce6_block(F val, unsigned n, unsigned grid_size)
{
    __shared__ double sd[256];
    const unsigned tid = threadIdx.x;
    double acc = 0;
    for (unsigned i = blockIdx.x * 512 + tid; i < n; i += grid_size) {
        if (i + 256 < n) acc += val(i) + val(i + 256);
        else acc += val(i);
    }
    sd[tid] = acc;
    __syncthreads();
    for (unsigned h = 128; h >= 1; h >>= 1) {
        if (tid < h) sd[tid] += sd[tid + h];
        __syncthreads();
    }
    const double r = sd[0];
    __syncthreads();
    return r;
}

// Compute_{u,v}Residual_AD (ADSolver.cu:122-160): |new - old| on interior
// cells with iBlank == 1, 0 elsewhere; pass 1 of Reduction for u and v.
__global__ __launch_bounds__(256) void kc_l1(int nx, int ny, const double *iblank,
                                             const double *a, const double *b, const double *c,
                                             const double *d, double *part)
{
    const unsigned n = (unsigned)(nx * ny), gs = 512u * gridDim.x;
    auto val = [&](const double *x, const double *y) {
        return [=](unsigned id) {
            const int i = (int)id % nx, j = (int)id / nx;
            return (i > 0 && i < nx - 1 && j > 0 && j < ny - 1 && iblank[id] == 1) ? fabs(x[id] - y[id]) : 0.0;
        };
    };
    const double su = reduce6_block(val(a, b), n, gs);
    const double sv = reduce6_block(val(c, d), n, gs);
    if (threadIdx.x == 0) {
        part[2 * blockIdx.x] = su;
        part[2 * blockIdx.x + 1] = sv;
    }
}

// Pass 2 of Reduction over nb block sums (stride 2: u and v interleaved).
__global__ __launch_bounds__(256) void kc_finish(const double *part, int nb, int stride, double *out)
{
    const double s0 = reduce6_block([=](unsigned k) { return part[stride * k]; }, (unsigned)nb, 512u);
    double s1 = 0.0;
    if (stride == 2) s1 = reduce6_block([=](unsigned k) { return part[2 * k + 1]; }, (unsigned)nb, 512u);
    if (threadIdx.x == 0) {
        out[0] = s0;
        out[1] = s1;
    }
}

// jacobiIteration, PPESolver.cu:13-31 (boundary copied, no RHS).
__global__ void kc_jacobi(int nx, int ny, const double *cxp, const double *cxm, const double *cyp,
                          const double *cym, const double *p, double *pn)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= nx * ny) return;
    const int i = id % nx, j = id / nx;
    pn[id] = p[id];
    if (i > 0 && i < nx - 1 && j > 0 && j < ny - 1) {
        const double ap = -1 * ((cxp[i] + cxm[i]) + (cyp[j] + cym[j]));
        pn[id] = -(p[id + 1] * cxp[i] + p[id - 1] * cxm[i] + p[id + nx] * cyp[j] + p[id - nx] * cym[j]) / ap;
    }
}

// Compute_Residual, PPESolver.cu:33-50: signed A.p per interior cell (0 on
// the ring), pass 1 of Reduction.
__global__ __launch_bounds__(256) void kc_presid(int nx, int ny, const double *cxp,
                                                 const double *cxm, const double *cyp,
                                                 const double *cym, const double *p, double *part)
{
    const unsigned n = (unsigned)(nx * ny), gs = 512u * gridDim.x;
    const double r = reduce6_block(
        [=](unsigned id) {
            const int i = (int)id % nx, j = (int)id / nx;
            if (!(i > 0 && i < nx - 1 && j > 0 && j < ny - 1)) return 0.0;
            const double ap = -1 * ((cxp[i] + cxm[i]) + (cyp[j] + cym[j]));
            return p[id] * ap + p[id + 1] * cxp[i] + p[id - 1] * cxm[i] + p[id + nx] * cyp[j] +
                   p[id - nx] * cym[j];
        },
        n, gs);
    if (threadIdx.x == 0) part[blockIdx.x] = r;
}

// set_pressure_BC, PPESolver.cu:54-71.
__global__ void kc_pbc(int nx, int ny, double *p)
{
    const int id = blockIdx.x * blockDim.x + threadIdx.x;
    if (id >= nx * ny) return;
    const int i = id % nx, j = id / nx;
    if (i == 0 || j == 0) p[id] = 100.0;
}

// ---------------------------------------------------------------------------
// One-workgroup forms of ADsolver and PPESolver for grids whose fields fit in
// the LDS of one CU (the reference's own deck: 52 x 52 cells with ghosts).
// At this size a pass is waits, not work: launched kernel by kernel, one
// Poisson iteration took 21 us (four launches, a copy and a host wait for
// 2,704 cells).  Here the whole call is one launch; an iteration costs its
// LDS reads, its FP64 arithmetic and one (Poisson) or four (AD) barriers.
//
// Wave w owns the cells id = 512 w + lane + 64 q, q = 0..7: exactly the cells
// of block w of reduce6's first pass, so that pass's fold needs no LDS and no
// barrier (h = 128 and 64 fall on a lane's own cells, h = 32..1 are lane
// exchanges), and every sum has the bits of the launch-by-launch form.
//
// LDS is indexed from its array by integer offsets, never through pointers
// chosen at run time: those become flat accesses, whose base the compiler may
// place below the array (the south neighbour of a first-row cell, 64 q cells
// on in the immediate offset), outside the LDS aperture the hardware tests.
// ---------------------------------------------------------------------------
constexpr int kOneCells = 8192;       // 16 waves x 512 cells
constexpr int kOneReg = 4096;         // 8 waves, 256 registers a lane
constexpr int kOneQ = 8;              // cells per lane
// iterations per launch at most: a Poisson launch lasts up to 18 ms at 52 x 52
// cells and 45 ms at 90 x 91; an ADsolver call is one launch, 6.2 and 24 us an
// iteration (calls that allow more iterations than this run launch by launch)
constexpr int kOneIters = 16384;
constexpr size_t kOneLds = 160 * 1024;

// Lane l's value plus that of lane l ^ h for h = 32, 16, ..: in lane 0 the
// order of the fold s[t] += s[t + h] (each step adds the same two numbers).
template <int CTRL>
__device__ __forceinline__ double dpp_add(double v)
{
    const int lo = __builtin_amdgcn_mov_dpp(__double2loint(v), CTRL, 0xF, 0xF, true);
    const int hi = __builtin_amdgcn_mov_dpp(__double2hiint(v), CTRL, 0xF, 0xF, true);
    return v + __hiloint2double(hi, lo);
}
// h = 8, 4, 2, 1 within rows of 16 lanes (row rotations)
__device__ __forceinline__ double fold16(double v)
{
    v = dpp_add<0x128>(v);
    v = dpp_add<0x124>(v);
    v = dpp_add<0x122>(v);
    return dpp_add<0x121>(v);
}
__device__ __forceinline__ double fold64(double v)
{
    v += __shfl_xor(v, 32, 64);
    v += __shfl_xor(v, 16, 64);
    return fold16(v);
}
__device__ __forceinline__ double lane0(double v)
{
    return __hiloint2double(__builtin_amdgcn_readfirstlane(__double2hiint(v)),
                            __builtin_amdgcn_readfirstlane(__double2loint(v)));
}

// Pass 1 of Reduction over a wave's 512 values (zero past the end): thread t
// of the reference's block adds val(t) + val(t + 256), which are this lane's
// values q and q + 4.
__device__ __forceinline__ double fold512(const double (&val)[kOneQ])
{
    return fold64(((val[0] + val[4]) + (val[2] + val[6])) + ((val[1] + val[5]) + (val[3] + val[7])));
}

// Pass 2 over at most 16 block sums (the others are zero), in every wave.
__device__ __forceinline__ double fold_parts(const double *lds, int part, int lane)
{
    return lane0(fold16(lane < 16 ? lds[part + lane] : 0.0));
}

// x / b, correctly rounded, from y = RN(1 / b): q = x y is within one ulp, the
// remainder x - q b is exact in an FMA, and RN(q + remainder y) is the
// correctly rounded quotient (P. Markstein, "Computation of elementary
// functions on the IBM RISC System/6000 processor", IBM J. Res. Dev. 34, 1990,
// theorem 7.2), unless b's mantissa is all ones or an operation leaves the
// normal range: those take the division.
// Three operations where the division takes about 25, in a loop that is made
// of one division per cell.
__device__ __forceinline__ bool div_special(double b)
{
    const unsigned long long m = (unsigned long long)__double_as_longlong(b) & 0xfffffffffffffull;
    const double a = fabs(b);
    return m == 0xfffffffffffffull || !(a > 1e-60 && a < 1e60);
}
__device__ __forceinline__ double div_by(double x, double b, double y)
{
    const double q = x * y;
    return __builtin_fma(__builtin_fma(-q, b, x), y, q);
}
__device__ __forceinline__ double div_by(double x, double b, double y, bool special)
{
    const double a = fabs(x);
    return (special || !((a > 1e-200 && a < 1e200) || a == 0.0)) ? x / b : div_by(x, b, y);
}

// A compile-time distance between the LDS buffers puts a buffer's offset into
// the instructions.
constexpr int kOneStride = kOneReg + 1;

// PPESolver's loop (PPESolver.cu:164-195), at most kOneReg cells.  Iteration
// k reads p_k once: the same four products give its residual (the stop test
// of iteration k) and p_{k+1}, which goes to the other LDS buffer.  The
// test's sum is complete after the iteration's one barrier; a stop at k
// stores p_k from registers.  Everything a cell needs is in registers (8
// waves, 256 registers a lane) and the loop has no branch per cell: a ring
// cell, or one past the end, has zero coefficients, reads an interior cell's
// neighbours and stores to a spare cell.  The deck's 14,807 iterations on 52 x
// 52 cells take 16.1 ms (312 launch by launch, 27.8 with a branch per cell): of an
// iteration's 2,600 cycles the FP64 instructions (17 per cell) are 1,090 on the
// SIMDs that hold two of the six waves, the rest is the chain of the fold, its
// LDS write, the barrier and the second fold.
__global__ __launch_bounds__(512) void kc_ppe_one(int nx, int ny, const double *vx, const double *vy, double *p,
                                                  int iter0, int itermax, int most, double tol, double *out)
{
    __shared__ __align__(16) double lds[2 * kOneStride + 32];
    constexpr int part = 2 * kOneStride;  // [2][16]
    const int n = nx * ny;
    const double *cxp = vx + 5 * nx, *cxm = vx + 6 * nx, *cyp = vy + 5 * ny, *cym = vy + 6 * ny;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int id0 = 512 * w + lane;
    double xp[kOneQ], xm[kOneQ], yp[kOneQ], ym[kOneQ], own[kOneQ], y[kOneQ], ap[kOneQ];
    int cs[kOneQ], cw[kOneQ], cn[kOneQ], to[kOneQ];  // south, west, north neighbour; where the cell is stored
    bool special = false;
    if (threadIdx.x < 32) lds[part + threadIdx.x] = 0.0;
#pragma unroll
    for (int q = 0; q < kOneQ; q++) {
        const int id = id0 + 64 * q;
        own[q] = 0.0;
        int j = 0, i = 0;
        if (id < n) {
            j = id / nx;
            i = id - j * nx;
            double v = p[id];
            if (i == 0 || j == 0) {  // set_pressure_BC
                v = 100.0;
                p[id] = v;
            }
            own[q] = v;
            lds[id] = v;
            lds[kOneStride + id] = v;
        }
        const bool in = i > 0 && i < nx - 1 && j > 0 && j < ny - 1;
        const int c = in ? id : nx + 1;
        cs[q] = c - nx;
        cw[q] = c - 1;
        cn[q] = c + nx;
        to[q] = in ? id : kOneReg;
        if (!in) own[q] = 0.0;
        xp[q] = in ? cxp[i] : 0.0;
        xm[q] = in ? cxm[i] : 0.0;
        yp[q] = in ? cyp[j] : 0.0;
        ym[q] = in ? cym[j] : 0.0;
        ap[q] = in ? -1 * ((xp[q] + xm[q]) + (yp[q] + ym[q])) : 1.0;
        special = special || div_special(ap[q]);
        y[q] = 1.0 / ap[q];
        __builtin_amdgcn_sched_barrier(0);
    }
    __syncthreads();
    double res = 1.0;
    int k = iter0;
    bool stopped = k >= itermax;
    // iteration k, p_k in buffer B; true: no further one
    auto iteration = [&]<int B>() -> bool {
        constexpr int b = B * kOneStride, nb = kOneStride - b;
        double r[kOneQ], nv[kOneQ], small = 1.0, large = 1.0;
#pragma unroll
        for (int q = 0; q < kOneQ; q++) {
            const double e = lds[b + cw[q] + 2] * xp[q], ww = lds[b + cw[q]] * xm[q];
            const double nn = lds[b + cn[q]] * yp[q], s = lds[b + cs[q]] * ym[q];
            r[q] = own[q] * ap[q] + e + ww + nn + s;
            const double t = -(e + ww + nn + s);
            nv[q] = div_by(t, ap[q], y[q]);
            // (a cell without coefficients has t = 0 and is left out)
            small = fmin(small, to[q] == kOneReg ? 1.0 : fabs(t));
            large = fmax(large, fabs(t));
        }
        if (__any(special || !(small > 1e-200 && large < 1e200))) {
            __builtin_amdgcn_sched_barrier(0);
#pragma unroll
            for (int q = 0; q < kOneQ; q++) {
                const double e = lds[b + cw[q] + 2] * xp[q], ww = lds[b + cw[q]] * xm[q];
                const double nn = lds[b + cn[q]] * yp[q], s = lds[b + cs[q]] * ym[q];
                nv[q] = -(e + ww + nn + s) / ap[q];
                __builtin_amdgcn_sched_barrier(0);
            }
        }
        // the next iterate, before the test is known; the buffer's former
        // contents were last read before the previous barrier
#pragma unroll
        for (int q = 0; q < kOneQ; q++) lds[nb + to[q]] = nv[q];
        const double f = fold512(r);
        if (lane == 0) lds[part + 16 * B + w] = f;
        __syncthreads();
        if (k > iter0) {  // (iter0: nothing done yet, or decided by the launch before)
            res = fold_parts(lds, part + 16 * B, lane);
            stopped = !(res > tol) || k >= itermax;
        }
        if (stopped || k - iter0 >= most) return true;
#pragma unroll
        for (int q = 0; q < kOneQ; q++) own[q] = nv[q];
        k++;
        return false;
    };
    while (!stopped)
        if (iteration.template operator()<0>() || iteration.template operator()<1>()) break;
#pragma unroll
    for (int q = 0; q < kOneQ; q++)
        if (to[q] != kOneReg) p[to[q]] = own[q];
    if (threadIdx.x == 0) {
        out[0] = res;
        out[1] = (double)k;
        out[2] = stopped ? 1.0 : 0.0;
    }
}

// The same for up to kOneCells cells (16 waves, 128 registers a lane), with
// the coefficients read from LDS.
__global__ __launch_bounds__(1024) void kc_ppe_wide(int nx, int ny, const double *vx, const double *vy,
                                                               double *p, int iter0, int itermax, int most, double tol,
                                                               double *out)
{
    extern __shared__ __align__(16) double lds[];
    const int n = nx * ny;
    // offsets in lds: the two iterates from 0 and n; the block sums, [2][16];
    // cxp, cxm and cyp, cym
    const int part = 2 * n, lx = part + 32, ly = lx + 2 * nx;
    const double *cxp = vx + 5 * nx, *cxm = vx + 6 * nx, *cyp = vy + 5 * ny, *cym = vy + 6 * ny;
    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int id0 = 512 * w + lane;
    double own[kOneQ], y[kOneQ];
    int ij[kOneQ];  // i in the low half, j in the high half
    unsigned in = 0;
    bool special = false;
    {
        for (int k = threadIdx.x; k < 2 * nx; k += blockDim.x) lds[lx + k] = cxp[k];  // cxp, cxm are adjacent
        for (int k = threadIdx.x; k < 2 * ny; k += blockDim.x) lds[ly + k] = cyp[k];
    }
    if (threadIdx.x < 32) lds[part + threadIdx.x] = 0.0;
#pragma unroll
    for (int q = 0; q < kOneQ; q++) {
        const int id = id0 + 64 * q;
        own[q] = y[q] = 0.0;
        ij[q] = 0;
        if (id < n) {
            const int j = id / nx, i = id - j * nx;
            ij[q] = i | (j << 16);
            double v = p[id];
            if (i == 0 || j == 0) v = 100.0;  // set_pressure_BC
            own[q] = v;
            lds[id] = v;
            lds[n + id] = v;
            if (i > 0 && i < nx - 1 && j > 0 && j < ny - 1) {
                in |= 1u << q;
                const double a = -1 * ((cxp[i] + cxm[i]) + (cyp[j] + cym[j]));
                special = special || div_special(a);
                y[q] = 1.0 / a;
            }
        }
    }
    __syncthreads();
    double res = 1.0;
    int k = iter0;
    bool stopped = k >= itermax;
    // k - iter0 iterations done; p_k is iterate (k - iter0) & 1
    while (!stopped) {
        const int b = ((k - iter0) & 1) * n, nb = n - b;
        double r[kOneQ], nv[kOneQ];
#pragma unroll
        for (int q = 0; q < kOneQ; q++) {
            r[q] = 0.0;
            nv[q] = own[q];
            if (in & (1u << q)) {
                const int id = b + id0 + 64 * q;
                double xp, xm, yp, ym, a;
                const int i = ij[q] & 0xffff, j = ij[q] >> 16;
                xp = lds[lx + i];
                xm = lds[lx + nx + i];
                yp = lds[ly + j];
                ym = lds[ly + ny + j];
                a = -1 * ((xp + xm) + (yp + ym));
                const double e = lds[id + 1] * xp, ww = lds[id - 1] * xm, nn = lds[id + nx] * yp, s = lds[id - nx] * ym;
                r[q] = own[q] * a + e + ww + nn + s;
                nv[q] = div_by(-(e + ww + nn + s), a, y[q], special);
            }
        }
        // the next iterate, before the test is known: a stop keeps p_k, which
        // is in own; the buffer's former contents were last read before the
        // previous barrier
#pragma unroll
        for (int q = 0; q < kOneQ; q++)
            if (in & (1u << q)) lds[nb + id0 + 64 * q] = nv[q];
        const double f = fold512(r);
        if (lane == 0) lds[part + 16 * (k & 1) + w] = f;
        __syncthreads();
        if (k > iter0) {  // (iter0: nothing done yet, or decided by the launch before)
            res = fold_parts(lds, part + 16 * (k & 1), lane);
            if (!(res > tol) || k >= itermax) stopped = true;
        }
        if (stopped || k - iter0 >= most) break;
#pragma unroll
        for (int q = 0; q < kOneQ; q++) own[q] = nv[q];
        k++;
    }
#pragma unroll
    for (int q = 0; q < kOneQ; q++)
        if (id0 + 64 * q < n) p[id0 + 64 * q] = own[q];
    if (threadIdx.x == 0) {
        out[0] = res;
        out[1] = (double)k;
        out[2] = stopped ? 1.0 : 0.0;
    }
}

// Per-lane coefficients of its cells: held in registers (REG, at most
// kOneReg cells) or read from the axis vectors.
template <bool REG>
struct OneCoef {
    double xp[REG ? kOneQ : 1], xm[REG ? kOneQ : 1], yp[REG ? kOneQ : 1], ym[REG ? kOneQ : 1];
};

// ADsolver (ADSolver.cu:268-395) on one workgroup.  u and v live in LDS, in
// place: a sweep holds its new values in registers until every cell has been
// read.  The reference's second buffer matters only through its ring, which
// keeps the values of two iterations ago: those are kept apart (alt) and
// change places with the ring after each sweep.  The deck's ten calls of five
// iterations: 0.65 ms (3.5 launch by launch); 88 x 88 cells 2.7 ms (5.5).
template <bool REG>
__global__ __launch_bounds__(REG ? 512 : 1024) void kc_ad_one(int nx, int ny, const double *vx, const double *vy,
                                                              double *u, double *v, double *uf, double *vf, double dt,
                                                              double w_ad, double tol, int itermax, double *out)
{
    extern __shared__ __align__(16) double lds[];
    const int n = nx * ny, nr = 2 * (nx + ny);
    // offsets in lds: u and v from 0 and n; the other buffers' rings, [2][nr];
    // the block sums, [2 fields][16]
    const int alt = 2 * n, part = alt + 2 * nr;
    const double *dx = vx, *dy = vy;
    const double *axp = vx + 2 * nx, *axm = vx + 3 * nx, *px = vx + 4 * nx;
    const double *ayp = vy + 2 * ny, *aym = vy + 3 * ny, *py = vy + 4 * ny;
    const int tid = threadIdx.x, nt = blockDim.x, lane = tid & 63, w = tid >> 6;
    const int id0 = 512 * w + lane;
    const int nuf = (nx - 1) * (ny - 2), nvf = (nx - 2) * (ny - 1);

    // Compute_velf (kc_velf's expressions)
    auto velf = [&]() {
        for (int id = tid; id < (nuf > nvf ? nuf : nvf); id += nt) {
            if (id < nuf) {
                const int j = id / (nx - 1), i = id - j * (nx - 1);
                const int idc = j * nx + i;
                uf[id] = 1.0 / (dx[i] + dx[i + 1]) * (lds[idc + nx + 1] * dx[i] + lds[idc + nx] * dx[i + 1]);
            } else {
                const int j = id / (nx - 2), i = id - j * (nx - 2);
                const int idc = j * nx + i;
                vf[id] = 1.0 / (dy[j + 1] + dy[j]) * (lds[n + idc + nx + 1] * dy[j] + lds[n + idc + 1] * dy[j + 1]);
            }
        }
    };
    // set_velocity_BC (kc_bc) on both fields
    auto bc = [&]() {
        for (int k = tid; k < 2 * (nx + ny - 4); k += nt) {
            const int c = k >= nx + ny - 4, kk = k - c * (nx + ny - 4);
            const int o = c * n;
            const double two = (c ? 0.0 : 1.0) * 2.0;
            if (kk < ny - 2) {
                const int j = 1 + kk;
                const int ww = j * nx, e = nx - 1 + j * nx;
                const double old_w = lds[o + ww];
                const double nw = -lds[o + ww + 1] + two, ne = -lds[o + e - 1] + two;
                lds[o + ww] = nw;
                lds[o + e] = ne;
                if (j == 1) lds[o + 0] = -old_w + two;
                if (j == ny - 2) lds[o + (ny - 1) * nx] = -nw + two;
                if (j == ny - 2) lds[o + nx - 1 + (ny - 1) * nx] = -ne + two;
            } else {
                const int i = 1 + (kk - (ny - 2));
                const double ns = -lds[o + i + nx] + two;
                lds[o + i] = ns;
                lds[o + i + (ny - 1) * nx] = -lds[o + i + (ny - 2) * nx] + two;
                if (i == nx - 2) lds[o + nx - 1] = -ns + two;
            }
        }
    };
    // ring index -> cell: south row, north row, west and east columns
    auto ring = [&](int k) {
        if (k < nx) return k;
        if (k < 2 * nx) return (ny - 1) * nx + (k - nx);
        if (k < 2 * nx + ny - 2) return (k - 2 * nx + 1) * nx;
        return (k - 2 * nx - (ny - 2) + 1) * nx + nx - 1;
    };
    const int nring = 2 * nx + 2 * (ny - 2);

    for (int k = tid; k < n; k += nt) {
        lds[k] = u[k];
        lds[n + k] = v[k];
    }
    for (int k = tid; k < 2 * nr; k += nt) lds[alt + k] = 0.0;  // fresh scratch (:275-287)
    if (tid < 32) lds[part + tid] = 0.0;
    __syncthreads();
    velf();  // :298, before the BC (stale ghosts)
    __syncthreads();
    bc();  // :304
    __syncthreads();

    // ADSource (kc_source's expressions) of the owned cells, coefficients
    OneCoef<REG> C;
    double s[2][kOneQ], y[kOneQ], ap[REG ? kOneQ : 1];
    int ij[kOneQ];
    unsigned in = 0;
    bool special = false;
#pragma unroll
    for (int q = 0; q < kOneQ; q++) {
        const int id = id0 + 64 * q;
        s[0][q] = s[1][q] = y[q] = 0.0;
        ij[q] = 0;
        if constexpr (REG) C.xp[q] = C.xm[q] = C.yp[q] = C.ym[q] = ap[q] = 0.0;
        if (id >= n) continue;
        const int j = id / nx, i = id - j * nx;
        ij[q] = i | (j << 16);
        if (!(i > 0 && i < nx - 1 && j > 0 && j < ny - 1)) continue;
        in |= 1u << q;
        const double dx_i = dx[i], dx_ip1 = dx[i + 1], dx_im1 = dx[i - 1];
        const double dy_j = dy[j], dy_jp1 = dy[j + 1], dy_jm1 = dy[j - 1];
        const double ufe = uf[i + (j - 1) * (nx - 1)], ufw = uf[i - 1 + (j - 1) * (nx - 1)];
        const double vfn = vf[i - 1 + j * (nx - 2)], vfs = vf[i - 1 + (j - 1) * (nx - 2)];
#pragma unroll
        for (int c = 0; c < 2; c++) {
            const int a = c * n;
            s[c][q] =
                (lds[a + id] - (dt / dx_i) * 0.5 * (((1 / (dx_i + dx_ip1)) * (lds[a + id + 1] * dx_i + lds[a + id] * dx_ip1) * ufe)
                                              - ((1 / (dx_i + dx_im1)) * (lds[a + id] * dx_im1 + lds[a + id - 1] * dx_i) * ufw)))
                - (dt / dy_j) * 0.5 * (((1 / (dy_j + dy_jp1)) * (lds[a + id + nx] * dy_j + lds[a + id] * dy_jp1) * vfn)
                                       - ((1 / (dy_j + dy_jm1)) * (lds[a + id] * dy_jm1 + lds[a + id - nx] * dy_j) * vfs));
        }
        const double d = px[i] + py[j];
        special = special || div_special(d);
        y[q] = 1.0 / d;
        if constexpr (REG) {
            C.xp[q] = axp[i];
            C.xm[q] = axm[i];
            C.yp[q] = ayp[j];
            C.ym[q] = aym[j];
            ap[q] = d;
        }
    }
    __syncthreads();  // uf, vf read before the loop rewrites them

    double ures = 1.0, vres = 1.0;
    int iter = 0;
    while (ures + vres > tol && iter < itermax) {  // :315
        bc();                                       // :317
        __syncthreads();
        velf();  // :321
        double nv[2][kOneQ], r[2][kOneQ];
#pragma unroll
        for (int q = 0; q < kOneQ; q++) {
            r[0][q] = r[1][q] = nv[0][q] = nv[1][q] = 0.0;
            if (!(in & (1u << q))) continue;
            const int id = id0 + 64 * q;
            double xp, xm, yp, ym, d;
            if constexpr (REG) {
                xp = C.xp[q];
                xm = C.xm[q];
                yp = C.yp[q];
                ym = C.ym[q];
                d = ap[q];
            } else {
                const int i = ij[q] & 0xffff, j = ij[q] >> 16;
                xp = axp[i];
                xm = axm[i];
                yp = ayp[j];
                ym = aym[j];
                d = px[i] + py[j];
            }
#pragma unroll
            for (int c = 0; c < 2; c++) {
                const int a = c * n;
                const double t = s[c][q] + xp * lds[a + id + 1] + xm * lds[a + id - 1] + yp * lds[a + id + nx] + ym * lds[a + id - nx];
                double x = div_by(t, d, y[q], special);
                if (w_ad != 1.0) x = (1.0 - w_ad) * lds[a + id] + w_ad * x;
                nv[c][q] = x;
                r[c][q] = fabs(x - lds[a + id]);
            }
        }
        const double fu = fold512(r[0]), fv = fold512(r[1]);
        if (lane == 0) {
            lds[part + w] = fu;
            lds[part + 16 + w] = fv;
        }
        __syncthreads();
        ures = fold_parts(lds, part, lane);  // :350-366
        vres = fold_parts(lds, part + 16, lane);
        // the new interior, and the ring of the other buffer (:337 changed
        // only the old buffer's corner (0,0), from its ghost (0,1))
#pragma unroll
        for (int q = 0; q < kOneQ; q++)
            if (in & (1u << q)) {
                lds[id0 + 64 * q] = nv[0][q];
                lds[n + id0 + 64 * q] = nv[1][q];
            }
        for (int k = tid; k < 2 * nring; k += nt) {
            const int c = k >= nring, kk = k - c * nring;
            const int id = ring(kk);
            double old = lds[c * n + id];
            const double a = lds[alt + c * nr + kk];
            if (kk == 0) old = -lds[c * n + nx] + (c ? 0.0 : 1.0) * 2.0;
            if (kk != 2 * nx) lds[c * n + id] = a;  // (0,1) is written below, after the corner has read it
            lds[alt + c * nr + kk] = kk == 2 * nx ? lds[alt + c * nr + kk] : old;
        }
        __syncthreads();
        if (tid < 2) {  // ghost (0,1)
            const double a = lds[alt + tid * nr + 2 * nx];
            lds[alt + tid * nr + 2 * nx] = lds[tid * n + nx];
            lds[tid * n + nx] = a;
        }
        iter++;
        __syncthreads();
    }
    for (int k = tid; k < n; k += nt) {
        u[k] = lds[k];
        v[k] = lds[n + k];
    }
    if (tid == 0) {
        out[0] = ures;
        out[1] = vres;
        out[2] = (double)iter;
    }
}

// ---------------------------------------------------------------------------
CompatCase::~CompatCase()
{
    if (st) hipStreamSynchronize(st);
    if (mem) hipFree(mem);
    if (h_out) hipHostFree(h_out);
    if (st) hipStreamDestroy(st);
}

if_status CompatCase::create(const if_case_desc &d)
{
    int ndev = 0;
    if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
        return fail(IF_ERR_NODEV, "no HIP device available");
    if (d.nxf < 3 || d.nyf < 3 || !d.xf || !d.yf) return fail(IF_ERR_ARG, "case: bad grid");
    nx = d.nxf + 1;
    ny = d.nyf + 1;
    dt = d.dt;
    re = d.re;
    ad_itermax = d.ad_itermax;
    ppe_itermax = d.ppe_itermax;
    w_ad = d.ad_omega > 0 ? d.ad_omega : 1.0;
    xc.resize(nx);
    dx.resize(nx);
    yc.resize(ny);
    dy.resize(ny);
    grid_metric(d.nxf, d.xf, xc.data(), dx.data());
    grid_metric(d.nyf, d.yf, yc.data(), dy.data());
    IFF_HIP(hipStreamCreate(&st));
    const size_t N = (size_t)nx * ny;
    nblk = (int)((N + 255) / 256);
    // per-axis vectors: dx, dy, xc, yc, AD (xp xm px / yp ym py), PPE (cxp cxm / cyp cym)
    std::vector<double> ax(8 * nx, 0.0), ay(8 * ny, 0.0);
    const double k = dt / re;
    auto fill = [&](std::vector<double> &V, const std::vector<double> &w,
                    const std::vector<double> &c, int n, bool is_x) {
        for (int i = 0; i < n; i++) { V[i] = w[i]; V[n + i] = c[i]; }
        for (int i = 1; i < n - 1; i++) {
            const double di = w[i], dp = w[i + 1], dm = w[i - 1];
            V[2 * n + i] = k * (2 / (di * (di + dp)));
            V[3 * n + i] = k * (2 / (di * (di + dm)));
            V[4 * n + i] = is_x ? 1.0 + k * ((2 / (di * (di + dp))) + (2 / (di * (di + dm))))
                                : k * ((2 / (di * (di + dp))) + (2 / (di * (di + dm))));
            V[5 * n + i] = (2 / (di * (di + dp)));
            V[6 * n + i] = (2 / (di * (di + dm)));
        }
    };
    fill(ax, dx, xc, nx, true);
    fill(ay, dy, yc, ny, false);
    const size_t nuf = (size_t)(nx - 1) * (ny - 2), nvf = (size_t)(nx - 2) * (ny - 1);
    const size_t total = 12 * N + nuf + nvf + 8 * (size_t)(nx + ny) + 2 * (size_t)nblk + 4;
    IFF_HIP(hipMalloc(&mem, total * sizeof(double)));
    IFF_HIP(hipMemsetAsync(mem, 0, total * sizeof(double), st));
    double *m = mem;
    for (int b = 0; b < 2; b++) { u[b] = m; m += N; }
    for (int b = 0; b < 2; b++) { v[b] = m; m += N; }
    for (int b = 0; b < 2; b++) { p[b] = m; m += N; }
    sx = m; m += N;
    sy = m; m += N;
    iblank = m; m += N;
    pres = m; m += N;  // unused spare (keeps the layout simple)
    m += 2 * N;
    uf = m; m += nuf;
    vf = m; m += nvf;
    vx = m; m += 8 * nx;
    vy = m; m += 8 * ny;
    part = m; m += 2 * nblk;
    scal = m; m += 4;
    IFF_HIP(hipMemcpyAsync(vx, ax.data(), ax.size() * 8, hipMemcpyHostToDevice, st));
    IFF_HIP(hipMemcpyAsync(vy, ay.data(), ay.size() * 8, hipMemcpyHostToDevice, st));
    IFF_HIP(hipHostMalloc((void **)&h_out, 4 * sizeof(double), hipHostMallocDefault));
    // the one-workgroup forms, where the fields fit in one CU's LDS
    if (N <= (size_t)kOneCells) {
        lds_ad = sizeof(double) * (2 * N + 4 * (size_t)(nx + ny) + 32);
        lds_ppe = N <= (size_t)kOneReg ? 0 : sizeof(double) * (2 * N + 32 + 2 * (size_t)(nx + ny));
        one_ad = lds_ad <= kOneLds && ad_itermax <= kOneIters;
        one_ppe = lds_ppe <= kOneLds;
        for (const void *k : {(const void *)kc_ad_one<true>, (const void *)kc_ad_one<false>,
                              (const void *)kc_ppe_wide})
            IFF_HIP(hipFuncSetAttribute(k, hipFuncAttributeMaxDynamicSharedMemorySize, (int)kOneLds));
    }
    hipLaunchKernelGGL(kc_init, dim3(nblk), dim3(256), 0, st, nx, ny, vx + nx, vy + ny, u[0], v[0],
                       p[0], iblank);
    IFF_HIP(hipGetLastError());
    IFF_HIP(hipStreamSynchronize(st));
    return IF_OK;
}

void CompatCase::bc(double *uu, double *vv)
{
    const int nb = (nx + ny + 255) / 256;
    hipLaunchKernelGGL(kc_bc, dim3(nb), dim3(256), 0, st, nx, ny, uu, 1.0);
    hipLaunchKernelGGL(kc_bc, dim3(nb), dim3(256), 0, st, nx, ny, vv, 0.0);
}

void CompatCase::velf(const double *uu, const double *vv)
{
    const int n = std::max((nx - 1) * (ny - 2), (nx - 2) * (ny - 1));
    hipLaunchKernelGGL(kc_velf, dim3((n + 255) / 256), dim3(256), 0, st, nx, ny, vx, vy, uu, vv, uf, vf);
}

// ImmerseFlow::ADsolver, ADSolver.cu:268-395.
if_status CompatCase::ad_step(if_step_stats *stt)
{
    const double *xp = vx + 2 * nx, *xm = vx + 3 * nx, *px = vx + 4 * nx;
    const double *yp = vy + 2 * ny, *ym = vy + 3 * ny, *py = vy + 4 * ny;
    if (one_ad) {
        const dim3 wg(64 * ((nx * ny + 511) / 512));
        const double tol = std::pow(10.0, -6.0);
        auto *k = nx * ny <= kOneReg ? kc_ad_one<true> : kc_ad_one<false>;
        hipLaunchKernelGGL(k, dim3(1), wg, lds_ad, st, nx, ny, vx, vy, u[cur], v[cur], uf, vf, dt, w_ad, tol,
                           ad_itermax, h_out);
        IFF_HIP(hipGetLastError());
        IFF_HIP(hipStreamSynchronize(st));
        steps++;
        if (stt) {
            std::memset(stt, 0, sizeof(*stt));
            stt->steps = 1;
            stt->ad_iters = (int)h_out[2];
            stt->ad_res = h_out[0] + h_out[1];
            stt->total_ad_iters = stt->ad_iters;
        }
        return IF_OK;
    }
    // fresh per-call scratch (cudaMalloc'd in the reference, :275-287)
    IFF_HIP(hipMemsetAsync(u[1 - cur], 0, sizeof(double) * nx * ny, st));
    IFF_HIP(hipMemsetAsync(v[1 - cur], 0, sizeof(double) * nx * ny, st));
    velf(u[cur], v[cur]);  // :298, before the BC (stale ghosts)
    bc(u[cur], v[cur]);    // :304
    hipLaunchKernelGGL(kc_source, dim3(nblk), dim3(256), 0, st, nx, ny, vx, vy, dt, u[cur], v[cur],
                       uf, vf, sx, sy);  // :308
    double ures = 1.0, vres = 1.0;
    int iter = 0;
    while (ures + vres > std::pow(10.0, -6.0) && iter < ad_itermax) {  // :315
        bc(u[cur], v[cur]);                                             // :317
        velf(u[cur], v[cur]);                                           // :321
        hipLaunchKernelGGL(kc_sweep, dim3(nblk), dim3(256), 0, st, nx, ny, xp, xm, px, yp, ym, py,
                           iblank, sx, sy, u[cur], v[cur], u[1 - cur], v[1 - cur], w_ad);  // :326,:331
        bc(u[cur], v[cur]);                                             // :337 (old buffer)
        cur = 1 - cur;                                                  // :342-348
        hipLaunchKernelGGL(kc_l1, dim3(nblk), dim3(256), 0, st, nx, ny, iblank, u[cur], u[1 - cur],
                           v[cur], v[1 - cur], part);                   // :350-358
        hipLaunchKernelGGL(kc_finish, dim3(1), dim3(256), 0, st, part, nblk, 2, scal);
        IFF_HIP(hipMemcpyAsync(h_out, scal, 2 * sizeof(double), hipMemcpyDeviceToHost, st));
        IFF_HIP(hipStreamSynchronize(st));                              // :360-366
        ures = h_out[0];
        vres = h_out[1];
        iter += 1;
    }
    IFF_HIP(hipGetLastError());
    steps++;
    if (stt) {
        std::memset(stt, 0, sizeof(*stt));
        stt->steps = 1;
        stt->ad_iters = iter;
        stt->ad_res = ures + vres;
        stt->total_ad_iters = iter;
    }
    return IF_OK;
}

// ImmerseFlow::PPESolver loop, PPESolver.cu:164-195.
if_status CompatCase::ppe_solve(if_step_stats *stt)
{
    const double *cxp = vx + 5 * nx, *cxm = vx + 6 * nx, *cyp = vy + 5 * ny, *cym = vy + 6 * ny;
    if (one_ppe) {
        const dim3 wg(64 * ((nx * ny + 511) / 512));
        auto *k = nx * ny <= kOneReg ? kc_ppe_one : kc_ppe_wide;
        h_out[0] = 1.0;
        h_out[1] = h_out[2] = 0.0;
        do {  // a launch runs at most kOneIters iterations
            hipLaunchKernelGGL(k, dim3(1), wg, lds_ppe, st, nx, ny, vx, vy, p[pcur], (int)h_out[1],
                               ppe_itermax, kOneIters, std::pow(10.0, -6.0), h_out);
            IFF_HIP(hipGetLastError());
            IFF_HIP(hipStreamSynchronize(st));
        } while (h_out[2] == 0.0);
        if (stt) {
            std::memset(stt, 0, sizeof(*stt));
            stt->ppe_sweeps = (int)h_out[1];
            stt->ppe_res = h_out[0];
            stt->total_ppe_sweeps = stt->ppe_sweeps;
        }
        return IF_OK;
    }
    IFF_HIP(hipMemsetAsync(p[1 - pcur], 0, sizeof(double) * nx * ny, st));
    hipLaunchKernelGGL(kc_pbc, dim3(nblk), dim3(256), 0, st, nx, ny, p[pcur]);
    double residual = 1.0;
    int iter = 0;
    while (residual > std::pow(10.0, -6.0) && iter < ppe_itermax) {
        hipLaunchKernelGGL(kc_jacobi, dim3(nblk), dim3(256), 0, st, nx, ny, cxp, cxm, cyp, cym,
                           p[pcur], p[1 - pcur]);
        pcur = 1 - pcur;
        hipLaunchKernelGGL(kc_presid, dim3(nblk), dim3(256), 0, st, nx, ny, cxp, cxm, cyp, cym,
                           p[pcur], part);
        hipLaunchKernelGGL(kc_finish, dim3(1), dim3(256), 0, st, part, nblk, 1, scal);
        IFF_HIP(hipMemcpyAsync(h_out, scal, sizeof(double), hipMemcpyDeviceToHost, st));
        IFF_HIP(hipStreamSynchronize(st));
        residual = h_out[0];
        iter += 1;
    }
    hipLaunchKernelGGL(kc_pbc, dim3(nblk), dim3(256), 0, st, nx, ny, p[pcur]);
    IFF_HIP(hipGetLastError());
    IFF_HIP(hipStreamSynchronize(st));
    if (stt) {
        std::memset(stt, 0, sizeof(*stt));
        stt->ppe_sweeps = iter;
        stt->ppe_res = residual;
        stt->total_ppe_sweeps = iter;
    }
    return IF_OK;
}

if_status CompatCase::get_field(int which, double *out, size_t n)
{
    const size_t N = (size_t)nx * ny;
    const double *src = nullptr;
    size_t need = N;
    switch (which) {
    case IF_FIELD_U: src = u[cur]; break;
    case IF_FIELD_V: src = v[cur]; break;
    case IF_FIELD_P: src = p[pcur]; break;
    case IF_FIELD_UF: src = uf; need = (size_t)(nx - 1) * (ny - 2); break;
    case IF_FIELD_VF: src = vf; need = (size_t)(nx - 2) * (ny - 1); break;
    case IF_FIELD_IBLANK: src = iblank; break;
    default: return fail(IF_ERR_ARG, "get_field: field not available in compat mode");
    }
    if (!out || n != need) return fail(IF_ERR_ARG, "get_field: size mismatch");
    IFF_HIP(hipStreamSynchronize(st));
    IFF_HIP(hipMemcpy(out, src, need * sizeof(double), hipMemcpyDeviceToHost));
    return IF_OK;
}

if_status CompatCase::set_field(int which, const double *in, size_t n)
{
    const size_t N = (size_t)nx * ny;
    double *dst = nullptr;
    size_t need = N;
    switch (which) {
    case IF_FIELD_U: dst = u[cur]; break;
    case IF_FIELD_V: dst = v[cur]; break;
    case IF_FIELD_P: dst = p[pcur]; break;
    case IF_FIELD_UF: dst = uf; need = (size_t)(nx - 1) * (ny - 2); break;
    case IF_FIELD_VF: dst = vf; need = (size_t)(nx - 2) * (ny - 1); break;
    default: return fail(IF_ERR_ARG, "set_field: field not settable");
    }
    if (!in || n != need) return fail(IF_ERR_ARG, "set_field: size mismatch");
    IFF_HIP(hipStreamSynchronize(st));
    IFF_HIP(hipMemcpy(dst, in, need * sizeof(double), hipMemcpyHostToDevice));
    return IF_OK;
}

}  // namespace iff
