// Persistent zebra line SOR: a chunk of K sweeps in one launch.
//
// One launch per colour (k_line_sor) reads its row's factors, fields and flags
// again each time and takes 7.6 us on a 256^2 grid, where a row's dependent
// chain (B fused multiply-adds forward and back, six reduction levels across
// the lanes) is a fifth of that.  Here a wave owns a row for the whole chunk and
// a lane its segment of it: the row, its right side and its factors stay
// in registers, the rows above and below come from the neighbouring waves
// through LDS.  A block's NW rows include a halo of 2M rows on either side:
// each half-sweep leaves one row less of it exact, so M sweeps run before the
// blocks exchange rows (device scope, as in the register-tile sweep: stage
// counters, bounded waits).
// Same operations in the same order per row as k_line_sor.  Measured, 256^2 FP64:
// 3.8 us per sweep against 15.2; bound by the row's chain (four half-sweeps of
// about 1.1 us a stage) and the exchange after each stage (about 3 us).
#include "common.h"
#include "kernels.h"
#include "line.h"

namespace iff {

template <typename T, int B, int NW, int M>
__global__ __launch_bounds__(64 * NW) void k_line_pers(const CaseDev *cs, const int2 *blocks, int K, PersArgs pa)
{
    constexpr int H = 2 * M, NS = NW - 2 * H;     // halo rows a side, stored rows
    constexpr int RY = (H + NS - 1) / NS;         // blocks a side that the halo reaches
    static_assert(NS > 0 && 2 * RY < 64, "block shape");
    __shared__ T xr[NW + 2][B][64];  // rows of the block; the slots beyond it stay 0
    const int2 bl = blocks[blockIdx.x];
    const CaseDev &c = cs[bl.x];
    const Ctrl *ct = c.ctrl;
    if (!ct->active || ct->ppe_done) return;  // every block of the case alike
    int kexec = c.ppe_itermax - ct->ppe_sweeps;
    if (kexec > K) kexec = K;
    if (kexec <= 0) return;
    const int nx = c.nx, ny = c.ny, P = c.P, n = nx - 2, S = c.lS, m = S - 1;
    const int lane = (int)threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
    const int j = 1 + bl.y * NS - H + w;
    const bool rowin = j >= 1 && j <= ny - 2, stored = rowin && w >= H && w < H + NS;
    T *buf[2];
    const T *rhs;
    T om;
    const bool zero_src = sizeof(T) == 4;  // a mixed chunk starts from e = 0
    if constexpr (sizeof(T) == 8) {
        buf[0] = c.p[ct->ppe_base & 1];
        buf[1] = c.p[(ct->ppe_base + 1) & 1];
        rhs = c.rhs;
        om = c.omega;
    } else {
        buf[0] = c.e[0];
        buf[1] = c.e[1];
        rhs = c.r32;
        om = c.omega_f;
    }
    const int len = lane < S - 1 ? B - 1 : (lane == S - 1 ? n - (S - 1) * B : 0);
    const int i0 = 1 + lane * B;

    // the row, its right side and its factors.  A lane with fewer cells (the
    // row's last segment, and the lanes behind it) gets factors that pass the
    // recurrences' values through: r = 0, -l r = 1 forward, -u r = 0 backward.
    T p[B], rh[B], fr[B], fn[B], fc[B], fh[B], fq[B];
    T pal[kLinePcrLevels], pga[kLinePcrLevels], prb = (T)0, snl = (T)0, snu = (T)0;
    unsigned nb_n = 0, nb_s = 0, solved = 0, in = 0;  // bit t: open faces, solved, inside the row
    T yN = (T)0, yS = (T)0;
#pragma unroll
    for (int t = 0; t < B; t++) {
        p[t] = rh[t] = fr[t] = fc[t] = fh[t] = fq[t] = (T)0;
        fn[t] = (T)1;
    }
#pragma unroll
    for (int q = 0; q < kLinePcrLevels; q++) pal[q] = pga[q] = (T)0;
    const size_t row = (size_t)(rowin ? j : 1) * P;
    if (rowin) {
        const LineMetric<T> mt(c);
        yN = G(mt.yp)[j];
        yS = G(mt.ym)[j];
        const auto F = G((const T *)c.lf + (size_t)j * line_row_stride(B));
        const auto pcr = F + (size_t)kLinePlanes * B * 64;
#pragma unroll
        for (int q = 0; q < kLinePcrLevels; q++) {
            if ((1 << q) >= m) break;
            pal[q] = pcr[(2 * q) * 64 + lane];
            pga[q] = pcr[(2 * q + 1) * 64 + lane];
        }
        prb = pcr[(2 * kLinePcrLevels) * 64 + lane];
        if (lane < m) {
            snl = F[((size_t)kLfR * B + B - 1) * 64 + lane];
            snu = F[((size_t)kLfNlr * B + B - 1) * 64 + lane];
        }
#pragma unroll
        for (int t = 0; t < B; t++) {
            if (t < len) {
                fr[t] = F[((size_t)kLfR * B + t) * 64 + lane];
                fn[t] = F[((size_t)kLfNlr * B + t) * 64 + lane];
                fh[t] = F[((size_t)kLfH * B + t) * 64 + lane];
                fq[t] = F[((size_t)kLfQ * B + t) * 64 + lane];
                if (t < len - 1) fc[t] = F[((size_t)kLfNcp * B + t) * 64 + lane];
            }
            if (i0 + t <= n) {
                const int i = i0 + t;
                in |= 1u << t;
                const unsigned f = G(c.flags)[row + i];
                if (!zero_src) p[t] = G((const T *)buf[0])[row + i];
                rh[t] = G(rhs)[row + i];
                T l, b, u;
                if (LineMetric<T>::cell(f, G(mt.xp)[i], G(mt.xm)[i], yN, yS, l, b, u)) solved |= 1u << t;
                if (f & F_OPEN_N) nb_n |= 1u << t;
                if (f & F_OPEN_S) nb_s |= 1u << t;
            }
        }
    }
    if (w == 0) {
#pragma unroll
        for (int t = 0; t < B; t++) xr[0][t][lane] = xr[NW + 1][t][lane] = (T)0;
    }

    // one half-sweep of this wave's row
    auto solve = [&]() __attribute__((always_inline)) {
        T g[B], d[B];
#pragma unroll
        for (int t = 0; t < B; t++) {
            const T un = xr[w + 2][t][lane], us = xr[w][t][lane];
            const T aN = nb_n >> t & 1u ? yN : (T)0, aS = nb_s >> t & 1u ? yS : (T)0;
            d[t] = solved >> t & 1u ? (aN * un + aS * us) - rh[t] : p[t];
        }
        // forward gp = fma(-l r, gp, d r)
        T gp = (T)0;
#pragma unroll
        for (int t = 0; t < B; t++) {
            const T dr = d[t] * fr[t];
            gp = t == 0 ? dr : fmaT(fn[t], gp, dr);
            g[t] = gp;
        }
        const T glast = gp;
        // backward g = fma(-u r, g, gp)
#pragma unroll
        for (int t = B - 2; t >= 0; t--) g[t] = fmaT(fc[t], g[t + 1], g[t]);
        // separators, cyclic reduction
        const T gR = from_east(g[0]);
        T D = lane < m ? fmaT(snu, gR, fmaT(snl, glast, d[B - 1])) : (T)0;
#pragma unroll
        for (int q = 0; q < kLinePcrLevels; q++) {
            const int sg = 1 << q;
            if (sg >= m) break;
            T Dm_, Dp_;
            if (q == 0) {
                Dm_ = from_west(D);
                Dp_ = from_east(D);
            } else if (q == 1) {
                Dm_ = from_west(from_west(D));
                Dp_ = from_east(from_east(D));
            } else {
                Dm_ = shfl_up_t(D, sg);
                Dp_ = shfl_down_t(D, sg);
            }
            const T Dm = lane >= sg ? Dm_ : (T)0, Dp = lane + sg < m ? Dp_ : (T)0;
            if (lane < m) D = fmaT(pga[q], Dp, fmaT(pal[q], Dm, D));
        }
        const T xs = lane < m ? D * prb : (T)0;
        const T xw = from_west(xs);
        const T xL = lane >= 1 ? xw : (T)0, xR = lane < m ? xs : (T)0;
        // x = fma(q, xR, fma(h, xL, g)), separators xs; relax
#pragma unroll
        for (int t = 0; t < B; t++) {
            T x = fmaT(fq[t], xR, fmaT(fh[t], xL, g[t]));
            if (t == B - 1 && lane < m) x = xs;
            if (solved >> t & 1u) p[t] = p[t] + om * (x - p[t]);
            xr[w + 1][t][lane] = p[t];
        }
    };
    // the row to a buffer at device scope
    auto put = [&](T *out) __attribute__((always_inline)) {
#pragma unroll
        for (int t = 0; t < B; t++)
            if (in >> t & 1u)
                __hip_atomic_store(out + row + i0 + t, p[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    };

    const int nblk = (ny - 2 + NS - 1) / NS, b0 = (int)blockIdx.x - bl.y;
    unsigned *const flags = pa.flags + b0;
    const unsigned f0 = __hip_atomic_load(&flags[bl.y], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    int nb = -1;  // the blocks whose rows the halo holds (a lane of wave 0 each)
    if (w == 0 && lane < 2 * RY) {
        const int q = bl.y + (lane < RY ? lane - RY : lane - RY + 1);
        if (q >= 0 && q < nblk) nb = q;
    }
    // Stages of at most M sweeps, stage l into buffer (l + 1) & 1: as many as
    // leave the chunk's result where kexec single sweeps do
    int rest = kexec, left = (kexec + M - 1) / M;
    if ((left ^ kexec) & 1) left++;
    for (int l = 0;; l++) {
        const int me = min(M, rest - (left - 1));
#pragma unroll
        for (int t = 0; t < B; t++) xr[w + 1][t][lane] = p[t];
        __syncthreads();
        for (int h = 0; h < 2 * me; h++) {  // odd rows first
            if (rowin && (j & 1) != (h & 1) && w > h && NW - 1 - w > h) solve();
            __syncthreads();
        }
        rest -= me;
        left--;
        T *const out = buf[(l + 1) & 1];
        if (stored && (rest == 0 || w < 2 * H || w >= NS)) put(out);
        if (rest == 0) break;
        __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
        __syncthreads();
        if (threadIdx.x == 0)
            __hip_atomic_store(&flags[bl.y], f0 + (unsigned)(l + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool bad = w == 0 && wait_neighbours(flags, nb, f0 + (unsigned)(l + 1), pa.bar);
        if (__builtin_amdgcn_readfirstlane(__syncthreads_or(bad))) break;
        if (rowin && !stored) {
#pragma unroll
            for (int t = 0; t < B; t++)
                if (in >> t & 1u)
                    p[t] = __hip_atomic_load(out + row + i0 + t, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    // counters of all blocks of the case agree when a launch starts
    __syncthreads();
    int ns = (kexec + M - 1) / M;
    if ((ns ^ kexec) & 1) ns++;
    if (threadIdx.x == 0)
        __hip_atomic_store(&flags[bl.y], f0 + (unsigned)ns, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// Waves of a block, sweeps per stage and rows stored: 16 waves have 128
// registers each; where a segment's factors take more, 12 (168; 4 cells in
// FP64 spill at 128) or 8 (256).  From 9 cells a lane they no longer fit.
template <typename T, int B> struct LineShape {
    static constexpr int NW = sizeof(T) == 4 || B < 4 ? 16 : B < 6 ? 12 : 8, M = NW == 8 ? 1 : 2, NS = NW - 4 * M;
    static int capacity()
    {
        static int cap = -1;  // one device type per process
        if (cap < 0) {
            int per_cu = 0, dev = 0, cus = 0;
            if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_line_pers<T, B, NW, M>, 64 * NW, 0) !=
                    hipSuccess ||
                hipGetDevice(&dev) != hipSuccess ||
                hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
                return 0;
            cap = per_cu * cus;
        }
        return cap;
    }
};

#define IFF_LINE_B(X) X(2) X(3) X(4) X(5) X(6) X(7) X(8)

int line_pers_rows(int prec, int B)
{
#define IFF_LR(B_) \
    if (B == B_) return prec == IF_FP64 ? LineShape<double, B_>::NS : LineShape<float, B_>::NS;
    IFF_LINE_B(IFF_LR)
#undef IFF_LR
    return 0;
}

bool line_pers_fits(int prec, int B, int nblocks)
{
#define IFF_LF(B_) \
    if (B == B_)   \
        return nblocks <= (prec == IF_FP64 ? LineShape<double, B_>::capacity() : LineShape<float, B_>::capacity());
    IFF_LINE_B(IFF_LF)
#undef IFF_LF
    return false;
}

void launch_line_pers(hipStream_t st, int prec, int B, const CaseDev *cs, const int2 *blocks, int nblocks, int K,
                      const PersArgs &pa)
{
    const dim3 grid((unsigned)nblocks);
#define IFF_LL(B_)                                                                                                  \
    if (B == B_) {                                                                                                  \
        if (prec == IF_FP64)                                                                                        \
            hipLaunchKernelGGL((k_line_pers<double, B_, LineShape<double, B_>::NW, LineShape<double, B_>::M>), grid, \
                               dim3(64 * LineShape<double, B_>::NW), 0, st, cs, blocks, K, pa);                     \
        else                                                                                                        \
            hipLaunchKernelGGL((k_line_pers<float, B_, LineShape<float, B_>::NW, LineShape<float, B_>::M>), grid,   \
                               dim3(64 * LineShape<float, B_>::NW), 0, st, cs, blocks, K, pa);                      \
    }
    IFF_LINE_B(IFF_LL)
#undef IFF_LL
}

}  // namespace iff
