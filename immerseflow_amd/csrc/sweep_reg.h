// Register-tile red-black SOR for gfx950.
//
// A workgroup of NW (4, 8 or 16) wave64s owns a tile of 128 columns by NW*NRW rows
// (halo H = 2M on every side included): lane l of every wave holds the
// column pair (c0+2l, c0+2l+1) -- one red and one black cell of each row --
// and wave w holds rows w*NRW .. w*NRW+NRW-1, all in registers.  In a
// half-sweep each lane therefore updates exactly one cell per row, and
// which of its two cells that is depends only on the row, so the whole
// wave follows one path with every lane busy:
//   * east/west neighbours: the lane's other cell, or the adjacent lane's
//     through a DPP wave shift;
//   * north/south neighbours: the lane's own registers, except at the
//     wave's first and last row, whose neighbours come from the adjacent
//     waves through a small LDS exchange (one barrier per half-sweep).
// Every cell takes one branch-free form, with the metric itself as its
// coefficients (x: per lane, y: per row) and 0 held in every cell the sweep
// keeps.  FP64: the oracle's update, bit for bit.  FP32 (the mixed path's
// error sweeps): the general form or, on a grid with one coefficient value
// per axis, the five-operation one.  Every kernel computes the same expression per case
// (sor.h), so the result does not depend on the path, the tile shape, the
// kernel or the batch a case is in.  The cells' weights come from a table
// indexed by the flag byte (uniform grids) or per cell (FP32: loaded once
// per launch; FP64: formed once per launch); WM, the launch's weight mode,
// picks the form at compile time.
//
// M sweeps per launch on the tile with its 2M halo (temporal blocking):
// after half-sweep h only the tile plus a ring of 2M-1-h cells is still
// exact, so after 2M half-sweeps the interior (TW x TY) is, and only it is
// stored.  Reads come from buffer src and writes go to dst (ping-pong), so
// tiles never read halos that other tiles are writing.  HBM traffic is one
// read of the unknown, the right side and the flags (or FP32 weights),
// plus the halo, and one write of the unknown per M sweeps.
#pragma once
#include "common.h"
#include "kernels.h"
#include "sor.h"
#include "stages.h"

#include <type_traits>
#include <utility>

namespace iff {

namespace {

template <typename T, int NRW>
struct RegTile {
    T pa[NRW], pb[NRW];  // unknown, slots a (even column) and b (odd column)
    T ra[NRW], rb[NRW];  // right side (FP32: w r once the weights are formed)
    T cyp[NRW], cym[NRW];
    T wa[NRW], wb[NRW];  // the cell's weight om/sa, 0 for a cell the sweep does not update
};

// A wave-uniform value held in scalar registers (the row coefficients are
// the same in every lane; in SGPRs they cost no vector registers and enter
// the multiplies as scalar operands).
__device__ __forceinline__ float uniform(float x)
{
    return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(x)));
}
__device__ __forceinline__ double uniform(double x)
{
    const long long b = __double_as_longlong(x);
    const int lo = __builtin_amdgcn_readfirstlane((int)(b & 0xffffffffLL));
    const int hi = __builtin_amdgcn_readfirstlane((int)(b >> 32));
    return __longlong_as_double(((long long)hi << 32) | (unsigned int)lo);
}

__device__ __forceinline__ int uniform(int x) { return __builtin_amdgcn_readfirstlane(x); }
__device__ __forceinline__ void *uniform_ptr(void *p)
{
    const unsigned long long b = (unsigned long long)p;
    const unsigned lo = __builtin_amdgcn_readfirstlane((unsigned)b);
    const unsigned hi = __builtin_amdgcn_readfirstlane((unsigned)(b >> 32));
    return (void *)(((unsigned long long)hi << 32) | lo);
}

// a if face bit F of flags f is set, else +0: the bit, sign-extended to a
// full mask, ANDed with a's bits (two VALU operations, no compare).
template <typename T, int F>
__device__ __forceinline__ T face_coef(int f, T a)
{
    const int m = __builtin_amdgcn_sbfe(f, __builtin_ctz(F), 1);
    if constexpr (sizeof(T) == 8)
        return __longlong_as_double(__double_as_longlong(a) & (long long)m);
    else
        return __int_as_float(__float_as_int(a) & m);
}

// One cell of a half-sweep, FP32 (the error equation of the mixed path).
// Every cell takes this one branch-free form: the error is zero in every
// non-fluid cell (each solve starts from zero and never updates them), and
// a face is closed exactly when it lies on the domain boundary or next to a
// non-fluid cell, so the metric coefficients (zeroed on boundary faces)
// give the same neighbour sum as the flagged ones.  The closed faces enter
// through the cell's weight w = om / sa (sa over the open faces), formed
// once per launch with wr = w r; w = 0 leaves a non-fluid cell at zero.
// (a1, p1) is the neighbour held by the adjacent lane: the lane shift
// folds into that product (v_mul_f32 with DPP).
__device__ __forceinline__ float reg_cell_w(float pc, float wr, float a1, float p1, float a2, float p2, float pN,
                                            float pS, float cyp, float cym, float w, float c1)
{
    return sor_cell_w(pc, wr, a1, p1, a2, p2, cyp, pN, cym, pS, w, c1);
}

// One cell of a half-sweep, FP64, with the cell's weight w = om / sa formed
// once per launch (w = 0: a cell the sweep keeps).  As in FP32 one branch-free
// form: the tile holds 0 in every cell the sweep keeps, so the metric
// coefficients (zeroed on boundary faces) give the neighbour sum of the
// flagged ones (0 times the neighbour's value across a closed face), and the
// kept cells' own values stay where they are in memory, in both buffers
// (k_faces_rhs).  With the oracle's rule evaluated per cell instead, a row
// holding any such cell took 2.5 times the operations in one dependent chain,
// and every tile waited for the tiles around the body.
__device__ __forceinline__ double reg_cell(double pc, double r, double pE, double pW, double pN, double pS, double cxp,
                                           double cxm, double cyp, double cym, double w, double c1)
{
    const double sum = (cxp * pE + cxm * pW) + (cyp * pN + cym * pS);
    return sor_cell_w64(pc, r, sum, w, c1);
}

// One row's cells of a half-sweep.  c1 = 1 - om; the cells' weights are in R
// (UNI, FP32: K = w ax, the five-operation form with ratio = ay / ax).
template <typename T, int NRW, int Q, int k, bool UNI = false>
__device__ __forceinline__ void reg_row(RegTile<T, NRW> &R, T sv, T nv, T cxpa, T cxma, T cxpb, T cxmb,
                                        T c1, T ratio = (T)0)
{
    constexpr int ks = k > 0 ? k - 1 : 0, kn = k < NRW - 1 ? k + 1 : 0;
    if constexpr ((k & 1) == Q) {
        const T pS = k == 0 ? sv : R.pa[ks];
        const T pN = k == NRW - 1 ? nv : R.pa[kn];
        const T pE = R.pb[k], pW = from_west(R.pb[k]);
        if constexpr (sizeof(T) == 4 && UNI)
            R.pa[k] = sor_cell_u(R.pa[k], R.ra[k], pW, pE, pN, pS, R.wa[k], ratio, c1);
        else if constexpr (sizeof(T) == 4)  // slot a: odd column, west neighbour in lane l-1
            R.pa[k] = reg_cell_w(R.pa[k], R.ra[k], cxma, pW, cxpa, pE, pN, pS, R.cyp[k], R.cym[k], R.wa[k], c1);
        else
            R.pa[k] = reg_cell(R.pa[k], R.ra[k], pE, pW, pN, pS, cxpa, cxma, R.cyp[k], R.cym[k], R.wa[k], c1);
    } else {
        const T pS = k == 0 ? sv : R.pb[ks];
        const T pN = k == NRW - 1 ? nv : R.pb[kn];
        const T pE = from_east(R.pa[k]), pW = R.pa[k];
        if constexpr (sizeof(T) == 4 && UNI)
            R.pb[k] = sor_cell_u(R.pb[k], R.rb[k], pW, pE, pN, pS, R.wb[k], ratio, c1);
        else if constexpr (sizeof(T) == 4)  // slot b: even column, east neighbour in lane l+1
            R.pb[k] = reg_cell_w(R.pb[k], R.rb[k], cxpb, pE, cxmb, pW, pN, pS, R.cyp[k], R.cym[k], R.wb[k], c1);
        else
            R.pb[k] = reg_cell(R.pb[k], R.rb[k], pE, pW, pN, pS, cxpb, cxmb, R.cyp[k], R.cym[k], R.wb[k], c1);
    }
}

// The slot of row k that half-sweep type Q updates.
template <typename T, int NRW, int Q, int k>
__device__ __forceinline__ T updated(const RegTile<T, NRW> &R)
{
    return (k & 1) == Q ? R.pa[k] : R.pb[k];
}

// A wave's rows in a half-sweep (row<k>() updates row k), in the order that
// keeps the exchange off the critical path: the first half of the rows
// between (they hide the LDS read of the neighbour rows), the first and the
// last row, their publication, the other rows (they hide its LDS write).  Left
// to itself the compiler moves the rows of the next half-sweep up before the
// publication, and every wave of the block waits for it.
template <int NRW, typename ROW, typename PUB>
__device__ __forceinline__ void fast_rows(ROW &&row, PUB &&publish)
{
    constexpr int A = (NRW - 1) / 2;  // rows 1 .. A before, A + 1 .. NRW - 2 after
    [&]<int... K>(std::integer_sequence<int, K...>) {
        (row.template operator()<K + 1>(), ...);
    }(std::make_integer_sequence<int, (A < NRW - 2 ? A : NRW - 2)>{});
    __builtin_amdgcn_sched_barrier(0);
    row.template operator()<0>();
    row.template operator()<NRW - 1>();
    publish();
    __builtin_amdgcn_sched_barrier(0);
    [&]<int... K>(std::integer_sequence<int, K...>) {
        (row.template operator()<K + A + 1>(), ...);
    }(std::make_integer_sequence<int, (NRW - 2 > A ? NRW - 2 - A : 0)>{});
    __builtin_amdgcn_sched_barrier(0);
}

// Synchronisation of the persistent sweep.  Between stages a tile's border
// strips go to its neighbours through strip buffers that the readers poll
// (k_rbsor_reg); every tile has a stage counter (flags[t]), which counts the
// stages over all launches, so that all counters of a case agree when a launch
// starts; the FP64 solve's checks wait for them.  Strips are written and read
// at device scope (sc1: write-through, and loads that miss in the per-XCD
// L2), so no cache flush is needed.  All waits are bounded: past
// bar->timeout ticks of the 100 MHz real-time counter bar->err is set, every
// later wait ends soon and every block stops at its next stage boundary, so
// the kernel always ends; the host checks err after the step.
constexpr unsigned kRsrc3 = 0x00020000;              // buffer resource word 3 (gfx9)

// wait_neighbours (sor.h) for all n tiles of a case, by all threads of the block (the
// answer is this wave's)
__device__ __forceinline__ bool wait_all(const unsigned *flags, int n, unsigned target, GridBar *bar)
{
    const unsigned long long t0 = __builtin_amdgcn_s_memrealtime();
    const unsigned long long tmo = bar->timeout;
    while (true) {
        bool ok = true;
        for (int i = threadIdx.x; i < n; i += blockDim.x)
            ok = ok && (int)(__hip_atomic_load(&flags[i], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) - target) >= 0;
        const unsigned err = __hip_atomic_load(&bar->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (__any(err != 0)) return true;
        if (__all(ok)) return false;
        if (__builtin_amdgcn_s_memrealtime() - t0 > tmo) {
            __hip_atomic_store(&bar->err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            return true;
        }
        __builtin_amdgcn_s_sleep(1);
    }
}

}  // namespace

// PERS: one launch runs the chunk's K sweeps as stages of M
// sweeps.  The tile stays in registers; after each stage a block sends the
// border strips (depth 2M) of its stored region and takes its halo ring from its
// neighbours' strips.  The last stage leaves the whole stored region where
// launches of M sweeps leave it (FP32 e[n & 1], FP64 p[(ppe_base + n) & 1] after
// n of them), so the checks read the same buffer either way.
//
// The second launch bound holds the FP32 per-stage 128 x 128 blocks (16
// waves x 8 rows) at 8 waves per SIMD, i.e. 64 VGPRs and two blocks per CU:
// left free, some of them take a few more registers and run at one block
// per CU, a third slower.
template <typename T, int M, int NW, int NRW, bool PERS, int WM>
constexpr bool two_per_cu = sizeof(T) == 4 && NW == 16 &&
                            (PERS ? M <= 8 && (WM == 1 || (WM == 0 && NRW <= 6)) : NRW == 8 && WM != 2);

// PERS: neighbours poll the strips themselves; where the registers for it
// are not there (two blocks per CU, FP64 from 5 rows a wave: spills cost up to
// 1.9 us per sweep), each tile's stage counter (flags) tells them
template <typename T, int M, int NW, int NRW, int WM>
constexpr bool polls = NW == 16 && (sizeof(T) == 4 ? !two_per_cu<T, M, NW, NRW, true, WM> : NRW <= 4);

template <typename T, int M, int NW, int NRW, bool PERS, int WM>
__global__ __launch_bounds__(64 * NW, (two_per_cu<T, M, NW, NRW, PERS, WM>) ? 8 : 1)
void k_rbsor_reg(const CaseDev *cs, const int2 *tiles, int ntiles, int ntiles_pad, int s, int K, PersArgs pa)
{
    constexpr bool kPoll = PERS && polls<T, M, NW, NRW, WM>;
    constexpr int H = 2 * M;
    constexpr int TW = 128 - 2 * H;   // stored columns per tile
    constexpr int TY = NW * NRW - 2 * H;  // stored rows per tile
    static_assert(TY > 0 && NRW <= 32, "tile shape");
    using V2 = typename VecT<T, 2>::type;
    // [parity][1 + wave][first row, last row][lane]; slots 0 and NW + 1 stay
    // zero (the rows beyond the first and last wave), so every wave reads its
    // neighbour rows unconditionally.  A half-sweep reads only neighbours of
    // the other colour, which the half-sweep before it updated: one slot per
    // lane and row is exchanged, the one just updated.  (Exchanging both
    // moved twice the bytes: 32 KB per half-sweep of a 16-wave FP32 block,
    // 256 LDS cycles, where three rows of updates take about 160.)
    __shared__ T xch[2][NW + 2][2][64];
    const int t = tile_of_block(ntiles_pad);
    GridBar *const bar = pa.bar;
    unsigned *const flags = pa.flags;
    const bool solve = PERS && sizeof(T) == 8 && pa.nchunk > 0;
    if constexpr (PERS) {
        bool run = false;
        if (t < ntiles) {
            const CaseDev &cr = cs[tiles[t].x];
            const Ctrl *cc = cr.ctrl;
            run = cr.ppe_solver == IF_PPE_RBSOR && cc->active && !cc->ppe_done && cr.ppe_itermax > cc->ppe_sweeps;
        }
        if (!run) {  // whole workgroup, every tile of the case alike
            if (solve && t < ntiles && tiles[t].y == 0 && threadIdx.x == 0) {
                const Ctrl *cc = cs[tiles[t].x].ctrl;
                check_case(pa.ncase, false, cc->active && !cc->ad_done, bar);
            }
            return;
        }
    } else {
        if (t >= ntiles) return;  // whole workgroup
    }
    // wave-uniform throughout, and marked so: loop counts, row tests and field
    // addresses then live in scalar registers
    const int2 tl = make_int2(uniform(tiles[t].x), uniform(tiles[t].y));
    const CaseDev &c = cs[tl.x];
    const Ctrl *ct = c.ctrl;
    if (c.ppe_solver != IF_PPE_RBSOR || !ct->active || ct->ppe_done) return;  // (PERS: never taken)
    int kexec = uniform(c.ppe_itermax - ct->ppe_sweeps);
    if (kexec > K) kexec = K;
    if (s >= kexec) return;  // (PERS: s = 0 < kexec)
    int meff = kexec - s;
    if (meff > M) meff = M;
    const int nst = 2 * meff;  // half-sweeps of this launch
    const int L = s / M;       // launch index inside the chunk

    const int nx = uniform(c.nx), ny = uniform(c.ny), P = uniform(c.P);
    const T *src;
    T *dst;
    const T *rhs;
    const T *cxp_, *cxm_, *cyp_, *cym_;
    bool zero_src = false;
    T om;
    if constexpr (sizeof(T) == 8) {
        src = c.p[(ct->ppe_base + L) & 1];
        dst = c.p[(ct->ppe_base + L + 1) & 1];
        rhs = c.rhs;
        cxp_ = c.x.cp; cxm_ = c.x.cm; cyp_ = c.y.cp; cym_ = c.y.cm;
        om = c.omega;
    } else {
        src = c.e[L & 1];
        dst = c.e[(L + 1) & 1];
        zero_src = (L == 0);
        rhs = c.r32;
        cxp_ = c.xf.cp; cxm_ = c.xf.cm; cyp_ = c.yf.cp; cym_ = c.yf.cm;
        om = c.omega_f;
    }
    const int ntxs = (nx - 2 + TW - 1) / TW;
    const int tx = tl.y % ntxs, ty = tl.y / ntxs;
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int c0 = 1 + tx * TW - H;            // first tile column
    const int jt0 = 1 + ty * TY - H + w * NRW;  // first row of this wave
    const int ga = c0 + 2 * lane;               // slot a column; slot b is ga + 1
    const bool ina = ga >= 1 && ga <= nx - 2;
    const bool inb = ga + 1 >= 1 && ga + 1 <= nx - 2;
    // x coefficients of the fast path: zero on the domain boundary faces
    // and outside the interior.  A slot outside the interior has weight 0:
    // its value stays finite, is never stored and is only ever multiplied
    // by the zero coefficient of a boundary face.
    const T cxpa = (ina && ga != nx - 2) ? G(cxp_)[ga] : (T)0;
    const T cxma = (ina && ga != 1) ? G(cxm_)[ga] : (T)0;
    const T cxpb = (inb && ga + 1 != nx - 2) ? G(cxp_)[ga + 1] : (T)0;
    const T cxmb = (inb && ga + 1 != 1) ? G(cxm_)[ga + 1] : (T)0;
    // WM, the weight mode of the launch (kernels rather than runtime
    // branches, which would hold both forms' registers at once):
    //   1: every case has a weight table (wtab / wtab64): the weights are
    //      looked up by flag pattern instead of loaded per cell (FP32: w32)
    //      or formed with a division on every launch (FP64); FP32 takes the
    //      five-operation form (every such case is uni);
    //   0: per-cell weights, the general form;
    //   2 (FP32): per-cell weights, the form each case's uni flag picks (a
    //      batch mixing uniform and stretched grids).
    RegTile<T, NRW> R;
    int lf[NRW];  // FP64: flags, slot a in bits 0-7, slot b in bits 8-15
    // FP32: the cells' weights om / sa (k_weights32: once for a resident set,
    // every step with moving bodies),
    // or on a grid with one value per coefficient the weight of the cell's
    // flag pattern: lane q holds the table's entry q, and each cell reads
    // its entry across the wave (ds_bpermute)
    const float *w32 = c.w32;
    static_assert(WM == 0 || WM == 1 || (WM == 2 && sizeof(T) == 4), "weight mode");
    constexpr bool wuni = WM == 1;
    // FP32 with one coefficient value per axis: the five-operation update,
    // K = w ax held in place of w
    const bool uni = sizeof(T) == 4 && (WM == 1 || (WM == 2 && c.uni));
    const T uax = sizeof(T) == 4 ? (T)c.uax : (T)0, uratio = sizeof(T) == 4 ? (T)c.uratio : (T)0;
    int wtv = 0, wtv_hi = 0;  // FP32: K = w ax; FP64: w (low and high halves)
    if constexpr (wuni) {
        if constexpr (sizeof(T) == 4) {
            wtv = __float_as_int(G(c.wtab)[lane]);
        } else {
            const double d = G(c.wtab64)[lane];
            wtv = __double2loint(d);
            wtv_hi = __double2hiint(d);
        }
    }
    // Loads.  A tile lying inside the interior (the common case) loads
    // every row with aligned 8-byte vectors and no per-lane tests.
    const bool tile_in = c0 >= 1 && c0 + 127 <= nx - 2 && jt0 >= 1 && jt0 + NRW - 1 <= ny - 2;
    if (tile_in) {
#pragma unroll
        for (int k = 0; k < NRW; k++) {
            const size_t ro = (size_t)(jt0 + k) * P;  // wave-uniform row offset
            const V2 pv = zero_src ? V2{(T)0, (T)0} : gload_vec<V2>(src + ro + ga);
            const V2 rv = gload_vec<V2>(rhs + ro + ga);
            R.pa[k] = pv[0];
            R.pb[k] = pv[1];
            R.ra[k] = rv[0];
            R.rb[k] = rv[1];
            if constexpr (sizeof(T) == 4) {
                if constexpr (wuni) {
                    const u8x2 fb = gload_vec<u8x2>(c.flags + ro + ga);
                    lf[k] = (int)fb[0] | ((int)fb[1] << 8);
                } else {
                    const V2 wv = gload_vec<V2>(w32 + ro + ga);
                    R.wa[k] = wv[0];
                    R.wb[k] = wv[1];
                    lf[k] = 0;
                }
            } else {
                const u8x2 fb = gload_vec<u8x2>(c.flags + ro + ga);
                lf[k] = (int)fb[0] | ((int)fb[1] << 8);
            }
        }
    } else {
#pragma unroll
        for (int k = 0; k < NRW; k++) {
            const int gj = jt0 + k;
            const bool rowin = gj >= 0 && gj < ny;
            const bool rowint = gj >= 1 && gj <= ny - 2;
            T a = (T)0, b = (T)0, x = (T)0, y = (T)0, wa = (T)0, wb = (T)0;
            int f = 0;
            if (rowin) {
                const size_t o = (size_t)gj * P + ga;
                if (!zero_src) {
                    if (ga >= 0 && ga + 1 < nx) {
                        const V2 v = gload_vec<V2>(src + o);
                        a = v[0];
                        b = v[1];
                    } else {
                        if (ga >= 0 && ga < nx) a = G(src)[o];
                        if (ga + 1 >= 0 && ga + 1 < nx) b = G(src)[o + 1];
                    }
                }
                if (rowint) {
                    if (ina && inb) {
                        const V2 v = gload_vec<V2>(rhs + o);
                        x = v[0];
                        y = v[1];
                        if (sizeof(T) == 4 && !wuni) {
                            const V2 wv = gload_vec<V2>(w32 + o);
                            wa = wv[0];
                            wb = wv[1];
                        } else {
                            const u8x2 fb = gload_vec<u8x2>(c.flags + o);
                            f = (int)fb[0] | ((int)fb[1] << 8);
                        }
                    } else {
                        if (ina) {
                            x = G(rhs)[o];
                            if (sizeof(T) == 4 && !wuni)
                                wa = G(w32)[o];
                            else
                                f = G(c.flags)[o];
                        }
                        if (inb) {
                            y = G(rhs)[o + 1];
                            if (sizeof(T) == 4 && !wuni)
                                wb = G(w32)[o + 1];
                            else
                                f |= (int)G(c.flags)[o + 1] << 8;
                        }
                    }
                }
            }
            R.pa[k] = a;
            R.pb[k] = b;
            R.ra[k] = x;
            R.rb[k] = y;
            if constexpr (sizeof(T) == 4) {
                R.wa[k] = wa;
                R.wb[k] = wb;
            }
            lf[k] = f;
        }
    }

    // Per-row coefficients and the cells' weights (0 for a cell the sweep
    // keeps: outside the interior, not fluid, or without an open face; its
    // value in the tile is 0).  FP32 weights come from k_weights32; wr = w r
    // is formed here.
    // FP64, solve: the cells' open faces for the residual (flag bits 0-5 of
    // slot a in bits 0-5, of slot b in 6-11, two rows a register)
    unsigned of[PERS && sizeof(T) == 8 ? (NRW + 1) / 2 : 1] = {};
    unsigned smask = 0;  // FP64: rows holding an interior cell that is kept
#pragma unroll
    for (int k = 0; k < NRW; k++) {
        const int gj = jt0 + k;
        const bool rowint = gj >= 1 && gj <= ny - 2;
        const T yp = (rowint && gj != ny - 2) ? G(cyp_)[gj] : (T)0;
        const T ym = (rowint && gj != 1) ? G(cym_)[gj] : (T)0;
        R.cyp[k] = uniform(yp);
        R.cym[k] = uniform(ym);
        if constexpr (sizeof(T) == 4) {
            // the five-operation form holds K = w ax in place of w; r32
            // holds r' = r / ax for such a case, so K r' stands for w r
            if constexpr (wuni) {  // a cell outside the interior has flags 0: weight 0
                R.wa[k] = __int_as_float(__builtin_amdgcn_ds_bpermute((lf[k] & 63) << 2, wtv));
                R.wb[k] = __int_as_float(__builtin_amdgcn_ds_bpermute(((lf[k] >> 8) & 63) << 2, wtv));
            } else if (uni) {
                R.wa[k] = R.wa[k] * uax;
                R.wb[k] = R.wb[k] * uax;
            }
            R.ra[k] = R.wa[k] * R.ra[k];
            R.rb[k] = R.wb[k] * R.rb[k];
        } else {
            // the weight om / sa over the open faces.  With a table: the entry
            // of the cell's flag pattern, formed with the same expression (a
            // cell outside the interior has flags 0)
            const int f = lf[k], fa = f & 0xff, fb = f >> 8;
            if constexpr (wuni) {
                auto look = [&](int q) {
                    const int i = (q & 63) << 2;
                    return __hiloint2double(__builtin_amdgcn_ds_bpermute(i, wtv_hi),
                                            __builtin_amdgcn_ds_bpermute(i, wtv));
                };
                R.wa[k] = look(fa);
                R.wb[k] = look(fb);
            } else {
                const T sa_a = (face_coef<T, F_OPEN_E>(fa, cxpa) + face_coef<T, F_OPEN_W>(fa, cxma)) +
                               (face_coef<T, F_OPEN_N>(fa, yp) + face_coef<T, F_OPEN_S>(fa, ym));
                const T sa_b = (face_coef<T, F_OPEN_E>(fb, cxpb) + face_coef<T, F_OPEN_W>(fb, cxmb)) +
                               (face_coef<T, F_OPEN_N>(fb, yp) + face_coef<T, F_OPEN_S>(fb, ym));
                R.wa[k] = (rowint && (fa & F_FLUID) && sa_a != (T)0) ? sor_weight64(sa_a, om) : (T)0;
                R.wb[k] = (rowint && (fb & F_FLUID) && sa_b != (T)0) ? sor_weight64(sa_b, om) : (T)0;
            }
            if constexpr (PERS) of[k / 2] |= (unsigned)((fa & 63) | (fb & 63) << 6) << (16 * (k & 1));
            if (rowint && __any((ina && R.wa[k] == (T)0) || (inb && R.wb[k] == (T)0))) smask |= 1u << k;
            R.pa[k] = R.wa[k] != (T)0 ? R.pa[k] : (T)0;
            R.pb[k] = R.wb[k] != (T)0 ? R.pb[k] : (T)0;
        }
    }
    const T c1 = (T)1 - om;

    const int Z = (c0 + jt0) & 1;  // parity of slot a in the wave's first row
    // Half-sweep h has colour h & 1, and slot a of row k has parity Z + k,
    // so rows with (k & 1) == Q update slot a where Q = (Z ^ h) & 1.  Within
    // a half-sweep every updated cell reads only cells of the other colour,
    // so the row order (fast_rows) changes no result.
    if (w == 0) {
#pragma unroll
        for (int b = 0; b < 2; b++)
#pragma unroll
            for (int r = 0; r < 2; r++) {
                xch[b][0][r][lane] = (T)0;
                xch[b][NW + 1][r][lane] = (T)0;
            }
    }
    // Tile row rr holds the value of the full sweep after half-sweep h only
    // while rr > h and NW * NRW - 1 - rr > h: each half-sweep loses one
    // row at each edge of the tile.  A wave none of whose rows can still
    // be valid (all of them in the halo, which is H = 2M deep) skips the
    // update and the publish and only joins the barrier; the rows next to
    // it read its stale values only when they are no longer valid either.
    // That frees issue slots for the other workgroup on the CU; the
    // persistent form (one workgroup per CU, every wave waiting at the
    // barrier for the slowest SIMD) runs every wave.
    auto live = [&](int h) { return PERS || (w * NRW + NRW - 1 > h && NW * NRW - 1 - w * NRW > h); };
    // publish the first and last row's slot that a half-sweep of type Q updates
    auto publish = [&]<int Q>(int b) {
        xch[b][w + 1][0][lane] = updated<T, NRW, Q, 0>(R);
        xch[b][w + 1][1][lane] = updated<T, NRW, Q, NRW - 1>(R);
    };
    auto half = [&]<int Q, bool UNI>(int h) {
        const int b = h & 1;
        if (live(h)) {
            const T sv = xch[b][w][1][lane], nv = xch[b][w + 2][0][lane];
            fast_rows<NRW>(
                [&]<int k>() {
                    reg_row<T, NRW, Q, k, UNI>(R, sv, nv, cxpa, cxma, cxpb, cxmb, c1, uratio);
                },
                [&]() { publish.template operator()<Q>(b ^ 1); });
        }
        __syncthreads();
    };
    // nst is even: the half-sweeps run in pairs whose colour order is fixed
    // per wave, so each loop body is straight-line code
    auto pairs = [&]<bool UNI>(int n, auto &&after) {
        if (Z == 0)
            publish.template operator()<1>(0);
        else
            publish.template operator()<0>(0);
        __syncthreads();
        after();
        if (Z == 0) {
            for (int h = 0; h < n; h += 2) {
                half.template operator()<0, UNI>(h);
                half.template operator()<1, UNI>(h + 1);
            }
        } else {
            for (int h = 0; h < n; h += 2) {
                half.template operator()<1, UNI>(h);
                half.template operator()<0, UNI>(h + 1);
            }
        }
    };
    // n half-sweeps (n even); after() runs once every wave of the block is here
    auto sweeps = [&](int n, auto &&after) {
        if constexpr (WM == 2) {
            if (uni)
                pairs.template operator()<true>(n, after);
            else
                pairs.template operator()<false>(n, after);
        } else {
            pairs.template operator()<sizeof(T) == 4 && WM == 1>(n, after);
        }
    };
    // store the stored region of the tile (rows H .. H+TY-1, columns H ..
    // H+TW-1)
    auto store = [&](T *out) {
        if (lane >= H / 2 && lane < 64 - H / 2) {
#pragma unroll
            for (int k = 0; k < NRW; k++) {
                const int rr = w * NRW + k;
                const int gj = jt0 + k;
                if (rr < H || rr >= H + TY || gj > ny - 2) continue;
                T *row = out + (size_t)gj * P;  // wave-uniform
                if (sizeof(T) == 8 && ((smask >> k) & 1u)) {  // kept cells are not written
                    if (R.wa[k] != (T)0) GW(row)[ga] = R.pa[k];
                    if (R.wb[k] != (T)0) GW(row)[ga + 1] = R.pb[k];
                } else if (ga + 1 <= nx - 2)
                    gstore_vec<V2>(row + ga, V2{R.pa[k], R.pb[k]});
                else if (ga <= nx - 2)
                    GW(row)[ga] = R.pa[k];
            }
        }
    };
    if constexpr (PERS) {
        using U2 = unsigned __attribute__((ext_vector_type(2)));
        using U4 = unsigned __attribute__((ext_vector_type(4)));
        // A tile without neighbours needs no stages: no halo of it is ever
        // read, so it runs the whole chunk at once, and leaves its output in
        // the last stage's buffer
        const int ntys = (ny - 2 + TY - 1) / TY;
        const bool alone = ntxs * ntys == 1;
        const unsigned f0 = __hip_atomic_load(&flags[t], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        // the tiles of the case that this one's halo reaches into (a lane of
        // wave 0 each): the next columns of tiles, and RY rows of them where
        // the tile is lower than its halo
        constexpr int RY = (H + TY - 1) / TY, NB = 3 * (2 * RY + 1) - 1;
        static_assert(TW >= H && NB < 64, "halo reach");
        int nb = -1;
        if (!kPoll && w == 0 && lane < NB) {
            const int d = lane < NB / 2 ? lane : lane + 1;  // without the centre
            const int qx = tx + d % 3 - 1, qy = ty + d / 3 - RY;
            if (qx >= 0 && qx < ntxs && qy >= 0 && qy < ntys) nb = t - tl.y + qy * ntxs + qx;
        }
        const int nrec = P * ny * (int)sizeof(T);  // bytes of a field
        // The wave's rows, as wave-uniform masks: stored rows in the domain,
        // those of them in the top and bottom strips, halo rows in the domain
        unsigned m_st = 0, m_strip = 0, m_halo = 0;
#pragma unroll
        for (int k = 0; k < NRW; k++) {
            const int rr = w * NRW + k, gj = jt0 + k;
            const bool st = rr >= H && rr < H + TY;
            if (gj < 1 || gj > ny - 2) continue;
            if (st) m_st |= 1u << k;
            if (st && !(rr >= 2 * H && rr < TY)) m_strip |= 1u << k;
            if (!st) m_halo |= 1u << k;
        }
        // Buffer offsets: the lane's column in the vector offset, the row
        // (wave-uniform) in the scalar offset.  Accesses are not masked: a lane
        // that stores or loads nothing has an offset past every field, which the
        // buffer's bounds check drops.  An exec mask and its branches per row
        // made a stage's stores and loads about 600 instructions a wave.
        constexpr int kDrop = 0x7fffff00;
        const bool stl = lane >= H / 2 && lane < 64 - H / 2;  // stored lanes
        // Offsets and lane masks are formed from an opaque copy of the column
        // where they are used, and the rows' masks made opaque there: held over
        // the sweeps they do not fit in the registers.
        auto column = [&]() {
            int q = ga;
            asm volatile("" : "+v"(q));
            return q;
        };
        auto opaque = [](unsigned &a, unsigned &b) {
            asm volatile("" : "+v"(a), "+v"(b));
            a = (unsigned)uniform((int)a);
            b = (unsigned)uniform((int)b);
        };
        // the launch reads its first values from buf0 and leaves its result in
        // one of the two
        void *buf0, *buf1;
        if constexpr (sizeof(T) == 8) {
            buf0 = c.p[ct->ppe_base & 1];
            buf1 = c.p[(ct->ppe_base + 1) & 1];
        } else {
            buf0 = c.e[0];
            buf1 = c.e[1];
        }
        // the descriptors are built from wave-uniform (readfirstlane)
        // pointers: held in scalar registers, with no per-lane loop around
        // the buffer accesses
        const __amdgpu_buffer_rsrc_t rs0 = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(buf0), 0, nrec, kRsrc3);
        const __amdgpu_buffer_rsrc_t rs1 = __builtin_amdgcn_make_buffer_rsrc(uniform_ptr(buf1), 0, nrec, kRsrc3);
        // Solve (FP64, pa.nchunk > 0): the launch runs chunks of K sweeps until
        // the residual of the case passes its stopping rule, it runs out of
        // sweeps, or pa.nchunk are done.  A chunk's last stage does at most
        // M - 1 sweeps, so that a ring of exact cells is left around the
        // stored region and the tile has its residual from its registers;
        // the maxima meet at the stage's flags, waited for by the case's tiles all
        // together.  A launch for each chunk and for each check cost 28 us
        // per 10 sweeps of a 256^2 grid, of which 11 were sweeps.
        Ctrl *const ctw = c.ctrl;
        const int left = uniform(c.ppe_itermax - ct->ppe_sweeps);
        const int base = uniform(ct->ppe_base);
        // the residual's maximum over the stored cells, from the tile after a
        // stage's last sweep: k_ppe_resid's expression and operand order, with
        // the open faces' coefficients (a kept cell is held as 0, and its
        // faces are closed).  xch[1 - c] holds the neighbour rows' cells of
        // colour c.
        auto residual = [&]() __attribute__((always_inline)) {
            double m = 0.0;
            if constexpr (sizeof(T) == 8) {
                const int cn = (Z + NRW - 1) & 1;
                const T sa = xch[Z][w][1][lane], sb = xch[1 - Z][w][1][lane];
                const T na = xch[cn][w + 2][0][lane], nb_ = xch[1 - cn][w + 2][0][lane];
                auto cell = [&](unsigned f, T pc, T r, T pE, T pW, T pN, T pS, T cxp, T cxm, T cyp, T cym) {
                    const T aE = face_coef<T, F_OPEN_E>((int)f, cxp), aW = face_coef<T, F_OPEN_W>((int)f, cxm);
                    const T aN = face_coef<T, F_OPEN_N>((int)f, cyp), aS = face_coef<T, F_OPEN_S>((int)f, cym);
                    const T ap = -((aE + aW) + (aN + aS));
                    const T sum = (aE * pE + aW * pW) + (aN * pN + aS * pS);
                    return absinf(r - (ap * pc + sum));
                };
#pragma unroll
                for (int k = 0; k < NRW; k++) {
                    if (!((m_st >> k) & 1u)) continue;
                    // (opaque: the coefficients of all rows, formed once before
                    // the loop, would not fit in the registers)
                    asm volatile("" : "+v"(of[k / 2]));
                    const unsigned f = of[k / 2] >> (16 * (k & 1));
                    const T pSa = k == 0 ? sa : R.pa[k > 0 ? k - 1 : 0], pSb = k == 0 ? sb : R.pb[k > 0 ? k - 1 : 0];
                    const T pNa = k == NRW - 1 ? na : R.pa[k < NRW - 1 ? k + 1 : k];
                    const T pNb = k == NRW - 1 ? nb_ : R.pb[k < NRW - 1 ? k + 1 : k];
                    const T ma = cell(f & 63, R.pa[k], R.ra[k], R.pb[k], from_west(R.pb[k]), pNa, pSa, cxpa, cxma,
                                      R.cyp[k], R.cym[k]);
                    const T mb = cell(f >> 6 & 63, R.pb[k], R.rb[k], from_east(R.pa[k]), R.pa[k], pNb, pSb, cxpb, cxmb,
                                      R.cyp[k], R.cym[k]);
                    if (stl && R.wa[k] != (T)0) m = fmax(m, ma);
                    if (stl && R.wb[k] != (T)0) m = fmax(m, mb);
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            return wave_max(m);
        };
        // output at device scope: the border strips, or (the end of the case) the
        // whole stored region
        auto put = [&](const __amdgpu_buffer_rsrc_t ro, bool whole) __attribute__((always_inline)) {
            const int q = column(), ln = (q - c0) >> 1;
            const bool st = ln >= H / 2 && ln < 64 - H / 2;
            const int vo_all = st && q + 1 <= nx - 2 ? q * (int)sizeof(T) : kDrop;
            const int vo_side = ln < H || ln >= 64 - H ? vo_all : kDrop;
            const unsigned m_all = whole ? m_st : m_strip;
            // a last interior column without a partner (odd widths)
            const int vo_one = st && q == nx - 2 ? q * (int)sizeof(T) : kDrop;
            const bool one = __any(st && q == nx - 2);
#pragma unroll
            for (int k = 0; k < NRW; k++) {
                const int srow = (jt0 + k) * P * (int)sizeof(T);  // uniform: scalar offset
                if (!((m_st >> k) & 1u)) continue;
                const int vo = ((m_all >> k) & 1u) ? vo_all : vo_side;
                if constexpr (sizeof(T) == 4) {
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, V2{R.pa[k], R.pb[k]}), ro, vo, srow,
                                                          kDev);
                } else if ((smask >> k) & 1u) {  // kept cells are not written
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, R.pa[k]), ro,
                                                          R.wa[k] != (T)0 ? vo : kDrop, srow, kDev);
                    __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, R.pb[k]), ro,
                                                          R.wb[k] != (T)0 ? vo : kDrop, srow + 8, kDev);
                } else {
                    __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(U4, V2{R.pa[k], R.pb[k]}), ro, vo, srow,
                                                           kDev);
                }
            }
            if (one) {  // (a right edge tile: its last column is in the right strip)
#pragma unroll
                for (int k = 0; k < NRW; k++) {
                    const int srow = (jt0 + k) * P * (int)sizeof(T);
                    if (!((m_st >> k) & 1u)) continue;
                    if constexpr (sizeof(T) == 4)
                        __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(R.pa[k]), ro, vo_one, srow, kDev);
                    else
                        __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(U2, R.pa[k]), ro,
                                                              R.wa[k] != (T)0 ? vo_one : kDrop, srow, kDev);
                }
            }
        };
        // The exchange by polling.  A stage's strips go to one of three buffers
        // laid out as the field, stage g (counted over launches) to buffer
        // strip_of(g), and a reader polls the cells themselves: a word of all ones,
        // which no value has (kHole, a NaN that cap() maps to its neighbour),
        // means not yet written.  So a stage costs a store, its way to the reader
        // and the reader's load; with a counter behind the strips it is a round
        // trip and two barriers more.  FP32 256^2 0.60 -> 0.56 us per sweep,
        // 611^2 0.71 -> 0.64, stretched 2048 x 1024 1.32 -> 1.19; FP64 800^2
        // 1.55 -> 1.27.
        // Buffer strip_of(g + 1) is emptied during stage g: what it holds, stage
        // g - 2, has been read, since the neighbours' stage g - 1, sent after
        // that, has arrived in every wave of this block; and it is empty
        // before stage g is sent, so a neighbour that has stage g finds
        // it empty or stage g + 1 in it.
        constexpr unsigned kHole = 0xffffffffu;
        auto cap = [](unsigned x) { return x < kHole ? x : kHole - 1u; };
        auto strip_buf = [&](unsigned g) {
            return __builtin_amdgcn_make_buffer_rsrc(uniform_ptr((char *)c.xb + (size_t)strip_of(g) * (size_t)nrec), 0, nrec,
                                                     kRsrc3);
        };
        auto send = [&](const __amdgpu_buffer_rsrc_t xo, auto empty) __attribute__((always_inline)) {
            // the strips, in column pairs: every stored column in the top and
            // bottom strips' rows, else the left and right strips' columns
            unsigned ms = m_st, mp = m_strip;
            opaque(ms, mp);
            const int q = column(), ln = (q - c0) >> 1;
            const bool on = q >= 1 && q <= nx - 2 && ln >= H / 2 && ln < 64 - H / 2;
            const int vs_all = on ? q * (int)sizeof(T) : kDrop;
            const int vs_side = on && (ln < H || ln >= 64 - H) ? q * (int)sizeof(T) : kDrop;
#pragma unroll
            for (int k = 0; k < NRW; k++) {
                const int srow = (jt0 + k) * P * (int)sizeof(T);
                if (!((ms >> k) & 1u)) continue;
                const int vo = ((mp >> k) & 1u) ? vs_all : vs_side;
                if constexpr (sizeof(T) == 4) {
                    U2 v = {kHole, kHole};
                    if constexpr (!decltype(empty)::value)
                        v = U2{cap(__float_as_uint(R.pa[k])), __float_as_uint(R.pb[k])};
                    __builtin_amdgcn_raw_buffer_store_b64(v, xo, vo, srow, kDev);
                } else {  // (two atoms of 8 bytes)
                    U4 v = {kHole, kHole, kHole, kHole};
                    if constexpr (!decltype(empty)::value) {
                        const U2 a = __builtin_bit_cast(U2, R.pa[k]), b = __builtin_bit_cast(U2, R.pb[k]);
                        v = U4{a[0], cap(a[1]), b[0], cap(b[1])};
                    }
                    __builtin_amdgcn_raw_buffer_store_b128(v, xo, vo, srow, kDev);
                }
            }
        };
        using XV = std::conditional_t<sizeof(T) == 4, U2, U4>;
        // this wave's part of the halo ring: the cells of the tile outside its
        // stored region that lie in the domain's interior.  true: give up.
        // Four rows at once, without branches: their loads are in flight
        // together.  (A lane that takes nothing, and every lane of a row outside
        // the domain, has an offset past the field: 0.)
        auto receive = [&](const __amdgpu_buffer_rsrc_t xi) __attribute__((always_inline)) {
            constexpr int kGroup = NRW <= 6 ? NRW : 4;
            unsigned long long t0 = 0;
            for (unsigned tries = 1;; tries++) {
                asm volatile("" ::: "memory");  // (load again)
                bool hole = false;
                unsigned mh = m_halo, ms = m_st;
                opaque(mh, ms);
                const int q = column(), ln = (q - c0) >> 1;
                const bool h_all = q >= 1 && q <= nx - 2, h_side = h_all && (ln < H / 2 || ln >= 64 - H / 2);
                const int vh_all = h_all ? q * (int)sizeof(T) : kDrop, vh_side = h_side ? q * (int)sizeof(T) : kDrop;
#pragma unroll
                for (int k0 = 0; k0 < NRW; k0 += kGroup) {
                    XV x[kGroup];
#pragma unroll
                    for (int r = 0; r < kGroup && k0 + r < NRW; r++) {
                        const int k = k0 + r, srow = strip_row(jt0 + k, ny) * P * (int)sizeof(T);
                        const int vo = (mh >> k) & 1u ? vh_all : (ms >> k) & 1u ? vh_side : kDrop;
                        if constexpr (sizeof(T) == 4)
                            x[r] = __builtin_amdgcn_raw_buffer_load_b64(xi, vo, srow, kDev);
                        else
                            x[r] = __builtin_amdgcn_raw_buffer_load_b128(xi, vo, srow, kDev);
                    }
#pragma unroll
                    for (int r = 0; r < kGroup && k0 + r < NRW; r++) {
                        const int k = k0 + r;
                        const bool mine = (mh >> k) & 1u ? h_all : (ms >> k) & 1u && h_side;
                        const V2 v = __builtin_bit_cast(V2, x[r]);
                        if constexpr (sizeof(T) == 4) {
                            hole = hole || x[r][0] == kHole;
                            R.pa[k] = mine ? v[0] : R.pa[k];
                            R.pb[k] = mine ? v[1] : R.pb[k];
                        } else {  // kept cells stay 0
                            hole = hole || x[r][1] == kHole || x[r][3] == kHole;
                            R.pa[k] = mine ? (R.wa[k] != (T)0 ? v[0] : (T)0) : R.pa[k];
                            R.pb[k] = mine ? (R.wb[k] != (T)0 ? v[1] : (T)0) : R.pb[k];
                        }
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (!__any(hole)) return false;
                if (tries % 4 == 0 && __hip_atomic_load(&bar->err, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0)
                    return true;
                const unsigned long long now = __builtin_amdgcn_s_memrealtime();
                if (t0 == 0) t0 = now;
                if (now - t0 > bar->timeout) {
                    __hip_atomic_store(&bar->err, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    return true;
                }
            }
        };
        // The same from the output of a stage whose counters have been seen.
        // (A pair with a cell on the domain's ring loads that too: its value
        // only ever meets a zero coefficient.)
        auto reload = [&](const __amdgpu_buffer_rsrc_t ro) __attribute__((always_inline)) {
            const int q = column(), ln = (q - c0) >> 1;
            const bool ldl = q >= 0 && q <= nx - 2, ld_side = ldl && (ln < H / 2 || ln >= 64 - H / 2);
            auto halo = [&](unsigned rows) {
#pragma unroll
                for (int k = 0; k < NRW; k++) {
                    if (!((rows >> k) & 1u)) continue;
                    const int srow = (jt0 + k) * P * (int)sizeof(T);
                    V2 v;
                    if constexpr (sizeof(T) == 4)
                        v = __builtin_bit_cast(V2, __builtin_amdgcn_raw_buffer_load_b64(ro, q * 4, srow, kDev));
                    else
                        v = __builtin_bit_cast(V2, __builtin_amdgcn_raw_buffer_load_b128(ro, q * 8, srow, kDev));
                    if constexpr (sizeof(T) == 8) {  // kept cells stay 0
                        R.pa[k] = R.wa[k] != (T)0 ? v[0] : (T)0;
                        R.pb[k] = R.wb[k] != (T)0 ? v[1] : (T)0;
                    } else {
                        R.pa[k] = v[0];
                        R.pb[k] = v[1];
                    }
                }
            };
            if (ld_side) halo(m_st);
            if (ldl) halo(m_halo);
        };
        __shared__ int stuck;  // a wave of the block has given up
        if (threadIdx.x == 0) stuck = 0;
        __shared__ double red[sizeof(T) == 8 ? NW : 1];
        int done = 0, chunk = 0;      // sweeps and chunks behind the running chunk
        int kc = kexec, rest = kexec;  // sweeps of the running chunk, and what is left of them
        bool whole = false;
        unsigned sent = 3u;  // bit q: stage g - 1 - q used its strip buffer (before the launch: maybe)
        int l = 0;
        for (;; l++) {
            int me = alone || rest < M ? rest : M;
            if (solve && !alone && rest == M) me = (M + 1) / 2;
            const unsigned g = f0 + (unsigned)l;
            sweeps(2 * me, [&] {
                if constexpr (kPoll)
                    if (!alone && (sent & 2u)) send(strip_buf(g + 1u), std::true_type{});
            });
            rest -= me;
            // after a timed-out wait anywhere in the launch, stop sweeping: the
            // fields in memory are finite, the step reports the failure and
            // the solve resumes from the current pressure
            if (kPoll && __builtin_amdgcn_readfirstlane(stuck)) {
                if (solve && tl.y == 0 && threadIdx.x == 0) {
                    ctw->ppe_done = 2;
                    check_case(pa.ncase, false, false, bar);
                }
                break;
            }
            const bool check = solve && rest == 0;
            const bool last = !solve && rest == 0;
            // (a plain launch leaves its output where launches of M sweeps do)
            const __amdgpu_buffer_rsrc_t ro = ((solve || !alone ? l + 1 : (kexec + M - 1) / M) & 1) ? rs1 : rs0;
            if (check) {
                const double m = residual();
                if (lane == 0) red[w] = m;
                __syncthreads();
            }
            // at a check the tiles wait for each other all together anyway: the
            // strips go with the counters
            const bool poll = kPoll && !check;
            sent = sent << 1 | (poll ? 1u : 0u);
            if (kPoll && !last && poll && !alone) {
                __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);  // (the emptied strips)
                send(strip_buf(g), std::false_type{});
            } else if (!alone || last) {
                put(ro, last);
            }
            if (last) break;
            if (check && threadIdx.x == 0) {
                double m = red[0];
#pragma unroll
                for (int q = 1; q < NW; q++) m = fmax(m, red[sizeof(T) == 8 ? q : 0]);
                __hip_atomic_store(&pa.vals[(size_t)(chunk & 1) * ntiles + t], m, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
            if (!alone && !poll) {
                // the stage's counter, behind this block's stores; wait for the
                // tiles the halo reaches, at a check for all tiles of the case
                __builtin_amdgcn_s_waitcnt(kWaitVmcnt0);
                __syncthreads();
                if (threadIdx.x == 0)
                    __hip_atomic_store(&flags[t], g + 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                const bool bad = check ? wait_all(flags + (t - tl.y), ntxs * ntys, g + 1u, bar)
                                       : w == 0 && wait_neighbours(flags, nb, g + 1u, bar);
                if (__builtin_amdgcn_readfirstlane(__syncthreads_or(bad))) {
                    // (at a check other tiles may have seen every counter and
                    // end here: this one leaves its part of the result too)
                    whole = check;
                    if (solve && tl.y == 0 && threadIdx.x == 0) {
                        ctw->ppe_done = 2;
                        check_case(pa.ncase, false, false, bar);
                    }
                    break;
                }
            }
            if (check) {
                double m = 0.0;
                if (alone) {
                    for (int q = lane; q < NW; q += 64) m = red[sizeof(T) == 8 ? q : 0];
                } else {
                    for (int q = lane; q < ntxs * ntys; q += 64)
                        m = fmax(m, __hip_atomic_load(&pa.vals[(size_t)(chunk & 1) * ntiles + (t - tl.y) + q],
                                                      __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
                }
                const double res = c.dt * uniform(wave_max(m));
                done += kc;
                chunk++;
                const bool failed = !(res <= 1.0e300);
                const bool stop = !(res > c.ppe_tol) || done >= left || failed;
                if (stop || chunk == pa.nchunk) {
                    whole = true;
                    if (tl.y == 0 && threadIdx.x == 0) {
                        ctw->ppe_sweeps += done;
                        ctw->tot_ppe += done;
                        ctw->ppe_base = (base + l + 1) & 1;
                        ctw->ppe_res = res;
                        if (failed) ctw->failed = 1;
                        if (stop) ctw->ppe_done = 1;
                        check_case(pa.ncase, !stop, false, bar);
                    }
                    break;
                }
                kc = rest = min(K, left - done);
                if (alone) __syncthreads();  // red is read before the next chunk's maxima
            }
            if (alone) continue;
            if (poll) {
                if constexpr (kPoll)
                    if (receive(strip_buf(g))) stuck = 1;
            } else {
                reload(ro);
            }
        }
        if (solve) {
            if (whole) put((l + 1) & 1 ? rs1 : rs0, true);
        } else if (!alone && threadIdx.x == 0) {
            // (a case's counters agree when a launch starts)
            __hip_atomic_store(&flags[t], f0 + (unsigned)(l + 1), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        return;
    }
    sweeps(nst, [] {});
    store(dst);
}

}  // namespace iff
