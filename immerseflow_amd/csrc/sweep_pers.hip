// Persistent launches of the register-tile red-black SOR (sweep_reg.h).
#include "sweep_reg.h"

#include <functional>
#include <iterator>

namespace iff {

// Blocks of the persistent form that can be resident at once: resident
// blocks per CU (occupancy calculator) times the CUs, per shape and weight
// mode.
template <typename T, int M, int NW, int NRW, int WM>
static int pers_capacity()
{
    static int capacity = -1;  // one device type per process
    if (capacity < 0) {
        int per_cu = 0, dev = 0, cus = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, k_rbsor_reg<T, M, NW, NRW, true, WM>, 64 * NW,
                                                         0) != hipSuccess ||
            hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return 0;
        capacity = per_cu * cus;
    }
    return capacity;
}

template <typename T, int M, int NW, int NRW>
static void pers_one(hipStream_t st, const CaseDev *cs, const int2 *tiles, int nt, int K, const PersArgs &pa, int wt)
{
    const int pad = ((nt + 7) / 8) * 8;
#define IFF_PLW(WM_)                                                                                           \
    hipLaunchKernelGGL((k_rbsor_reg<T, M, NW, NRW, true, WM_>), dim3(pad), dim3(64 * NW), 0, st, cs, tiles, nt, \
                       pad, 0, K, pa)
    if (wt == 1)
        IFF_PLW(1);
    else if (sizeof(T) == 4 && wt == 2)
        IFF_PLW(sizeof(T) == 4 ? 2 : 0);
    else
        IFF_PLW(0);
#undef IFF_PLW
}

// the shapes with a persistent form: (waves, sweeps per stage, tile_y,
// rows per wave), FP32 and FP64; the last ones of each only for the
// default's low tiles (reg_auto_shape)
#define IFF_PERS_SHAPES32(X)                                                                                \
    X(float, 16, 8, 96, 8) X(float, 16, 8, 64, 6) X(float, 16, 4, 48, 4) X(float, 8, 8, 32, 8) X(float, 8, 4, 32, 6) \
    X(float, 16, 12, 16, 4) X(float, 16, 16, 32, 6) X(float, 16, 12, 48, 6)
#define IFF_PERS_SHAPES64(X)                                                                        \
    X(double, 16, 4, 80, 6) X(double, 16, 4, 64, 5) X(double, 16, 4, 48, 4) X(double, 16, 8, 32, 4) \
    X(double, 16, 8, 64, 6) X(double, 16, 12, 16, 4) X(double, 16, 8, 48, 5)

// The default launch shape of kernel 4, for cases whose tiles at (tile_y,
// sweeps per stage) are counted by tiles: the first shape that fits on the
// device as one persistent launch, in this order.  A small grid is bound by
// the latency of its half-sweeps and of the exchange after each stage, not by
// arithmetic: low tiles (few rows per wave) shorten the one, deep stages the
// other, and the halo they recompute costs nothing on idle CUs; from about
// one tile per CU on the recomputation counts.  Measured (us per sweep, uniform
// n x n, one circle):
//   FP32   n   64: 64 x 8 (one tile) 0.46, 16 x 12 0.54, 32 x 16 0.60
//             256: 16 x 12 0.56, 32 x 16 0.60, 48 x 12 0.66, 64 x 8 0.86, 96 x 8 1.02
//             611: 32 x 16 0.64 (200 tiles), 48 x 12 0.70, 16 x 12 0.80 (312), 64 x 8 0.94
//             800: 48 x 12 0.72 (170), 64 x 8 0.94, 32 x 16 1.15 (325, per stage)
//            1024: 64 x 8 0.97 (176), 48 x 12 1.12 (286), 96 x 8 1.12
//            1400: 96 x 8 1.29 (225), 64 x 8 1.34 (330, two per CU)
//            1948: 96 x 8 1.88 (441, two per CU); per stage 64 x 8 2.8
//   stretched 2048 x 1024: 96 x 8 1.19 (242), 64 x 8 1.60 (352)
//   FP64   n   64: 64 x 4 (one tile) 0.96, 16 x 12 1.06
//             256: 16 x 12 1.05, 32 x 8 1.15, 48 x 8 1.57
//             800: 32 x 8 1.27 (225), 48 x 8 1.65, 64 x 8 1.81
//            1024: 48 x 8 1.80 (242), 64 x 8 1.92, 48 x 4 2.2
//   stretched 2048 x 1024: only 80 x 4 fits, 2.9
// False: none fits.
bool reg_auto_shape(int prec, int wt, const std::function<int(int, int, int *)> &tiles, int *ty, int *m)
{
    struct Shape {
        int ty, m, per_cu;  // tiles per CU it is chosen at, at most
        bool single;        // only where every case is one tile
    };
    static const Shape s32[] = {{64, 8, 2, true}, {16, 12, 1, false}, {32, 16, 1, false}, {48, 12, 1, false},
                                {64, 8, 1, false}, {96, 8, 1, false},  {64, 8, 2, false},  {96, 8, 2, false}};
    static const Shape s64[] = {{64, 4, 1, true}, {16, 12, 1, false}, {32, 8, 1, false}, {48, 8, 1, false},
                                {64, 8, 1, false}, {80, 4, 1, false}};
    static int cus = -1;  // one device type per process
    if (cus < 0) {
        int dev = 0, n = 0;
        if (hipGetDevice(&dev) != hipSuccess ||
            hipDeviceGetAttribute(&n, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
            return false;
        cus = n;
    }
    const Shape *const list = prec == IF_FP64 ? s64 : s32;
    const int count = (int)(prec == IF_FP64 ? std::size(s64) : std::size(s32));
    for (int k = 0; k < count; k++) {
        const Shape &s = list[k];
        int most = 0;  // tiles of the largest case
        const int nt = tiles(s.ty, s.m, &most);
        if ((s.single && most > 1) || nt > s.per_cu * cus || !pers_fits(prec, 16, s.ty, s.m, nt, wt)) continue;
        *ty = s.ty;
        *m = s.m;
        return true;
    }
    return false;
}

int pers_blocks(int prec, int waves, int ty, int m, int wt)
{
#define IFF_PB(T_, W_, M_, TY_, NRW_)                                                      \
    if (waves == W_ && m == M_ && ty == TY_)                                               \
        return wt == 1                       ? pers_capacity<T_, M_, W_, NRW_, 1>()        \
               : wt == 2 && sizeof(T_) == 4 ? pers_capacity<T_, M_, W_, NRW_, sizeof(T_) == 4 ? 2 : 0>() \
                                             : pers_capacity<T_, M_, W_, NRW_, 0>();
    if (prec == IF_FP64) {
        IFF_PERS_SHAPES64(IFF_PB)
    } else {
        IFF_PERS_SHAPES32(IFF_PB)
    }
#undef IFF_PB
    return 0;
}

bool pers_polls(int prec, int waves, int ty, int m, int wt)
{
#define IFF_PP(T_, W_, M_, TY_, NRW_)                                    \
    if (waves == W_ && m == M_ && ty == TY_)                             \
        return wt == 1                       ? polls<T_, M_, W_, NRW_, 1> \
               : wt == 2 && sizeof(T_) == 4 ? polls<T_, M_, W_, NRW_, 2> \
                                             : polls<T_, M_, W_, NRW_, 0>;
    if (prec == IF_FP64) {
        IFF_PERS_SHAPES64(IFF_PP)
    } else {
        IFF_PERS_SHAPES32(IFF_PP)
    }
#undef IFF_PP
    return false;
}

bool pers_fits(int prec, int waves, int ty, int m, int nt, int wt)
{
    const int pad = ((nt + 7) / 8) * 8;
    return pad <= pers_blocks(prec, waves, ty, m, wt);
}

void launch_ppe_sweep_pers(hipStream_t st, int prec, int waves, int ty, int m, const CaseDev *cs,
                           const int2 *tiles, int nt, int K, const PersArgs &pa, int wt)
{
#define IFF_PL(T_, W_, M_, TY_, NRW_)                                      \
    if (waves == W_ && m == M_ && ty == TY_) {                            \
        pers_one<T_, M_, W_, NRW_>(st, cs, tiles, nt, K, pa, wt); \
        return;                                                           \
    }
    if (prec == IF_FP64) {
        IFF_PERS_SHAPES64(IFF_PL)
    } else {
        IFF_PERS_SHAPES32(IFF_PL)
    }
#undef IFF_PL
}

}  // namespace iff
