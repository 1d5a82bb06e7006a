// Persistent launches of the register-tile red-black SOR (sweep_reg.h).
#include <algorithm>

#include "sweep_reg.h"

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
static void pers_one(hipStream_t st, const CaseDev *cs, const int2 *tiles, int nt, int K, GridBar *bar,
                     unsigned *flags, int wt)
{
    const int pad = ((nt + 7) / 8) * 8;
#define IFF_PLW(WM_)                                                                                           \
    hipLaunchKernelGGL((k_rbsor_reg<T, M, NW, NRW, true, WM_>), dim3(pad), dim3(64 * NW), 0, st, cs, tiles, nt, \
                       pad, 0, K, bar, flags)
    if (wt == 1)
        IFF_PLW(1);
    else if (sizeof(T) == 4 && wt == 2)
        IFF_PLW(sizeof(T) == 4 ? 2 : 0);
    else
        IFF_PLW(0);
#undef IFF_PLW
}

// the shapes with a persistent form: (waves, sweeps per stage, tile_y,
// rows per wave), FP32 and FP64
#define IFF_PERS_SHAPES32(X) \
    X(float, 16, 8, 96, 8) X(float, 16, 8, 64, 6) X(float, 16, 4, 48, 4) X(float, 8, 8, 32, 8) X(float, 8, 4, 32, 6) \
    X(float, 16, 8, 16, 3) X(float, 16, 8, 32, 4) X(float, 16, 8, 48, 5) X(float, 16, 12, 32, 5) X(float, 16, 12, 48, 6) \
    X(float, 16, 12, 80, 8) X(float, 16, 16, 32, 6) X(float, 16, 16, 64, 8) X(float, 16, 4, 16, 2) X(float, 16, 4, 32, 3) \
    X(float, 16, 4, 80, 6) X(float, 16, 4, 112, 8) X(float, 16, 6, 72, 6) X(float, 16, 6, 104, 8) X(float, 16, 6, 24, 3) X(float, 16, 6, 40, 4)
#define IFF_PERS_SHAPES64(X) X(double, 16, 4, 80, 6) X(double, 16, 4, 64, 5) X(double, 16, 4, 48, 4) \
    X(double, 16, 4, 16, 2) X(double, 16, 4, 32, 3) X(double, 16, 6, 24, 3) X(double, 16, 6, 40, 4) X(double, 16, 8, 16, 3) \
    X(double, 16, 8, 32, 4) X(double, 16, 8, 48, 5) X(double, 16, 8, 64, 6) X(double, 16, 6, 56, 5) X(double, 16, 6, 72, 6) X(double, 16, 3, 20, 2) X(double,16,2,24,2) X(double, 8,4,16,4) X(double,8,4,32,6) X(double,8,2,24,4) X(double,8,4,48,8) X(double,8,3,36,6)
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

bool pers_fits(int prec, int waves, int ty, int m, int nt, int wt)
{
    const int pad = ((nt + 7) / 8) * 8;
    return pad <= pers_blocks(prec, waves, ty, m, wt);
}

void launch_ppe_sweep_pers(hipStream_t st, int prec, int waves, int ty, int m, const CaseDev *cs,
                           const int2 *tiles, int nt, int K, GridBar *bar, unsigned *flags, int wt)
{
#define IFF_PL(T_, W_, M_, TY_, NRW_)                                      \
    if (waves == W_ && m == M_ && ty == TY_) {                            \
        pers_one<T_, M_, W_, NRW_>(st, cs, tiles, nt, K, bar, flags, wt); \
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
