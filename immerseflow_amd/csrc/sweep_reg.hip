// Per-stage launches of the register-tile red-black SOR (sweep_reg.h).
#include "sweep_reg.h"

namespace iff {

template <typename T, int M, int NW, int NRW>
static void reg_one(hipStream_t st, const CaseDev *cs, const int2 *tiles, int nt, int s, int K, int wt)
{
    const int pad = ((nt + 7) / 8) * 8;
#define IFF_RL(WM_)                                                                                             \
    hipLaunchKernelGGL((k_rbsor_reg<T, M, NW, NRW, false, WM_>), dim3(pad), dim3(64 * NW), 0, st, cs, tiles, nt, \
                       pad, s, K, PersArgs{})
    if (wt == 1)
        IFF_RL(1);
    else if (sizeof(T) == 4 && wt == 2)
        IFF_RL(sizeof(T) == 4 ? 2 : 0);
    else
        IFF_RL(0);
#undef IFF_RL
}

// Stored tile: 128 - 4M columns by tile_y rows; tile_y + 4M rows per
// workgroup, split over its waves (4, 8 or 16).  M = 8 (8- and 16-wave
// tiles) trades a wider halo for half the loads per sweep.  The FP64 tile
// of 16 waves x 8 rows does not fit the 128 registers a 1024-lane
// workgroup allows, so that shape is FP32 (mixed precision) only, as are
// its deeper forms: 9 to 12 sweeps on the same 128 x 128 cells (92, 88, 84
// and 80 stored rows and columns), fewer loads per sweep for more
// recomputed halo.
bool reg_variant_ok(int prec, int waves, int ty, int m)
{
    if (waves == 4) return (m == 1 || m == 2 || m == 4) && (ty == 16 || ty == 32 || ty == 48);
    if (waves == 8)
        return (m == 2 && (ty == 24 || ty == 40 || ty == 56)) || (m == 4 && (ty == 32 || ty == 48 || ty == 64)) ||
               (m == 8 && (ty == 32 || ty == 48 || ty == 64));
    if (waves == 16)
        return (m == 4 && (ty == 48 || ty == 64 || ty == 80)) ||
               (m == 8 && (ty == 32 || ty == 64 || (ty == 96 && prec != IF_FP64))) ||
               (prec != IF_FP64 && ((m == 9 && ty == 92) || (m == 10 && ty == 88) || (m == 11 && ty == 84) ||
                                    (m == 12 && ty == 80))) ||
               // the default's low tiles (reg_auto_shape)
               (m == 12 && ty == 16) || (prec == IF_FP64 && m == 8 && ty == 48) ||
               (prec != IF_FP64 && ((m == 16 && ty == 32) || (m == 12 && ty == 48)));
    return false;
}

int reg_out_cols(int m) { return 128 - 4 * m; }

void launch_ppe_sweep_reg(hipStream_t st, int prec, int waves, int ty, int m, const CaseDev *cs,
                          const int2 *tiles, int nt, int s, int K, int wt)
{
#define IFF_RG(T, W_, M_, TY_)                                                            \
    if (waves == W_ && m == M_ && ty == TY_) {                                            \
        reg_one<T, M_, W_, (TY_ + 4 * M_) / W_>(st, cs, tiles, nt, s, K, wt);            \
        return;                                                                           \
    }
#define IFF_RG_ALL(T)                                                                     \
    IFF_RG(T, 4, 1, 16) IFF_RG(T, 4, 1, 32) IFF_RG(T, 4, 1, 48)                           \
    IFF_RG(T, 4, 2, 16) IFF_RG(T, 4, 2, 32) IFF_RG(T, 4, 2, 48)                           \
    IFF_RG(T, 4, 4, 16) IFF_RG(T, 4, 4, 32) IFF_RG(T, 4, 4, 48)                           \
    IFF_RG(T, 8, 2, 24) IFF_RG(T, 8, 2, 40) IFF_RG(T, 8, 2, 56)                           \
    IFF_RG(T, 8, 4, 32) IFF_RG(T, 8, 4, 48) IFF_RG(T, 8, 4, 64)                           \
    IFF_RG(T, 8, 8, 32) IFF_RG(T, 8, 8, 48) IFF_RG(T, 8, 8, 64)                           \
    IFF_RG(T, 16, 4, 48) IFF_RG(T, 16, 4, 64) IFF_RG(T, 16, 4, 80) IFF_RG(T, 16, 8, 32) IFF_RG(T, 16, 8, 64)
    // (the default's low tiles come last in each list: without the persistent
    // form, mostly after a neighbour wait timed out)
    if (prec == IF_FP64) {
        IFF_RG_ALL(double)
        IFF_RG(double, 16, 12, 16)
        IFF_RG(double, 16, 8, 48)
    } else {
        IFF_RG_ALL(float)
        IFF_RG(float, 16, 8, 96)
        IFF_RG(float, 16, 9, 92)
        IFF_RG(float, 16, 10, 88)
        IFF_RG(float, 16, 11, 84)
        IFF_RG(float, 16, 12, 80)
        IFF_RG(float, 16, 12, 16)
        IFF_RG(float, 16, 16, 32)
        IFF_RG(float, 16, 12, 48)
    }
#undef IFF_RG_ALL
#undef IFF_RG
}

}  // namespace iff
