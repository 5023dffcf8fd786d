// The class launchers on bin pairs of given sizes, for their launch shapes (nothing runs).
#include "tgpu_device.h"

extern "C" int emu_launch_1000(int n_part, const int *n_bra, const int *n_ket, int variant, int mixed)
{
    JKArgs a{};
    a.kcol_max[0] = 8;  // K rows of 8 columns
    a.kcol = a.kcol_map = n_bra;
    a.kcol_lofs[1] = 8;
    for (int l = 2; l < TGPU_LMAX + 2; ++l) a.kcol_lofs[l] = 8;
    a.krow_min_kets = 256;
    JKPart parts[TGPU_MAX_PARTS + 1] = {};
    for (int k = 0; k < n_part; ++k) {
        parts[k].n_bra = n_bra[k];
        parts[k].n_ket_max = parts[k].n_ket_avg = n_ket[k];
        parts[k].bra_start = k;
    }
    return tgpu_launch_jk_1000(a, parts, n_part, variant, mixed, nullptr);
}

extern "C" void emu_schwarz_10(int start, int n)
{
    tgpu_launch_schwarz_10(DevPairs{}, DevPrims{}, start, n, nullptr, nullptr, 0, 0, nullptr);
}
