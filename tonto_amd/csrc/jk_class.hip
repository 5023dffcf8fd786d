// One angular-momentum class pair of the J/K build per translation unit, so that the
// classes compile in parallel.  Built with -DTGPU_LP=.. -DTGPU_LQ=.. -DTGPU_LR=..
// -DTGPU_LS=.. -DTGPU_HEAVY=0|1.
#include <algorithm>

#include "launch_plan.h"
#include "tgpu_device.h"

#define TGPU_STR2(x) #x
#define TGPU_STR(x) TGPU_STR2(x)
#define TGPU_CAT5(a, b, c, d, e) a##b##c##d##e
#define TGPU_CAT3(a, b, c) a##b##c
#define TGPU_GEN_FILE(a, b, c, d) TGPU_STR(gen/eri_##a##b##c##d.inc)
#define TGPU_GEN_FILE_X(a, b, c, d) TGPU_GEN_FILE(a, b, c, d)
#include TGPU_GEN_FILE_X(TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS)

#define TGPU_LAUNCH_NAME_X(a, b, c, d) TGPU_CAT5(tgpu_launch_jk_, a, b, c, d)
#define TGPU_SCHWARZ_NAME_X(a, b) TGPU_CAT3(tgpu_launch_schwarz_, a, b)
#define TGPU_WS_NAME_X(a, b, c, d) TGPU_CAT5(tgpu_wave_ws_, a, b, c, d)

// Launches the class pair over `parts` (one per bin pair, every one with bra and ket pairs).
int TGPU_LAUNCH_NAME_X(TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS)(const JKArgs &a, const JKPart *parts, int n_part,
                                                         int variant, bool mixed, hipStream_t s)
{
    if (n_part <= 0) return TGPU_OK;
    if (n_part > TGPU_MAX_PARTS) return TGPU_E_ARG;
#if !TGPU_HEAVY
    if (variant == 0) {
        // parts in the LDS-row form, then the others four bra pairs per work-group
        JKLaunch rows, glob;
        rows.a = glob.a = a;
        size_t lds = 0, wlds = 0;
        // The LDS-row form for single molecules with long ket segments (>= 4 rounds of 64 by
        // default, so that the four wavefronts of one bra pair have work): as many of the
        // bra pair's K rows as fit the work-group's LDS budget next to the Rys table and
        // the ket queue, and at least a quarter of them ((fd|ps) at 4160 functions: 7 of
        // 16 rows in LDS, 120 -> 71 ms against every K update global).  A row holds the
        // columns of the ket shells' two angular momenta only.  Not built for (ff|ss): its FP64 instantiation
        // gives wrong K on every cluster tested while its mixed twin and the global-atomic
        // form are exact (cause not found), so that class pair updates K globally.
        bool rows_ok = false;
#if !(TGPU_LP == 3 && TGPU_LQ == 3 && TGPU_LR == 0 && TGPU_LS == 0)
        constexpr int NP = ncart(TGPU_LP), NQ = ncart(TGPU_LQ);
        constexpr int NRT = EriBody<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, double>::NROOT;
        constexpr size_t kStatic = rys_block_size(NRT) * sizeof(double) + (TGPU_COMPACT ? 4 * 128 * 8 : 0);
        constexpr size_t kMaxLds = 155 * 1024;
        static bool attr_set = false;
        if (!attr_set) {
            // dynamic LDS above the 64 KiB default has to be allowed per kernel
            (void)hipFuncSetAttribute((const void *)jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, false, KR_GROUP>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kMaxLds - kStatic));
            (void)hipFuncSetAttribute((const void *)jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, true, KR_GROUP>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kMaxLds - kStatic));
            (void)hipFuncSetAttribute((const void *)jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, false, KR_WAVE>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kMaxLds - kStatic));
            (void)hipFuncSetAttribute((const void *)jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, true, KR_WAVE>,
                                      hipFuncAttributeMaxDynamicSharedMemorySize, (int)(kMaxLds - kStatic));
            attr_set = true;
        }
        const size_t budget = a.krow_budget > 0 && (size_t)a.krow_budget < kMaxLds ? (size_t)a.krow_budget : kMaxLds;
        const int nR = a.kcol_lofs[TGPU_LR + 1] - a.kcol_lofs[TGPU_LR];
        const int W = TGPU_LR == TGPU_LS ? nR : nR + a.kcol_lofs[TGPU_LS + 1] - a.kcol_lofs[TGPU_LS];
        const size_t row_bytes = (size_t)W * sizeof(double);
        const int fit = a.kcol_map && W > 0 && budget > kStatic ? (int)((budget - kStatic) / row_bytes) : 0;
        const int nkr = fit < NP + NQ ? fit : NP + NQ;
        // (no K digested, as in the UHF ket-side J pass: no rows)
        rows_ok = a.kp != HUGE_VAL && nkr > 0 && 4 * nkr >= NP + NQ;
        if (rows_ok) {
            JKArgs &b = rows.a;
            b.krow_rows = nkr;
            // (..|ss) class pairs: density rows in the LDS left after the K rows, when all
            // of both fit
            const int pfit = (int)((budget - kStatic - (size_t)nkr * row_bytes) / row_bytes);
            b.prow_rows = TGPU_LR == 0 && TGPU_LS == 0 && a.prow_enable && nkr == NP + NQ && pfit >= NP + NQ
                              ? NP + NQ
                              : 0;
            lds = (size_t)(nkr + b.prow_rows) * row_bytes;
            // the bra pair's two P_max rows, in what is left, unless they lower the number of
            // work-groups a CU holds ((pp|ss) at 4160 functions: 2 -> 1, 99 -> 130 ms; (ds|ps),
            // at one either way: 259 -> 239 ms)
            const size_t pm_bytes = 2 * (size_t)a.n_shell * sizeof(double);
            constexpr size_t kCuLds = 160 * 1024;
            b.pmrow = a.pmrow && a.n_shell > 0 && budget >= kStatic + lds + pm_bytes &&
                              kCuLds / (kStatic + lds + pm_bytes) == kCuLds / (kStatic + lds)
                          ? 1
                          : 0;
            if (b.pmrow) lds += pm_bytes;
        }
        // The others: the rows of the wavefronts' own bra pairs in LDS, at most kWaveRowsLds per
        // work-group if all of them then fit (two work-groups per CU), else as many as fit one,
        // down to a quarter of them; global updates only for (ff|ss) (as above), where K is not
        // digested, and for molecules too large for a quarter.
        constexpr size_t kWaveRowsLds = 76 * 1024;
        const size_t Wmax = a.kcol_max[TGPU_LR] + (TGPU_LR == TGPU_LS ? 0 : a.kcol_max[TGPU_LS]);
        const size_t row4 = 4 * Wmax * sizeof(double);  // one row of each wavefront
        const size_t room = budget > kStatic ? budget - kStatic : 0;
        const size_t small = budget < kWaveRowsLds ? room : kWaveRowsLds - kStatic;
        int nwr = row4 ? (int)std::min<size_t>(NP + NQ, small / row4) : 0;
        if (nwr < NP + NQ && row4) nwr = (int)std::min<size_t>(NP + NQ, room / row4);
        if (a.kp != HUGE_VAL && a.kcol && 4 * nwr >= NP + NQ) {
            glob.a.krow_rows = nwr;
            glob.a.krow_stride = (int)(nwr * Wmax);
            wlds = nwr * row4;
        }
#endif
        auto in_rows = [&](const JKPart &p) { return rows_ok && p.n_ket_avg >= a.krow_min_kets; };
        long long groups[TGPU_MAX_PARTS];
        for (int k = 0; k < n_part; ++k) {
            groups[k] = in_rows(parts[k]) ? parts[k].n_bra : (parts[k].n_bra + 3LL) / 4;
            if (groups[k] > kMostThreads / 256) return TGPU_E_UNSUPPORTED;
        }
        for (int k0 = 0, k1; k0 < n_part; k0 = k1) {
            k1 = launch_end(groups, n_part, k0, kMostThreads / 256);
            int rows_grid = 0, glob_grid = 0;
            rows.clear();
            glob.clear();
            for (int k = k0; k < k1; ++k) {
                const bool r = in_rows(parts[k]);
                int &grid = r ? rows_grid : glob_grid;
                JKPart &p = (r ? rows : glob).add(parts[k], grid);
                p.gx = p.gy = 1;
                grid += (int)groups[k];
            }
#if !(TGPU_LP == 3 && TGPU_LQ == 3 && TGPU_LR == 0 && TGPU_LS == 0)
            if (rows_grid > 0) {
                if (mixed) jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, true, KR_GROUP><<<rows_grid, 256, lds, s>>>(rows);
                else jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, false, KR_GROUP><<<rows_grid, 256, lds, s>>>(rows);
            }
            if (glob_grid > 0 && wlds) {
                if (mixed) jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, true, KR_WAVE><<<glob_grid, 256, wlds, s>>>(glob);
                else jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, false, KR_WAVE><<<glob_grid, 256, wlds, s>>>(glob);
                continue;
            }
#endif
            if (glob_grid > 0) {
                if (mixed) jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, true, KR_GLOBAL><<<glob_grid, 256, 0, s>>>(glob);
                else jk_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, false, KR_GLOBAL><<<glob_grid, 256, 0, s>>>(glob);
            }
        }
        return TGPU_OK;
    }
#endif
    (void)variant;
#if TGPU_LP <= 2
    using namespace rows_form;
    constexpr bool kGB = false;
    constexpr long long kWS = 0;
#else
    using namespace level_form;
    using C = WaveCfg<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS>;
    constexpr bool kGB = C::GB;  // transfer buffers in the workspace
    constexpr long long kWS = C::WS;
#endif
    JKLaunch L;
    L.a = a;
    // FP64 over the kets before the FP32 split of each prefix (all of it in an FP64 build),
    // then FP32 over the rest
    if (!mixed) L.a.fp32_thr = 0.0;
    long long slots = 0;
    if (kGB) {
        slots = ws_slot_count(a.ws_doubles, kWS);
        // the caller sizes the workspace for at least one slot of every class it launches;
        // with fewer slots than parts, each part takes all of them in a launch of its own
        if (slots <= 0 || !a.ws) return TGPU_E_STATE;
        if (slots < n_part) {
            for (int k = 0; k < n_part; ++k)
                if (int rc = TGPU_LAUNCH_NAME_X(TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS)(a, parts + k, 1, 1, mixed, s))
                    return rc;
            return TGPU_OK;
        }
    }
    WavePlan plan[TGPU_MAX_PARTS];
    long long groups[TGPU_MAX_PARTS];
    auto chunk = [](const JKPart &p) { return p.ket_chunk > 0 && p.ket_chunk <= 64 ? p.ket_chunk : 64; };  // one lane per ket
    for (int k = 0; k < n_part; ++k) {
        const int nk = parts[k].n_ket_max, kc = chunk(parts[k]);
        plan[k] = WavePlan{parts[k].n_bra, nk > 0 ? (nk + kc - 1) / kc : 1, 0, 0};
    }
    plan_wave(plan, n_part, slots);
    for (int k = 0; k < n_part; ++k) {
        groups[k] = plan[k].gx * plan[k].gy;
        if (groups[k] > kMostThreads / 64) return TGPU_E_UNSUPPORTED;
    }
    for (int k0 = 0, k1; k0 < n_part; k0 = k1) {
        k1 = launch_end(groups, n_part, k0, kMostThreads / 64);
        int grid = 0;
        L.clear();
        for (int k = k0; k < k1; ++k) {
            JKPart &p = L.add(parts[k], grid);
            p.ket_chunk = chunk(p);
            p.gx = (int)plan[k].gx;
            p.gy = (int)plan[k].gy;
            grid += (int)groups[k];
        }
        jk_wave_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, double><<<grid, 64, 0, s>>>(L);
        if (mixed) jk_wave_kernel<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS, float><<<grid, 64, 0, s>>>(L);
    }
    return TGPU_OK;
}

size_t TGPU_WS_NAME_X(TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS)()
{
#if TGPU_LP <= 2
    return 0;
#else
    return level_form::WaveCfg<TGPU_LP, TGPU_LQ, TGPU_LR, TGPU_LS>::WS;
#endif
}

#if TGPU_LP == TGPU_LR && TGPU_LQ == TGPU_LS
void TGPU_SCHWARZ_NAME_X(TGPU_LP, TGPU_LQ)(const DevPairs &pr, const DevPrims &pm, int start, int n,
                                          double *maxI, double *ws, long long ws_doubles, int sph, hipStream_t s)
{
#if TGPU_HEAVY && TGPU_LP <= 2
    (void)ws;
    (void)ws_doubles;
    constexpr int T = rows_form::WaveCfg<TGPU_LP, TGPU_LQ, TGPU_LP, TGPU_LQ>::TEAMS;
    rows_form::schwarz_wave_kernel<TGPU_LP, TGPU_LQ><<<(n + T - 1) / T, 64, 0, s>>>(pr, pm, start, n, maxI, sph);
#elif TGPU_HEAVY
    using namespace level_form;
    using C = WaveCfg<TGPU_LP, TGPU_LQ, TGPU_LP, TGPU_LQ>;
    const long long slots = ws_slot_count(ws_doubles, C::WS);
    const int grid = C::GB ? (int)(n < slots ? n : slots) : n;
    if (grid > 0) schwarz_wave_kernel<TGPU_LP, TGPU_LQ><<<grid, 64, 0, s>>>(pr, pm, start, n, maxI, ws, sph);
#else
    (void)ws;
    (void)ws_doubles;
    constexpr int kSplit = 16;
    // (the lanes are numbered in an int)
    in_chunks(n, (1LL << 31) / kSplit, [&](long long at, long long count) {
        const int grid = (int)((count + 64 / kSplit - 1) / (64 / kSplit));
        schwarz_kernel<TGPU_LP, TGPU_LQ, kSplit><<<grid, 64, 0, s>>>(pr, pm, start + (int)at, (int)count, maxI, sph);
    });
#endif
}
#endif
