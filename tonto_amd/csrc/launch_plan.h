// Shapes of the class launches: host code without HIP, so that it can be tested on its own.
#pragma once
#include <algorithm>

// One bin pair of a wavefront-form launch: n_bra bra pairs, `chunks` ket chunks in the longest
// ket segment.  Its grid is (gx, gy): work-group (x, y) takes bra pairs x, x + gx, ... and, of
// each, the ket chunks y, y + gy, ...
struct WavePlan {
    long long n_bra, chunks, gx, gy;
};

// Fills gx and gy.  slots == 0 (no workspace): gy splits long prefixes when there are few bra
// pairs, so that a part's grid holds about 65536 work-groups.  Else a work-group takes a slot
// of the workspace, the grids together at most `slots` >= n of them: every part what it can
// use where that fits, else shares in proportion to bra pairs times chunks.  (Even shares
// left (ff|fp) with most of its kets in one of two parts at one work-group per bra pair there,
// each over the whole prefix: FP64 builds of (H2O)64/cc-pVTZ 127 against 53 ms, of (H2O)32
// 10.4 against 6.9.)
inline void plan_wave(WavePlan *p, int n, long long slots)
{
    constexpr long long kWaveGrid = 65536;
    double total = 0.0;
    for (int k = 0; k < n; ++k) total += (double)p[k].n_bra * (double)p[k].chunks;
    long long left = slots;
    for (int k = 0; k < n; ++k) {
        const double want = (double)p[k].n_bra * (double)p[k].chunks;
        long long gx = p[k].n_bra, gy = p[k].chunks;
        if (slots == 0) {
            gy = std::min(gy, std::max(1LL, (kWaveGrid + gx - 1) / gx));
        } else if (total > (double)slots) {
            // (a slot stays for each part that follows, whatever the rounding)
            const long long share =
                std::min(1 + (long long)((double)(slots - n) * (want / total)), left - (n - 1 - k));
            gx = std::min(gx, share);
            gy = std::min(gy, std::max(1LL, share / gx));
            left -= gx * gy;
        }
        p[k].gx = gx;
        p[k].gy = gy;
    }
}

// A launch has to have fewer than 2^32 threads along x.
constexpr long long kMostThreads = 0xffffffffLL;

// The bin pairs [first, end) go into one launch of at most `most` work-groups; a bin pair that
// has more by itself is alone.  (A class pair's 16 bin pairs together can exceed the limit that
// each keeps to: (ps|ss) from about 4.2 million bra pairs.)
inline int launch_end(const long long *groups, int n, int first, long long most)
{
    long long sum = groups[first];
    int end = first + 1;
    while (end < n && sum + groups[end] <= most) sum += groups[end++];
    return end;
}

// f(at, count) for consecutive parts of n items, at most `most` each
template <typename F>
inline void in_chunks(long long n, long long most, F f)
{
    for (long long at = 0; at < n; at += most) f(at, std::min(most, n - at));
}
