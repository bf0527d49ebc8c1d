// runs.h -- how many rows of a sequence one workgroup of a recurrence walks, who walks an attention's keys and in which order its tiles
// are listed (host code, without HIP).
//
// A short step's few runs are walked by a few CUs, each row waiting for the one before; where the chip is full short runs only
// add carries.
#pragma once
#include <algorithm>
#include <climits>
#include <cmath>
#include <cstdint>
#include <vector>

namespace pgmi {

constexpr int kRunCUs = 256;

// lanes of a scan workgroup of 256 that share a channel of N states
constexpr int scan_lanes(int N) { return N <= 16 ? 1 : N <= 32 ? 2 : N <= 64 ? 4 : N <= 128 ? 8 : 16; }
// What a run of C channels takes of a round of kRunCUs: 256 channels of one lane each, and as much of two and four, which wait on
// each other's sums and leave room for as many more workgroups; 8 and 16 lanes fill the chip two and four times as fast.
// Measured, 2,048 channels, us a layer by run lengths 64 / 32 / 16: 500 rows of 64 states 114 / 95 / 93, of 128 144 / 138 / 140, of 256
// 261 / 267 / 288; 1,540 rows 172 / 171 / 180, 282 / 286 / 308, 655 / 682 / 758.
constexpr long scan_columns(int C, int N) { return ((long)C + 255) / 256 * std::max(1, scan_lanes(N) / 4); }
constexpr long gru_columns(int C) { return ((long)C + 127) / 128; }
// the scan's workgroups for a run of C channels
constexpr long scan_workgroups(int C, int N) { return ((long)C * scan_lanes(N) + 255) / 256; }

inline long runs_of(const int32_t* lens, int n_seq, int rows) {
    long n = 0;
    for (int r = 0; r < n_seq; ++r) n += (lens[r] + rows - 1) / rows;
    return n;
}

// Sequences that are walked whole take one launch where runs take three, two of them walks: the longest of the sequences if that
// pays, else 0.  Up to 40 rows it does, and up to 64 where whole sequences fill half the chip; `workgroups` of one run, 0 where
// only the first counts.  us a layer, whole / in the best runs: 2,048 channels of 16 states, 17 rows 42 / 52, 40 rows 52 / 53, 64 rows 63 /
// 54; 8 x 64 rows of 4,096 channels 79 / 83, of 2,048 of 64 states 81 / 97, of 512 of 16 states 61 / 54; minGRU of 1,024, 17 rows 17 / 21,
// 40 rows 22 / 22, 64 rows 27 / 22, 32 x 40 rows 28 / 31.
inline int whole_rows(const int32_t* lens, int n_seq, long workgroups) {
    const int most = *std::max_element(lens, lens + n_seq);
    return most <= 40 || (most <= 64 && n_seq * workgroups >= kRunCUs / 2) ? most : 0;
}

// The scan takes the length whose rounds walk the fewest rows, a workgroup's start costing about 8.  us of its three launches,
// 64- / 16-row runs: 500 rows of 2,048 channels of 16 states 86 / 41, 300 rows 69 / 35; 64 rows / this rule: 1,540 rows of 4,096
// channels (50-row runs) 98 / 92.  columns, workgroups: of the layer with the most.
inline int scan_run_rows(const int32_t* lens, int n_seq, long columns, long workgroups) {
    if (const int whole = whole_rows(lens, n_seq, workgroups)) return whole;
    int best = 64;
    long least = LONG_MAX;
    for (int ct = 64; ct >= 16; ct -= 2) {
        const long cost = (runs_of(lens, n_seq, ct) * columns + kRunCUs - 1) / kRunCUs * (ct + 8);
        if (cost < least) { least = cost; best = ct; }
    }
    return best;
}

// A step as the scan sees it: its sequences, and the runs that they would be cut into
struct ScanStep {
    int n_seq = 0, longest = 0, run_rows = 0, most_runs = 0;  // most_runs: of one sequence
    long rows = 0, padded = 0, runs = 0;                      // padded: every sequence's rows in whole blocks of 16
};
inline ScanStep scan_step_of(const int32_t* lens, int n_seq, int run_rows) {
    ScanStep s;
    s.n_seq = n_seq;
    s.run_rows = run_rows;
    for (int r = 0; r < n_seq; ++r) {
        const int n = (lens[r] + run_rows - 1) / run_rows;
        s.longest = std::max(s.longest, (int)lens[r]);
        s.most_runs = std::max(s.most_runs, n);
        s.rows += lens[r];
        s.padded += (lens[r] + 15) / 16 * 16;
        s.runs += n;
    }
    return s;
}
// Whether a layer walks its sequences with a lane per state (k_scan_walk: every exponential once, one launch) rather than in runs
// with a lane per channel (k_scan: twice, three launches): by the predicted time, in us.  A walk takes what its longest sequence
// takes alone, or what the chip takes for all of them (a CU's share of the workgroups, each with its start and its steps); runs take
// their launches, the rows' traffic, the rounds of rows walked one after the other and the carries.  The constants are fitted to 196
// steps of 64 to 8,192 channels and 33 to 4,096 rows: the rule loses 0.2 % of the better form on average, 22 % at most (runs kept for 700
// fp32 rows of 64 channels), and no walk that it takes is slower than runs by more than 1.3 %
// (nor by more than 3 % of 144 steps of other channels and 9 to 15 states).  us a layer, runs / walk: 1,024 + 387 + 129 rows of 4,096 channels
// 70.5 / 38.1, 512 rows 34.0 / 16.5, 8 x 512 rows 145 / 89, 500 rows of 2,048 fp32 channels 31.3 / 21.1; 4,096 rows of 2,048 channels
// 83 / 113, 64 x 33 rows of 4,096 50 / 116, 1,000 rows of 1,000 channels of 12 states 32.8 / 38.7 (1,024 of 16: 31 / 27).
inline bool scan_walks(const ScanStep& s, int C, int N, bool f32) {
    if (N <= 8 || N > 16) return false;
    const double per_cu = (C + 15) / 16 / (double)kRunCUs;
    const int odd = (C % 16 != 0) + (N != 16);  // single elements: channels that are no whole workgroups, states that are no 16
    const double walk = (f32 ? 5 : 3) + std::max((f32 ? 0.035 + 0.0035 * odd : 0.024 + 0.006 * odd) * s.longest,
                                                 per_cu * (0.5 * s.n_seq + (f32 ? 0.029 : 0.023) * (double)s.padded));
    const double rounds = (double)((s.runs * ((C + 255) / 256) + kRunCUs - 1) / kRunCUs);
    const double runs = s.most_runs == 1 ? 10 + rounds * s.run_rows * (f32 ? 0.44 : 0.3)
                                         : (f32 ? 18.9 + 8.5e-6 * C * (double)s.rows : 17.6 + 7.1e-6 * C * (double)s.rows) +
                                               rounds * (s.run_rows + 8) * (f32 ? 0.21 : 0.048) + 0.093 * s.most_runs;
    return walk < runs;
}

// minGRU: the longest runs, down to 8 rows, that still give every CU a workgroup of 128 channels; of one sequence no more than 84,
// which the carry walks one after the other (us a layer on runs of 32 / 24 / 16 / 8 rows, 64 channels: 300 rows 30 / 28 / 26 / 24, 700
// rows 32 / 29 / 27 / 28, 2,000 rows 36 / 35 / 35 / 41, 5,000 rows 50 / 51 / 55 / 76)
inline int gru_run_rows(const int32_t* lens, int n_seq, long columns) {
    if (const int whole = whole_rows(lens, n_seq, 0)) return whole;
    const int most = *std::max_element(lens, lens + n_seq);
    int ct = 32;
    for (const int k : {24, 16, 8}) {
        if (runs_of(lens, n_seq, ct) * columns >= kRunCUs || (most + k - 1) / k > 84) break;
        ct = k;
    }
    return ct;
}

// Whether a minGRU layer walks its sequences whole (k_gru_walk, one launch) rather than in the runs above: as scan_walks, by the
// predicted time in us, fitted to 180 steps of 44 to 4,096 channels and 17 to 4,096 rows.  It leans to the runs: it loses 2.1 % of the
// better form on average, up to 37 % where runs are kept for 2,000 rows of up to 256 channels, and 12 % at most where a walk is taken
// (4,096 fp32 rows of 2,048 channels).  us a layer, runs / walk: 1,024 + 387 + 129 rows of 2,048 channels 21.7 / 12.6, 500 rows of 1,024 fp32
// channels 14.7 / 6.8, 60 rows of 2,048 11.0 / 5.7, 8 x 512 rows 30.1 / 22.5; 64 x 33 rows 10.9 / 40, 4,096 rows of 1,024 channels 30 / 34.
inline bool gru_walks(const ScanStep& s, int C, bool f32) {
    const double per_cu = (C + 15) / 16 / (double)kRunCUs, traffic = (f32 ? 3.4e-6 : 1.65e-6) * C * (double)s.rows;
    const double row = C % 16 == 0 ? 0.008 : f32 ? 0.011 : 0.0135;  // (channels that are no whole workgroups: single elements)
    const double walk = 4.5 + std::max(row * s.longest, per_cu * (0.5 * s.n_seq + (f32 ? 0.0135 : 0.0095) * (double)s.padded));
    const double runs = traffic + (s.most_runs == 1 ? 3.6 + 0.11 * s.run_rows : 8.2 + 0.21 * s.run_rows + 0.07 * s.most_runs);
    return walk < runs;
}

// The tiles of a prompt's attention, `rows` (position, head) pairs of one sequence each: by the 64 keys that the last position's fall in,
// so fewest keys first whatever the window, then by sequence.
struct AttnTile { int seq, first; };
inline std::vector<AttnTile> attn_tiles(const int32_t* starts, const int32_t* lens, int n_seq, int R, int rows) {
    std::vector<AttnTile> t;
    std::vector<int> end;
    long lo = LONG_MAX, hi = 0;
    for (int r = 0; r < n_seq; ++r)
        for (int f = 0, n = lens[r] * R; f < n; f += rows) {
            end.push_back(starts[r] / 64 + (starts[r] % 64 + (std::min((long)f + rows, (long)n) - 1) / R) / 64);
            lo = std::min(lo, (long)end.back());
            hi = std::max(hi, (long)end.back());
            t.push_back({r, f});
            if (n - f <= rows) break;
        }
    if (n_seq == 1) return t;
    std::vector<int> at(hi - lo + 2);
    for (const int e : end) ++at[e - lo + 1];
    for (size_t k = 1; k < at.size(); ++k) at[k] += at[k - 1];
    std::vector<AttnTile> sorted(t.size());
    for (size_t k = 0; k < t.size(); ++k) sorted[at[end[k] - lo]++] = t[k];
    return sorted;
}

// Whether a prompt's attention gives each tile of 64 (position, head) pairs to two teams of four waves, which take its 64-key tiles in
// turn, rather than to one: by the predicted time, in us of heads of 128 (narrower and wider ones take a like share more or less of every
// term).  A step takes what its longest tile's chain takes, or what the chip takes for all tiles and keys; two teams halve the chain,
// but fill a CU (heads of up to 64: half of it), so that tiles past 256 (512) wait for others to end.  Fitted to 627 steps of 1 to 16
// sequences, 60 to 5,000 rows, heads of 32 to 256, windows of 256 to 4,096: the rule loses 0.3 % of the better form on average, 12 % at
// most.  us, one team / two, 16 heads of 128 in 2 groups, window 1,024, distance bias: 1,024 + 387 + 129 rows 31.3 / 25.7, 500 rows 18.5 /
// 16.0, 600 + 500 rows 21.6 / 18.7; 4 x 300 rows 14.5 / 17.5, 8 x 512 rows 37.1 / 46.4, 2,048 rows 46.5 / 50.3; 4 x 130 rows of 32 heads
// in 8 groups 12.8 / 16.9; heads of 64, 2 x 1,000 rows 23.3 / 19.8.
inline bool wattn_teams(const int32_t* starts, const int32_t* lens, int n_seq, int heads, int groups, int dim, int vdim, int window, int keep) {
    const double most = (double)window + keep, R = heads / groups;
    auto pairs = [&](double n) { return n <= most ? n * (n + 1) / 2 : most * (most + 1) / 2 + (n - most) * most; };  // of positions 0 .. n - 1
    double tiles = 0, keys = 0, longest = 0;  // the last two in tiles of 64
    for (int r = 0; r < n_seq; ++r) {
        const double end = (double)starts[r] + lens[r];
        tiles += groups * std::ceil(lens[r] * R / 64);
        keys += groups * R * ((pairs(end) - pairs(starts[r])) / 4096 + 0.5 * lens[r] / 64);
        longest = std::max(longest, std::ceil(std::min(end, most) / 64) + (end > most));
    }
    const bool half = dim <= 64 && vdim <= 64;
    const double one = std::max(6.5 + 1.6 * longest, (2 * tiles + 1.45 * keys) / kRunCUs);
    const double two = std::max(std::max(7.5 + 2.2 * std::ceil(longest / 2), tiles > (half ? 2 : 1) * kRunCUs ? 2 * (7.5 + 2.2) : 0.0),
                                ((half ? 4.8 : 7.3) * tiles + 1.25 * keys) / kRunCUs);
    return two < one;
}

}  // namespace pgmi
