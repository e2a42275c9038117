// The order in which a launch deals the pieces (rows, chunks of rows) of a large buffer to the eight XCDs.  No device code in it
// apart from xcd_piece, so that a host compiler takes it alone.
#pragma once

#include <stdint.h>

#include <initializer_list>

#ifdef __HIPCC__
#define TRLK_HOST_DEVICE __host__ __device__ __forceinline__
#else
#define TRLK_HOST_DEVICE inline
#endif

namespace trlk {

// Pieces of a large buffer in address order, dealt to the workgroups of a launch.  The hardware deals consecutive workgroups to
// the eight XCDs in turn; workgroup w of XCD w mod 8 takes the XCD's pieces in order, and those are runs of `run` neighbouring
// pieces, every eighth run of the buffer: what an XCD reads and writes at a time is one narrow window, and eight neighbouring
// windows move through the buffer together.  (Single pieces in turn have no such windows.  One contiguous eighth of the buffer
// per XCD has, but gives each XCD whole sequences: with completions of 1/16 of the longest to the longest an XCD gets up to a
// fifth more bytes than the mean, and the launch waits for it.)
TRLK_HOST_DEVICE int64_t xcd_piece(unsigned w, unsigned run) {
    const unsigned q = w >> 3, k = q / run;
    return (int64_t(k) * 8 + (w & 7)) * run + (q - k * run);
}
// The length of a run for `total` pieces, `period` of them per sequence, where `want` is wanted: short enough for 10 runs per XCD,
// and such that an XCD does not meet the same part of every sequence, one XCD the padding and another none.  That happens when
// the 8 runs of a round are about a sequence, or half of one: 1025 rows of 151936 16-bit logits per sequence, runs of 17 to
// 25 rows 2665-2680 us, 32 2716-2732, 64 2793, 128 2934-2950.  Rounds far shorter than a sequence cannot do it; longer ones
// are brought to a whole number of sequences and 0.382 or 0.618 of one (the golden section: the part of the sequence that
// an XCD meets keeps moving), the nearest that leaves 10 runs.  At last the rounds are made equally long: 12.4 of them give some
// XCDs 13 runs and others 12.  bf16, three draws of completions of 1/16 of the longest to the longest: [20, 585, 50264]
// 10 rounds 416 / 421 / 419 us, 12.3 407 / 416, 13.0 409 / 407 / 403, 17 409 / 406 / 403, 33 412 / 417 / 411; [10, 137, 151936] 7.2 rounds
// 182 / 171, 9.6 177 / 176 / 149, 15.7 180 / 167 / 151.
inline unsigned xcd_run(int64_t total, int64_t want, int64_t period) {
    const int64_t most = total < (int64_t(1) << 30) ? total / 80 : 1;
    int64_t run = want < most ? want : most;
    if (run <= 1) return 1u;
    const double round = 8.0 * double(run) / double(period), whole = double(int64_t(round));  // in sequences
    if (round > 0.382) {
        double best = 0.382;
        for (double c : {whole - 0.382, whole + 0.382, whole + 0.618, whole + 1.382}) {
            if (c <= 0.0 || c * double(period) > 8.0 * double(most)) continue;
            const double is = c < round ? round / c : c / round, was = best < round ? round / best : best / round;
            if (is < was) best = c;
        }
        run = int64_t(best * double(period) / 8.0 + 0.5);
        run = run < 1 ? 1 : run < most ? run : most;
    }
    const int64_t rounds = (total + 8 * run - 1) / (8 * run);
    return unsigned((total + 8 * rounds - 1) / (8 * rounds));
}
// Workgroups of the launch: whole rounds of runs; the pieces from `total` on do not exist.
inline unsigned xcd_grid(int64_t total, unsigned run) { return unsigned((total + 8 * run - 1) / (8 * run) * (8 * run)); }

}  // namespace trlk
