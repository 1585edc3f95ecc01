// Plain FP32 putative matching by a certified sieve: an int8 score pass finds the few pairs whose
// score can matter, those are scored exactly.
#pragma once
#include <hip/hip_runtime.h>

#include "v3dm_kernels.h"

namespace v3dm {

// Which scores can matter: a query is accepted when its best b1 > minScore and
// (2 - 2 b1) / max(0.001, 2 - 2 b2) < minRatio.  With b1 > minScore every second best
// b2 <= T = 1 - (1 - minScore) / minRatio passes the ratio, so a pair whose score is at most
// min(minScore, T) changes no decision.
//
// The sieve's rows: q = round(256 x) in [-127, 127] (SIFT components stay below 0.5), kept with
// r = ||x - q / 256||, so that x y <= q_x q_y / 65536 + r_x ||y|| + (||x|| + r_x) r_y whatever
// the rows hold.  The int8 products are exact in int32.
//
// Rule: sets in the range of the split pass (finite rows, v3dm_split.h), certification on, and
// T >= kSieveMin.  Unrelated SIFT descriptors score below that, so a query has a handful of
// candidates; with a lower T most pairs would be candidates and the full score pass is faster.
constexpr float kSieveMin = 0.75f;
constexpr float kSieveScale = 256.0f;
constexpr int kSieveTile = 32;
constexpr int kSieveTileBytes = kSieveTile * 128;
constexpr int kSieveGroup = 8;  // rows that share one residual (their largest)

// True with the bound *T where scores of at most *T cannot matter.
bool sieve_bound(float minScore, float minRatio, float* T);

// One side: n rows as int8 tiles (kSieveTileBytes per 32 rows: [16 components][row]), residuals
// per kSieveGroup rows, the FP32 rows.
struct SieveSet {
    signed char const* q;
    float const* res;
    float const* X;
    int n;
};

// Per query (left, then right at offR): the candidates' best as score bits << 32 | ~index, and
// the second best's bits.  Zero before a pass; the decisions leave them zero.  Features of a
// block whose list overflowed hold kSieveFlood and are listed for the exact re-check (flags:
// left ones from 0, right ones from offR, counted at cntL and cntR; null: the decisions list
// them).
constexpr unsigned long long kSieveFlood = ~0ull;

struct SieveBest {
    unsigned long long* best;
    unsigned* second;
    int offR;
    int* flags;
    int* cntL;
    int* cntR;
};

struct SievePlan {
    int groups = 1, splits = 1, tiles = 1;
};
SievePlan plan_sieve(int nL, int nR);

// bits: guided-matching bitmap (removed pairs are no candidates), or null.
void launch_sieve(SieveSet const& L, SieveSet const& R, SievePlan const& p, unsigned const* maxNormBits, float T,
                  SieveBest const& b, unsigned const* bits, int ldi, hipStream_t st);
// Decisions of all queries and the exact re-check of the listed ones, in one launch (buffers as
// launch_recheck_exact).
void launch_sieve_finish(float const* L, float const* R, int nL, int nR, SieveBest const& b, int const* flagList,
                         int rowsL, int rowsR, int const* counters, float minScore, float minRatio, int* colMax,
                         int* rowMax, Top2* part, int* tickets, unsigned const* gbits, int ldi, hipStream_t st);

}  // namespace v3dm
