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
// candidates; with a low T most pairs would be candidates and the full score pass is faster.
// Finds in us by T, sieve / full pass (FP32 uploads; uint8 ones): 4096 x 4096 0.6: 103 / 54 (42),
// 0.65: 34 / 52 (41), 0.75: 33 / 47 (41); 16384 x 16384 0.6: 415 / 292 (181), 0.65: 72 / 233 (143),
// 0.75: 56 / 206 (134).  The line lies above the crossing of synthetic SIFT sets, for sets whose
// unrelated descriptors score higher.
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
// wave whose list overflowed hold kSieveFlood and are listed for the exact re-check (flags:
// left ones from 0, right ones from offR, counted at cntL and cntR; null: the decisions list
// them).
//
// Sets with many nearly equal rows, or rows that int8 holds badly, can have any number of
// candidates, and the full pass serves any sets at the same speed.  So a wave scores at most
// `limit` of them, the features of the waves that have more are re-checked exactly, and both have
// a bound: where the candidates of the waves with more than one round of them (64), summed in
// *scored, pass `mostScored`, or a side's listed features times the other side's count pass
// `mostListed`, the call is given to the full pass: *gate is set (for the kernels and the host that
// follow), its decisions are void, and the remaining waves neither score nor list.  gate null:
// no bound.
constexpr unsigned long long kSieveFlood = ~0ull;
constexpr int kSieveList = 512;  // a pair's largest limit

struct SieveBest {
    unsigned long long* best;
    unsigned* second;
    int offR;
    int limit;
    int* flags;
    int* cntL;
    int* cntR;
    unsigned* scored;
    unsigned mostScored;
    long long mostListed;
    int* gate;
};

// The bounds of `pairs` scores: about the full pass's time each (45 us of launches and a second
// wait, and 1.3 * 10^6 scores per us).  The card takes 3000 candidates per us, with their listing
// and entering, and re-checks 60000 pairs per us.  A wave's candidates are a chain of rounds of 64
// of about 10 us: one and a half for the short runs of small sets, whose full pass is short too,
// eight for long ones, which may hold a small cluster by themselves (SIFT sets have about ten
// candidates a wave).  Calls in us with a share of both sides in one cluster of nearly equal rows,
// 0 / 2 / 5 / 10 / 50%: 16384 x 16384 60 / 99 / 465 / 334 / 332, 8192 x 8192 41 / 48 / 106 / 281 / 154,
// 2048 x 2048 30 / 30 / 36 / 86 / 76; with lists of 2048 and no bounds 61 / 93 / 257 / 857 / 15555,
// 40 / 46 / 94 / 252 / 5885 and 29 / 29 / 35 / 54 / 435; with the FP32 instruction 740, 245 and 80 at
// any share.  Lower limits move the two lower figures of the middle up, higher ones the third.
__host__ __device__ inline unsigned sieve_most_scored(double pairs) { return (unsigned)(120000.0 + pairs / 700); }
inline long long sieve_most_listed(double pairs) { return (1LL << 20) + (long long)(pairs / 32); }
inline int sieve_limit(long long pairs)  // of a wave of `pairs` scores
{
    return pairs < 96 * 64 ? 96 : pairs < kSieveList * 64 ? (int)(pairs / 64) : kSieveList;
}

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
