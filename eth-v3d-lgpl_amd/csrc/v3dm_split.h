// The FP32 score pass on FP16 matrix instructions: descriptors split in two FP16 parts.
#pragma once
#include <hip/hip_runtime.h>

#include "v3dm_kernels.h"

namespace v3dm {

// A descriptor component x is held as x * 2^14 = hi + lo, hi = fp16(x * 2^14) and lo =
// fp16(x * 2^14 - hi), both to nearest even (the difference is exact in FP32): 22 to 24
// significant bits.  A dot product is the sum of hi hi + hi lo + lo hi (products of FP16
// numbers are exact in FP32, the sums are FP32), i.e. 2^28 times the score.
//
// Range rule: the fixed scale needs |x| < 2 (2^15 in FP16) and parts well above the smallest
// FP16 number 2^-24.  Sets whose rows all have a norm of 0 or in [kSplitNormMin,
// kSplitNormMax) are taken (SIFT descriptors are unit vectors); any other set (NaN, infinite,
// tiny, huge or widely scaled rows) goes to the FP32 instruction (v3dm_fp32.hip).
//
// Error: |x 2^14 - hi - lo| <= 2^-22 |x| 2^14 + 2^-25 and the dropped lo lo is at most 2^-22
// of its product, so with 24 FP32 accumulations |score error| <= (3 * 2^-22 + 24 * 2^-23)
// ||q|| ||c|| + 2^-39 sqrt(128) (||q|| + ||c||), and with norms of at least 2^-10 the last
// term is below 2^-24 ||q|| max||c||: within the 2^-15 that the certified decisions assume.
// Measured on unit descriptors it is below the FP32 instruction's (v3dm_split.hip).
//
// The certified decisions take epsRel (2^-15 unless the caller sets it), the FP32 instruction's
// bound with a factor 2, times kSplitEps for split rows (2^-17: a factor 2 on the bound above)
// and kIntEps for integer rows (2^-21: |score - exact| <= 5.01 * 2^-24 score), so that fewer
// queries are left open (16384 x 16384: 16 of 32768 at 2^-15).
constexpr float kSplitEps = 0.25f;
constexpr float kIntEps = 0.015625f;
constexpr float kSplitScale = 16384.0f;
constexpr float kSplitBack = 3.7252902984619140625e-09f;  // 2^-28
constexpr float kSplitNormMin = 0.0009765625f;            // 2^-10
constexpr float kSplitNormMax = 2.0f;
constexpr int kIntRowBytes = 256;    // integer components in FP16
constexpr int kSplitRowBytes = 512;  // per half (64 components): 128 B of hi, 128 B of lo
constexpr int kSplitRowPad = 256;    // split buffers hold a multiple of 256 rows
constexpr int kSplitTile = 32;       // right features per tile
constexpr int kSplitMaxTiles = 1 << 16;  // tiles of one work unit: their byte offsets fit 32 bits

// One feature set in one launch: its FP32 rows X (copied from the device array src, or
// dequantised from the uint8 rows src as SIFT_Feature::normalizeDescriptor, or in place), the
// norms and the set's largest norm (as launch_norms), the sieve's int8 rows and residuals
// (v3dm_sieve.h) and the scales of uint8 rows.  n: a multiple of 32.  maxNorm: 8 bytes, the norm's
// bits under the epoch, which grows from call to call (the 8 bytes start at zero); *hostFit
// (mapped host memory): set to 0 when the set is out of the split pass's range.
enum RowSource { kRowsInPlace, kRowsF32, kRowsU8 };
constexpr int kPrepGroups = 256;
void launch_prep_rows(RowSource from, void const* src, float* X, int n, float* norm, unsigned int* maxNorm,
                      unsigned epoch, float* scale, signed char* q8, float* res, int* hostFit, hipStream_t st);

// The rows of the full pass of two sets in range: split rows, and of sets with scales the
// components as FP16 integers (ints null: none).
struct SplitRowsOf {
    float const* X;
    float const* scale;
    unsigned char* split;
    unsigned char* ints;
    int n;
};
// gated: the call's counters, for a launch that does nothing unless its sieve gave the call to the
// full pass (counters[kCntGate]); null: always.  The same for `gate` below.
void launch_split_sets(SplitRowsOf const& a, SplitRowsOf const& b, int* gated, hipStream_t st);

// One side of a score pass: n split rows, and for sets uploaded as uint8 their components as
// FP16 integers with the rows' scales (else null).  All padded to kSplitRowPad rows.
struct SplitSet {
    unsigned char const* split;
    unsigned char const* ints;
    float const* scale;
    int n;
};

// Score pass of two sets in range: colPart[split][i], rowPart[leftBlock][j] as
// launch_fused_fp32, with left blocks of 256 features and tiles of 32 right features; on the
// integers where both sides have them.  bits: guided-matching bitmap (pairs scored -1e20), or
// null.  A partial's index is -1 where its best does not exceed minScore.
FusedPlan plan_split(int nL, int nR);
void launch_split_pass(SplitSet const& L, SplitSet const& R, FusedPlan const& p, Top2* colPart, int ldc,
                       Top2* rowPart, int ldr, unsigned const* bits, int ldi, float minScore, hipStream_t st,
                       int const* gate = nullptr);

// Measurement: the scores of the split pass, out[i * nCols + j] (as launch_score_block).
void launch_score_block_split(unsigned char const* L, unsigned char const* R, int nRows, int nCols, float* out,
                              hipStream_t st);

}  // namespace v3dm
