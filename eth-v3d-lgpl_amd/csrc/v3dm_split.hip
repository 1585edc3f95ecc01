// Plain FP32 putative matching on FP16 matrix instructions (gfx950): the fused score pass of
// v3dm_fp32.hip with every descriptor split in two FP16 parts (v3dm_split.h).
//
// v_mfma_f32_32x32x2_f32 runs at 1/16 of v_mfma_f32_32x32x16_f16's rate; three FP16
// products per score give the FP32 product's accuracy at 3/16 of its matrix time.
//
// Reference path: V3D_CUDA::SIFT_Matching::findPutativeMatches
// (V3D/CUDA/v3d_cudamatching.cu:522-552); as there, scores, best and second best are FP32.
#include <type_traits>

#include "v3dm_batch.h"
#include "v3dm_device.h"
#include "v3dm_kernels.h"
#include "v3dm_split.h"

namespace v3dm {

typedef _Float16 v8h __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) void lds_void;

// ------------------------------------------------------------------------------ score pass
// Work-group: kW waves of 64 left features each (two 32-column blocks whose hi and lo parts
// are the resident B operands, 128 VGPRs), streaming 32-row tiles of right features through
// two LDS stages filled by direct global->LDS loads.  Why this shape: a tile's parts (16 KiB)
// are read from LDS once per wave for two column blocks, so 48 matrix instructions (1536
// cycles) stand against 16 KiB of operand reads, 16 KiB of the score transpose below (256
// LDS cycles a wave together, 1024 of the CU's per tile) and about 190 vector instructions
// (760 cycles) that the SIMD's other wave overlaps; 256 VGPRs leave two waves per SIMD, and
// the 76 KiB of LDS two work-groups per CU, which drift apart and fill each other's gaps.
// Counts are multiples of 32, so no tile and no column block is partial; a wave's second (or
// every) block past nL is skipped.
//
// Lane l holds column c = l % 32 and rows j = 8 (r / 4) + 4 (l / 32) + r % 4 of each 32x32
// block.  Per left feature the running top-2 stays in registers (the position
// looked for only where it can matter, see Selection); per right feature each wave
// writes its scores to its own LDS rows, reads them back a row per lane pair, and the waves'
// partial top-2 of a tile are merged by one of them after the next tile's barrier, so a tile
// costs one barrier.
//
// k index of matrix step s: h*64 + 8*s + v (h = l / 32); the parts of one score are added
// small products first (lo hi, hi lo, then hi hi) step by step.
//
// What bounds it: matrix instructions on real descriptors, which draw the card's power limit
// (the three products of 16384 x 16384 run at 1.13 PFLOP/s here; a loop of nothing but the
// instruction reaches 1.48, the library's 8192^3 product 1.2); the products and operand reads
// alone take 164 us of the 182.  16384 x 16384: 182 us against 605-635 us of k_fused_fp32;
// 8192 x 7936: 58 against 185 us.  One tile's selection after its products instead of beside
// the next tile's: 210 against 196 us; every position tracked instead of looked for: 215
// against 195 us; second bests left to the compiler's order (spills): 196 against 182 us.
// Most calls take the sieve (v3dm_sieve.h: 37 us); this pass serves low minimum scores, a zero
// error bound and blocks of scores.
//
// Integer rows (kInt): descriptors uploaded as uint8 are their integer components q times the
// row's scale d, the scale leaves the sum, and FP16 holds the integers exactly: ONE product per
// score gives the exact integer sum I <= 128 * 255^2 < 2^24, and the score is fl(fl(I d_j) d_i)
// (two roundings and the rows' own: |score - exact| <= 5.01 * 2^-24 score).  16 matrix
// instructions per wave and tile instead of 48, two multiplications per score more; the tile
// is 8 KiB, the B operands 64 VGPRs, and the right scales of a tile are loaded while the tile
// is multiplied, behind the last use of the previous tile's.
constexpr int kTRow = 36;  // floats per row of the transposed block

template <bool kInt>
struct SplitRows {
    static constexpr int kBytes = kInt ? kIntRowBytes : kSplitRowBytes;
    static constexpr int kTileBytes = kSplitTile * kBytes;
    static constexpr int kLoadRows = 1024 / kBytes;  // rows of one 1 KiB direct load
    static constexpr int kLoadStep = 1024 + 16;
    static constexpr int kStage = (kSplitTile / kLoadRows) * kLoadStep;
};

template <bool kInt, int kW>
struct SplitLds {
    __attribute__((aligned(16))) unsigned char stage[2][SplitRows<kInt>::kStage];
    __attribute__((aligned(16))) float trans[kW][2][kSplitTile * kTRow];
    float absent[kSplitTile * kTRow];  // where column blocks past nL write their scores
    float rowB1[2][kW][kSplitTile], rowB2[2][kW][kSplitTile];
    int rowA1[2][kW][kSplitTile];
};

// Stage layout: a direct load fills 1 KiB (two split rows or four integer rows as they lie in
// memory, lane L at +16 L) and the next load starts 16 bytes further on.  Within a load each
// lane fetches the chunk that belongs at its slot: split rows have hi and lo swapped in odd
// rows, integer row r has its 16 chunks at slot c ^ (4 (r % 4)).  The 16 rows that a group of
// lanes reads one chunk of then lie on distinct 16-byte columns of the 256 bytes of banks
// (with the 64-byte halves of split rows swapped instead, a quarter of the LDS cycles were
// conflicts), and a lane's chunks need two addresses with constant offsets: hi and lo, or
// steps 0-3 and 4-7.
template <bool kInt>
__device__ __forceinline__ int split_src(int tid)
{
    return kInt ? (tid * 16) ^ ((tid & 48) << 2) : (tid * 16) ^ ((tid & 32) << 2);
}

// One direct load of 1 KiB.  R (`bytes` long) as a raw buffer resource: a tile's loads take one
// scalar offset and the 32-bit lane offset (64-bit lane addresses would not leave room for the
// operands).
__device__ __forceinline__ void load_to_lds(unsigned char const* R, int bytes, unsigned char* to, int lane, int at)
{
    __builtin_amdgcn_raw_ptr_buffer_load_lds(
        __builtin_amdgcn_make_buffer_rsrc(const_cast<unsigned char*>(R), 0, bytes, 0x00027000), (lds_void*)to, 16, lane,
        at, 0, 0);
}

template <bool kInt, int kW>
__device__ __forceinline__ void split_stage(unsigned char const* __restrict__ R, int bytes, int t,
                                            unsigned char* stage, int src, int wv)
{
    using Rows = SplitRows<kInt>;
#pragma unroll
    for (int p = 0; p < kSplitTile / (Rows::kLoadRows * kW); ++p)
        load_to_lds(R, bytes, stage + (kW * p + wv) * Rows::kLoadStep, src, t * Rows::kTileBytes + p * (1024 * kW));
}

// Best and second best of a stream of scores, without the position: 13 instructions per 8
// scores (two triples by max3 / med3, a pair, three states merged by max3 / med3) where
// pushing them one by one with the position took 32.
struct Best2 {
    float b1, b2;
};

__device__ __forceinline__ float max3(float a, float b, float c) { return fmaxf(fmaxf(a, b), c); }

__device__ __forceinline__ Best2 best2_of8(float const (&x)[8])
{
    float const h0 = max3(x[0], x[1], x[2]), m0 = __builtin_amdgcn_fmed3f(x[0], x[1], x[2]);
    float const h1 = max3(x[3], x[4], x[5]), m1 = __builtin_amdgcn_fmed3f(x[3], x[4], x[5]);
    float const h2 = fmaxf(x[6], x[7]), m2 = fminf(x[6], x[7]);
    return Best2{max3(h0, h1, h2), fmaxf(__builtin_amdgcn_fmed3f(h0, h1, h2), max3(m0, m1, m2))};
}

__device__ __forceinline__ Best2 best2_merge(Best2 a, Best2 b)
{
    return Best2{fmaxf(a.b1, b.b1), max3(a.b2, b.b2, fminf(a.b1, b.b1))};
}

// A best or second best in score units; the initial state stays kInit.
__device__ __forceinline__ float split_back(float b, float back) { return b > -1e29f ? b * back : kInit; }

// The partial top-2 of tile t's right features from the waves' LDS entries.
template <bool kInt, int kW>
__device__ __forceinline__ void split_merge_rows(SplitLds<kInt, kW> const& lds, int t, int lane,
                                                 Top2* __restrict__ rowPart)
{
    if (lane >= kSplitTile) return;
    Top2 s = top2_init();
#pragma unroll
    for (int w = 0; w < kW; ++w)
        s = top2_merge(s, Top2{lds.rowB1[t & 1][w][lane], lds.rowB2[t & 1][w][lane], lds.rowA1[t & 1][w][lane]});
    if (!kInt) {
        s.b1 = split_back(s.b1, kSplitBack);
        s.b2 = split_back(s.b2, kSplitBack);
    }
    // transposed row 16 h + r holds row 8 (r / 4) + 4 h + r % 4 of the tile
    rowPart[t * kSplitTile + 8 * ((lane & 15) >> 2) + 4 * (lane >> 4) + (lane & 3)] = s;
}

// Computes x here: left to itself the compiler moves a second best past the rare branches to
// its next use and keeps every score it comes from in a register until then (spills).
__device__ __forceinline__ void settle(float& x) { __asm__ volatile("" : "+v"(x)); }

// Running state of one left feature: at = 16 * tile + r of the best, kept only while the
// best exceeds the caller's minimum score.
struct ColState {
    Best2 s;
    int at;
};

// Where a lane's stream position p (a multiple of 4) lies in its wave's transposed blocks.
constexpr int split_tr(int p) { return (p >> 4) * (kSplitTile * kTRow) + (p & 15); }

// The selection of one tile (both directions) in eight parts, one per matrix step of the
// next tile: parts 0-3 the left features (and the scores to LDS), parts 4-7 the right
// features, read back a part ahead.
//
// A position is looked for only where a new best exceeds thr (the caller's minimum score):
// a query whose best does not is rejected or re-checked exactly whatever the position, and a
// query that is accepted has its best above it.  At the usual 0.9 one tile in twenty of a
// wave holds such a score; with a minimum below most scores the search costs what tracking
// the position of every score would.
struct Selection {
    Best2 row;
    float old;
    float4 next[2];  // the coming columns
};

// What a tile's scores need besides the products: the guided bits of the lane's columns, or
// the scales of the lane's rows (element r: row 8 (r / 4) + 4 h + r % 4) of integer rows.
template <bool kInt>
struct TileSide {
    unsigned gw[2];
};
template <>
struct TileSide<true> {
    float4 d[4];
    __device__ __forceinline__ float scale(int r) const
    {
        float4 const v = d[r >> 2];
        return (r & 3) == 0 ? v.x : (r & 3) == 1 ? v.y : (r & 3) == 2 ? v.z : v.w;
    }
};

template <bool kGuided, bool kInt, int kW>
__device__ __forceinline__ void select_part(int part, Selection& x, v16f (&acc)[2], TileSide<kInt> const& side,
                                            float const (&dl)[2], ColState (&col)[2], int t, float* const (&tw)[2],
                                            float const* tr, SplitLds<kInt, kW>& lds, int wv, int lane, int i0,
                                            float thr)
{
    if (part < 4) {
        int const cb = part >> 1, r0 = 8 * (part & 1);
        float v[8];
#pragma unroll
        for (int r = 0; r < 8; ++r) {
            int const e = r0 + r;
            if constexpr (kInt) acc[cb][e] *= side.scale(e);
            else if (kGuided)
                acc[cb][e] = ((side.gw[cb] >> (8 * (e >> 2) + (e & 3))) & 1u) ? -1e20f / kSplitBack : acc[cb][e];
            v[r] = acc[cb][e];
            tw[cb][e * kTRow] = kInt ? v[r] * dl[cb] : v[r];
        }
        if (r0 == 0) x.old = col[cb].s.b1;
        col[cb].s = best2_merge(col[cb].s, best2_of8(v));
        settle(col[cb].s.b2);
        if (r0 != 0) {
            float const b = col[cb].s.b1;
            bool const better = b > x.old && (kInt ? b * dl[cb] : b) > thr;
            if (__builtin_expect(__builtin_amdgcn_ballot_w64(better) != 0, 0)) {
                int at = 0;
#pragma unroll
                for (int r = 15; r >= 0; --r) at = acc[cb][r] == b ? r : at;  // the first of equal bests
                col[cb].at = better ? 16 * t + at : col[cb].at;
            }
        }
        // the wave's own LDS rows: its writes come before its reads (LDS operations of one
        // wave are in order)
        if (part == 3) __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    } else {
        float const v[8] = {x.next[0].x, x.next[0].y, x.next[0].z, x.next[0].w,
                            x.next[1].x, x.next[1].y, x.next[1].z, x.next[1].w};
        Best2 const b = best2_of8(v);
        x.row = part == 4 ? b : best2_merge(x.row, b);
        settle(x.row.b2);
    }
    if (part >= 3 && part < 7) {
        x.next[0] = *reinterpret_cast<float4 const*>(tr + split_tr(8 * (part - 3)));
        x.next[1] = *reinterpret_cast<float4 const*>(tr + split_tr(8 * (part - 3) + 4));
    }
    if (part == 7) {
        // the two halves of the wave hold 32 columns of a row each; both end with the merged
        // state and write it
        float const o1 = __shfl_xor(x.row.b1, 32), o2 = __shfl_xor(x.row.b2, 32);
        Best2 const both = best2_merge(x.row, Best2{o1, o2});
        int a1 = -1;
        if (__builtin_expect(__builtin_amdgcn_ballot_w64(both.b1 > thr) != 0, 0)) {
            // position p of the lane's stream: column block p / 16, column 16 h + p % 16
            int q = 64;
#pragma unroll
            for (int p = 28; p >= 0; p -= 4) {
                float4 const v = *reinterpret_cast<float4 const*>(tr + split_tr(p));
                q = v.w == both.b1 ? p + 3 : q;
                q = v.z == both.b1 ? p + 2 : q;
                q = v.y == both.b1 ? p + 1 : q;
                q = v.x == both.b1 ? p : q;
            }
            int at = q == 64 ? 0x7fffffff : i0 + (q >> 4) * 32 + 16 * (lane >> 5) + (q & 15);
            at = min(at, __shfl_xor(at, 32));  // the first of equal bests
            a1 = both.b1 > thr ? at : -1;
        }
        lds.rowB1[t & 1][wv][lane & 31] = both.b1;
        lds.rowB2[t & 1][wv][lane & 31] = both.b2;
        lds.rowA1[t & 1][wv][lane & 31] = a1;
    }
}

// One work unit: left block lb (64 * kW features) against right tiles [t0, t1) -> colPart[i],
// rowPart[j] (the caller's split and left block offsets applied).  dL, dR: the rows' scales
// (kInt).
template <bool kGuided, bool kInt, int kW>
__device__ __forceinline__ void split_block(unsigned char const* __restrict__ L, unsigned char const* __restrict__ R,
                                            float const* __restrict__ dL, float const* __restrict__ dR, int nL, int lb,
                                            int t0, int t1, Top2* __restrict__ colPart, Top2* __restrict__ rowPart,
                                            unsigned const* __restrict__ bits, int ldi, SplitLds<kInt, kW>& lds,
                                            float thr)
{
    using Rows = SplitRows<kInt>;
    static_assert((long long)kSplitMaxTiles * Rows::kTileBytes < (1LL << 31), "32-bit offsets of a unit's tiles");
    // an opaque copy of the thread index: in the persistent kernel it keeps the per-lane
    // offsets derived from it inside the item loop instead of live across it
    int tid = threadIdx.x;
    __asm__ volatile("" : "+v"(tid));
    int const lane = tid & 63;
    int const wv = __builtin_amdgcn_readfirstlane(tid >> 6);
    int const h = lane >> 5;
    int const c32 = lane & 31;
    int const i0 = lb * (64 * kW) + wv * 64;
    int const nBlk = min(max((nL - i0) / 32, 0), 2);  // column blocks of this wave that exist

    int const src = split_src<kInt>(tid);
    // the resource spans the unit's own tiles: their offsets fit 32 bits (kSplitMaxTiles), an
    // image's need not (a tile of split rows is 16 KiB: from 2^17 tiles on they would not)
    R += (size_t)t0 * Rows::kTileBytes;
    int const bytes = (t1 - t0) * Rows::kTileBytes;
    split_stage<kInt, kW>(R, bytes, 0, lds.stage[0], src, wv);

    // rows past nL are inside the buffer (a multiple of kSplitRowPad rows) and never used
    v8h bh[2][8], bl[2][8];
    float dl[2] = {0.0f, 0.0f};
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        uint4 const* p = reinterpret_cast<uint4 const*>(L + (size_t)(i0 + cb * 32 + c32) * Rows::kBytes +
                                                        h * (Rows::kBytes / 2));
#pragma unroll
        for (int s = 0; s < 8; ++s) {
            bh[cb][s] = __builtin_bit_cast(v8h, p[s]);
            if (!kInt) bl[cb][s] = __builtin_bit_cast(v8h, p[8 + s]);
        }
        if (kInt) dl[cb] = dL[i0 + cb * 32 + c32];
    }

    // scores of a column block past nL go to `absent`; the rows read for it hold -3e30, below
    // the initial state, and never count
    float* tw[2];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        float* const own = lds.trans[wv][cb];
        tw[cb] = (cb < nBlk ? own : lds.absent) + 16 * h * kTRow + c32;
        if (cb >= nBlk)
            for (int k = lane; k < kSplitTile * kTRow; k += 64) own[k] = -3e30f;
    }
    float const* const tr = lds.trans[wv][0] + c32 * kTRow + 16 * h;

    ColState col[2];
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) col[cb] = ColState{Best2{kInit, kInit}, -1};
    TileSide<kInt> side{};  // of the tile whose selection comes next

    // the lane's half row of a stage
    int const at = kInt ? (c32 >> 2) * Rows::kLoadStep + (c32 & 3) * 256 + ((128 * h) ^ (64 * (c32 & 3)))
                        : (c32 >> 1) * Rows::kLoadStep + (c32 & 1) * 512 + h * 256;

    // Tile t's products into acc beside the selection of tile t - 1 from prev
    auto step = [&](int t, v16f(&acc)[2], v16f(&prev)[2], auto select) {
        wait_lds_loads();
        __syncthreads();  // tile t is staged; every wave is done with the other stage
        int const cur = (t - t0) & 1;
        if (t + 1 < t1) split_stage<kInt, kW>(R, bytes, t + 1 - t0, lds.stage[cur ^ 1], src, wv);
        // the partials of tile t - 2 were written before this barrier
        if (t >= t0 + 2 && wv == t % kW) split_merge_rows<kInt, kW>(lds, t - 2, lane, rowPart);
        TileSide<kInt> now{};
        if constexpr (kGuided && !kInt) {
#pragma unroll
            for (int cb = 0; cb < 2; ++cb)
                if (cb < nBlk) now.gw[cb] = bits[(size_t)t * ldi + i0 + cb * 32 + c32] >> (4 * h);
        }
        unsigned char const* const st = lds.stage[cur];
        acc[0] = v16f{};
        acc[1] = v16f{};
        Selection x;
        if constexpr (kInt) {
            // steps 0-3 and 4-7: the chunk's bit 6 is swapped with the row's
            unsigned char const* const A0 = st + at;
            unsigned char const* const A1 = st + at + ((c32 & 1) ? -64 : 64);
            v8h a = *reinterpret_cast<v8h const*>(A0);
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                v8h const b = a;
                if (s < 7) a = *reinterpret_cast<v8h const*>((s < 3 ? A0 : A1) + 16 * ((s + 1) & 3));
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b, bh[0][s], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(b, bh[1][s], acc[1], 0, 0, 0);
                if (decltype(select)::value) {
                    select_part<kGuided, kInt, kW>(s, x, prev, side, dl, col, t - 1, tw, tr, lds, wv, lane, i0, thr);
#pragma unroll
                    for (int k = 0; k < 2; ++k) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x080, 4, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 18, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
                if (s == 4) {  // the previous tile's scales are used up
#pragma unroll
                    for (int q = 0; q < 4; ++q)
                        side.d[q] = *reinterpret_cast<float4 const*>(dR + t * kSplitTile + 8 * q + 4 * h);
                }
            }
        } else {
            unsigned char const* const Ah = st + at + 128 * (c32 & 1);
            unsigned char const* const Al = st + at + 128 * (~c32 & 1);
            v8h al = *reinterpret_cast<v8h const*>(Al), ah = *reinterpret_cast<v8h const*>(Ah);
#pragma unroll
            for (int s = 0; s < 8; ++s) {
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh[0][s], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh[1][s], acc[1], 0, 0, 0);
                if (s < 7) al = *reinterpret_cast<v8h const*>(Al + 16 * (s + 1));
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl[0][s], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl[1][s], acc[1], 0, 0, 0);
                acc[0] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh[0][s], acc[0], 0, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh[1][s], acc[1], 0, 0, 0);
                if (s < 7) ah = *reinterpret_cast<v8h const*>(Ah + 16 * (s + 1));
                if (decltype(select)::value) {
                    select_part<kGuided, kInt, kW>(s, x, prev, side, dl, col, t - 1, tw, tr, lds, wv, lane, i0, thr);
                    // one matrix instruction per six of the selection's; nothing moves between steps
#pragma unroll
                    for (int k = 0; k < 6; ++k) {
                        __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
                        __builtin_amdgcn_sched_group_barrier(0x080, 2, 0);
                        __builtin_amdgcn_sched_group_barrier(0x002, 6, 0);
                    }
                    __builtin_amdgcn_sched_barrier(0);
                }
            }
            if constexpr (kGuided) side = now;
        }
    };
    v16f accA[2], accB[2];
    step(t0, accA, accB, std::false_type{});
    if constexpr (kInt) {
        int t = t0 + 1;
        for (; t + 1 < t1; t += 2) {
            step(t, accB, accA, std::true_type{});
            step(t + 1, accA, accB, std::true_type{});
        }
        if (t < t1) {
            step(t, accB, accA, std::true_type{});
            accA[0] = accB[0];
            accA[1] = accB[1];
        }
    } else {
        // one body and a copy: two bodies' addresses would not fit beside the operands
        for (int t = t0 + 1; t < t1; ++t) {
            step(t, accB, accA, std::true_type{});
            accA[0] = accB[0];
            accA[1] = accB[1];
        }
    }
    {
        Selection x;
#pragma unroll
        for (int s = 0; s < 8; ++s)
            select_part<kGuided, kInt, kW>(s, x, accA, side, dl, col, t1 - 1, tw, tr, lds, wv, lane, i0, thr);
    }
    __syncthreads();  // the last tiles' partials (and, in a persistent kernel, the stages)
    if (wv == t1 % kW) split_merge_rows<kInt, kW>(lds, t1 - 1, lane, rowPart);
    if (t1 - t0 >= 2 && wv == (t1 + 1) % kW) split_merge_rows<kInt, kW>(lds, t1 - 2, lane, rowPart);
#pragma unroll
    for (int cb = 0; cb < 2; ++cb) {
        int const p = col[cb].at;
        int const j = p < 0 ? -1 : (p >> 4) * kSplitTile + 8 * ((p & 15) >> 2) + 4 * h + (p & 3);
        Top2 cs{col[cb].s.b1, col[cb].s.b2, j};
        cs = top2_merge(cs, top2_shfl_xor(cs, 32));
        float const back = kInt ? dl[cb] : kSplitBack;
        cs.b1 = split_back(cs.b1, back);
        cs.b2 = split_back(cs.b2, back);
        if (h == 0 && cb < nBlk) colPart[i0 + cb * 32 + c32] = cs;
    }
}

template <bool kGuided, bool kInt>
__global__ __launch_bounds__(256, 2) void k_split_pass(unsigned char const* __restrict__ L,
                                                       unsigned char const* __restrict__ R,
                                                       float const* __restrict__ dL, float const* __restrict__ dR,
                                                       int nL, int nR, int leftBlocks, int tilesPerSplit,
                                                       Top2* __restrict__ colPart, int ldc,
                                                       Top2* __restrict__ rowPart, int ldr,
                                                       unsigned const* __restrict__ bits, int ldi, float thr,
                                                       int const* __restrict__ gate)
{
    if (gate && !*gate) return;
    __shared__ SplitLds<kInt, 4> lds;
    // neighbouring work-groups of one XCD share a split's right tiles in its L2
    int const b = xcd_block(blockIdx.x, gridDim.x);
    int const split = b / leftBlocks, lb = b - split * leftBlocks;
    int const t0 = split * tilesPerSplit;
    int const t1 = min(t0 + tilesPerSplit, nR / kSplitTile);
    split_block<kGuided, kInt, 4>(L, R, dL, dR, nL, lb, t0, t1, colPart + (size_t)split * ldc,
                                  rowPart + (size_t)lb * ldr, bits, ldi, lds, thr);
}

// Persistent form over a batch (as k_batch_fused_fp32): item = (pair, left block of 64 * kW
// features, split, 64-row right tiles per split).
template <bool kInt, int kW>
__global__ __launch_bounds__(64 * kW, 2) void k_batch_split(BatchDev b, int4 const* __restrict__ items, int nItems,
                                                            int const* __restrict__ nItemsDev,
                                                            int* __restrict__ queue, Top2* __restrict__ part,
                                                            float thr)
{
    __shared__ SplitLds<kInt, kW> lds;
    __shared__ int sItem;
    if (nItemsDev) nItems = __builtin_amdgcn_readfirstlane(min(nItems, *nItemsDev));  // written by an earlier kernel
    for (;;) {
        if (threadIdx.x == 0) sItem = atomicAdd(queue, 1);
        __syncthreads();  // also: every wave is done with the LDS of the previous item
        int const it = __builtin_amdgcn_readfirstlane(sItem);  // uniform: keeps the item in SGPRs
        __syncthreads();
        if (it >= nItems) break;
        int4 const w = items[it];
        BatchSeg const sl = b.seg[w.x];
        BatchSeg const sr = b.seg[b.nPairs + w.x];
        size_t const l0 = b.imgBase[sl.img], r0 = b.imgBase[sr.img];
        int const t0 = w.z * w.w * 2;
        int const t1 = min(t0 + 2 * w.w, sr.n / kSplitTile);
        split_block<false, kInt, kW>(b.split + l0 * SplitRows<kInt>::kBytes, b.split + r0 * SplitRows<kInt>::kBytes,
                                     kInt ? b.denom + l0 : nullptr, kInt ? b.denom + r0 : nullptr, sl.n, w.y, t0, t1,
                                     part + sl.partOff + (size_t)w.z * sl.ld, part + sr.partOff + (size_t)w.y * sr.ld,
                                     nullptr, 0, lds, thr);
    }
}

void launch_batch_split(BatchDev const& b, bool ints, int4 const* items, int nItems, int* queue, Top2* part, int grid,
                        int leftRows, float minScore, hipStream_t st, int const* nItemsDev)
{
    if (nItems <= 0) return;
    float const thr = ints ? minScore : minScore / kSplitBack;  // exact: a power of two
    dim3 const g(grid), t(leftRows);
    if (ints && leftRows == 256)
        hipLaunchKernelGGL((k_batch_split<true, 4>), g, t, 0, st, b, items, nItems, nItemsDev, queue, part, thr);
    else if (ints)
        hipLaunchKernelGGL((k_batch_split<true, 2>), g, t, 0, st, b, items, nItems, nItemsDev, queue, part, thr);
    else if (leftRows == 256)
        hipLaunchKernelGGL((k_batch_split<false, 4>), g, t, 0, st, b, items, nItems, nItemsDev, queue, part, thr);
    else
        hipLaunchKernelGGL((k_batch_split<false, 2>), g, t, 0, st, b, items, nItems, nItemsDev, queue, part, thr);
}

// The pass's scores of one 32x32 block per wave, written out (v3dm_score_block): the same
// operands, instructions and order as split_block.
__global__ __launch_bounds__(64) void k_split_scores(unsigned char const* __restrict__ L,
                                                     unsigned char const* __restrict__ R, int nRows, int nCols,
                                                     float* __restrict__ out)
{
    int const lane = threadIdx.x;
    int const h = lane >> 5;
    int const c32 = lane & 31;
    int const i0 = blockIdx.y * 32, j0 = blockIdx.x * 32;
    uint4 const* q = reinterpret_cast<uint4 const*>(L + (size_t)(i0 + c32) * kSplitRowBytes + h * 256);
    uint4 const* c = reinterpret_cast<uint4 const*>(R + (size_t)(j0 + c32) * kSplitRowBytes + h * 256);
    v16f acc = v16f{};
    for (int s = 0; s < 8; ++s) {
        v8h const ah = __builtin_bit_cast(v8h, c[s]), al = __builtin_bit_cast(v8h, c[8 + s]);
        v8h const bh = __builtin_bit_cast(v8h, q[s]), bl = __builtin_bit_cast(v8h, q[8 + s]);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(al, bh, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bl, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x16_f16(ah, bh, acc, 0, 0, 0);
    }
    int const i = i0 + c32;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
        int const j = j0 + 8 * (r >> 2) + 4 * h + (r & 3);
        if (i < nRows && j < nCols) out[(size_t)i * nCols + j] = acc[r] * kSplitBack;
    }
}

void launch_score_block_split(unsigned char const* L, unsigned char const* R, int nRows, int nCols, float* out,
                              hipStream_t st)
{
    dim3 const grid((nCols + 31) / 32, (nRows + 31) / 32);
    hipLaunchKernelGGL(k_split_scores, grid, dim3(64), 0, st, L, R, nRows, nCols, out);
}

// Splits of the right features: the work-groups run in rounds of 512 (two per CU), so the
// pass takes about ceil(groups / 512) * (tiles per split + the operand load and the column
// merge, about two tiles); the smallest of that, fewer splits on a tie.
FusedPlan plan_split(int nL, int nR)
{
    FusedPlan p;
    p.leftBlocks = (nL + 255) / 256;
    int const nTiles = nR / kSplitTile;
    int best = 0x7fffffff;
    for (int s = 1; s <= kMaxSplits && s <= nTiles; ++s) {
        int const tiles = (nTiles + s - 1) / s;
        int const splits = (nTiles + tiles - 1) / tiles;
        int const rounds = (int)(((long long)p.leftBlocks * splits + 511) / 512);
        int const cost = rounds * (tiles + 2);
        if (cost < best) {
            best = cost;
            p.splits = splits;
            p.tilesPerSplit = tiles;
        }
    }
    return p;
}

void launch_split_pass(SplitSet const& L, SplitSet const& R, FusedPlan const& p, Top2* colPart, int ldc,
                       Top2* rowPart, int ldr, unsigned const* bits, int ldi, float minScore, hipStream_t st,
                       int const* gate)
{
    if (L.n <= 0 || R.n <= 0) return;
    dim3 const grid(p.leftBlocks * p.splits);
    bool const ints = L.ints && R.ints && !bits;
    float const thr = ints ? minScore : minScore / kSplitBack;  // exact: a power of two
    if (ints)
        hipLaunchKernelGGL((k_split_pass<false, true>), grid, dim3(256), 0, st, L.ints, R.ints, L.scale, R.scale, L.n,
                           R.n, p.leftBlocks, p.tilesPerSplit, colPart, ldc, rowPart, ldr, bits, ldi, thr, gate);
    else if (bits)
        hipLaunchKernelGGL((k_split_pass<true, false>), grid, dim3(256), 0, st, L.split, R.split, nullptr, nullptr,
                           L.n, R.n, p.leftBlocks, p.tilesPerSplit, colPart, ldc, rowPart, ldr, bits, ldi, thr, gate);
    else
        hipLaunchKernelGGL((k_split_pass<false, false>), grid, dim3(256), 0, st, L.split, R.split, nullptr, nullptr,
                           L.n, R.n, p.leftBlocks, p.tilesPerSplit, colPart, ldc, rowPart, ldr, bits, ldi, thr, gate);
}

}  // namespace v3dm
