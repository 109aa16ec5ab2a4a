// Split query tiles of the pipelined prefill: when a launch splits them, which piece a workgroup
// runs, and the merge of the pieces. Shared by the tile launch (prefill_attn.hip) and the decode
// merge launch that takes the tile merge along (decode_attn.hip). Inline device code in
// namespace ptile; the kernels stay in those files.
//
// A tile workgroup walks its whole visible range, so a launch with fewer workgroups than CUs
// leaves CUs idle for as long as its longest tile takes. Where the batch fills at most half of
// them, the longest tile is cut into c = 256 / workgroups pieces (c workgroups for every one of
// that size are one round of the chip), the others into pieces of at most that length P, never
// under kSplitMinTiles. Each piece is a workgroup of its own that leaves unnormalised fp32 rows
// and (m, l) pairs for the merge.
//
// A key tile takes ~1.3 us at head dim 128 (half that at 64), while a split costs the merge
// (4-10 us) and a prologue per piece: tiles are split where that saves at least kSplitGain of
// them. Whole -> split, us a call replayed from a graph: 1 x (12,345 cached + 1,024 new) 32q/8kv
// 276 -> 213, 2 x (20,000 + 16) 32q/8kv 396 -> 63, 1 x (2,000 + 512) 16q/8kv 68 -> 41, 1 x 2,048
// 16q/8kv 56 -> 44, 1 x (900 + 200) 32q/8kv 36 -> 26, head dim 64 1 x (3,000 + 100) 32q/8kv
// 56 -> 31, fp8 1 x (8,000 + 1,024) 32q/8kv 249 -> 164. With 176-280 workgroups (2 x (1,000 + 700),
// 1 x 1,536 and 1 x 2,048 at 32q/8kv) pieces of unequal rounds and the merge lost 6-8 us, hence
// the half; at savings of 8-12 key tiles the two sides are even. An estimate of each of 16 piece
// lengths from a histogram of the pieces, on the device, found little better lengths and took
// 5 us itself.
//
// The host knows the widths of the table rows, not the lengths, so it can only tell that a launch
// may split (SplitRule); most such launches of short prompts over wide tables do not. The lengths
// are read where they are used: every wavefront of a tile workgroup and of the merge derives the
// plan from query_start_loc and context_lens, one request a lane, and no list is kept. At up to
// 2,048 positions such a launch needs no planner, which pays for the merge: 16q/8kv on a table of
// 128 blocks, without splits -> now, 1 x 200 new tokens 18.1 -> 15.0 us, 8 x 200 19.8 -> 16.5.
// Wider tables need it for the decode items, whose merge then takes the tiles' along: on 2,048
// blocks 1 x 200 21.3 -> 22.0, 8 x 200 22.9 -> 24.6, 4 x 200 with four single-token requests
// 27.5 -> 28.9 (the merge now comes after the tiles, with a wavefront per possible row). A word of
// the planner that spares both the plan where nothing splits took 0.3-0.9 us off these and cost
// every other prompt 0.2-0.4 (the tile kernel's start). An in-launch merge by the last piece would
// need agent-scope fences, which write back and invalidate the L2.
#pragma once

#include "attn_common.hpp"

namespace ccinfer::hipk::ptile {

constexpr int kKeysPerTile = 64;

// Heads per workgroup: the 8 wavefronts split as HPW heads x (8/HPW) row groups.
__host__ __device__ inline int heads_per_wg(int G) {
    return (G % 4 == 0) ? 4 : ((G % 2 == 0) ? 2 : 1);
}

// The pipelined tile kernel's workgroup.
template <int D>
struct PipeShape {
    static constexpr int kRows = 32;                     // query rows per wavefront
    static constexpr int kWaves = 8;
    static constexpr int kThreads = 64 * kWaves;
    static constexpr int kCPR = D / 8;                   // 16-byte chunks per K/V row
    static constexpr int kLoads = kKeysPerTile * kCPR / kThreads;  // per K or V
    static_assert(kKeysPerTile * kCPR % kThreads == 0, "staging must split evenly");
};

// The softmax reference of a row without a key yet.
constexpr float kMaxInit = -1.0e30f;

constexpr int kSplitCus = 256;
constexpr int kSplitMinTiles = 4;
constexpr int kSplitGain = 14;       // key tiles at head dim 128
constexpr int kSplitRequests = 64;   // one request a lane
constexpr int kWhole = 0x7fffffff;

// What the host passes of a launch that may split; batch = 0: it may not.
struct SplitRule {
    const int32_t* qsl = nullptr;
    const int32_t* context_lens = nullptr;
    int batch = 0;
    int total_tokens = 0;
    int tile_tokens = 0;
    int units = 0;    // workgroups per tile
    int gain = 0;     // key tiles a split has to save
    int key_cap = 0;  // positions a table row can hold
};

// The piece length P (key tiles) for `tiles` query tiles whose longest has `longest` key tiles
// (kWhole: no split). The host calls it with the fewest tiles and the longest table row possible,
// to see whether a launch may split at all. At most kSplitCus / units pieces come out: a tile has
// at most c of them.
__host__ __device__ inline int split_length(int tiles, int units, int longest, int gain) {
    const int wgs = tiles * units;
    const int c = wgs > 0 ? kSplitCus / wgs : kSplitCus;
    if (c < 2) return kWhole;
    int P = (longest + c - 1) / c;
    if (P < kSplitMinTiles) P = kSplitMinTiles;
    return longest - P >= gain ? P : kWhole;
}

// A workgroup's work (times the head units): the query tile from row t0 of request req on (query
// rows qb .. qb + rows, after `prefix` cached positions), against the key tiles [kt0, kt1) of its
// range (or to the range's end, if that comes first). pieces: those of the query tile; with more
// than one, the partial rows go to slot `slot`.
struct TilePiece {
    int req, qb, rows, prefix;
    int t0, kt0, kt1, slot, pieces;
};

__device__ __forceinline__ int key_tiles(const SplitRule& a, int keys) {
    return (min(keys, a.key_cap) - 1) / kKeysPerTile + 1;
}

// The plan of a batch: lane b holds request b's first query row, rows, cached prefix and query
// tiles (n, inclusive sums in incl); single-token requests have none. The rest is the same in
// every lane.
struct SplitPlan {
    int qb, rows, prefix, n, incl;
    int total;  // query tiles
    int P;      // key tiles a piece may have (kWhole: tiles are whole)
    int per;    // pieces the longest tile has
};

__device__ __forceinline__ SplitPlan split_plan(const SplitRule& a) {
    const int lane = threadIdx.x & 63;
    SplitPlan s{0, 0, 0, 0, 0, 0, kWhole, 1};
    int longest = 0;
    if (lane < a.batch) {
        s.qb = a.qsl[lane];
        const int qe = a.qsl[lane + 1];
        const int qlen = qe - s.qb;
        s.rows = min(qe, a.total_tokens) - s.qb;
        s.prefix = a.context_lens[lane] - qlen;
        if (qlen > 1 && s.prefix >= 0 && s.qb >= 0 && s.rows > 0) {
            s.n = (s.rows + a.tile_tokens - 1) / a.tile_tokens;
            longest = key_tiles(a, s.prefix + s.rows);
        }
    }
    // Sums and maxima up to each lane by DPP moves (row_shr 1 / 2 / 4 / 8 in rows of 16 lanes,
    // then each row's last lane to the rows after it): shuffles through LDS took 1-2 us here.
    s.incl = s.n;
#define CCI_SCAN(ctrl, rows)                                                                     \
    s.incl += __builtin_amdgcn_update_dpp(0, s.incl, ctrl, rows, 0xf, false);                     \
    longest = max(longest, __builtin_amdgcn_update_dpp(0, longest, ctrl, rows, 0xf, false))
    CCI_SCAN(0x111, 0xf);
    CCI_SCAN(0x112, 0xf);
    CCI_SCAN(0x114, 0xf);
    CCI_SCAN(0x118, 0xf);
    CCI_SCAN(0x142, 0xa);
    CCI_SCAN(0x143, 0xc);
#undef CCI_SCAN
    s.total = __builtin_amdgcn_readlane(s.incl, 63);
    longest = __builtin_amdgcn_readlane(longest, 63);
    s.P = __builtin_amdgcn_readfirstlane(split_length(s.total, a.units, longest, a.gain));
    if (s.P != kWhole) s.per = __builtin_amdgcn_readfirstlane((longest + s.P - 1) / s.P);
    return s;
}

// Piece k of query tile `tile`; false where there is none. The first cost % c of a tile's c
// pieces have cost / c + 1 key tiles, the others cost / c.
__device__ __forceinline__ bool split_piece(const SplitRule& a, const SplitPlan& s, int tile, int k,
                                            TilePiece* out) {
    if (tile >= s.total) return false;
    const int b = __builtin_popcountll(__builtin_amdgcn_ballot_w64(s.incl <= tile));
    const int first = __builtin_amdgcn_readlane(s.incl, b) - __builtin_amdgcn_readlane(s.n, b);
    const int t0 = (tile - first) * a.tile_tokens;
    const int rows = __builtin_amdgcn_readlane(s.rows, b);
    const int prefix = __builtin_amdgcn_readlane(s.prefix, b);
    const int cost = key_tiles(a, prefix + min(t0 + a.tile_tokens, rows));
    const int c = s.P == kWhole ? 1 : __builtin_amdgcn_readfirstlane((cost + s.P - 1) / s.P);
    if (k >= c) return false;
    const int len = __builtin_amdgcn_readfirstlane(cost / c);
    const int more = cost - len * c;
    const int kt0 = k * len + min(k, more);
    const int kt1 = kt0 + len + (k < more ? 1 : 0);
    const int qb = __builtin_amdgcn_readlane(s.qb, b);
    *out = TilePiece{b, qb, rows, prefix, t0, kt0, kt1, tile * s.per + k, c};
    return true;
}

// The arguments of a tile merge: rows of a launch's split tiles, from the partials to `out`.
struct TileMerge {
    SplitRule rule;
    __bf16* out = nullptr;
    const float* part_o = nullptr;
    const float* part_ml = nullptr;
    int hq = 0, hkv = 0, dr = 0;
    int max_tiles = 0;  // query tiles at most
};

// Workgroups (of four wavefronts) of a merge: a tile has units * 8 * D / 32 wavefronts (a multiple
// of four).
inline int tile_merge_wgs(const TileMerge& t, int D) {
    const int tiles = t.max_tiles < kSplitCus / 2 / t.rule.units ? t.max_tiles
                                                                  : kSplitCus / 2 / t.rule.units;
    return tiles * t.rule.units * (PipeShape<64>::kWaves * (D / 32) / 4);
}

// Log-sum-exp merge of the pieces of split tiles. One wavefront (wi) per (query tile, unit,
// wavefront of the tile kernel, 32-dim block n): it reads the partials in the tile kernel's own
// lane layout, so every load is a whole kilobyte, and stores the rows as that kernel's epilogue
// does. Wavefronts of tiles that are whole, or not there, leave at once. Bound by the latency of
// its loads: with the pieces of a batch loaded together, 2 x (20,000 + 16) takes 10 % less a call
// than with a loop left to the scheduler (8 pieces at a time: the same; 1 x 2,048, whose tiles have
// two pieces, then 4 % more).
template <int D, bool kPad>
__device__ __forceinline__ void merge_tile_pieces(const TileMerge& t, int wi) {
    constexpr int kPipeWaves = PipeShape<D>::kWaves;
    constexpr int kPipeRows = PipeShape<D>::kRows;
    constexpr int NT2 = D / 32;
    const int ds = kPad ? t.dr : D;
    const int G = t.hq / t.hkv;
    const int HPW = heads_per_wg(G);
    const int WPH = kPipeWaves / HPW;
    const int U = t.rule.units;
    const int lane = threadIdx.x & 63;
    const int n = wi % NT2;
    const int wave = wi / NT2 % kPipeWaves;
    const int u = wi / (NT2 * kPipeWaves) % U;
    const SplitPlan plan = split_plan(t.rule);
    TilePiece st;
    if (!split_piece(t.rule, plan, wi / (NT2 * kPipeWaves * U), 0, &st) || st.pieces < 2) return;
    const int tw = st.t0 + (wave % WPH) * kPipeRows;
    if (tw >= st.rows) return;
    const int q_head = u / (G / HPW) * G + u % (G / HPW) * HPW + wave / WPH;
    const int c32 = lane & 31;
    const int h32 = lane >> 5;
    const int64_t wv0 = (static_cast<int64_t>(st.slot) * U + u) * kPipeWaves + wave;
    const int64_t step = static_cast<int64_t>(U) * kPipeWaves;
    float mmax = kMaxInit;
#pragma unroll 8
    for (int p = 0; p < st.pieces; ++p)
        mmax = fmaxf(mmax, t.part_ml[((wv0 + p * step) * kPipeRows + c32) * 2]);
    f32x4 acc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
    float l = 0.f;
    // kBatch pieces' loads in flight at a time (past the last piece: a repeat of it, which is not
    // added: a row that V made infinite would become NaN by 0 * Inf)
    constexpr int kBatch = 4;
    for (int p0 = 0; p0 < st.pieces; p0 += kBatch) {
        f32x2 ml[kBatch];
        f32x4 o[kBatch][4];
#pragma unroll
        for (int x = 0; x < kBatch; ++x) {
            const int64_t wv = wv0 + min(p0 + x, st.pieces - 1) * step;
            ml[x] = *reinterpret_cast<const f32x2*>(t.part_ml + (wv * kPipeRows + c32) * 2);
            const f32x4* po = reinterpret_cast<const f32x4*>(t.part_o) + wv * (NT2 * 4 * 64) +
                              n * 4 * 64 + lane;
#pragma unroll
            for (int i = 0; i < 4; ++i) o[x][i] = po[i * 64];
        }
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int x = 0; x < kBatch; ++x) {
            if (p0 + x >= st.pieces) break;
            const float w = __builtin_amdgcn_exp2f(ml[x][0] - mmax);
            l += ml[x][1] * w;
#pragma unroll
            for (int i = 0; i < 4; ++i) acc[i] = acc[i] + o[x][i] * w;
        }
    }
    const int tq = tw + c32;
    if (tq >= st.rows) return;
    const float inv = l > 0.f ? 1.f / l : 0.f;
    __bf16* o = t.out + (static_cast<int64_t>(st.qb + tq) * t.hq + q_head) * ds;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
        if (kPad && 32 * n + 8 * i + 4 * h32 >= t.dr) continue;  // padded dims
        u32x2 w;
        w[0] = pack_bf16x2(acc[i][0] * inv, acc[i][1] * inv);
        w[1] = pack_bf16x2(acc[i][2] * inv, acc[i][3] * inv);
        *reinterpret_cast<u32x2*>(o + 32 * n + 8 * i + 4 * h32) = w;
    }
}

}  // namespace ccinfer::hipk::ptile
