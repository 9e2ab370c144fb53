// C-ABI host dispatch for the gfx950 attention forward.
//
// Mirrors the reference dispatch src/bshd.hip:1-38: the same argument checks
// in the same order (all before any HIP call), config 0 -> auto selection,
// config -> kernel instantiation, and hipGetLastError() after the launch.
#include "fav4_bshd.h"
#include "bshd_kernel.hpp"

#include <algorithm>
#include <atomic>
#include <climits>
#include <cmath>
#include <cstdint>

namespace {

// Most workgroups in a grid dimension.  Larger decode chunk and merge grids loop
// inside the kernel, the other kernels take a second dimension (item_grid).
constexpr int64_t MAX_GRID = int64_t(1) << 22;

// CU count of the current device (256 if it cannot be read), cached per
// device after the first query.
int device_cus() {
    static std::atomic<int> cache[64];
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess) return 256;
    const bool slot = dev >= 0 && dev < 64;
    if (slot && (cus = cache[dev].load(std::memory_order_relaxed)) > 0) return cus;
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    if (slot) cache[dev].store(cus, std::memory_order_relaxed);
    return cus;
}

// One workgroup per item, in rows of at most MAX_GRID (a grid dimension holds
// fewer than 2^32 threads).
dim3 item_grid(int64_t total) {
    const int64_t rows = (total + MAX_GRID - 1) / MAX_GRID;
    return dim3(unsigned((total + rows - 1) / rows), unsigned(rows));
}

template <int WAVES, int BN, int STAGES, bool PIPE, bool CAUSAL>
int launch(const Fav4Args& a, const fav4::Layout& L, hipStream_t stream) {
    constexpr int BM = WAVES * 32;
    const int tiles = (a.sq + BM - 1) / BM;
    const int64_t bh = int64_t(a.batch) * a.heads;
    // Causal q tiles go in pairs of equal cost unless each has a CU of its own
    // (B3 H5 S1500, 180 q tiles: 33.8 us paired, 29.4 not; B4 H16 S2048 in
    // config 1, 1024 q tiles: 82 and 113).
    const bool paired = CAUSAL && bh * tiles > device_cus();
    const int64_t total = bh * fav4::items_per_head(tiles, paired);
    if (total > INT_MAX) return hipErrorInvalidValue;
    const dim3 grid = item_grid(total);
    if (a.lse)
        hipLaunchKernelGGL((fav4::fwd_kernel<WAVES, BN, CAUSAL, true, STAGES, PIPE>), grid, dim3(WAVES * 64), 0,
                           stream, a, L, tiles, int(total), paired);
    else
        hipLaunchKernelGGL((fav4::fwd_kernel<WAVES, BN, CAUSAL, false, STAGES, PIPE>), grid, dim3(WAVES * 64), 0,
                           stream, a, L, tiles, int(total), paired);
    return hipGetLastError();
}

template <bool CAUSAL>
int dispatch(const Fav4Args& a, const fav4::Layout& L, int config, hipStream_t stream) {
    switch (config) {
    case 1: return launch<4, 64, 2, false, CAUSAL>(a, L, stream);
    case 2: return launch<8, 64, 2, false, CAUSAL>(a, L, stream);
    case 3: return launch<8, 64, 3, true, CAUSAL>(a, L, stream);
    default: return hipErrorInvalidValue;
    }
}

// Argument checks of src/bshd.hip:27-34, in the same order, before any HIP call.
// kv_heads: heads of K/V (0 = heads, the reference's case); the key-side
// overflow limit counts those, as K/V rows are kv_heads * 256 bytes apart.
int validate(const Fav4Args* a, int causal, int config, int kv_heads = 0) {
    if (!a || !a->q || !a->k || !a->v || !a->o || a->batch <= 0 || a->heads <= 0 || a->sq <= 0 ||
        a->sk <= 0 || (causal != 0 && causal != 1) || config < 0 || config > 3 ||
        !std::isfinite(a->scale) || a->scale <= 0)
        return hipErrorInvalidValue;
    if (kv_heads == 0) kv_heads = a->heads;
    if (kv_heads < 0 || kv_heads > a->heads || a->heads % kv_heads != 0) return hipErrorInvalidValue;
    if (a->batch > INT_MAX / a->heads || a->heads > INT_MAX / 128 ||
        a->sq > INT_MAX / (a->heads * 128) || a->sk > INT_MAX / (kv_heads * 128) ||
        ((reinterpret_cast<uintptr_t>(a->q) | reinterpret_cast<uintptr_t>(a->k) |
          reinterpret_cast<uintptr_t>(a->v) | reinterpret_cast<uintptr_t>(a->o)) & 15))
        return hipErrorInvalidValue;
    return hipSuccess;
}

// Contiguous BSHD Q/O [B, Sq, H, 128] and K/V [B, Sk, kv_heads, 128].
fav4::Layout bshd_layout(const Fav4Args& a, int kv_heads) {
    fav4::Layout L;
    const int64_t row = int64_t(a.heads) * fav4::ROW_BYTES, kvrow = int64_t(kv_heads) * fav4::ROW_BYTES;
    L.qr = L.orow = uint32_t(row);
    L.kr = L.vr = uint32_t(kvrow);
    L.qb = L.ob = row * a.sq;
    L.kb = L.vb = kvrow * a.sk;
    L.qh = L.oh = L.kh = L.vh = fav4::ROW_BYTES;
    L.group = a.heads / kv_heads;
    return L;
}

// One tensor's element strides, checked: non-negative, multiples of 8
// elements (every row starts 16-byte aligned), the rows of one (batch, head)
// slice within a 4 GiB buffer bound, and the whole view within 2^48 bytes (so
// no address computation can overflow).
bool stride_ok(const Fav4Strides* st, int batch, int heads, int rows) {
    if (!st || st->batch < 0 || st->seq <= 0 || st->head < 0 || ((st->batch | st->seq | st->head) & 7))
        return false;
    if ((int64_t(rows) - 1) * static_cast<__int128>(st->seq) * 2 + fav4::ROW_BYTES > int64_t(UINT32_MAX))
        return false;
    const __int128 span = static_cast<__int128>(batch - 1) * st->batch + static_cast<__int128>(heads - 1) * st->head +
                          static_cast<__int128>(rows - 1) * st->seq + fav4::D;
    return span * 2 <= (static_cast<__int128>(1) << 48);
}

// ---- split-KV -------------------------------------------------------------
constexpr int MIN_TILES_PER_SPLIT = 4;   // Auto keeps >= 4 key tiles per chunk
constexpr int MAX_SPLIT_SQ = 1 << 22;    // keeps a chunk's O rows under a 4 GiB buffer bound
constexpr int DECODE_SQ = 32;            // up to this many queries: the one-wave decode shape

// Tile shape that a plan assumes: 8 waves x 256-row q tiles x 64-key tiles (one
// workgroup fills a CU), or for decode 1 wave x 32 rows x 32-key tiles (three
// workgroups per CU, each with 48 KiB of LDS).  Packed and paged prefill may
// run 128-row tiles instead (packed_prefill_run).
struct SplitShape {
    int bm, bn, wgs_per_cu, auto_max;
};
SplitShape split_shape(const Fav4Args& a) {
    if (a.sq <= DECODE_SQ) return {32, 32, 3, 128};
    return {256, 64, 1, 64};
}

struct SplitPlan {
    int splits, tps;   // chunks and key tiles per chunk
    SplitShape shape;
    int tiles;         // q tiles per item
    int64_t items;     // (batch, head) items, or (batch, K/V head) groups for decode
    int ranges = 0;    // decode over equal ranges of the packed keys: workgroups per (K/V head, q tile); 0: not
};

// Auto for prefill (Sq > 32).  Filling the CUs is not enough: on the small
// grids where splitting is considered, the unsplit forward runs 128-row q
// tiles two per CU, while the split kernel runs 256-row (q tile, chunk) items
// one per CU with higher fixed costs.  Auto therefore keeps, among
// 1..max_splits chunks, the count with the lowest predicted time.  The model
// (microseconds) was fitted to graph-timed MI355X runs of 23 shapes (B1-4, H1-64,
// Sq 256-16384, Sk up to 65536) with earlier kernels, whose causal forward
// always paired a heavy q tile with a light one and whose packed forward
// launched every q tile up to the longest sequence.  With the present ones, on
// 70 random shapes of that range, its choice is 4.7% behind the fastest
// measured on average: 49 shapes within 2%, 13 over 10%, the worst 1.5x (B4 H1
// 510 x 1495 dense unsplit 29.6 us, in 6 chunks 19.5), none slower than with the
// kernels that it was fitted to by more than 3%:
//  * unsplit: rounds * (9 + c per 64-key tile of an item), an item being a
//    q tile (dense; c = 0.9 with at most one workgroup per CU, else 1.0) or
//    the heaviest tile pair (causal; c = 1.0);
//  * split: rounds * (F + c per 64-key tile of a chunk) + 5 for the merge,
//    F = 19 and c = 1.8 dense, F = 18 and c = 1.5 causal;
// where rounds = work items / resident workgroups, rounded up.
// Bottom-right causal (br): the packed (varlen) entry point runs one chunk
// on its unsplit kernel, one item per (sequence, head, q tile) and no pairs
// (br_unsplit; priced as rounds * 9 plus the larger of the average work per
// workgroup slot and the heaviest item); the paged entry point runs one chunk
// on the split kernels (priced as split_time(1)).
int prefill_auto_splits(const Fav4Args& a, int causal, int max_splits, int ktiles, bool br, bool br_unsplit) {
    const int64_t cus = device_cus();
    const int64_t bh = int64_t(a.batch) * a.heads;
    const int keys = causal ? std::min(a.sk, a.sq) : a.sk;
    // Key tiles visible to a q tile whose rows end at rows_end (bottom-right:
    // the last row sees keys up to rows_end - 1 + sk - sq).
    auto vis_tiles = [&](int64_t rows_end) {
        int64_t vis = causal ? std::min<int64_t>(keys, rows_end) : keys;
        if (br) vis = std::min<int64_t>(keys, std::max<int64_t>(0, std::min<int64_t>(rows_end, a.sq) + a.sk - a.sq));
        return int((vis + 63) / 64);
    };
    const int nt128 = (a.sq + 127) / 128;
    double best;
    if (causal) {
        const int npairs = (nt128 + 1) / 2;
        int heavy = 0;
        for (int i = 0; i < npairs; ++i) {
            const int j = nt128 - 1 - i;
            heavy = std::max(heavy, vis_tiles(128LL * (i + 1)) + (j != i ? vis_tiles(128LL * (j + 1)) : 0));
        }
        best = double((bh * npairs + 2 * cus - 1) / (2 * cus)) * (9.0 + 1.0 * heavy);
    } else {
        const int64_t items = bh * nt128;
        best = double((items + 2 * cus - 1) / (2 * cus)) * (9.0 + (items <= cus ? 0.9 : 1.0) * ktiles);
    }
    const double fixed = causal || br ? 18.0 : 19.0, per_tile = causal || br ? 1.5 : 1.8;
    const int nt256 = (a.sq + 255) / 256;
    auto split_time = [&](int s) {
        const int tps = (ktiles + s - 1) / s;
        int64_t items = 0;
        for (int i = 0; i < nt256; ++i) items += (vis_tiles(256LL * (i + 1)) + tps - 1) / tps;
        return double((bh * items + cus - 1) / cus) * (fixed + per_tile * tps) + 5.0;
    };
    if (br && br_unsplit) {
        // fwd_kernel_varlen's tile rule: 128-row tiles for sq <= 1024 or when
        // 256-row tiles would leave CUs idle (two workgroups per CU), else 256.
        const bool small = a.sq <= 1024 || bh * ((a.sq + 255) / 256) < cus;
        const int bm = small ? 128 : 256;
        const int nt = (a.sq + bm - 1) / bm;
        const int64_t slots = small ? 2 * cus : cus;
        int64_t sum = 0;
        int heavy = 0;
        for (int i = 0; i < nt; ++i) {
            const int w = vis_tiles(int64_t(bm) * (i + 1));
            sum += w;
            heavy = std::max(heavy, w);
        }
        const int64_t rounds = (bh * nt + slots - 1) / slots;
        best = double(rounds) * 9.0 + std::max(double(bh * sum) / double(slots), double(heavy));
    } else if (br) {
        best = split_time(1);
    }
    int pick = 1;
    for (int s = 2; s <= max_splits; ++s) {
        const double t = split_time(s);
        if (t < best) best = t, pick = s;
    }
    return pick;
}

// Chunking of the key range a row can see (top-left causal never shows a key
// past sq - 1); `req` = 0 picks enough chunks to fill the CUs once (the
// shape's resident workgroups per CU; more chunks only add merge traffic and
// per-chunk pipeline fill), for prefill then the model above.  The
// count is then rounded so that no chunk starts past that range.
// The decode shape packs the query heads that share a K/V head into one row
// space of (heads / kv_heads) * sq rows per (batch, K/V head).
SplitPlan split_plan(const Fav4Args& a, int kv_heads, int causal, int req, bool br = false, bool br_unsplit = false) {
    const SplitShape sh = split_shape(a);
    const bool pack = sh.bm == 32;
    const int rows = pack ? (a.heads / kv_heads) * a.sq : a.sq;
    const int tiles = (rows + sh.bm - 1) / sh.bm;
    const int64_t items = int64_t(a.batch) * (pack ? kv_heads : a.heads);
    const int keys = causal ? std::min(a.sk, a.sq) : a.sk;
    const int ktiles = (keys + sh.bn - 1) / sh.bn;
    int64_t splits = req;
    if (splits == 0) {
        const int64_t units = items * tiles;
        // Decode with one or two (batch, K/V head) tiles (B1 MQA / two K/V
        // heads, long caches) runs faster on up to 256 chunks (measured on
        // MI355X, 128 -> 256: B1 H8 KVH1 Sk200000 52.6 -> 39.9 us, B1 H8 KVH2
        // Sk262144 65.6 -> 59.6 us; with four tiles 256 lost, 54.3 -> 62.4 us).
        const int auto_max = pack && units <= 2 ? fav4::MAX_SPLITS : sh.auto_max;
        splits = (int64_t(device_cus()) * sh.wgs_per_cu + units - 1) / units;
        splits = std::min<int64_t>(splits, std::min(auto_max, std::max(1, ktiles / MIN_TILES_PER_SPLIT)));
        if (!pack && splits > 1) splits = prefill_auto_splits(a, causal, int(splits), ktiles, br, br_unsplit);
    }
    splits = std::max<int64_t>(1, std::min<int64_t>(splits, ktiles));
    const int tps = int((ktiles + splits - 1) / splits);
    return {(ktiles + tps - 1) / tps, tps, sh, tiles, items};
}

// The chunks that Auto runs of a decode plan `p` (which sizes the workspace and
// is what the select calls report): equal chunks run side by side, so a second
// round of a few of them costs as much as the first, and no more are taken than
// fit at once (H32 KVH8, graph-timed, by workgroups: B5 Sk16384 800 -> 760
// 73.7 -> 56.8 us, B13 Sk30000 832 -> 728 294 -> 247, B7 Sk8192 784 -> 728
// 54.1 -> 42.9, B11 Sk4096 792 -> 704 42.7 -> 36.1).  Where that makes 32
// chunks or more of each row, two workgroups per CU do: the merge of three
// costs more than they gain (768 and 512: B1 Sk65536 50.0 and 47.9, B2 Sk8192
// 18.9 and 16.9, B2 Sk50000 71.6 and 68.7; B4 Sk4096, 24 and 16 chunks of a
// row, 17.6 and 19.3, B4 Sk16384 46.9 and 49.3).  Never one chunk: that would
// be the unpacked forward, a stream per query head.  max_tps: key tiles a
// chunk may span.
SplitPlan decode_run(const Fav4Args& a, const SplitPlan& p, int max_tps = INT_MAX) {
    if (p.shape.bm != 32 || p.splits <= 2) return p;
    const int64_t ktiles = (int64_t(a.sk) + p.shape.bn - 1) / p.shape.bn;
    const int64_t cus = device_cus(), units = p.items * p.tiles, two = cus * 2 / units;
    int64_t splits = two >= 32 ? two : std::max<int64_t>(2, cus * p.shape.wgs_per_cu / units);
    splits = std::max(splits, (ktiles + max_tps - 1) / max_tps);
    if (splits >= p.splits) return p;
    SplitPlan run = p;
    run.tps = int((ktiles + splits - 1) / splits);
    run.splits = int((ktiles + run.tps - 1) / run.tps);
    return run;
}

int64_t split_workspace(const Fav4Args& a, const SplitPlan& p) {
    if (p.splits <= 1) return 0;
    return int64_t(p.splits) * a.batch * a.heads * a.sq * (fav4::D * 4 + 2 * 4);
}

// Shape-only checks for the split-KV queries (no buffers needed yet).
int split_shape_ok(const Fav4Args* a, int kv_heads, int causal, int splits) {
    if (!a || a->batch <= 0 || a->heads <= 0 || a->sq <= 0 || a->sk <= 0 || (causal != 0 && causal != 1) ||
        kv_heads <= 0 || kv_heads > a->heads || a->heads % kv_heads != 0 ||
        a->batch > INT_MAX / a->heads || a->heads > INT_MAX / 128 || a->sq > INT_MAX / (a->heads * 128) ||
        a->sk > INT_MAX / (kv_heads * 128) || splits < 0 || splits > fav4::MAX_SPLITS || a->sq > MAX_SPLIT_SQ)
        return hipErrorInvalidValue;
    // Decode packs a group's (heads / kv_heads) * sq rows into one row space,
    // whose FP32 partial rows must fit a 4 GiB buffer bound.
    if (a->sq <= DECODE_SQ && int64_t(a->heads / kv_heads) * a->sq * fav4::D * 4 > int64_t(UINT32_MAX))
        return hipErrorInvalidValue;
    return hipSuccess;
}

int split_args_ok(const Fav4Args* a, int kv_heads, int causal, int splits) {
    if (kv_heads <= 0) return hipErrorInvalidValue;
    const int st = validate(a, causal, 0, kv_heads);
    return st != hipSuccess ? st : split_shape_ok(a, kv_heads, causal, splits);
}

// Packed and paged prefill on 256-row tiles keeps two key tiles in flight
// (three LDS stages) where at most half of its waves have queries and a chunk is
// long enough to pay for the two tiles it prefetches in vain: it then waits for
// K/V.  One and two tiles in flight, K/V from memory (several caches in turn):
// 2 x 40 queries H8, chunks of 24 tiles 44.9 and 38.0 us, of 16 33.7 and 29.7;
// 4 x 80 H8, of 31 66.2 and 61.4, of 12 34.7 and 33.5, of 8 27.4 and 27.1; 64 x
// 64 H4, of 16 35.0 and 31.8.  With K/V in the memory-side cache they are even
// from 16 tiles on, and 5% apart the other way below 8.  4 x 1024 queries on
// 4096 keys H32 lose 3% by it.
constexpr int STREAM_SQ = 128;
constexpr int STREAM_TPS = 12;

// Prefill chunks: K/V in BSHD (KV 0), packed (1) or paged (2) layout.
template <bool CAUSAL, int KV, bool BR, int WAVES, int STAGES = 2>
void launch_chunks(const Fav4Args& a, int kv_heads, const SplitPlan& p, const fav4::SplitArgs& sp, int64_t total,
                   hipStream_t stream) {
    const int tiles = (a.sq + WAVES * 32 - 1) / (WAVES * 32);
    int key_bits = 1;
    while (p.tps >> key_bits) ++key_bits;
    auto go = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, item_grid(total), dim3(WAVES * 64), 0, stream, a, sp, kv_heads, tiles, int(total),
                           key_bits);
    };
    if (a.lse) go(fav4::fwd_kernel_chunk<CAUSAL, true, WAVES, KV, BR, STAGES>);
    else go(fav4::fwd_kernel_chunk<CAUSAL, false, WAVES, KV, BR, STAGES>);
}

// VARLEN: `a` holds the packed batch's shape (max lengths) and `sp` its
// sequence offsets.  PAGED: the same over paged K/V caches.
// Top-left causal decode (sq <= 32) sees at most 32 keys, one tile, so the
// plan never splits it: top-left causal launches use the prefill shape only.
// BR (packed only): bottom-right causal.
template <bool CAUSAL, bool VARLEN = false, bool PAGED = false, bool BR = false>
int launch_split(const Fav4Args& a, int kv_heads, const SplitPlan& p, void* ws, fav4::SplitArgs sp,
                 hipStream_t stream) {
    static_assert(!(CAUSAL && VARLEN) || BR, "top-left causal decode never splits");
    static_assert(!BR || (CAUSAL && VARLEN), "bottom-right causal is for packed calls");
    static_assert(!PAGED || VARLEN, "paged caches hold packed sequences");
    const bool decode = p.shape.bm == 32;
    const int64_t rows = int64_t(a.batch) * a.heads * a.sq;
    int64_t total = p.items * p.tiles * p.splits;
    if (total > INT_MAX || rows > INT_MAX || (VARLEN && !PAGED && !BR && !decode) || (CAUSAL && !BR && decode))
        return hipErrorInvalidValue;
    sp.o_part = static_cast<float*>(ws);
    sp.lse_part = sp.o_part + int64_t(p.splits) * rows * fav4::D;
    sp.splits = p.splits;
    sp.tps = p.tps;
    sp.bm = p.shape.bm;
    sp.mask = BR ? 2 : CAUSAL;
    // The FP32 sums only feed an LSE output.
    if (!decode) {
        if constexpr (!VARLEN || PAGED || BR) {
            constexpr int KV = PAGED ? 2 : VARLEN ? 1 : 0;
            // The sorted lists hold only the q tiles that exist.
            if (VARLEN && a.batch <= fav4::MAX_SORTED_SEQS)
                total = std::min(total, a.heads * p.splits *
                                            ((sp.total_q + int64_t(a.batch) * (p.shape.bm - 1)) / p.shape.bm));
            if constexpr (KV == 0) {
                launch_chunks<CAUSAL, KV, BR, 8, 3>(a, kv_heads, p, sp, total, stream);
            } else {
                if (p.shape.bm == 128) launch_chunks<CAUSAL, KV, BR, 4>(a, kv_heads, p, sp, total, stream);
                else if (a.sq <= STREAM_SQ && p.tps >= STREAM_TPS)
                    launch_chunks<CAUSAL, KV, BR, 8, 3>(a, kv_heads, p, sp, total, stream);
                else launch_chunks<CAUSAL, KV, BR, 8>(a, kv_heads, p, sp, total, stream);
            }
        }
    } else if (VARLEN && p.ranges > 0) {
        if constexpr (VARLEN) {
            const int ktiles = (a.sk + p.shape.bn - 1) / p.shape.bn;
            const int min_tiles = (ktiles + p.splits - 2) / (p.splits - 1);
            const dim3 grid(unsigned(kv_heads) * unsigned(p.tiles) * unsigned(p.ranges));
            if (a.lse)
                hipLaunchKernelGGL((fav4::fwd_kernel_ranges<true, PAGED, BR>), grid, dim3(64), 0, stream, a, sp,
                                   kv_heads, p.tiles, p.ranges, min_tiles);
            else
                hipLaunchKernelGGL((fav4::fwd_kernel_ranges<false, PAGED, BR>), grid, dim3(64), 0, stream, a, sp,
                                   kv_heads, p.tiles, p.ranges, min_tiles);
        }
    } else {
        const int grid = int(total < MAX_GRID ? total : MAX_GRID), tiles = p.tiles;
        auto go = [&](auto kernel) {
            hipLaunchKernelGGL(kernel, dim3(grid), dim3(64), 0, stream, a, sp, kv_heads, tiles, int(total));
        };
        if constexpr (!CAUSAL || BR) {
            if (a.lse) go(fav4::fwd_kernel_split<true, VARLEN, PAGED, BR>);
            else go(fav4::fwd_kernel_split<false, VARLEN, PAGED, BR>);
        }
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess || (!decode && p.splits == 1)) return e;
    // Lane groups per merged row: one per 8 chunks, at most 8 (one workgroup).
    const int per = p.splits <= 8 ? 1 : p.splits <= 16 ? 2 : p.splits <= 32 ? 4 : 8;
    const int64_t row_blocks = (rows * per + 7) / 8;
    const unsigned blocks = unsigned(row_blocks < MAX_GRID ? row_blocks : MAX_GRID);
    auto merge = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(blocks), dim3(256), 0, stream, a, sp); };
    auto merge_rows = [&](auto decode_c) {
        constexpr bool DECODE = decltype(decode_c)::value;
        if (per == 1) merge(fav4::combine_kernel<1, VARLEN, DECODE>);
        else if (per == 2) merge(fav4::combine_kernel<2, VARLEN, DECODE>);
        else if (per == 4) merge(fav4::combine_kernel<4, VARLEN, DECODE>);
        else merge(fav4::combine_kernel<8, VARLEN, DECODE>);
    };
    if (decode) merge_rows(std::true_type{});
    else merge_rows(std::false_type{});
    return hipGetLastError();
}

// causal = 2 on the packed calls: bottom-right causal (query i of a sequence
// with sq queries and sk keys sees keys j <= sk - sq + i).
constexpr int BOTTOM_RIGHT = 2;

// Up to this many items per resident workgroup (rounds), a causal packed batch's
// lists go by each q tile's own keys, else by its sequence's: with few rounds the
// last items decide (4 x 2048 tokens H16, 2 rounds: 77 us by tile, 97 by
// sequence; 8 x 4096 H8, 4 rounds: 264 and 313), with many the q tiles of a
// sequence profit from running together (32 x 1024..7168 H8, 16 rounds: 874 and
// 844; 8 x 4096 H32, 16 rounds: 1092 and 1065), the earlier the fewer they are.
// By sequence over by tile, means of 330 random batches: 2 or 3 q tiles, 2-4
// rounds 0.94 (0.87 at worst), up to 2 rounds 1.02; 4-7 tiles, 3-4 rounds 0.88,
// 2-3 rounds 1.10; 8 or more, 3-4 rounds 1.09.
int by_item_rounds(int tiles) { return tiles < 4 ? 2 : tiles < 8 ? 3 : 4; }

// The grid of a packed call's lists of n items a head (packed_head_rank's ids).
int64_t list_ids(int64_t n, int heads, int block_bits) {
    if ((heads & 7) == 0) return n * heads;
    const int64_t blocks = heads * ((n + (int64_t(1) << block_bits) - 1) >> block_bits);
    return ((blocks + 7) / 8 * 8) << block_bits;
}

template <int WAVES>
void launch_varlen(const Fav4VarlenArgs& a, int causal, int tiles, int64_t items, int key_bits, hipStream_t stream) {
    const int slots = device_cus() * 8 / WAVES;            // workgroups resident at once
    const bool by_item = causal && items <= int64_t(by_item_rounds(tiles)) * slots;
    // By sequence, sequences of up to 4 q tiles: the ranks go to the XCDs in blocks
    // of that many, so that a sequence's tiles share its K/V in one L2 and a short
    // last tile is not always the same XCD's (56 x 148 tokens dense H4 15.8 and
    // 12.4 us); with 16 blocks an XCD or more, to keep the XCDs even, and none
    // that would make one round two.  Longer ones: rank by rank (4 x 4096 causal
    // H20, 5 rounds, in blocks of 8 372 us, else 333).  -1: by tile.
    int block_bits = by_item ? -1 : 0;
    if (!by_item && tiles <= 4) {
        while ((1 << block_bits) < tiles) ++block_bits;
        if (items >> block_bits < 128 || (items <= slots && items + (8 << block_bits) > slots)) block_bits = 0;
    }
    const int total = int(key_bits ? list_ids(items / a.heads, a.heads, std::max(0, block_bits)) : items);
    const dim3 grid = item_grid(total), block(WAVES * 64);
    if (causal == BOTTOM_RIGHT && a.lse)
        hipLaunchKernelGGL((fav4::fwd_kernel_varlen<64, true, true, WAVES, true>), grid, block, 0, stream, a,
                           tiles, total, key_bits, block_bits);
    else if (causal == BOTTOM_RIGHT)
        hipLaunchKernelGGL((fav4::fwd_kernel_varlen<64, true, false, WAVES, true>), grid, block, 0, stream, a,
                           tiles, total, key_bits, block_bits);
    else if (causal && a.lse)
        hipLaunchKernelGGL((fav4::fwd_kernel_varlen<64, true, true, WAVES>), grid, block, 0, stream, a, tiles, total,
                           key_bits, block_bits);
    else if (causal)
        hipLaunchKernelGGL((fav4::fwd_kernel_varlen<64, true, false, WAVES>), grid, block, 0, stream, a, tiles, total,
                           key_bits, block_bits);
    else if (a.lse)
        hipLaunchKernelGGL((fav4::fwd_kernel_varlen<64, false, true, WAVES>), grid, block, 0, stream, a, tiles, total,
                           key_bits, block_bits);
    else
        hipLaunchKernelGGL((fav4::fwd_kernel_varlen<64, false, false, WAVES>), grid, block, 0, stream, a, tiles, total,
                           key_bits, block_bits);
}

// Checks of the packed-sequence arguments (before any HIP call); the shape
// checks alone serve the queries that take no buffers.  causal 0, 1 or
// BOTTOM_RIGHT.
int varlen_shape_ok(const Fav4VarlenArgs* a, int causal) {
    if (!a || a->batch <= 0 || a->heads <= 0 || a->kv_heads <= 0 || a->heads % a->kv_heads != 0 ||
        a->max_seqlen_q <= 0 || a->max_seqlen_k <= 0 || a->total_q <= 0 || a->total_k <= 0 ||
        causal < 0 || causal > BOTTOM_RIGHT || !std::isfinite(a->scale) || a->scale <= 0)
        return hipErrorInvalidValue;
    if (a->batch > INT_MAX - 1 || a->heads > INT_MAX / 256 ||
        int64_t(a->max_seqlen_q) * a->heads * 256 > int64_t(UINT32_MAX) ||
        int64_t(a->max_seqlen_k) * a->kv_heads * 256 > int64_t(UINT32_MAX))
        return hipErrorInvalidValue;
    return hipSuccess;
}

int varlen_ok(const Fav4VarlenArgs* a, int causal) {
    if (varlen_shape_ok(a, causal) != hipSuccess || !a->q || !a->k || !a->v || !a->o || !a->cu_seqlens_q ||
        !a->cu_seqlens_k ||
        ((reinterpret_cast<uintptr_t>(a->q) | reinterpret_cast<uintptr_t>(a->k) |
          reinterpret_cast<uintptr_t>(a->v) | reinterpret_cast<uintptr_t>(a->o)) & 15) ||
        ((reinterpret_cast<uintptr_t>(a->cu_seqlens_q) | reinterpret_cast<uintptr_t>(a->cu_seqlens_k)) & 3) ||
        (a->lse && (reinterpret_cast<uintptr_t>(a->lse) & 3)))
        return hipErrorInvalidValue;
    return hipSuccess;
}

// The packed batch as the split-KV kernels see it: sq / sk are the longest
// sequence's lengths, LSE is [heads, total_q].
Fav4Args varlen_shape(const Fav4VarlenArgs& v) {
    Fav4Args a{};
    a.q = v.q; a.k = v.k; a.v = v.v; a.o = v.o; a.lse = v.lse;
    a.batch = v.batch; a.heads = v.heads; a.sq = v.max_seqlen_q; a.sk = v.max_seqlen_k;
    a.scale = v.scale;
    return a;
}

// Split-KV of packed decode batches (max_seqlen_q <= 32; longer queries take
// one chunk, the plain packed forward).  Chunks are a fixed number of key
// tiles for every sequence, so a sequence has as many non-empty chunks as its
// keys need.  Auto takes the chunk size of the contiguous-batch Auto plan at
// the mean key length (total_k / batch), so a uniform batch gets exactly the
// contiguous plan.  A ragged batch (mean below 3/4 of the longest) gets
// chunks of at most RAGGED_TPS key tiles: its chunks differ in length, and
// more, shorter ones even out the CUs' finishing times (measured on MI355X,
// against the uncapped plan: +0.7%, +2% and +13% on three ragged batches;
// the same cap on uniform batches lost 3-25%).  Either is enlarged if the
// longest sequence would need more than MAX_SPLITS chunks.
constexpr int RAGGED_TPS = 64;

// `a` is the packed batch's shape (max lengths), total_k its key count.
SplitPlan packed_split_plan(const Fav4Args& a, int kv_heads, int64_t total_k, int causal, int req) {
    if (a.sq > DECODE_SQ) return {1, 1, split_shape(a), 1, 1};
    SplitPlan p = split_plan(a, kv_heads, causal, req == 0 ? 1 : req);
    if (req == 0) {
        Fav4Args mean = a;
        mean.sk = int(std::max<int64_t>(1, std::min<int64_t>(a.sk, (total_k + a.batch - 1) / a.batch)));
        const int keys = causal ? std::min(a.sk, a.sq) : a.sk;
        const int ktiles = (keys + p.shape.bn - 1) / p.shape.bn;
        int tps = split_plan(mean, kv_heads, causal, 0).tps;
        if (4 * int64_t(mean.sk) < 3 * int64_t(a.sk)) tps = std::min(tps, RAGGED_TPS);
        p.tps = std::max(tps, (ktiles + fav4::MAX_SPLITS - 1) / fav4::MAX_SPLITS);
        p.splits = (ktiles + p.tps - 1) / p.tps;
    }
    return p;
}

// How Auto runs the decode of a packed or paged batch whose plan is `p` (which
// sizes the workspace): equal ranges of the batch's keys, RANGE_WGS_PER_CU
// one-wave workgroups per CU (fwd_kernel_ranges), unless
//  * every sequence has the longest one's keys (the contiguous call's chunks
//    then, and its result bitwise);
//  * a range would be under MIN_RANGE_TILES key tiles, not counting its
//    sequences' own cost: the short ranges then gain nothing or lose (plan /
//    ranges, H32 KVH8: 10 tiles, 32 sequences of 64..2048 keys 28.6 / 22.7 us;
//    4.2 tiles, 3 of 2500..3000 14.1 / 14.0; 2.6 tiles, 8 of 100..2000 14.2 both;
//    0.3 - 1.4 tiles, 24 - 84 sequences of 30..110 9.5 - 12.9 / 11.3 - 14.2);
//  * the plan's chunks would not hold the ranges: a sequence of n tiles meets
//    at most (n - 2) / (range length) + 2 of them, so `splits` chunks suffice
//    for ranges of at least ktiles / (splits - 1) tiles, which the kernel keeps
//    to;
//  * the batch has more sequences than a wave's lanes list.
// Two workgroups per CU against three (the plan's): 32 sequences of 1k..32k
// keys 202 us both, 64 of 64..2048 40.9 and 41.5, 200 of 300..9000 346 and 349,
// 16 of 8 queries H64 on 1k..16k 121 and 130, 8 of 1k..32k 93 and 121.
constexpr int RANGE_WGS_PER_CU = 2;
constexpr int MIN_RANGE_TILES = 8;
SplitPlan packed_decode_run(const Fav4Args& a, int kv_heads, int64_t total_k, const SplitPlan& p,
                            int max_tps = INT_MAX) {
    if (total_k >= int64_t(a.batch) * a.sk) return decode_run(a, p, max_tps);
    if (a.batch > fav4::MAX_SORTED_SEQS || p.splits < 2) return p;
    const int64_t streams = int64_t(kv_heads) * p.tiles;
    const int64_t ranges = int64_t(device_cus()) * RANGE_WGS_PER_CU / streams;
    if (ranges < 2) return p;
    const int64_t ktiles = (a.sk + p.shape.bn - 1) / p.shape.bn;
    const int64_t range = (total_k / p.shape.bn + a.batch / 2 + ranges - 1) / ranges;
    if (range < MIN_RANGE_TILES || ktiles > range * (p.splits - 1)) return p;
    const int64_t full = range + int64_t(a.batch) * fav4::RANGE_SEQ_TILES / ranges;
    SplitPlan run = p;
    run.splits = int(std::min<int64_t>(p.splits, (ktiles + full - 1) / full + 2));
    run.ranges = int(ranges);
    return run;
}

// How the prefill of a packed or paged batch (max_seqlen_q > 32) with plan `p`
// runs: the q tile (128 or 256 rows) and, for Auto, the chunk count up to the
// plan's (which sizes the workspace) with the lowest predicted time.  The
// plan takes every sequence as long as the longest; this model takes the
// batch's means as well (microseconds; fitted to 1558 graph-timed runs on MI355X:
// 255 random batches of 1-64 sequences, 33-2048 queries, 64-60000 keys, H1-128,
// over up to 11 chunk counts and both tiles).  A chunk costs 7 plus c per key
// tile: 128-row tiles c = 1.1 with at most one workgroup per CU, 1.5 with two;
// 256-row ones 1.0 where half of their waves have no query, else 1.45.
//  * Chunks that are resident at once take one chunk's time (10% more where
//    some CUs have two).
//  * Lengths near the longest (mean >= 3/4): whole rounds of equal chunks; from
//    the third on their ends spread and half a round is left over.
//  * Other lengths: the average load per resident workgroup and a fifth of the
//    longest chunk (the lists start the long ones first), never less than that.
//  * Merging writes and reads FP32 partials: 4 x 1024 queries against 4096 keys
//    H32 217 us in one chunk, 290 in two.
// Other counts than the plan's are not taken where the caller does not know the
// key total (one less than the most), since the lengths may be anything: 43 of
// 24..94 queries on 6630..52830 keys H4 640 us in the chunks that equal lengths
// would want, 556 in the plan's 13.  On 396 other batches the choice is 1.8%
// behind the fastest of the runs on average (1.1% at a given chunk count), and 7
// are slower by more than 2% than the 256-row chunks of the plan's count that
// every batch once had, the worst by 17% (1.5x on average).  With 9 + 1.1 or 10 +
// 1.75 per tile and half a q tile counted for a sequence with fewer queries than
// one, it was 4.3% behind, the worst 1.8x.
SplitPlan packed_prefill_run(const Fav4Args& a, int64_t total_q, int64_t total_k, bool br, const SplitPlan& p,
                             bool choose) {
    const int ktiles = (a.sk + 63) / 64;
    const double cus = device_cus(), seqs = a.batch;
    const double mean_q = std::min<double>(a.sq, double(total_q) / seqs);
    const double mean_k = std::min<double>(a.sk, double(total_k) / seqs);
    const bool uniform = 4 * mean_k >= 3.0 * a.sk;
    const double mean = std::max(1.0, mean_k / 64 + 0.5 - (br ? 0.5 * mean_q / 64 : 0.0));   // key tiles per q tile
    auto predict = [&](int bm, int splits, int tps) {
        const double slots = bm == 256 ? cus : 2 * cus, fixed = 7.0;
        const double qtiles = a.heads * seqs * std::min<double>((a.sq + bm - 1) / bm, std::max(1.0, mean_q / bm + 0.5));
        const double chunks = std::max(1.0, uniform ? std::ceil(mean / tps - 0.25) : mean / tps + 0.4);
        const double items = qtiles * chunks, rounds = items / slots;
        const double alone = bm == 128 ? 1.1 : a.sq <= 128 ? 1.0 : 1.45;       // per key tile, one workgroup on the CU
        const bool shared = bm == 128 && items > cus;
        const double per_tile = shared ? 1.5 : alone, longest = fixed + alone * std::min(tps, ktiles);
        const double chunk = fixed + per_tile * std::min<double>(tps, mean);
        double t;
        if (rounds <= 1)
            t = fixed + (chunk - fixed) * (shared ? 1.1 : 1.0);
        else if (uniform)
            t = chunk * (rounds <= 2.02 ? 2.0 : rounds + 0.5);
        else
            t = qtiles * (chunks * fixed + per_tile * mean) / slots + 0.2 * (fixed + per_tile * std::min(tps, ktiles));
        t = std::max(t, longest);
        if (splits > 1)
            t += 3.5 + double(total_q) * a.heads * splits * 1040 / 3e6 * (uniform ? 1.0 : std::max(0.3, mean_k / a.sk));
        return t;
    };
    const bool unknown = a.batch > 1 && total_k == int64_t(a.batch) * a.sk - 1;
    const int fewest = choose && !unknown ? 1 : p.splits;
    SplitPlan best = p;
    double best_t = 0;
    bool first = true;
    for (int s = fewest; s <= p.splits; ++s) {
        const int tps = s == p.splits ? p.tps : (ktiles + s - 1) / s, splits = (ktiles + tps - 1) / tps;
        for (int bm : {256, 128}) {
            const double t = predict(bm, splits, tps);
            if (!first && t >= best_t) continue;
            first = false;
            best_t = t;
            best = {splits, tps, SplitShape{bm, 64, bm == 256 ? 1 : 2, 64}, (a.sq + bm - 1) / bm, p.items};
        }
    }
    return best;
}

// Bottom-right causal in the split-KV packed calls sees as many keys as a
// dense call, so it is planned like one.  Decode always runs the split
// kernels, also for one chunk (their one-wave shape streams a K/V head once
// for its whole query group); prefill with one chunk runs the unsplit packed
// forward, which takes this mask directly.

SplitPlan varlen_split_plan(const Fav4VarlenArgs& v, int causal, int req) {
    const Fav4Args a = varlen_shape(v);
    // Bottom-right prefill: the contiguous prefill plan at the max lengths.
    if (causal == BOTTOM_RIGHT && a.sq > DECODE_SQ) return split_plan(a, v.kv_heads, 0, req, true, true);
    return packed_split_plan(a, v.kv_heads, v.total_k, causal == BOTTOM_RIGHT ? 0 : causal, req);
}

int varlen_split_ok(const Fav4VarlenArgs* v, int causal, int splits, bool buffers) {
    const bool br = causal == BOTTOM_RIGHT;
    const int st = buffers ? varlen_ok(v, br ? 0 : causal) : varlen_shape_ok(v, br ? 0 : causal);
    if (st != hipSuccess) return st;
    if (splits < 0 || splits > fav4::MAX_SPLITS) return hipErrorInvalidValue;
    if (v->max_seqlen_q > DECODE_SQ && !br) return hipSuccess;
    const Fav4Args a = varlen_shape(*v);
    return split_shape_ok(&a, v->kv_heads, br ? 0 : causal, splits);
}

// Workspace of a packed plan; bottom-right decode needs it for one chunk too.
int64_t varlen_workspace(const Fav4VarlenArgs& v, const SplitPlan& p, int causal) {
    if (p.splits <= 1 && (causal != BOTTOM_RIGHT || v.max_seqlen_q > DECODE_SQ)) return 0;
    return int64_t(p.splits) * v.batch * v.heads * v.max_seqlen_q * (fav4::D * 4 + 2 * 4);
}

// ---- paged K/V caches ----------------------------------------------------
constexpr int PAGED_MAX_TPS = 64;          // key tiles per chunk: one page number per lane
constexpr int PAGED_MAX_KEYS = fav4::MAX_SPLITS * PAGED_MAX_TPS * 32;

// Decode (max_seqlen_q <= 32) needs page_size % 32 == 0 (a 32-key tile lies in
// one page), prefill page_size % 64 == 0 (64-key tiles).
int paged_shape_ok(const Fav4PagedArgs* a, int causal, int splits) {
    if (!a || a->batch <= 0 || a->heads <= 0 || a->kv_heads <= 0 || a->heads % a->kv_heads != 0 ||
        a->max_seqlen_q <= 0 || a->max_seqlen_q > MAX_SPLIT_SQ || a->max_seqlen_k <= 0 || a->total_q <= 0 ||
        a->total_k < 0 || a->num_pages <= 0 || a->page_size <= 0 ||
        a->page_size % (a->max_seqlen_q > DECODE_SQ ? 64 : 32) != 0 ||
        a->max_pages_per_seq <= 0 || (causal != 0 && causal != BOTTOM_RIGHT) || !std::isfinite(a->scale) ||
        a->scale <= 0 || splits < 0 ||
        splits > fav4::MAX_SPLITS)
        return hipErrorInvalidValue;
    if (a->batch > INT_MAX - 1 || a->heads > INT_MAX / 256 || a->max_seqlen_k > PAGED_MAX_KEYS ||
        int64_t(a->max_seqlen_k) > int64_t(a->max_pages_per_seq) * a->page_size ||
        int64_t(a->page_size) * a->kv_heads * 256 > int64_t(UINT32_MAX) ||
        int64_t(a->max_seqlen_q) * a->heads * 256 > int64_t(UINT32_MAX) ||
        (a->max_seqlen_q <= DECODE_SQ ? int64_t(a->heads / a->kv_heads) : 1) * a->max_seqlen_q * fav4::D * 4 >
            int64_t(UINT32_MAX) ||
        int64_t(a->batch) * a->heads * a->max_seqlen_q > INT_MAX)
        return hipErrorInvalidValue;
    return hipSuccess;
}

int paged_ok(const Fav4PagedArgs* a, int causal, int splits) {
    if (paged_shape_ok(a, causal, splits) != hipSuccess || !a->q || !a->k_cache || !a->v_cache || !a->o ||
        !a->cu_seqlens_q || !a->seqlens_k || !a->block_table ||
        ((reinterpret_cast<uintptr_t>(a->q) | reinterpret_cast<uintptr_t>(a->k_cache) |
          reinterpret_cast<uintptr_t>(a->v_cache) | reinterpret_cast<uintptr_t>(a->o)) & 15) ||
        ((reinterpret_cast<uintptr_t>(a->cu_seqlens_q) | reinterpret_cast<uintptr_t>(a->seqlens_k) |
          reinterpret_cast<uintptr_t>(a->block_table)) & 3) ||
        (a->lse && (reinterpret_cast<uintptr_t>(a->lse) & 3)))
        return hipErrorInvalidValue;
    return hipSuccess;
}

Fav4Args paged_shape(const Fav4PagedArgs& v) {
    Fav4Args a{};
    a.q = v.q; a.k = v.k_cache; a.v = v.v_cache; a.o = v.o; a.lse = v.lse;
    a.batch = v.batch; a.heads = v.heads; a.sq = v.max_seqlen_q; a.sk = v.max_seqlen_k;
    a.scale = v.scale;
    return a;
}

// The packed-batch plan, with chunks capped at 64 key tiles (a decode chunk's
// page numbers fit the lanes of one wave; the prefill chunks and the ranges,
// which may be longer, load them 64 at a time); one chunk still runs the split
// kernels.
SplitPlan paged_plan(const Fav4PagedArgs& v, int causal, int req) {
    const Fav4Args a = paged_shape(v);
    // Prefill: the contiguous prefill plan at the max lengths (bottom-right
    // causal with the key count its q tiles see).
    SplitPlan p = a.sq > DECODE_SQ ? split_plan(a, v.kv_heads, 0, req, causal == BOTTOM_RIGHT)
                                   : packed_split_plan(a, v.kv_heads, v.total_k, 0, req);
    if (p.tps > PAGED_MAX_TPS) {
        const int ktiles = (v.max_seqlen_k + p.shape.bn - 1) / p.shape.bn;
        p.tps = PAGED_MAX_TPS;
        p.splits = (ktiles + p.tps - 1) / p.tps;
    }
    return p;
}

int64_t paged_workspace(const Fav4PagedArgs& v, const SplitPlan& p) {
    return int64_t(p.splits) * v.batch * v.heads * v.max_seqlen_q * (fav4::D * 4 + 2 * 4);
}

// Auto: 128-row workgroups (config 1; two per CU, so one's prologue and
// epilogue overlap the other's key loop) for query lengths up to 768 (dense)
// or 1024 (causal), and wherever 256-row workgroups (config 2) would leave
// CUs without a work item (items: q tiles; causal: q-tile pairs); else
// config 2.  Measured on MI355X (graph-timed, config 1 vs 2, row-contiguous
// O stores): dense Sq 512 config 1 wins by 5%, Sq 768 they are equal, Sq 1024
// config 2 wins by 1.7-6.5% (B32 H8, B16 H8, B8 H8, B4 H16); causal config 1
// wins or ties up to Sq 1024 (by 26% at B8 H8 and B4 H16 Sq 1024, 17% at B32
// H8 Sq 768).  With fewer config-2 items than CUs config 1 wins by 28-46%
// (B1 H8 S2048..S4096, causal B1 H8 S8192, B2 H8 S4096); with one item per
// CU or more config 2 wins by 6-8% (dense B2 H8 S4096, B1 H32 S4096, causal
// B1 H32 S4096).
int auto_config(const Fav4Args& a, int causal) {
    if (a.sq <= (causal ? 1024 : 768)) return 1;
    const int64_t tiles = (int64_t(a.sq) + 255) / 256;
    const int64_t items = int64_t(a.batch) * a.heads * (causal ? (tiles + 1) / 2 : tiles);
    return items < device_cus() ? 1 : 2;
}

}  // namespace

// Replaces src/bshd.hip:23-25 (the dense choice; the forward calls
// auto_config with its mask).
extern "C" __attribute__((visibility("default"))) int fav4_bshd_select_config(const Fav4Args* a) {
    if (!a) return -1;
    return auto_config(*a, 0);
}

// The same for a call with this mask (no counterpart in the reference, whose
// Auto ignores the mask): the config fav4_bshd_forward runs for config 0.
extern "C" __attribute__((visibility("default"))) int fav4_bshd_select_config_masked(const Fav4Args* a,
                                                                             int causal) {
    if (!a || (causal != 0 && causal != 1)) return -1;
    return auto_config(*a, causal);
}

// Replaces src/bshd.hip:26-38.
extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward(const Fav4Args* a, int causal, int config,
                                                                hipStream_t stream) {
    const int st = validate(a, causal, config);
    if (st != hipSuccess) return st;
    if (config == 0) config = auto_config(*a, causal);
    const fav4::Layout L = bshd_layout(*a, a->heads);
    return causal ? dispatch<true>(*a, L, config, stream) : dispatch<false>(*a, L, config, stream);
}

// Arbitrary strides (no counterpart in the reference).
extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward_strided(
    const Fav4Args* a, int kv_heads, const Fav4Strides* q, const Fav4Strides* k, const Fav4Strides* v,
    const Fav4Strides* o, int causal, int config, hipStream_t stream) {
    if (!a || !a->q || !a->k || !a->v || !a->o || a->batch <= 0 || a->heads <= 0 || a->sq <= 0 || a->sk <= 0 ||
        (causal != 0 && causal != 1) || config < 0 || config > 3 || !std::isfinite(a->scale) || a->scale <= 0 ||
        kv_heads <= 0 || kv_heads > a->heads || a->heads % kv_heads != 0 || a->batch > INT_MAX / a->heads ||
        ((reinterpret_cast<uintptr_t>(a->q) | reinterpret_cast<uintptr_t>(a->k) |
          reinterpret_cast<uintptr_t>(a->v) | reinterpret_cast<uintptr_t>(a->o)) & 15) ||
        (a->lse && (reinterpret_cast<uintptr_t>(a->lse) & 3)) ||
        !stride_ok(q, a->batch, a->heads, a->sq) || !stride_ok(o, a->batch, a->heads, a->sq) ||
        !stride_ok(k, a->batch, kv_heads, a->sk) || !stride_ok(v, a->batch, kv_heads, a->sk))
        return hipErrorInvalidValue;
    fav4::Layout L;
    L.qb = q->batch * 2; L.qh = q->head * 2; L.qr = uint32_t(q->seq * 2);
    L.kb = k->batch * 2; L.kh = k->head * 2; L.kr = uint32_t(k->seq * 2);
    L.vb = v->batch * 2; L.vh = v->head * 2; L.vr = uint32_t(v->seq * 2);
    L.ob = o->batch * 2; L.oh = o->head * 2; L.orow = uint32_t(o->seq * 2);
    L.group = a->heads / kv_heads;
    if (config == 0) config = auto_config(*a, causal);
    return causal ? dispatch<true>(*a, L, config, stream) : dispatch<false>(*a, L, config, stream);
}

// Packed variable-length sequences (no counterpart in the reference).
extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward_varlen(const Fav4VarlenArgs* a, int causal,
                                                                       hipStream_t stream) {
    const int st = varlen_ok(a, causal);
    if (st != hipSuccess) return st;
    // Tile rule on the longest sequence: 128-row tiles (4 waves) for
    // max_seqlen_q <= 1024 or when 256-row tiles would give fewer
    // (sequence, head, q tile) items than CUs; else 256-row tiles.
    const int64_t tiles256 = (int64_t(a->max_seqlen_q) + 255) / 256;
    const bool small = a->max_seqlen_q <= 1024 || int64_t(a->batch) * a->heads * tiles256 < device_cus();
    const int bm = small ? 128 : 256;
    const int tiles = (a->max_seqlen_q + bm - 1) / bm;
    int64_t total = int64_t(a->batch) * a->heads * tiles;
    if (total > INT_MAX) return hipErrorInvalidValue;
    // The sorted item lists' key_bits: the bits of the key tiles that a q tile
    // can see; 0 means no lists.  Batches of one q tile and one key tile a
    // sequence have nothing to sort, and the search would cost their short items
    // 4-10% (sorted and not: H32 KVH8 256 x 16 tokens 73.4 and 68.9 us, 211 of
    // 5..41 causal on up to 1934 keys 76.6 and 69.0).  Two key tiles go either
    // way: H16 KVH8 43 of 56..72 tokens 13.7 and 15.2, H10 KVH5 165 of 12..98
    // causal on up to 2028 keys 28.4 and 26.4.
    const int keys = causal == 1 ? std::min(a->max_seqlen_q, a->max_seqlen_k) : a->max_seqlen_k;
    const int key_tiles = (keys + 63) / 64;
    int key_bits = 0;
    if (a->batch <= fav4::MAX_SORTED_SEQS && (tiles > 1 || key_tiles > 1)) {
        while (key_tiles >> key_bits) ++key_bits;
        // The lists hold only the q tiles that exist, and no batch of total_q
        // rows has more than this many of them.
        total = std::min(total, a->heads * ((a->total_q + int64_t(a->batch) * (bm - 1)) / bm));
    }
    if (small)
        launch_varlen<4>(*a, causal, tiles, total, key_bits, stream);
    else
        launch_varlen<8>(*a, causal, tiles, total, key_bits, stream);
    return hipGetLastError();
}

// Grouped-query / multi-query attention (no counterpart in the reference).
extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward_gqa(const Fav4Args* a, int kv_heads,
                                                                    int causal, int config, hipStream_t stream) {
    if (kv_heads <= 0) return hipErrorInvalidValue;
    const int st = validate(a, causal, config, kv_heads);
    if (st != hipSuccess) return st;
    if (config == 0) config = auto_config(*a, causal);
    const fav4::Layout L = bshd_layout(*a, kv_heads);
    return causal ? dispatch<true>(*a, L, config, stream) : dispatch<false>(*a, L, config, stream);
}

// Split-KV entry points (no counterpart in the reference; see the header).
// The MHA ones are the GQA ones with kv_heads = heads.
extern "C" __attribute__((visibility("default"))) int fav4_bshd_splitkv_gqa_select(const Fav4Args* a, int kv_heads,
                                                                           int causal) {
    if (split_shape_ok(a, kv_heads, causal, 0) != hipSuccess) return -1;
    return split_plan(*a, kv_heads, causal, 0).splits;
}

extern "C" __attribute__((visibility("default"))) long long fav4_bshd_splitkv_gqa_workspace_size(const Fav4Args* a,
                                                                                              int kv_heads,
                                                                                              int causal,
                                                                                              int splits) {
    if (split_shape_ok(a, kv_heads, causal, splits) != hipSuccess) return -1;
    return split_workspace(*a, split_plan(*a, kv_heads, causal, splits));
}

extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward_splitkv_gqa(const Fav4Args* a, int kv_heads,
                                                                            int causal, int splits,
                                                                            void* workspace,
                                                                            size_t workspace_bytes,
                                                                            hipStream_t stream) {
    const int st = split_args_ok(a, kv_heads, causal, splits);
    if (st != hipSuccess) return st;
    SplitPlan p = split_plan(*a, kv_heads, causal, splits);
    if (p.splits == 1) return fav4_bshd_forward_gqa(a, kv_heads, causal, 0, stream);
    const int64_t need = split_workspace(*a, p);
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255) || uint64_t(need) > workspace_bytes)
        return hipErrorInvalidValue;
    if (splits == 0) p = decode_run(*a, p);
    const fav4::SplitArgs sp{};
    return causal ? launch_split<true>(*a, kv_heads, p, workspace, sp, stream)
                  : launch_split<false>(*a, kv_heads, p, workspace, sp, stream);
}

extern "C" __attribute__((visibility("default"))) int fav4_bshd_splitkv_select(const Fav4Args* a, int causal) {
    return a ? fav4_bshd_splitkv_gqa_select(a, a->heads, causal) : -1;
}

extern "C" __attribute__((visibility("default"))) long long fav4_bshd_splitkv_workspace_size(const Fav4Args* a,
                                                                                          int causal, int splits) {
    return a ? fav4_bshd_splitkv_gqa_workspace_size(a, a->heads, causal, splits) : -1;
}

extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward_splitkv(const Fav4Args* a, int causal,
                                                                        int splits, void* workspace,
                                                                        size_t workspace_bytes,
                                                                        hipStream_t stream) {
    if (!a) return hipErrorInvalidValue;
    return fav4_bshd_forward_splitkv_gqa(a, a->heads, causal, splits, workspace, workspace_bytes, stream);
}

// Split-KV of packed variable-length batches (no counterpart in the reference).
extern "C" __attribute__((visibility("default"))) int fav4_bshd_splitkv_varlen_select(const Fav4VarlenArgs* a,
                                                                              int causal) {
    if (varlen_split_ok(a, causal, 0, false) != hipSuccess) return -1;
    return varlen_split_plan(*a, causal, 0).splits;
}

extern "C" __attribute__((visibility("default"))) long long fav4_bshd_splitkv_varlen_workspace_size(
    const Fav4VarlenArgs* a, int causal, int splits) {
    if (varlen_split_ok(a, causal, splits, false) != hipSuccess) return -1;
    return varlen_workspace(*a, varlen_split_plan(*a, causal, splits), causal);
}

extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward_splitkv_varlen(const Fav4VarlenArgs* a,
                                                                               int causal, int splits,
                                                                               void* workspace,
                                                                               size_t workspace_bytes,
                                                                               hipStream_t stream) {
    const int st = varlen_split_ok(a, causal, splits, true);
    if (st != hipSuccess) return st;
    SplitPlan p = varlen_split_plan(*a, causal, splits);
    // Top-left causal decode (max_seqlen_q <= 32) sees at most 32 keys, one
    // tile: the plan never splits it.  One-chunk bottom-right prefill needs
    // no merge either.
    const bool br = causal == BOTTOM_RIGHT;
    const bool unsplit = br ? p.splits == 1 && a->max_seqlen_q > DECODE_SQ : p.splits == 1 || causal;
    if (unsplit) return fav4_bshd_forward_varlen(a, causal, stream);
    const Fav4Args shape = varlen_shape(*a);
    const int64_t need = varlen_workspace(*a, p, causal);
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255) || uint64_t(need) > workspace_bytes)
        return hipErrorInvalidValue;
    fav4::SplitArgs sp{};
    sp.cu_q = a->cu_seqlens_q;
    sp.cu_k = a->cu_seqlens_k;
    sp.total_q = a->total_q;
    sp.total_k = a->total_k;
    if (br && shape.sq > DECODE_SQ)
        return launch_split<true, true, false, true>(
            shape, a->kv_heads, packed_prefill_run(shape, a->total_q, a->total_k, true, p, splits == 0), workspace, sp,
            stream);
    if (splits == 0) p = packed_decode_run(shape, a->kv_heads, a->total_k, p);
    return br ? launch_split<true, true, false, true>(shape, a->kv_heads, p, workspace, sp, stream)
              : launch_split<false, true>(shape, a->kv_heads, p, workspace, sp, stream);
}

// Split-KV decode over paged K/V caches (no counterpart in the reference).
extern "C" __attribute__((visibility("default"))) int fav4_bshd_splitkv_paged_select(const Fav4PagedArgs* a,
                                                                             int causal) {
    if (paged_shape_ok(a, causal, 0) != hipSuccess) return -1;
    return paged_plan(*a, causal, 0).splits;
}

extern "C" __attribute__((visibility("default"))) long long fav4_bshd_splitkv_paged_workspace_size(
    const Fav4PagedArgs* a, int causal, int splits) {
    if (paged_shape_ok(a, causal, splits) != hipSuccess) return -1;
    return paged_workspace(*a, paged_plan(*a, causal, splits));
}

extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward_splitkv_paged(const Fav4PagedArgs* a,
                                                                              int causal, int splits,
                                                                              void* workspace,
                                                                              size_t workspace_bytes,
                                                                              hipStream_t stream) {
    const int st = paged_ok(a, causal, splits);
    if (st != hipSuccess) return st;
    SplitPlan p = paged_plan(*a, causal, splits);
    const int64_t need = paged_workspace(*a, p);
    if (!workspace || (reinterpret_cast<uintptr_t>(workspace) & 255) || uint64_t(need) > workspace_bytes)
        return hipErrorInvalidValue;
    fav4::SplitArgs sp{};
    sp.cu_q = a->cu_seqlens_q;
    sp.total_q = a->total_q;
    sp.seqlens_k = a->seqlens_k;
    sp.block_table = a->block_table;
    sp.page_size = a->page_size;
    sp.max_pages = a->max_pages_per_seq;
    sp.num_pages = a->num_pages;
    const Fav4Args shape = paged_shape(*a);
    const bool br = causal == BOTTOM_RIGHT;
    if (shape.sq > DECODE_SQ) p = packed_prefill_run(shape, a->total_q, a->total_k, br, p, splits == 0);
    else if (splits == 0) p = packed_decode_run(shape, a->kv_heads, a->total_k, p, PAGED_MAX_TPS);
    return br ? launch_split<true, true, true, true>(shape, a->kv_heads, p, workspace, sp, stream)
              : launch_split<false, true, true>(shape, a->kv_heads, p, workspace, sp, stream);
}

// ---- Split-KV without a caller workspace ------------------------------------
// For callers that cannot allocate (code under HIP graph capture, serving
// loops, harnesses that forbid it): the chunk partials live in a fixed
// device-resident array, one copy per GPU, held until the process ends.
constexpr size_t SCRATCH_BYTES = size_t(64) << 20;
static __device__ __align__(256) unsigned char scratch[SCRATCH_BYTES];

namespace {

// Device address of the current device's `scratch` (in host code the array's
// name is only a stand-in, never a device address), looked up once per device
// with that device current and kept per device.
hipError_t scratch_address(void** out) {
    static std::atomic<void*> cache[64];
    int dev = 0;
    hipError_t e = hipGetDevice(&dev);
    if (e != hipSuccess) return e;
    if (dev < 0 || dev >= 64) return hipErrorInvalidDevice;
    void* p = cache[dev].load(std::memory_order_acquire);
    if (!p) {
        e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
        if (e != hipSuccess) return e;
        if (!p) return hipErrorInvalidSymbol;
        cache[dev].store(p, std::memory_order_release);
    }
    *out = p;
    return hipSuccess;
}

}  // namespace

extern "C" __attribute__((visibility("default"))) int fav4_bshd_forward_splitkv_gqa_noalloc(const Fav4Args* a,
                                                                                    int kv_heads, int causal,
                                                                                    int splits,
                                                                                    hipStream_t stream) {
    const int st = split_args_ok(a, kv_heads, causal, splits);
    if (st != hipSuccess) return st;
    SplitPlan p = split_plan(*a, kv_heads, causal, splits);
    if (p.splits == 1) return fav4_bshd_forward_gqa(a, kv_heads, causal, 0, stream);
    if (split_workspace(*a, p) > int64_t(SCRATCH_BYTES)) return hipErrorInvalidValue;
    if (splits == 0) p = decode_run(*a, p);
    void* ws = nullptr;
    const hipError_t e = scratch_address(&ws);
    if (e != hipSuccess) return e;
    // Every partial row the merge reads is written by the partial kernel
    // first, so the array needs no clearing between calls.
    const fav4::SplitArgs sp{};
    return causal ? launch_split<true>(*a, kv_heads, p, ws, sp, stream)
                  : launch_split<false>(*a, kv_heads, p, ws, sp, stream);
}
