// Internal interfaces between the kernel translation units and the C-ABI host layer.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>

#include "rgkc_device.h"

namespace rgkc {

constexpr int kScanTile = 4096;      // elements per workgroup tile in the device scans
constexpr int kP1Threads = 256;      // phase-1 workgroup size (one read segment per thread)
constexpr int kSegKmers = 128;       // k-mers per read segment (long reads are cut into segments)
constexpr int kMaxParts = 1024;      // partitions supported by the LDS histograms of phase 1
constexpr int kSubIds = 4096;         // minimizer sub-bucket ids per partition (12 bits)
constexpr uint32_t kGroupSegments = 64;  // count stage: record segments per bucket in the grouping kernels, at most
// packed stream-mode cursor: records in the low kRecBits bits, bytes above
constexpr int kRecBits = 28;
constexpr unsigned long long kRecMask = (1ull << kRecBits) - 1;

// ---- utilities (k_util.hip) ------------------------------------------------------------------
// Exclusive scan of n uint64 values; `tmp` must hold scan_tmp_words(n) uint64 words.
size_t scan_tmp_words(size_t n);
hipError_t scan_u64(const uint64_t* in, uint64_t* out, size_t n, uint64_t* tmp, hipStream_t s);
// Per-row exclusive scan of a rows x cols uint32 matrix (row-major), in place; row totals to
// `totals` (uint64, rows entries).
hipError_t rowscan_u32(uint32_t* m, uint64_t* totals, int rows, uint32_t cols, hipStream_t s);
// out[i] = a[i] + b[i] (n entries)
hipError_t add_u64(const uint64_t* a, const uint64_t* b, uint64_t* out, size_t n, hipStream_t s);

// Rows [r0, r1) of the dense (partition after partition) table into a host buffer: of the n_parts
// <= kGatherParts partitions that hold them, partition i has dense rows [first[i], first[i + 1]), which
// start at row src[i] & ~(1 << 63) of the main table (bit 63 clear) or the second one. dst_keys and
// dst_counts (either may be null) get row r at r - r0.
constexpr int kGatherParts = 1024;
struct GatherArgs {
    const uint64_t* first;
    const uint64_t* src;
    int n_parts;
    const void *keys, *keys2;
    const uint32_t *counts, *counts2;
    uint64_t r0, r1;
    void* dst_keys;
    uint32_t* dst_counts;
};
hipError_t launch_gather_rows(const GatherArgs& a, int key_bytes, hipStream_t s);

// ---- phase 1 (k_phase1.hip) ------------------------------------------------------------------
struct SegTable {
    uint32_t* seg_read = nullptr;   // read index of each segment
    uint32_t* seg_first = nullptr;  // first k-mer of each segment (read-relative)
    uint64_t n_seg = 0;
};

hipError_t launch_pack(const uint8_t* reads, uint64_t n_bytes, uint32_t* bases2, hipStream_t s);
hipError_t launch_seg_count(const uint64_t* offs, uint64_t n_reads, int k, uint64_t* nseg, hipStream_t s);
hipError_t launch_seg_fill(const uint64_t* offs, const uint64_t* seg_off, uint64_t n_reads, int k,
                           uint32_t* seg_read, uint32_t* seg_first, hipStream_t s);

struct P1Args {
    const uint32_t* bases2;
    const uint64_t* offs;
    const uint32_t* seg_read;
    const uint32_t* seg_first;
    uint64_t n_seg;
    uint64_t n_bases;  // bases in the batch (bases2 holds n_bases/16 + 2 words)
    int k, p, parts;
    FastDivU32 pdiv;  // division by parts
    // count mode: per-(partition, workgroup) histograms, partition-major [parts][n_wg]
    uint32_t* h_bytes;
    uint32_t* h_recs;
    uint32_t* h_kmers;
    uint32_t n_wg;
    // emit mode
    const uint64_t* part_off;   // byte region start of each partition in `store`
    const uint64_t* part_end;   // byte region end (capacity check)
    const uint64_t* rec_off;    // side-descriptor region start of each partition
    const uint64_t* rec_end;
    const uint32_t* wg_byte_off;  // exact mode: [parts][n_wg] exclusive prefixes (nullptr: atomics)
    const uint32_t* wg_rec_off;
    unsigned long long* pos_cursor;   // atomic mode: bytes << kRecBits | records (relative to part_off / rec_off)
    uint8_t* store;
    uint32_t* side;
    uint32_t* err;
    uint32_t* mm_hist;  // optional: k-mer-weighted histogram of minimizer prefixes (top 8 bases)
    int hist_shift;     // mm >> hist_shift is the bin
    // stream mode (persistent, batched input): segment count on the device, k-mer totals
    const uint64_t* n_seg_dev;
    unsigned long long* kmer_cursor;
    // superkmer lists (exact mode, optional): the count pass leaves each workgroup's superkmers in
    // skm_list[wg * skm_cap ...] as 8-byte entries (skm_entry) and their number in skm_n[wg]; the
    // emit pass writes records from the list instead of scanning again. skm_n[wg] > skm_cap marks
    // a workgroup whose list did not fit, or held a superkmer an entry cannot describe: the emit
    // pass rescans its segments.
    uint64_t* skm_list;
    uint32_t* skm_n;
    uint32_t skm_cap;
    uint32_t* wg_rescan;        // count pass: tiles whose list overflowed, n_rescan[0] of them
    uint32_t* n_rescan;
    uint32_t* n_listorder;      // list emit: tiles with too many entries for store order (written in list order)
    const uint32_t* wg_map;     // scanning emit: tile of each workgroup (nullptr: blockIdx.x)
    uint32_t n_map;             // persistent scanning emit: tiles in wg_map
    const uint32_t* n_map_dev;  // their number on the device instead (batched input)
    uint32_t list_reserve;      // list emit: reserve each tile's runs with pos_cursor from its raw
                                // histogram columns (capacity-sized regions) instead of exact offsets
};
// list entry: minimizer | segment within the workgroup << 32 | (b - segment's first k-mer) << 40 |
// k-mers << 47 (the owned superkmer [b, b + k-mers) starts inside its segment: b - s0 < kSegKmers)
constexpr int kSkmKmerBits = 17;
static_assert(kSegKmers <= 128, "list entries keep b - s0 in 7 bits");
hipError_t launch_p1_count(const P1Args& a, hipStream_t s);
hipError_t launch_p1_emit(const P1Args& a, uint32_t n_rescan, hipStream_t s);
hipError_t launch_p1_emit_stream(const P1Args& a, unsigned grid, hipStream_t s);
// Capacity-sized regions from superkmer lists: the list emit over all tiles (list_reserve), then
// the persistent scanning emit over the n_rescan tiles whose list overflowed (a.wg_map).
hipError_t launch_p1_emit_sized(const P1Args& a, uint32_t n_rescan, hipStream_t s);
// Batched input: pack + segment table from a device header ([0] reads, [1] bases; [2] set to the
// segment count; n_rescan[0], the last batch's, added to n_rescan[2] and cleared), all launched over the batch capacity.
hipError_t launch_batch_prep(const uint8_t* reads, const uint64_t* offs, uint64_t* hdr, uint64_t cap_reads,
                             uint64_t cap_bases, int k, uint32_t* bases2, uint64_t* nseg, uint64_t* seg_off,
                             uint64_t* scan_tmp, uint32_t* seg_read, uint32_t* seg_first, uint32_t* n_rescan,
                             hipStream_t s);
hipError_t launch_p1_batch(const P1Args& a, hipStream_t s);

// ---- count (k_group.hip, k_count.hip) ----------------------------------------------------------
// A unit of more than this many unit_caps is expanded into keys: the count stage takes 12.5 ms with 1 and
// 12.1 with 2 (1.2 G k-mers at 30x), 2.43 and 1.96 (188 M, k=25): a unit is read once per sweep.
constexpr uint32_t kDirectSlices = 2;
constexpr uint32_t kMaxKeySlices = 127; // hash slices (key regions) of an expanded unit
// A unit counted from its records goes in shares of at most this many unit_caps (hash slices, a work item
// each): one workgroup took all sweeps of a large one. 13 M k-mers of 7 minimizers (k=21, p=3) without
// expansion 2270 ms, so 25; 12 M (k=55, p=5) 513, 17; 11 M of low complexity 301, 8.0.
// A share's sweeps are a whole number, so that smaller ones read the records more often.
constexpr uint32_t kShareCaps = 4;
__host__ __device__ inline uint32_t unit_shares(uint32_t inst, uint32_t cap) {
    const uint64_t most = (uint64_t)cap * kShareCaps, n = (inst + most - 1) / most;
    return (uint32_t)(n < (1u << 16) ? n : 1u << 16);
}
constexpr int kSmallUnits = 1024;       // units of a bucket that the small grouping kernel takes
enum { kPlanItems, kPlanKeySlots, kPlanKeyUnits, kPlanKeyItems, kPlanSeenInst, kPlanSeenDistinct, kPlanWords };
// A unit of work: sub-buckets of one partition whose records lie together.
struct UnitDesc {
    uint32_t part, inst, n_rec, n_word;  // partition, k-mer instances, records, their 2-bit words
    uint64_t desc, word;                 // first record descriptor and first word
    uint32_t q, share;                   // its hash slices: key regions, or work items and which of them
};
// An expanded unit: key regions of 1 + cs slots per slice (the fill count, then keys) from slot key0 on.
struct KeyUnit {
    UnitDesc u;
    uint64_t key0, item0;
    uint32_t cs, pad;
};
struct KeyItem {
    uint32_t part, n, slice, q;
    uint64_t keys, pad;  // address of the slice's keys
};
// key slots of a slice region: the slice's share of instances with a margin (slices are hash slices: a
// share above 1.25x + 256 is far in the tail; a fuller slice gets an exact region in a second pass)
__host__ __device__ inline uint32_t key_region(uint32_t inst, uint32_t q) {
    return ((inst + q - 1) / q / 4 * 5 + 256 + 63) & ~63u;
}
struct CountArgs {
    const uint8_t* store;       // superkmer records
    const uint32_t* side;       // side descriptors, one per record, in store order
    const uint64_t* b_byte;     // bucket byte ranges [b_byte[i], b_byte[i+1])
    const uint64_t* b_rec;      // bucket record ranges [b_rec[i], b_rec[i+1])
    const uint64_t* b_byte_end; // optional explicit ends (regions with gaps); nullptr: next start
    const uint64_t* b_rec_end;
    const uint32_t* b_part;     // partition of each bucket
    uint32_t n_buckets;
    uint32_t n_segs;            // record segments per bucket (<= kGroupSegments)
    uint64_t rec_base;          // record index of desc[0] (the first record of the buckets counted)
    const uint64_t* row_base;   // per partition: first row of its region
    const uint64_t* row_end;    // per partition: end of its region
    unsigned long long* row_cursor;  // per partition: rows written so far
    void* out_keys;             // uint64 (k <= 32) or 2 x uint64 (k > 32) per row
    uint32_t* out_counts;
    int k;
    uint32_t cmin, cmax;
    uint32_t unit_cap;          // k-mer instances planned per sweep (distinct-capacity proxy)
    uint32_t* err;
    unsigned long long* stats;  // [0] sweeps, [1] overflow retries, [2] distinct (unfiltered)
    unsigned long long* part_distinct;  // per partition: distinct keys (unfiltered)
    unsigned long long* plan_n;         // [kPlanWords] totals of the plan, instances and distinct keys counted so far
    uint32_t* sub_inst;         // [n_buckets][kSubIds] k-mer instances of each sub-bucket
    unsigned long long* sub_rw; // [n_buckets][kSubIds] words << 32 | records of each sub-bucket
    uint16_t* sub_unit;         // [n_buckets][kSubIds] unit of each (non-empty) sub-bucket
    uint64_t* seg_bytes;        // [n_buckets][n_segs + 1] store bytes per record segment, then their prefix
    uint32_t* n_units;          // [n_buckets]
    unsigned long long* unit_cur;  // [n_buckets][kSubIds] words << 32 | records: next free place of each unit
    uint32_t* desc;             // k-mers of each record, unit after unit
    uint32_t* words;            // records re-encoded as word-aligned 2-bit bases, in the same order
    const uint64_t* b_word;     // [n_buckets + 1] word region of each bucket
    UnitDesc* unit_items;       // units counted from their records (plan_n[kPlanItems] of them)
    // Units far larger than a sweep are expanded into keys once (heavy_on), a region per hash slice:
    uint32_t heavy_on;
    KeyUnit* key_units;
    uint64_t* key_items;        // unit << 8 | slice
    KeyItem* key_desc;          // after expansion: each slice's keys
    uint64_t n_key_items;
    void* heavy_keys;           // key slots (8 or 16 bytes)
    // Slices whose region overflowed (a very frequent key) get an exact region in a second key area:
    uint64_t* ovf_n;            // [n_key_items + 1] keys of the item's exact region (0: none), their prefix in ovf_off
    uint64_t* ovf_off;
    void* ovf_keys;
};
hipError_t launch_hist(const CountArgs& a, hipStream_t s);
hipError_t launch_plan(const CountArgs& a, hipStream_t s);
hipError_t launch_group(const CountArgs& a, bool many, hipStream_t s);
hipError_t launch_expand(const CountArgs& a, uint64_t n_units, hipStream_t s);
// ovf_n of every key item (after launch_expand); then, with ovf_off and ovf_keys set, the exact regions
hipError_t launch_ovf_sizes(const CountArgs& a, hipStream_t s);
hipError_t launch_expand_ovf(const CountArgs& a, uint64_t n_units, hipStream_t s);
// the units counted from their records; the expanded units' slices
hipError_t launch_count_units(const CountArgs& a, hipStream_t s);
hipError_t launch_count_keys(const CountArgs& a, hipStream_t s);

// Side descriptors for a store that lacks them (host-provided partitions), over pieces of kIndexChunk
// bytes: record starts by the full/non-full byte rule, each record's minimizer from its first k-mer.
constexpr uint64_t kIndexChunk = 8192;
struct IndexArgs {
    const uint8_t* store;
    const uint64_t* part_byte;  // [n_parts+1]
    uint32_t n_parts, n_chunks;
    const uint32_t* chunk_part; // [n_chunks] partition of each piece
    const uint32_t* part_chunk; // [n_parts+1] first piece of each partition
    int k, p, parts_total;      // parts_total: the partition count the sub-bucket id is defined over
    uint32_t* side;             // out: one per record
    uint64_t* chunk_n;          // [n_chunks+1] records of each piece
    const uint64_t* chunk_rec;  // [n_chunks+1] their prefix
    uint64_t* rec_count;        // [n_parts][2] records, k-mers
    uint32_t* err;
};
hipError_t launch_index_count(const IndexArgs& a, hipStream_t s);
hipError_t launch_index_parts(const IndexArgs& a, hipStream_t s);  // rec_count[2 * i] once chunk_rec is there
hipError_t launch_index_fill(const IndexArgs& a, hipStream_t s);

// ---- row order (k_sort.hip) ------------------------------------------------------------------
constexpr int kSortDigitBits = 12;
constexpr uint32_t kSortChunk = 4096;  // rows per histogram / scatter workgroup
// A run of rows to sort: rows [start, start + len) of the table, or [toff, toff + len) of the
// scratch buffer when `where` is 1; the next digit is key bits [shift, shift + nbits).
struct SortSeg {
    uint64_t start, toff;
    uint32_t len;
    uint16_t shift;
    uint8_t nbits, where;
};
struct SortArgs {
    void* keys;           // the table (W bytes per row) and its counts
    uint32_t* counts;
    void* tkeys;          // scratch rows
    uint32_t* tcounts;
    const SortSeg* leaf;  // segments sorted in LDS
    const SortSeg* big;   // segments distributed by their next digit
    const uint32_t* chunk_seg;   // big segment of each chunk
    const uint32_t* seg_chunk0;  // first chunk of each big segment
    uint32_t* hist;       // [n_big][hstride] bucket sizes
    uint32_t* cursor;     // [n_big][hstride] next free row of each bucket (segment-relative)
    uint32_t hstride;     // bins per segment row: 1 << (widest digit of the round), <= 1 << kSortDigitBits
};
int sort_leaf_cap(int key_bytes);
hipError_t launch_sort_leaf(const SortArgs& a, uint32_t n_leaf, int key_bytes, hipStream_t s);
hipError_t launch_sort_hist(const SortArgs& a, uint32_t n_chunks, int key_bytes, hipStream_t s);
hipError_t launch_sort_scatter(const SortArgs& a, uint32_t n_chunks, int key_bytes, hipStream_t s);

// ---- load predictor network (k_mlp.hip) ---------------------------------------------------
// Flat parameter layout: W1[n_in x h1] b1[h1] W2[h1 x h2] b2[h2] W3[h2 x n_out] b3[n_out].
struct MlpDims {
    int n_in = 0, h1 = 0, h2 = 0, n_out = 0;
    __host__ __device__ size_t off_W1() const { return 0; }
    __host__ __device__ size_t off_b1() const { return (size_t)n_in * h1; }
    __host__ __device__ size_t off_W2() const { return off_b1() + h1; }
    __host__ __device__ size_t off_b2() const { return off_W2() + (size_t)h1 * h2; }
    __host__ __device__ size_t off_W3() const { return off_b2() + h2; }
    __host__ __device__ size_t off_b3() const { return off_W3() + (size_t)h2 * n_out; }
    __host__ __device__ size_t total() const { return off_b3() + n_out; }
};
hipError_t mlp_to_bf16(const float* w, void* wb, size_t n, hipStream_t s);
hipError_t mlp_forward(const MlpDims& d, const void* wb, const float* w32, const float* X, int B, float* H1, float* H2,
                       float* Y, hipStream_t s);
hipError_t mlp_backward(const MlpDims& d, const void* wb, const float* X, int B, const float* H1, const float* H2,
                        const float* Y, const float* T, const float* mask, float mask_sum, float* dY, float* dH1,
                        float* dH2, float* G, float* loss, hipStream_t s);
// The same for batches that go row by row (mlp_by_rows): `part` holds mlp_part_floats, row_loss B floats.
// T null: forward only; else the activations' gradients and each row's loss too, from which mlp_rows_grad
// makes the parameters' gradients and the loss.
bool mlp_by_rows(const MlpDims& d, int B, bool train);
size_t mlp_part_floats(const MlpDims& d, int B);
hipError_t mlp_rows_forward(const MlpDims& d, const void* wb, const float* w32, const float* X, int B, float* part,
                            const float* T, const float* mask, float mask_sum, float* H1, float* H2, float* Y, float* dY,
                            float* dH1, float* dH2, float* row_loss, hipStream_t s);
hipError_t mlp_rows_grad(const MlpDims& d, const float* X, int B, const float* H1, const float* H2, const float* dY,
                         const float* dH1, const float* dH2, const float* row_loss, float* G, float* loss, hipStream_t s);
hipError_t mlp_adam(size_t n, float* w, void* wb, const float* g, float* m1, float* m2, float lr, int step, float wd,
                    hipStream_t s);

}  // namespace rgkc
