// Count stage, first half, on gfx950: the records of a partition's store are cut into units of work
// and re-encoded for the counting kernels (k_count.hip).
//
//  1. k_hist: k-mer instances, records and 2-bit words of every minimizer sub-bucket (12 bits of
//     ~mm above the partition digits). All k-mers of a record share its minimizer, and the minimizer
//     is a function of the canonical k-mer, so sub-buckets hold disjoint key sets.
//  2. k_plan: a partition's sub-buckets become units: a sub-bucket of more than unit_cap instances
//     is one by itself, smaller ones are packed into runs of at most unit_cap. A unit's place in the
//     regrouped records, and one item descriptor per unit for the counting kernel.
//  3. k_group: every record's k-mer count goes to its unit's run of descriptors and its bases, re-encoded
//     from the reference's 3-bases-per-byte records into word-aligned 2-bit words (LSB-first), to the
//     unit's run of words, in the same order.
#include "rgkc_device.h"
#include "rgkc_internal.h"

namespace rgkc {
namespace {

constexpr int kPlanThreads = 1024;
constexpr int kSubPer = kSubIds / kPlanThreads;  // sub-buckets per thread of k_plan
static_assert(kSubPer == 4, "k_plan loads four sub-buckets per thread");

__device__ __forceinline__ uint32_t rec_words(uint32_t km, int k) { return (km + (uint32_t)k - 1u + 15u) >> 4; }

struct SegRange {
    uint32_t lo, hi;
};
// record segment sg of a bucket of nrec records
__device__ __forceinline__ SegRange group_seg(uint32_t nrec, uint32_t sg, uint32_t n_segs) {
    const uint32_t per = (nrec + n_segs - 1) / n_segs;
    const uint32_t lo = min(sg * per, nrec);
    return {lo, min(lo + per, nrec)};
}
__device__ __forceinline__ uint32_t bucket_nrec(const CountArgs& a, uint32_t bucket) {
    return (uint32_t)((a.b_rec_end ? a.b_rec_end[bucket] : a.b_rec[bucket + 1]) - a.b_rec[bucket]);
}

// ---------------------------------------------------------------------------------------------
// One workgroup per (bucket, record segment); sub_inst and sub_rw must be zero. Bound by the side
// descriptors' read (4 B per record) and its LDS atomics.
__global__ __launch_bounds__(1024) void k_hist(CountArgs a) {
    __shared__ uint32_t inst[kSubIds];
    __shared__ unsigned long long rw[kSubIds];
    __shared__ uint32_t tmp[1024 / 64 + 1];
    const uint32_t bucket = blockIdx.x / a.n_segs, sg = blockIdx.x % a.n_segs;
    const uint64_t rec0 = a.b_rec[bucket];
    const SegRange sr = group_seg(bucket_nrec(a, bucket), sg, a.n_segs);
    const int k = a.k;
    if (sr.lo >= sr.hi) {
        if (threadIdx.x == 0) a.seg_bytes[(size_t)bucket * (a.n_segs + 1) + sg] = 0;
        return;
    }
    for (int i = threadIdx.x; i < kSubIds; i += 1024) { inst[i] = 0; rw[i] = 0; }
    __syncthreads();
    uint32_t bytes = 0;
    for (uint32_t r = sr.lo + threadIdx.x; r < sr.hi; r += 1024) {
        const uint32_t sd = a.side[rec0 + r];
        const uint32_t s = side_sub(sd), km = side_kmers(sd);
        atomicAdd(&inst[s], km);
        atomicAdd(&rw[s], ((unsigned long long)rec_words(km, k) << 32) | 1ull);
        bytes += skm_nbytes(side_bm3(sd), km + (uint32_t)k - 1u);
    }
    uint32_t tb;
    (void)wg_exscan_u32(bytes, tmp, &tb);  // ends with a barrier
    for (int i = threadIdx.x; i < kSubIds; i += 1024)
        if (rw[i]) {
            atomicAdd(&a.sub_inst[(size_t)bucket * kSubIds + i], inst[i]);
            atomicAdd(&a.sub_rw[(size_t)bucket * kSubIds + i], rw[i]);
        }
    if (threadIdx.x == 0) a.seg_bytes[(size_t)bucket * (a.n_segs + 1) + sg] = tb;
}

// ---------------------------------------------------------------------------------------------
// One workgroup per bucket. Light sub-buckets (at most unit_cap instances) are packed greedily in
// sub-bucket order: their instances' prefix is laid out in LDS, every light sub-bucket finds by a
// binary search where a unit that began with it would end, and one thread follows those links from
// the first. A serial walk over the 4096 counts by one thread, run twice (to count and to fill), took
// 1.5 ms for 512 partitions; the links are a few hundred LDS reads.
// A unit of more than kDirectSlices * unit_cap instances gets a key region per hash slice (heavy_on)
// and is expanded by k_expand; every other unit is counted from its records (k_count.hip), a large one by
// several work items (unit_shares).
__global__ __launch_bounds__(kPlanThreads) void k_plan(CountArgs a) {
    __shared__ uint32_t pre[kSubIds + 1];             // instances of the light sub-buckets before each one
    __shared__ uint16_t nxt[kSubIds];                 // end of the unit that begins here, then the unit
    __shared__ uint32_t uinst[kSubIds];               // per unit: instances
    __shared__ unsigned long long urw[kSubIds];       // per unit: words << 32 | records
    __shared__ uint32_t tmp[2 * (kPlanThreads / 64) + 1];
    __shared__ unsigned long long base_d;
    const uint32_t bucket = blockIdx.x, t = threadIdx.x;
    const uint32_t cap = a.unit_cap;
    const size_t sb = (size_t)bucket * kSubIds;
    const uint4 iv = ((const uint4*)(a.sub_inst + sb))[t];
    const uint32_t inst[kSubPer] = {iv.x, iv.y, iv.z, iv.w};
    uint32_t nlh = 0, lsum = 0;  // light sub-buckets | heavy ones << 16; instances of the light ones
#pragma unroll
    for (int j = 0; j < kSubPer; j++) {
        const bool heavy = inst[j] > cap;
        nlh += heavy ? 0x10000u : (inst[j] ? 1u : 0u);
        lsum += heavy ? 0u : inst[j];
        uinst[t * kSubPer + j] = 0;
        urw[t * kSubPer + j] = 0;
    }
    uint32_t exlh, exs, totlh, tots;
    wg_exscan2_u32(nlh, lsum, tmp, exlh, exs, totlh, tots);
    const uint32_t nl = totlh & 0xFFFFu, nh = totlh >> 16;
    {
        uint32_t pos = exlh & 0xFFFFu, s = exs;
#pragma unroll
        for (int j = 0; j < kSubPer; j++)
            if (inst[j] && inst[j] <= cap) {
                pre[pos++] = s;
                s += inst[j];
            }
        if (t == 0) pre[nl] = tots;
    }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSubPer; j++) {
        const uint32_t i = t * kSubPer + j;
        if (i >= nl) break;
        uint32_t lo = i + 1, hi = nl;  // pre[lo] - pre[i] <= cap
        while (lo < hi) {
            const uint32_t m = (lo + hi + 1) >> 1;
            if (pre[m] - pre[i] <= cap) lo = m;
            else hi = m - 1;
        }
        nxt[i] = (uint16_t)lo;
    }
    __syncthreads();
    if (t == 0)
        for (uint32_t i = 0; i < nl;) {
            const uint32_t e = nxt[i];
            nxt[i] = (uint16_t)(e | 0x8000u);
            i = e;
        }
    __syncthreads();
    uint32_t nmark = 0;
#pragma unroll
    for (int j = 0; j < kSubPer; j++) {
        const uint32_t i = t * kSubPer + j;
        if (i < nl) nmark += nxt[i] >> 15;
    }
    uint32_t n_light;
    uint32_t um = wg_exscan_u32(nmark, tmp, &n_light);
#pragma unroll
    for (int j = 0; j < kSubPer; j++) {
        const uint32_t i = t * kSubPer + j;
        if (i < nl) {
            um += nxt[i] >> 15;
            nxt[i] = (uint16_t)(um - 1u);
        }
    }
    __syncthreads();
    {
        uint32_t pos = exlh & 0xFFFFu, hp = n_light + (exlh >> 16);
#pragma unroll
        for (int j = 0; j < kSubPer; j++) {
            if (!inst[j]) continue;
            const uint32_t s = t * kSubPer + j;
            const uint32_t u = inst[j] > cap ? hp++ : (uint32_t)nxt[pos++];
            a.sub_unit[sb + s] = (uint16_t)u;
            atomicAdd(&uinst[u], inst[j]);
            atomicAdd(&urw[u], a.sub_rw[sb + s]);
        }
    }
    __syncthreads();
    const uint32_t n_units = n_light + nh;
    // units of this thread: t * kSubPer ...
    uint32_t ui[kSubPer], ur[kSubPer], uw[kSubPer], sr = 0, sw = 0, nd = 0;
#pragma unroll
    for (int j = 0; j < kSubPer; j++) {
        const uint32_t u = t * kSubPer + j;
        ui[j] = uinst[u];
        ur[j] = (uint32_t)urw[u];
        uw[j] = (uint32_t)(urw[u] >> 32);
        sr += ur[j];
        sw += uw[j];
        const bool keyed = a.heavy_on && (uint64_t)ui[j] > (uint64_t)cap * kDirectSlices;
        nd += keyed ? 0u : unit_shares(ui[j], cap);
    }
    uint32_t er, ew, tr, tw, td;
    wg_exscan2_u32(sr, sw, tmp, er, ew, tr, tw);
    uint32_t ed = wg_exscan_u32(nd, tmp, &td);
    if (t == 0) {
        a.n_units[bucket] = n_units;
        if (tw > a.b_word[bucket + 1] - a.b_word[bucket]) raise_err(a.err, RGKC_ERR_SCRATCH);
        uint64_t acc = 0;  // store bytes before each segment
        uint64_t* const sg = a.seg_bytes + (size_t)bucket * (a.n_segs + 1);
        for (uint32_t i = 0; i <= a.n_segs; i++) {
            const uint64_t v = i < a.n_segs ? sg[i] : 0;
            sg[i] = acc;
            acc += v;
        }
        base_d = td ? atomicAdd(&a.plan_n[kPlanItems], (unsigned long long)td) : 0ull;
    }
    __syncthreads();
    const uint64_t desc0 = a.b_rec[bucket] - a.rec_base, word0 = a.b_word[bucket];
    const uint32_t part = a.b_part[bucket];
#pragma unroll
    for (int j = 0; j < kSubPer; j++) {
        const uint32_t u = t * kSubPer + j;
        if (u >= n_units) break;
        a.unit_cur[sb + u] = ((unsigned long long)ew << 32) | er;
        UnitDesc d;
        d.part = part;
        d.inst = ui[j];
        d.n_rec = ur[j];
        d.n_word = uw[j];
        d.share = 0;
        d.desc = desc0 + er;
        d.word = word0 + ew;
        if (a.heavy_on && (uint64_t)ui[j] > (uint64_t)cap * kDirectSlices) {
            const uint32_t q = (uint32_t)min(((uint64_t)ui[j] + cap - 1) / cap, (uint64_t)kMaxKeySlices);
            d.q = q;
            const uint32_t cs = key_region(ui[j], q);
            KeyUnit ku;
            ku.u = d;
            ku.cs = cs;
            ku.pad = 0;
            ku.key0 = atomicAdd(&a.plan_n[kPlanKeySlots], (unsigned long long)q * (cs + 1ull));
            const uint64_t ix = atomicAdd(&a.plan_n[kPlanKeyUnits], 1ull);
            ku.item0 = atomicAdd(&a.plan_n[kPlanKeyItems], (unsigned long long)q);
            a.key_units[ix] = ku;
            for (uint32_t s = 0; s < q; s++) a.key_items[ku.item0 + s] = (ix << 8) | s;
        } else {
            d.q = unit_shares(ui[j], cap);
            for (d.share = 0; d.share < d.q; d.share++) a.unit_items[base_d + ed++] = d;
        }
        er += ur[j];
        ew += uw[j];
    }
}

// ---------------------------------------------------------------------------------------------
// One workgroup per (bucket, record segment), over the segment's records in chunks. Per chunk: the
// records' store offsets (a scan over their byte counts); each record's place in its unit's part of the
// chunk (one packed LDS atomic: words << 12 | records); the units' parts laid out one after another
// (a scan over the units) and reserved in the units' runs (one packed atomic per unit, whose latency
// passes under the next step); a map from each of the chunk's words to its record; then lane i writes
// the chunk's i-th descriptor and word in unit order, so neighbouring lanes write neighbouring places.
// The chunk's store bytes are staged in LDS, their loads in flight while the places are worked out; a word is
// made from six of them.
// Before: records grouped by 1024 fixed groups, a thread re-encoding a whole record byte by byte out of
// staged LDS bytes; 3.6 ms for 114 M records (1.65 GB of store). With the bytes read where they lie, two
// unaligned loads a word: 2.35 ms, three fifths of it for the words (the chunks of a CU exceed its L1); now
// 1.5 ms.
constexpr uint32_t kGroupBytes = 17280;  // staged store bytes of a chunk: three workgroups of the small size share a CU
template <int TG, int CH, int WC, int UM>  // threads, records and words per chunk, units
__global__ __launch_bounds__(TG) void k_group(CountArgs a) {
    static_assert(CH < 4096 && WC < (1 << 16) && UM <= 4096 && UM % TG == 0 && CH % TG == 0, "packed fields");
    constexpr int RPT = CH / TG, UPT = UM / TG;
    constexpr uint32_t SB = kGroupBytes;
    constexpr int SPT = (int)((SB / 16u + TG - 1u) / TG);
    static_assert(SB % 16u == 0 && SB < (1u << 15) && WC * 16 < (1 << 17), "packed fields");
    __shared__ __align__(4) uint16_t umap[kSubIds];
    __shared__ uint32_t ucnt[UM];           // words << 12 | records of the chunk per unit, then their starts
    __shared__ uint32_t gw[UM], gr[UM];     // unit's run minus its start in the chunk: words, records
    __shared__ uint16_t wrec[WC];           // record (its place in the chunk) of each word
    __shared__ __align__(16) uint32_t stb[SB / 4 + 4]; // the chunk's store bytes, from a 16-byte boundary on
    __shared__ uint32_t rpos[CH];           // per place: first byte in stb | k-mers << 15
    __shared__ uint32_t rinfo[CH];          // per place: first word << 16 | unit << 2 | start % 3
    __shared__ uint32_t tmp[2 * (TG / 64) + 1];
    __shared__ unsigned long long sh_cut;   // records << 40 | store bytes of the chunk
    // Segments of a bucket go to one XCD (workgroup b runs on XCD b % 8): the runs that its chunks append
    // to then meet in one L2. Which one moves on by one every eight buckets: buckets of one residue mod 8
    // are of one minimizer residue and differ in size as a class (the largest held 1.25 times its share of 1.2 G
    // k-mers, which the other XCDs waited for).
    const uint32_t per_xcd = (a.n_buckets + 7) / 8 * a.n_segs;
    const uint32_t ix = blockIdx.x / 8u, row = ix / a.n_segs;
    const uint32_t bucket = row * 8u + ((blockIdx.x + row) & 7u), sg = ix % a.n_segs;
    if (ix >= per_xcd || bucket >= a.n_buckets) return;
    // all that the first chunk needs is loaded before anything is waited for or checked
    const uint64_t byte0 = a.b_byte[bucket];
    const uint64_t nbytes = (a.b_byte_end ? a.b_byte_end[bucket] : a.b_byte[bucket + 1]) - byte0;
    const uint64_t* const sgb = a.seg_bytes + (size_t)bucket * (a.n_segs + 1);
    const uint64_t seg0 = sgb[sg], segs_end = sgb[a.n_segs];
    const uint32_t n_units = a.n_units[bucket];
    const uint64_t rec0 = a.b_rec[bucket];
    const SegRange sr = group_seg(bucket_nrec(a, bucket), sg, a.n_segs);
    const uint32_t wcap = (uint32_t)min(a.b_word[bucket + 1] - a.b_word[bucket], (uint64_t)0xFFFFFFFFu);
    const int k = a.k;
    uint32_t* const words = a.words + a.b_word[bucket];
    uint32_t* const desc = a.desc + (rec0 - a.rec_base);
    unsigned long long* const ucur = a.unit_cur + (size_t)bucket * kSubIds;
    const uint8_t* store = a.store + byte0 + seg0;
    const uint8_t* const store_end = a.store + byte0 + nbytes;
    uint4 sv[SPT];
    auto load_bytes = [&](const uint8_t* from) {
        const uint8_t* const p = from - ((uintptr_t)from & 15u);
#pragma unroll
        for (int j = 0; j < SPT; j++) {
            const uint32_t o = 16u * (threadIdx.x + (uint32_t)j * TG);
            sv[j] = o < SB && p + o < store_end ? *(const uint4*)(p + o) : make_uint4(0, 0, 0, 0);  // (the store has slack past its end)
        }
    };
    uint32_t nsd[RPT], um[kSubIds / 2 / TG];
#pragma unroll
    for (int j = 0; j < RPT; j++) {
        const uint32_t r = sr.lo + threadIdx.x * RPT + j;
        nsd[j] = r < sr.hi ? a.side[rec0 + r] : 0u;
    }
#pragma unroll
    for (int j = 0; j < kSubIds / 2 / TG; j++)
        um[j] = ((const uint32_t*)(a.sub_unit + (size_t)bucket * kSubIds))[threadIdx.x + j * TG];
    load_bytes(store);
    if (segs_end != nbytes) {  // the records' sizes do not add up to the store
        if (threadIdx.x == 0) raise_err(a.err, RGKC_ERR_BAD_STORE);
        return;
    }
    if (n_units > (uint32_t)UM || (UM > kSmallUnits && n_units <= (uint32_t)kSmallUnits)) return;  // the other size
    if (sr.lo >= sr.hi) return;
#pragma unroll
    for (int j = 0; j < kSubIds / 2 / TG; j++) ((uint32_t*)umap)[threadIdx.x + j * TG] = um[j];
    for (uint32_t c0 = sr.lo; c0 < sr.hi;) {
        uint32_t sd[RPT], nb[RPT], nw[RPT], old[RPT], accb = 0, accw = 0;
        const uint32_t lead = (uint32_t)((uintptr_t)store & 15u);
#pragma unroll
        for (int j = 0; j < RPT; j++) {
            const uint32_t r = c0 + threadIdx.x * RPT + j;
            sd[j] = nsd[j];
            nb[j] = r < sr.hi ? skm_nbytes(side_bm3(sd[j]), side_kmers(sd[j]) + (uint32_t)k - 1u) : 0u;
            nw[j] = r < sr.hi ? rec_words(side_kmers(sd[j]), k) : 0u;
            accb += nb[j];
            accw += nw[j];
        }
#pragma unroll
        for (int j = 0; j < UPT; j++) ucnt[threadIdx.x + j * TG] = 0;
        if (threadIdx.x == 0) sh_cut = 0;
        uint32_t exb, exw, totb, totw;
        wg_exscan2_u32(accb, accw, tmp, exb, exw, totb, totw);  // ends with a barrier
        // the chunk: the leading records whose words fit the map and whose bytes are staged (at least one
        // record: a longer one is a chunk of its own)
        uint32_t off[RPT], mine = 0;
        {
            uint32_t eb = exb, ew = exw;
#pragma unroll
            for (int j = 0; j < RPT; j++) {
                off[j] = eb;
                eb += nb[j];
                ew += nw[j];
                const uint32_t r = c0 + threadIdx.x * RPT + j;
                if (r < sr.hi && ((ew <= (uint32_t)WC && lead + eb <= SB) || r == c0)) {
                    mine = j + 1;
                    old[j] = atomicAdd(&ucnt[umap[side_sub(sd[j])]], (min(nw[j], (uint32_t)WC) << 12) | 1u);
                }
            }
            // the highest record of each wave that is in
            const uint64_t bal = __ballot(mine != 0);
            if (mine && (bal >> (threadIdx.x & 63u)) == 1ull) {
                uint32_t cb = exb;
#pragma unroll
                for (int j = 0; j < RPT; j++)
                    if ((uint32_t)j < mine) cb += nb[j];
                atomicMax(&sh_cut, ((unsigned long long)(threadIdx.x * RPT + mine) << 40) | cb);
            }
        }
        __syncthreads();
        const uint32_t m = (uint32_t)(sh_cut >> 40);
        const uint32_t cbytes = (uint32_t)sh_cut;
        // the next chunk's descriptors, in flight from here on
#pragma unroll
        for (int j = 0; j < RPT; j++) {
            const uint32_t r = c0 + m + threadIdx.x * RPT + j;
            nsd[j] = r < sr.hi ? a.side[rec0 + r] : 0u;
        }
        // the units' parts of the chunk, unit after unit; their runs reserved (unit = thread * UPT + j)
        uint32_t uc[UPT], us = 0;
#pragma unroll
        for (int j = 0; j < UPT; j++) {
            uc[j] = ucnt[threadIdx.x * UPT + j];
            us += uc[j];
        }
        uint32_t utot;
        uint32_t ue = wg_exscan_u32(us, tmp, &utot);  // all have read ucnt before its barrier
        unsigned long long run[UPT];
        uint32_t ust[UPT];
        const bool alone = m == 1;  // a record whose words may exceed the map: reserved with its true words
#pragma unroll
        for (int j = 0; j < UPT; j++) {
            const uint32_t u = threadIdx.x * UPT + j;
            ust[j] = ue;
            ucnt[u] = ue;
            if (uc[j] && !alone)
                run[j] = atomicAdd(&ucur[u], ((unsigned long long)(uc[j] >> 12) << 32) | (uc[j] & 0xFFFu));
            ue += uc[j];
        }
#pragma unroll
        for (int j = 0; j < SPT; j++) {
            const uint32_t o = 4u * (threadIdx.x + (uint32_t)j * TG);
            if (o < SB / 4u) *(uint4*)&stb[o] = sv[j];
        }
        // the next chunk's descriptors are there by now; its bytes, before this chunk's stores
#pragma unroll
        for (int j = 0; j < RPT; j++) asm volatile("" : "+v"(nsd[j]));
        load_bytes(store + cbytes);
        __syncthreads();
        if (alone) {
            // one record: all threads make its words
            if (threadIdx.x == 0) {
                const uint32_t u = umap[side_sub(sd[0])];
                const unsigned long long o = atomicAdd(&ucur[u], ((unsigned long long)nw[0] << 32) | 1ull);
                gw[0] = (uint32_t)(o >> 32);
                gr[0] = (uint32_t)o;
                rpos[0] = side_kmers(sd[0]);
                rinfo[0] = side_bm3(sd[0]);
            }
            __syncthreads();
            const uint32_t w0 = gw[0], km1 = rpos[0], n1 = rec_words(km1, k);
            if (threadIdx.x == 0) desc[gr[0]] = km1;
            for (uint32_t i = threadIdx.x; i < n1; i += TG)
                if (w0 + i < wcap) words[w0 + i] = record_word(store, rinfo[0], 16u * i, km1 + (uint32_t)k - 1u);
        } else {
            // per place: the record's store byte, k-mers and words
#pragma unroll
            for (int j = 0; j < RPT; j++) {
                if ((uint32_t)j >= mine) break;
                const uint32_t u = umap[side_sub(sd[j])];
                const uint32_t st = ucnt[u];
                const uint32_t pl = (st & 0xFFFu) + (old[j] & 0xFFFu), w0 = (st >> 12) + (old[j] >> 12);
                rpos[pl] = (lead + off[j]) | (side_kmers(sd[j]) << 15);
                rinfo[pl] = (w0 << 16) | (u << 2) | side_bm3(sd[j]);
                for (uint32_t i = 0; i < nw[j]; i++) wrec[w0 + i] = (uint16_t)pl;
            }
#pragma unroll
            for (int j = 0; j < UPT; j++)
                if (uc[j]) {
                    const uint32_t u = threadIdx.x * UPT + j;
                    gw[u] = (uint32_t)(run[j] >> 32) - (ust[j] >> 12);
                    gr[u] = (uint32_t)run[j] - (ust[j] & 0xFFFu);
                }
            __syncthreads();
            const uint32_t nwc = utot >> 12;
            for (uint32_t i = threadIdx.x; i < m; i += TG) desc[gr[(rinfo[i] >> 2) & 0xFFFu] + i] = rpos[i] >> 15;
            for (uint32_t i = threadIdx.x; i < nwc; i += TG) {
                const uint32_t pl = wrec[i], inf = rinfo[pl];
                const uint32_t at = gw[(inf >> 2) & 0xFFFu] + i;
                const uint32_t ps = rpos[pl], bm3 = inf & 3u, t0 = 16u * (i - (inf >> 16));
                const uint32_t o = (ps & 0x7FFFu) + (bm3 + t0) / 3u, *const q = stb + (o >> 2);
                const uint32_t x0 = q[0], x1 = q[1], x2 = q[2];
                const RecordBytes rb = {__builtin_amdgcn_alignbyte(x1, x0, o & 3u), __builtin_amdgcn_alignbyte(x2, x1, o & 3u) & 0xFFFFu};
                const uint32_t v = record_word(rb, bm3, t0, (ps >> 15) + (uint32_t)k - 1u);
                if (at < wcap) words[at] = v;
            }
        }
        __syncthreads();
        store += cbytes;
        c0 += m;
    }
}

}  // namespace

hipError_t launch_hist(const CountArgs& a, hipStream_t s) {
    if (!a.n_buckets) return hipSuccess;
    hipLaunchKernelGGL(k_hist, dim3(a.n_buckets * a.n_segs), dim3(1024), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_plan(const CountArgs& a, hipStream_t s) {
    if (!a.n_buckets) return hipSuccess;
    hipLaunchKernelGGL(k_plan, dim3(a.n_buckets), dim3(kPlanThreads), 0, s, a);
    return hipGetLastError();
}

// Buckets of up to kSmallUnits units take the small kernel; `many`: some bucket may hold more.
hipError_t launch_group(const CountArgs& a, bool many, hipStream_t s) {
    if (!a.n_buckets) return hipSuccess;
    const dim3 grid((a.n_buckets + 7) / 8 * 8 * a.n_segs);
    hipLaunchKernelGGL((k_group<512, 1024, 3840, kSmallUnits>), grid, dim3(512), 0, s, a);
    if (many) hipLaunchKernelGGL((k_group<512, 1024, 3840, kSubIds>), grid, dim3(512), 0, s, a);
    return hipGetLastError();
}

}  // namespace rgkc
