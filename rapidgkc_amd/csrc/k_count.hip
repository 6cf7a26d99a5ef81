// Count stage, second half, on gfx950: exact (k-mer, count) tables from the units that k_group.hip
// laid out.
//
//  1. k_count_units, persistent: a workgroup takes units b, b + G, b + 2G, ... and counts each in
//     one or more sweeps over its records (of a large unit a share of its hash slices): chunks of records have their 2-bit words copied into LDS, the
//     k-mers are taken from there four at a time and counted in an open-addressing LDS table. A unit with
//     more distinct keys than the table holds is counted in hash slices, one sweep each, that read the
//     records again; their number follows the ratio of distinct keys to instances seen so far, and a sweep
//     that overflows all the same is cut further.
//  2. A unit of more than kDirectSlices sweeps would be read too often: k_expand extracts its k-mers once
//     and scatters their canonical keys to one region per hash slice, and k_count_keys counts a
//     slice from its region. A slice that received more keys than its margin (a very frequent k-mer) gets
//     an exact region in a second key area, filled by a second pass (k_ovf_sizes, k_expand<OVF>).
//  3. A sweep's distinct keys with min <= count <= max (utilities.hpp:190) are appended to the partition's
//     row region, one atomic per sweep. rgkc_sort_rows (k_sort.hip) puts a partition's rows in ascending
//     key order afterwards, the order of the reference's table (cpu_funcs.cpp:614-640).
//
// The canonical key is the smaller of the digit-reversed 2k-bit window and the complemented one
// (cpu_funcs.cpp:427-436, gpu_kmercounting.cu:63-74).
#include <stddef.h>

#include <algorithm>

#include "rgkc_device.h"
#include "rgkc_internal.h"

namespace rgkc {
namespace {

constexpr int kItemThreads = 1024; // count workgroup size (one per CU)
constexpr int kStack = 128;        // pending sweeps of one unit
constexpr uint32_t kMaxCut = 8;    // slices an overflowing sweep is cut into, at most
constexpr uint32_t kMaxSlices = 1u << 20;
constexpr int kProbes = 64;        // tries a key may take to find its slot
constexpr uint32_t kPiece = 4;     // consecutive k-mers of a record that one thread takes
// LDS table: 8192 x (8 + 4) or 6144 x (16 + 4) bytes: with the staging areas one workgroup of 16 waves takes a
// CU. 64-bit keys stage two records per thread, so that a unit is nearly always one chunk; with one record per thread
// and 10240 slots most units were two, the second one half empty (count kernel of 1.2 G k-mers: 9.2 ms, so 8.15). Two
// workgroups of 8 waves with half the table each were 4% slower: twice the sweeps, fewer equal records found.
//
// Hash: a 32-bit multiply per key word, its high half rotated down before the next word joins, and the
// high half folded into the low one at the end (two multiplies for 64-bit keys; a 64-bit multiply takes
// three and its carries). The table's group comes from the high half, the hash slice from the low one.
__device__ __forceinline__ uint32_t mix_in(uint32_t x) {
    x *= 0x9E3779B1u;
    return __builtin_amdgcn_alignbit(x, x, 16);
}
__device__ __forceinline__ uint32_t mix(uint32_t x) {
    x *= 0x85EBCA6Bu;
    return x ^ (x >> 16);
}
// a place below n < 2^16 from the hash's high half
__device__ __forceinline__ uint32_t place(uint32_t h, uint32_t n) { return __umul24(h >> 16, n) >> 16; }

template <typename K> struct KT;
template <> struct KT<uint64_t> {
    static constexpr uint32_t H = 8192;
    static constexpr int R = 2;  // records of a chunk per thread
    static __device__ __forceinline__ uint64_t empty() { return ~0ull; }
    static __device__ __forceinline__ uint32_t hash(uint64_t x) {
        return mix((mix_in((uint32_t)x) ^ (uint32_t)(x >> 32)));
    }
};
template <> struct KT<u128> {
    static constexpr uint32_t H = 6144;
    static constexpr int R = 1;
    static __device__ __forceinline__ u128 empty() { return ~(u128)0; }
    static __device__ __forceinline__ uint32_t hash(u128 v) {
        const uint64_t lo = (uint64_t)v, hi = (uint64_t)(v >> 64);
        uint32_t h = mix_in((uint32_t)lo) ^ (uint32_t)(lo >> 32);
        h = mix_in(h) ^ (uint32_t)hi;
        return mix(mix_in(h) ^ (uint32_t)(hi >> 32));
    }
};
// distinct keys a sweep is planned for: 80% of the slots (a key that spends kProbes tries, on full groups, lost claims
// and halves of other keys, flags the sweep)
template <typename K> constexpr float kFill = 0.80f * (float)KT<K>::H;

// A chunk of records: at most kItemThreads * R of them, W words, P pieces; S slots of its record set. A record of
// more than `Long` pieces is not cut into the piece map (record | piece << RecBits, 16 bits).
template <typename K> struct Chunk {
    static constexpr int R = KT<K>::R;
    static constexpr uint32_t W = R == 2 ? 6144 : 4096, P = 4096 * R, S = 2048 * R;
    static constexpr uint32_t RecBits = R == 2 ? 11 : 10, Long = 1u << (16 - RecBits);
    static constexpr uint32_t WBits = 13, WMask = (1u << WBits) - 1u;  // of a record's info: first word | k-mers << WBits
    static constexpr uint32_t MaxLong = W / (Long * kPiece / 16u);     // a long record has more words than this divides by
    static_assert(W <= WMask && kItemThreads * R <= (1 << RecBits) && W % kItemThreads == 0, "packed fields, whole words per thread");
    static_assert(0x3FFFFu < (1u << (32 - WBits)), "the k-mers of a record that its side descriptor holds");
};

// Hash slice of a key among n. Slice s of n is the union of the slices s * f ... s * f + f - 1 of n * f.
__device__ __forceinline__ uint32_t slice_of(uint32_t h, uint32_t n) {
    return __umulhi(__builtin_amdgcn_alignbit(h, h, 16), n);
}

__device__ __forceinline__ uint32_t rec_words(uint32_t km, int k) { return (km + (uint32_t)k - 1u + 15u) >> 4; }

// kPiece consecutive k-mers from base g on of an LSB-first 2-bit word array: key(j, ...) is the j-th
// one's canonical key, j = 0, 1, ... in order. The window of all of them is aligned once; the forward key
// (first base most significant) is digit-reversed once and then takes one base per step.
template <typename K> struct Window;
template <> struct Window<uint64_t> {
    uint32_t a0, a1, a2;
    uint64_t f;
    __device__ __forceinline__ void load(const uint32_t* bw, uint32_t g) {
        const uint32_t* const p = bw + (g >> 4);
        const uint32_t sh = 2u * (g & 15u);
        const uint32_t w1 = p[1], w2 = p[2];
        a0 = __builtin_amdgcn_alignbit(w1, p[0], sh);
        a1 = __builtin_amdgcn_alignbit(w2, w1, sh);
        a2 = __builtin_amdgcn_alignbit(p[3], w2, sh);
    }
    __device__ __forceinline__ uint64_t key(int j, int k, uint64_t m) {
        const uint32_t s = 2u * (uint32_t)j;
        const uint64_t y = ((uint64_t)__builtin_amdgcn_alignbit(a1, a0, s) |
                            ((uint64_t)__builtin_amdgcn_alignbit(a2, a1, s) << 32)) & m;
        if (j == 0) {
            uint64_t r = __builtin_bitreverse64(y);
            r = ((r >> 1) & 0x5555555555555555ull) | ((r & 0x5555555555555555ull) << 1);
            f = r >> (64 - 2 * k);
        } else {
            f = ((f << 2) | (y >> (2 * k - 2))) & m;
        }
        const uint64_t rc = y ^ m;
        return f < rc ? f : rc;
    }
};
template <> struct Window<u128> {
    uint32_t a[5];
    u128 f;
    __device__ __forceinline__ void load(const uint32_t* bw, uint32_t g) {
        const uint32_t* const p = bw + (g >> 4);
        const uint32_t sh = 2u * (g & 15u);
        uint32_t w = p[0];
#pragma unroll
        for (int i = 0; i < 5; i++) {
            const uint32_t n = p[i + 1];
            a[i] = __builtin_amdgcn_alignbit(n, w, sh);
            w = n;
        }
    }
    __device__ __forceinline__ u128 key(int j, int k, u128 m) {
        const uint32_t s = 2u * (uint32_t)j;
        uint32_t b[4];
#pragma unroll
        for (int i = 0; i < 4; i++) b[i] = __builtin_amdgcn_alignbit(a[i + 1], a[i], s);
        const uint64_t lo = (uint64_t)b[0] | ((uint64_t)b[1] << 32), hi = (uint64_t)b[2] | ((uint64_t)b[3] << 32);
        const u128 y = (((u128)hi << 64) | lo) & m;
        if (j == 0) {
            uint64_t rl = __builtin_bitreverse64((uint64_t)y), rh = __builtin_bitreverse64((uint64_t)(y >> 64));
            rl = ((rl >> 1) & 0x5555555555555555ull) | ((rl & 0x5555555555555555ull) << 1);
            rh = ((rh >> 1) & 0x5555555555555555ull) | ((rh & 0x5555555555555555ull) << 1);
            f = (((u128)rl << 64) | rh) >> (128 - 2 * k);
        } else {
            f = ((f << 2) | (y >> (2 * k - 2))) & m;
        }
        const u128 rc = y ^ m;
        return f < rc ? f : rc;
    }
};
template <typename K> __device__ __forceinline__ K key_mask(int k) {
    return (2 * k == 8 * (int)sizeof(K)) ? ~(K)0 : (((K)1 << (2 * k)) - 1);
}

// Adds w to the counts of the N keys of one thread (bit u of `valid`: key u counts), hashes h. Keys are never removed, so
// a slot holding a key keeps it for the whole sweep; a key that finds neither itself nor an empty slot
// among kProbes flags the sweep (*ovf = 1).
//
// 64-bit keys: groups of four slots (32 bytes, two 16-byte reads). A key is claimed with a CAS at its
// group's first empty slot, so a group's keys are always a prefix of it; the CAS's old value decides, and
// every lane inserting a key tries the same slots in the same order: a key is never held twice. (One CAS
// per slot in turn executed some lane's CAS for all four slots of every wave.)
constexpr uint32_t kGroupsOf4 = KT<uint64_t>::H / 4u;
// the slot of a group that holds the key, else 4; its first empty slot (4: none). Compares and selects
// that do not wait for one another.
__device__ __forceinline__ uint32_t find(ulonglong2 x, ulonglong2 y, uint64_t k, uint32_t& empty) {
    const uint32_t e0 = x.x == ~0ull ? 0u : 4u, e1 = x.y == ~0ull ? 1u : 4u, e2 = y.x == ~0ull ? 2u : 4u,
                   e3 = y.y == ~0ull ? 3u : 4u;
    const uint32_t i0 = x.x == k ? 0u : 4u, i1 = x.y == k ? 1u : 4u, i2 = y.x == k ? 2u : 4u, i3 = y.y == k ? 3u : 4u;
    empty = min(min(e0, e1), min(e2, e3));
    return min(min(i0, i1), min(i2, i3));
}
// One try for each of N keys; returns the keys that lost a claim to another key, or whose group is full.
template <int N>
__device__ __forceinline__ uint32_t insert_first(uint64_t* tk, uint32_t* tc, const uint64_t* key, const uint32_t* h,
                                                 uint32_t valid, uint32_t w) {
    uint32_t g[N], pend = 0;
    ulonglong2 q0[N], q1[N];
#pragma unroll
    for (int u = 0; u < N; u++) {
        g[u] = place(h[u], kGroupsOf4);
        const ulonglong2* const gs = (const ulonglong2*)&tk[4u * g[u]];
        q0[u] = gs[0];
        q1[u] = gs[1];
    }
#pragma unroll
    for (int u = 0; u < N; u++) {
        const uint32_t v = (valid >> u) & 1u;
        uint32_t e;
        uint32_t i = find(q0[u], q1[u], key[u], e);
        if (((i >> 2) & v) && e < 4u) {
            const unsigned long long o = atomicCAS((unsigned long long*)&tk[4u * g[u] + e], ~0ull, (unsigned long long)key[u]);
            i = ((o == ~0ull) | (o == key[u])) ? e : 4u;
        }
        pend |= ((i >> 2) & v) << u;
        if (v & ~(i >> 2)) atomicAdd(&tc[4u * g[u] + i], w);
    }
    return pend;
}
// The keys `pend` of N, on from their groups, in one loop (a lane's next key as soon as one has its slot):
// nearly every wave has some, few lanes more than one.
template <int N>
__device__ __forceinline__ void insert_rest(uint64_t* tk, uint32_t* tc, const uint64_t* key, const uint32_t* h, uint32_t pend,
                                            uint32_t w, uint32_t* ovf) {
    if (!pend) return;
    uint64_t kk = 0;
    uint32_t gg = 0;
    auto take = [&]() {
        const uint32_t u = (uint32_t)__builtin_ctz(pend);
        uint32_t hh = 0;
#pragma unroll
        for (int j = 0; j < N; j++)
            if (u == (uint32_t)j) { kk = key[j]; hh = h[j]; }
        gg = place(hh, kGroupsOf4);
    };
    take();
#pragma unroll 1
    for (int tries = 0;;) {
        const ulonglong2* const gs = (const ulonglong2*)&tk[4u * gg];
        uint32_t e;
        uint32_t i = find(gs[0], gs[1], kk, e);
        if ((i >> 2) && e < 4u) {
            const unsigned long long o = atomicCAS((unsigned long long*)&tk[4u * gg + e], ~0ull, (unsigned long long)kk);
            i = ((o == ~0ull) | (o == kk)) ? e : 4u;
        }
        if (i < 4u) {
            atomicAdd(&tc[4u * gg + i], w);
            pend &= pend - 1u;
            if (!pend) break;
            take();
            tries = 0;
        } else {
            if (e == 4u) gg = gg + 1u == kGroupsOf4 ? 0u : gg + 1u;
            if (++tries == kProbes) {
                *ovf = 1u;
                break;
            }
        }
    }
}
template <int N>
__device__ __forceinline__ void insert(uint64_t* tk, uint32_t* tc, const uint64_t* key, const uint32_t* h, uint32_t valid,
                                       uint32_t w, uint32_t* ovf) {
    insert_rest<N>(tk, tc, key, h, insert_first<N>(tk, tc, key, h, valid, w), w, ovf);
}
// 128-bit keys (126 bits at most) as two words of 63, neither ever ~0: the table holds the lower halves in groups
// of four, then the upper ones. A claim is a CAS of the lower half; the claimer writes the upper one next, and a
// key that meets its own lower half reads the upper one: ~0 until it is written, when the key tries again. Keys
// that differ in the lower half (the k-mer's last 31 bases), nearly all that share a group, never wait for each
// other. A slot of both words, marked busy until both were there and tried one by one: 392 M 128-bit keys
// 7.3 ms, so 5.8.
// The claimer writes in straight-line code before any lane of its wave tries again, and a full fence keeps the
// compiler from moving the write past the tries.
__device__ __forceinline__ uint64_t half0(u128 key) { return (uint64_t)key & (~0ull >> 1); }
__device__ __forceinline__ uint64_t half1(u128 key) { return (uint64_t)(key >> 63); }
constexpr uint32_t kGroups128 = KT<u128>::H / 4u;
__device__ __forceinline__ uint64_t load_half1(const uint64_t* ta, uint32_t s) {
    return __hip_atomic_load(ta + KT<u128>::H + s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
}
__device__ __forceinline__ void store_half1(uint64_t* ta, uint32_t s, uint64_t v) {
    __hip_atomic_store(ta + KT<u128>::H + s, v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_WORKGROUP);
}
template <int N>
__device__ __forceinline__ uint32_t insert_first(u128* tk, uint32_t* tc, const u128* key, const uint32_t* h, uint32_t valid,
                                                 uint32_t w) {
    uint64_t* const ta = (uint64_t*)tk;
    uint32_t g[N], at[N], pend = 0;
    ulonglong2 q0[N], q1[N];
#pragma unroll
    for (int u = 0; u < N; u++) {
        g[u] = 4u * place(h[u], kGroups128);
        const ulonglong2* const gs = (const ulonglong2*)&ta[g[u]];
        q0[u] = gs[0];
        q1[u] = gs[1];
    }
#pragma unroll
    for (int u = 0; u < N; u++) {
        const uint32_t v = (valid >> u) & 1u;
        const uint64_t ka = half0(key[u]);
        uint32_t e;
        uint32_t i = find(q0[u], q1[u], ka, e);
        if (((i >> 2) & v) && e < 4u) {
            const unsigned long long o = atomicCAS((unsigned long long*)&ta[g[u] + e], ~0ull, (unsigned long long)ka);
            if (o == ~0ull) store_half1(ta, g[u] + e, half1(key[u]));
            i = ((o == ~0ull) | (o == ka)) ? e : 4u;
        }
        at[u] = v ? i : 8u;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
    uint64_t kb[N];
#pragma unroll
    for (int u = 0; u < N; u++) kb[u] = load_half1(ta, g[u] + (at[u] & 3u));
#pragma unroll
    for (int u = 0; u < N; u++) {
        const bool hit = at[u] < 4u && kb[u] == half1(key[u]);
        if (hit) atomicAdd(&tc[g[u] + at[u]], w);
        pend |= (uint32_t)(!hit && at[u] < 8u) << u;
    }
    return pend;
}
template <int N>
__device__ __forceinline__ void insert_rest(u128* tk, uint32_t* tc, const u128* key, const uint32_t* h, uint32_t pend,
                                            uint32_t w, uint32_t* ovf) {
    if (!pend) return;
    uint64_t* const ta = (uint64_t*)tk;
    uint64_t ka = 0, kl = 0;
    uint32_t gg = 0, from = 0;  // slots of the group before `from` hold the lower half with another upper one
    auto take = [&]() {
        const uint32_t u = (uint32_t)__builtin_ctz(pend);
        uint32_t hh = 0;
#pragma unroll
        for (int j = 0; j < N; j++)
            if (u == (uint32_t)j) { ka = half0(key[j]); kl = half1(key[j]); hh = h[j]; }
        gg = place(hh, kGroups128);
        from = 0;
    };
    take();
#pragma unroll 1
    for (int tries = 0, waits = 0;;) {
        const ulonglong2* const gs = (const ulonglong2*)&ta[4u * gg];
        const ulonglong2 x = gs[0], y = gs[1];
        uint32_t e;
        (void)find(x, y, ka, e);
        uint32_t i = 4u;
        if (y.y == ka && from <= 3u) i = 3u;
        if (y.x == ka && from <= 2u) i = 2u;
        if (x.y == ka && from <= 1u) i = 1u;
        if (x.x == ka && from == 0u) i = 0u;
        if (i == 4u && e < 4u) {
            const unsigned long long o = atomicCAS((unsigned long long*)&ta[4u * gg + e], ~0ull, (unsigned long long)ka);
            if (o == ~0ull) store_half1(ta, 4u * gg + e, kl);
            i = ((o == ~0ull) | (o == ka)) ? e : 4u;
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        const uint64_t o = load_half1(ta, 4u * gg + (i & 3u));
        if (i < 4u && o == kl) {
            atomicAdd(&tc[4u * gg + i], w);
            pend &= pend - 1u;
            if (!pend) break;
            take();
            tries = waits = 0;
        } else if (i < 4u && o == ~0ull) {
            if (++waits > (1 << 16)) {  // reported as a failure, not retried
                *ovf = 2u;
                break;
            }
        } else {
            if (i < 4u) {
                from = i + 1u;
            } else if (e == 4u) {
                gg = gg + 1u == kGroups128 ? 0u : gg + 1u;
                from = 0;
            }
            if (++tries == kProbes) {
                *ovf = 1u;
                break;
            }
        }
    }
}
template <int N>
__device__ __forceinline__ void insert(u128* tk, uint32_t* tc, const u128* key, const uint32_t* h, uint32_t valid,
                                       uint32_t w, uint32_t* ovf) {
    insert_rest<N>(tk, tc, key, h, insert_first<N>(tk, tc, key, h, valid, w), w, ovf);
}

// Slot s of the table: its key (empty() if none), then empty again.
__device__ __forceinline__ uint64_t take_slot(uint64_t* tk, uint32_t s) {
    const uint64_t x = tk[s];
    tk[s] = ~0ull;
    return x;
}
__device__ __forceinline__ u128 take_slot(u128* tk, uint32_t s) {
    uint64_t* const ta = (uint64_t*)tk;
    const uint64_t x = ta[s], y = ta[KT<u128>::H + s];
    ta[s] = ta[KT<u128>::H + s] = ~0ull;
    return x == ~0ull ? KT<u128>::empty() : ((u128)y << 63) | x;
}

// ---------------------------------------------------------------------------------------------
// 2. One workgroup per expanded unit: every k-mer is extracted once and its canonical key goes to its
//    slice's key run. Per chunk of records the keys are counted per slice in LDS, each slice's run is
//    reserved from its LDS cursor, and a second pass writes the keys. Keys past a slice's capacity are
//    dropped while its cursor still counts them; the slice then gets an exact region in the overflow pass.
constexpr int kExpThreads = 256;
constexpr uint32_t kExpMap = 16u * kExpThreads;  // k-mers per expansion chunk
constexpr uint32_t kExpW = kExpMap / 4;          // and 2-bit words

template <typename K, bool OVF>
__global__ __launch_bounds__(kExpThreads, 6) void k_expand(CountArgs a) {
    // chunks of at most TC records and 16 k-mers per thread; keys are held in registers in rounds of 8
    // (64-bit) or 4 (128-bit) per thread, which keeps six workgroups on a CU
    constexpr int TC = kExpThreads, S = (int)kMaxKeySlices + 1;
    __shared__ uint32_t stw[kExpW + 8];
    __shared__ uint16_t kpos[kExpMap];
    __shared__ uint32_t cnt[S], gb[S], lcur[S], rcap[S];
    __shared__ uint64_t roff[S];  // first key slot of each slice's region (~0: none)
    __shared__ uint32_t sh_any;
    __shared__ uint32_t tmp2[2 * (TC / 64)], wn[TC / 64], inclw[TC], inclk[TC];
    const KeyUnit ku = a.key_units[blockIdx.x];
    const int k = a.k;
    const K m = key_mask<K>(k);
    K* const reg = (K*)(OVF ? a.ovf_keys : a.heavy_keys);
    if (threadIdx.x == 0) sh_any = 0;
    __syncthreads();
    if (threadIdx.x < (uint32_t)S) {
        const uint32_t j = threadIdx.x;
        uint64_t off = ~0ull;
        uint32_t cap = 0;
        if (j < ku.u.q) {
            if (!OVF) {
                off = ku.key0 + (uint64_t)j * (ku.cs + 1ull) + 1;
                cap = ku.cs;
            } else if (const uint64_t n = a.ovf_n[ku.item0 + j]) {
                off = a.ovf_off[ku.item0 + j];
                cap = (uint32_t)n;
                sh_any = 1;
            }
        }
        roff[j] = off;
        rcap[j] = cap;
        lcur[j] = 0;
    }
    __syncthreads();
    if (OVF && !sh_any) return;
    const uint32_t* const desc = a.desc + ku.u.desc;
    const uint32_t* words = a.words + ku.u.word;  // the chunk's first word
    const uint32_t n_rec = ku.u.n_rec, q = ku.u.q;
    for (uint32_t c0 = 0; c0 < n_rec;) {
        const uint32_t r = c0 + threadIdx.x;
        const uint32_t km = r < n_rec ? desc[r] : 0u;
        const uint32_t nw = r < n_rec ? rec_words(km, k) : 0u;
        // the chunk: the leading records whose words and k-mers fit the staging areas. Both inclusive
        // prefixes grow with the thread index, so the records that fit are threads [0, n).
        uint32_t exW, exK, totW, totK;
        wg_exscan2_u32(nw, km, tmp2, exW, exK, totW, totK);
        const bool in = (r < n_rec) && (exW + nw <= kExpW) && (exK + km <= kExpMap);
        const uint64_t bal = __ballot(in);
        if ((threadIdx.x & 63u) == 0) wn[threadIdx.x >> 6] = (uint32_t)__popcll(bal);
        inclw[threadIdx.x] = exW + nw;
        inclk[threadIdx.x] = exK + km;
        if (threadIdx.x < (uint32_t)S) cnt[threadIdx.x] = 0;
        __syncthreads();
        uint32_t n = 0;
#pragma unroll
        for (int w = 0; w < TC / 64; w++) n += wn[w];
        if (n == 0) {
            // the first record alone exceeds the staging area: its k-mers straight from HBM
            const uint32_t nk1 = inclk[0], nw1 = inclw[0];
            for (uint32_t x = threadIdx.x; x < nk1; x += TC) {
                Window<K> w;
                w.load(words, x);
                const K key = w.key(0, k, m);
                const uint32_t i = slice_of(KT<K>::hash(key), q);
                if (roff[i] == ~0ull) continue;
                const uint32_t idx = atomicAdd(&lcur[i], 1u);
                if (idx < rcap[i]) reg[roff[i] + idx] = key;
            }
            __syncthreads();
            c0 += 1;
            words += nw1;
            continue;
        }
        const uint32_t nwc = inclw[n - 1], nkc = inclk[n - 1];
        for (uint32_t i = threadIdx.x; i < nwc + 8; i += TC) stw[i] = i < nwc ? words[i] : 0u;
        if (in)
            for (uint32_t j = 0; j < km; j++) kpos[exK + j] = (uint16_t)(exW * 16u + j);
        __syncthreads();
        constexpr int KPT_ALL = (int)kExpMap / TC;
        constexpr int KPT = sizeof(K) == 8 ? KPT_ALL / 2 : KPT_ALL / 4;
        for (int rd = 0; rd < KPT_ALL / KPT; rd++) {
            if ((uint32_t)(rd * KPT * TC) >= nkc) break;  // no keys left for this round
            if (rd > 0) {
                if (threadIdx.x < (uint32_t)S) cnt[threadIdx.x] = 0;
                __syncthreads();
            }
            K kk[KPT];
            uint32_t ti[KPT];
#pragma unroll
            for (int u = 0; u < KPT; u++) {
                const uint32_t x = threadIdx.x + (uint32_t)(rd * KPT + u) * TC;
                ti[u] = ~0u;
                if (x < nkc) {
                    Window<K> w;
                    w.load(stw, kpos[x]);
                    kk[u] = w.key(0, k, m);
                    const uint32_t i = slice_of(KT<K>::hash(kk[u]), q);
                    if (!OVF || roff[i] != ~0ull) ti[u] = i | (atomicAdd(&cnt[i], 1u) << 8);  // slice | rank in the round
                }
            }
            __syncthreads();
            if (threadIdx.x < (uint32_t)S) {
                gb[threadIdx.x] = lcur[threadIdx.x];
                lcur[threadIdx.x] += cnt[threadIdx.x];
            }
            __syncthreads();
#pragma unroll
            for (int u = 0; u < KPT; u++) {
                if (ti[u] == ~0u) continue;
                const uint32_t i = ti[u] & 255u;
                const uint32_t idx = gb[i] + (ti[u] >> 8);
                if (idx < rcap[i]) reg[roff[i] + idx] = kk[u];
            }
            __syncthreads();
        }
        c0 += n;
        words += nwc;
    }
    __syncthreads();
    // each slice's key count (past its capacity too) into the slot before its keys
    if (!OVF && threadIdx.x < q) *(unsigned long long*)&reg[roff[threadIdx.x] - 1] = (unsigned long long)lcur[threadIdx.x];
}

// After expansion, one thread per slice: its descriptor, and the keys of an exact region if it received
// more than its own holds.
template <typename K>
__device__ __forceinline__ const K* key_slice(const CountArgs& a, uint64_t i, KeyUnit& ku, uint32_t& slice) {
    const uint64_t it = a.key_items[i];
    slice = (uint32_t)(it & 255u);
    ku = a.key_units[it >> 8];
    return (const K*)a.heavy_keys + ku.key0 + (uint64_t)slice * (ku.cs + 1ull);
}
template <typename K>
__global__ void k_ovf_sizes(CountArgs a) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i > a.n_key_items) return;
    uint64_t need = 0;
    if (i < a.n_key_items) {
        KeyUnit ku;
        uint32_t slice;
        const K* const reg = key_slice<K>(a, i, ku, slice);
        const uint64_t n = *(const unsigned long long*)reg;
        if (n > ku.cs) need = n;
    }
    a.ovf_n[i] = need;
}
template <typename K>
__global__ void k_key_desc(CountArgs a) {
    const uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= a.n_key_items) return;
    KeyUnit ku;
    uint32_t slice;
    const K* const reg = key_slice<K>(a, i, ku, slice);
    KeyItem d;
    d.part = ku.u.part;
    d.n = (uint32_t) * (const unsigned long long*)reg;
    d.slice = slice;
    d.q = ku.u.q;
    d.keys = d.n > ku.cs ? (uint64_t)((const K*)a.ovf_keys + a.ovf_off[i]) : (uint64_t)(reg + 1);
    d.pad = 0;
    a.key_desc[i] = d;
}

// ---------------------------------------------------------------------------------------------
// 1. / 3. The two persistent count kernels: workgroup b takes units (or expanded slices) b, b + G, ...
//     (G = grid size), each in one or more sweeps.
struct Cut {
    uint32_t slice, n;
};

// A sweep's end: every thread takes its table slots into registers and clears them. `occ` and `keep` are
// the wave's occupied slots and those that pass [cmin, cmax].
template <typename K> struct Slots {
    static constexpr int SPT = (int)KT<K>::H / kItemThreads;
    static_assert(KT<K>::H % kItemThreads == 0, "whole slots per thread");
    K key[SPT];
    uint32_t cnt[SPT];
    __device__ __forceinline__ bool kept(const CountArgs& a, int j) const {
        return key[j] != KT<K>::empty() && cnt[j] >= a.cmin && cnt[j] <= a.cmax;
    }
    __device__ __forceinline__ void take(const CountArgs& a, K* tkeys, uint32_t* tcnt, uint32_t& occ, uint32_t& keep) {
        occ = keep = 0;
#pragma unroll
        for (int j = 0; j < SPT; j++) {
            const uint32_t s = threadIdx.x + (uint32_t)j * kItemThreads;
            key[j] = take_slot(tkeys, s);
            cnt[j] = tcnt[s];
            tcnt[s] = 0;
        }
#pragma unroll
        for (int j = 0; j < SPT; j++) {
            occ += (uint32_t)__popcll(__ballot(key[j] != KT<K>::empty()));
            keep += (uint32_t)__popcll(__ballot(kept(a, j)));
        }
    }
    // The wave's kept rows from row `row` on, straight from registers: the kept ones of 64 slots go to
    // consecutive rows, so they leave in nearly whole lines.
    __device__ __forceinline__ void store(const CountArgs& a, uint64_t row) const {
#pragma unroll
        for (int j = 0; j < SPT; j++) {
            const bool keeps = kept(a, j);
            const uint64_t kb = __ballot(keeps);
            if (keeps) {
                const uint64_t r = row + __builtin_amdgcn_mbcnt_hi((uint32_t)(kb >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)kb, 0u));
                if constexpr (sizeof(K) == 8) ((uint64_t*)a.out_keys)[r] = (uint64_t)key[j];
                else ((ulonglong2*)a.out_keys)[r] = make_ulonglong2((uint64_t)key[j], (uint64_t)((u128)key[j] >> 64));
                a.out_counts[r] = cnt[j];
            }
            row += (uint32_t)__popcll(kb);
        }
    }
};
// the workgroup's totals and the kept rows of the waves before this one, from each wave's in wtot
__device__ __forceinline__ void slot_totals(const uint32_t* wtot, uint32_t wave, uint32_t& nd, uint32_t& kept, uint32_t& before) {
    nd = kept = before = 0;
#pragma unroll
    for (int w = 0; w < kItemThreads / 64; w++) {
        const uint32_t t = wtot[w];
        nd += t & 0xFFFFu;
        if ((uint32_t)w < wave) before += t >> 16;
        kept += t >> 16;
    }
}
// Cuts an overflowing sweep: f slices of it onto the stack, from the distinct keys held when it stopped and
// the share of its records or keys read until then. False (and an error) if it cannot be cut.
__device__ __forceinline__ bool cut_sweep(const CountArgs& a, uint32_t ovf, Cut c, uint32_t nd, float frac, float fill, Cut* stack,
                                          uint32_t& n_stack) {
    uint32_t f = (uint32_t)ceilf(1.2f * (float)nd / (fminf(frac, 1.0f) * fill));
    f = max(2u, min(f, kMaxCut));
    if (ovf >= 2u || (uint64_t)c.n * f > kMaxSlices || n_stack + f > (uint32_t)kStack) {
        raise_err(a.err, RGKC_ERR_COUNT_FAIL);
        return false;
    }
    for (uint32_t j = 0; j < f; j++) stack[n_stack++] = Cut{c.slice * f + j, c.n * f};
    return true;
}
// Row reservation of a sweep (thread 0): the rows its partition had before, and its first row from them, or ~0 (and
// an error) if they don't fit its region (apart, so that the atomic's latency can pass in between).
__device__ __forceinline__ uint64_t reserve_rows(const CountArgs& a, uint32_t part, uint32_t kept, uint32_t nd) {
    uint64_t rows = 0;
    if (kept) rows = atomicAdd(&a.row_cursor[part], (unsigned long long)kept);
    if (nd) atomicAdd(&a.part_distinct[part], (unsigned long long)nd);
    return rows;
}
__device__ __forceinline__ uint64_t first_row(const CountArgs& a, uint32_t part, uint64_t rows, uint32_t kept) {
    const uint64_t base = a.row_base[part], end = a.row_end[part];
    if (base + rows + kept <= end) return base + rows;
    raise_err(a.err, RGKC_ERR_ROW_OVERFLOW);
    return ~0ull;
}

// Units, from their records: chunk after chunk of up to kItemThreads * R records. A chunk is staged (record
// sizes scanned, words and record info to LDS) from registers whose loads were issued while the chunk
// before it was counted, across the ends of sweeps and units as well; a sweep's rows leave only after the
// next chunk is staged, so the row reservation's latency passes under the staging and the stores' under
// the next chunk's counting. (With the loads of a sweep's first chunk and its row stores in line, staging
// and row output took a third of the kernel.)
// Bound by LDS in the insert (random 32-byte reads, CAS and count atomics: a third of the time) and by the phases
// around it, one after another: equal records 15%, the wait for the slowest wave 14%, staging 11% (clocks of the
// first thread over 10 M reads at 30x). 1.2 G k-mers at 30x (360 M
// distinct): 7.7 ms, where expanding every k-mer took 6.5 and counting the keys 6.0; 188 M (k=25) 1.14 ms, before
// 1.2 + 0.85; 392 M 128-bit keys 5.4 ms, before 5.3 + 7.0. The loads take a uniform base and a thread's offset: with an
// address per load 27 registers went to scratch, 0.6 ms of the first.
template <typename K>
__global__ __launch_bounds__(kItemThreads, 4) void k_count_units(CountArgs a) {
    using C = Chunk<K>;
    constexpr int TC = kItemThreads, NW = TC / 64, R = C::R, WPT = (int)C::W / TC;
    __shared__ __align__(16) K tkeys[KT<K>::H];
    __shared__ uint32_t tcnt[KT<K>::H];
    __shared__ uint32_t stw[C::W + 8];
    // a chunk's records: first word | k-mers << WBits, how many equal ones; the hash set of the records, then
    // the pieces; the long records
    __shared__ uint32_t rinfo[TC * R], rmul[TC * R];
    __shared__ union { uint32_t same[C::S]; uint16_t pmap[C::P]; } mp;
    __shared__ uint16_t longs[C::MaxLong];
    __shared__ Cut stack[kStack];
    __shared__ uint32_t tmp2[2 * NW], wtot[NW];
    __shared__ unsigned long long sh_in;  // chunk: records << 20 | words
    __shared__ uint64_t sh_row_base;
    __shared__ uint32_t sh_ovf, sh_np, sh_long, sh_nstack, sh_next, sh_next_q;
    __shared__ uint32_t sh_first, sh_q0, sh_s0, sh_ns;  // next slice of the item, of q0 from slice s0 of ns on
    __shared__ Cut cur;
    uint32_t* const same = mp.same;
    uint16_t* const pmap = mp.pmap;

    const int k = a.k;
    const K m = key_mask<K>(k);
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    const uint64_t G = gridDim.x, it_end = a.plan_n[kPlanItems];
    uint64_t it = blockIdx.x;
    if (it >= it_end) return;
    // the workgroup's sweep, retry and distinct totals, added to the global counters once at the end;
    // instances and distinct keys of its sweeps are added to the shared totals every few sweeps
    unsigned long long n_sweeps = 0, n_retries = 0, n_distinct = 0, seen_i = 0, seen_d = 0;
    unsigned long long est_i = 0, est_d = 0;  // the shared totals, read one unit ahead by the last wave
    for (uint32_t i = threadIdx.x; i < KT<K>::H; i += TC) { tkeys[i] = KT<K>::empty(); tcnt[i] = 0; }

    // descriptors: lane i of every wave loads word i one unit ahead, and the fields are wave-uniform
    constexpr uint32_t DW = sizeof(UnitDesc) / 4;
    static_assert(DW <= 64, "a lane per word");
    const uint32_t* const items = (const uint32_t*)a.unit_items;
    auto fetch = [&](uint64_t i) { return (i < it_end && lane < DW) ? items[i * DW + lane] : 0u; };
    auto unit = [&](uint32_t v) {
        auto word = [&](int i) { return (uint32_t)__builtin_amdgcn_readlane((int)v, i); };
        UnitDesc d;
        d.part = word(0); d.inst = word(1); d.n_rec = word(2); d.n_word = word(3);
        d.desc = (uint64_t)word(4) | ((uint64_t)word(5) << 32);
        d.word = (uint64_t)word(6) | ((uint64_t)word(7) << 32);
        d.q = d.share = 0;
        return d;
    };
    constexpr int kQ = offsetof(UnitDesc, q) / 4, kShare = offsetof(UnitDesc, share) / 4;
    uint32_t ahead = fetch(it);
    UnitDesc ud = unit(ahead);
    // Initial hash slices of a unit's share: what its distinct keys should take by the ratio seen so far. The next unit's are
    // worked out by the last wave, which has the fewest records, while the others look for equal ones (at the sweep's
    // end by thread 0 they took 6% of the kernel).
    auto slices = [&](uint32_t v) {
        const uint32_t inst = (uint32_t)__builtin_amdgcn_readlane((int)v, 1), shares = max((uint32_t)__builtin_amdgcn_readlane((int)v, kQ), 1u);
        const float ratio = est_i > 4ull * a.unit_cap ? (float)est_d / (float)est_i : kFill<K> / (float)a.unit_cap;
        uint32_t q = (uint32_t)ceilf(1.1f * (float)inst * fminf(ratio, 1.0f) / kFill<K>);
        q = max(1u, min(q, kMaxSlices));
        if ((float)inst <= kFill<K>) q = 1u;
        est_i = __hip_atomic_load(&a.plan_n[kPlanSeenInst], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        est_d = __hip_atomic_load(&a.plan_n[kPlanSeenDistinct], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return shares == 1u ? q : (q + shares - 1u) / shares;
    };
    // thread 0: the item `v` begins, its share cut into q slices
    auto begin = [&](uint32_t v, uint32_t q) {
        sh_q0 = q;
        sh_s0 = (uint32_t)__builtin_amdgcn_readlane((int)v, kShare) * q;
        sh_ns = (uint32_t)__builtin_amdgcn_readlane((int)v, kQ) * q;
        sh_first = 1;
        cur = Cut{sh_s0, sh_ns};
    };
    bool planned = false;  // the next unit's slices are in sh_next_q
    {
        const uint32_t q = slices(ahead);
        if (threadIdx.x == 0) {
            sh_nstack = 0;
            begin(ahead, q);
            sh_ovf = 0;
        }
    }
    ahead = fetch(it + G);

    uint32_t dn[R], wn[WPT];  // the next chunk's descriptors and words of this thread
    auto load = [&](const UnitDesc& d, uint32_t c, uint32_t w) {
        const uint32_t* const pd = a.desc + d.desc + c;
        const uint32_t* const pw = a.words + d.word + w;
        const uint32_t ld = d.n_rec - c, lw = d.n_word - w;
#pragma unroll
        for (int j = 0; j < R; j++) {
            const uint32_t i = threadIdx.x * R + (uint32_t)j;
            dn[j] = i < ld ? pd[i] : 0u;
        }
#pragma unroll
        for (int u = 0; u < WPT; u++) {
            const uint32_t i = threadIdx.x + (uint32_t)u * TC;
            wn[u] = i < lw ? pw[i] : 0u;
        }
    };
    uint32_t n_in;  // this thread's records in the chunk
    auto pieces = [](uint32_t km) __attribute__((always_inline)) { return (km + kPiece - 1u) / kPiece; };
    // stages the loaded chunk (records c ... of the unit); `publish` runs in thread 0 before its last barrier
    auto stage = [&](uint32_t c, auto&& publish) {
        uint32_t nw[R], np[R], sw = 0, sp = 0;
#pragma unroll
        for (int j = 0; j < R; j++) {
            nw[j] = c + threadIdx.x * R + (uint32_t)j < ud.n_rec ? rec_words(dn[j], k) : 0u;
            np[j] = pieces(dn[j]);
            sw += nw[j];
            sp += np[j];
        }
        if (threadIdx.x == 0) { sh_in = 0; sh_np = 0; sh_long = 0; }
        uint32_t exW, exP, totW, totP;
        wg_exscan2_u32(sw, sp, tmp2, exW, exP, totW, totP);
        n_in = 0;
        uint32_t end = 0;
#pragma unroll
        for (int j = 0; j < R; j++) {
            const uint32_t r = threadIdx.x * R + (uint32_t)j;
            rinfo[r] = (exW & C::WMask) | (dn[j] << C::WBits);
            rmul[r] = 1u;
            exW += nw[j];
            exP += np[j];
            if (c + r < ud.n_rec && exW <= C::W && exP <= C::P) {
                n_in = (uint32_t)j + 1u;
                end = exW;
            }
        }
        const uint64_t bal = __ballot(n_in != 0);
        if (n_in && (bal >> lane) == 1ull) atomicMax(&sh_in, ((unsigned long long)(threadIdx.x * R + n_in) << 20) | end);
#pragma unroll
        for (int u = 0; u < WPT; u++) stw[threadIdx.x + (uint32_t)u * TC] = wn[u];
        for (uint32_t i = threadIdx.x; i < C::S; i += TC) same[i] = 0;
        if (threadIdx.x == 0) publish();
        __syncthreads();
    };
    load(ud, 0, 0);
    stage(0, [] {});
    uint32_t c0 = 0, w0 = 0;  // the staged chunk's first record and word in its unit
    for (;;) {
        const uint32_t n = (uint32_t)(sh_in >> 20), slice = cur.slice, ns = cur.n;
        const bool filt = ns > 1;
        // n == 0: the first record alone exceeds the staging area
        const uint32_t c1 = c0 + max(n, 1u), w1 = w0 + (n ? (uint32_t)sh_in & 0xFFFFFu : rec_words(rinfo[0] >> C::WBits, k));
        const bool last = c1 >= ud.n_rec;
        // the next chunk's loads: this sweep's, the unit's next sweep's, or the next unit's
        const bool again = sh_nstack > 0 || sh_first < sh_q0;
        if (!last) load(ud, c1, w1);
        else if (again) load(ud, 0, 0);
        else load(unit(ahead), 0, 0);
        if (!planned && wave == (uint32_t)NW - 1u) {
            const uint32_t q = slices(ahead);
            if (lane == 0) sh_next_q = q;
        }
        planned = true;
        auto single = [&](const uint32_t* bw, uint32_t g, uint32_t mul) {
            Window<K> w;
            w.load(bw, g);
            const K key = w.key(0, k, m);
            const uint32_t h = KT<K>::hash(key);
            insert<1>(tkeys, tcnt, &key, &h, !filt || slice_of(h, ns) == slice ? 1u : 0u, mul, &sh_ovf);
        };
        if (n == 0) {
            const uint32_t km1 = rinfo[0] >> C::WBits;  // its k-mers straight from HBM
            for (uint32_t x = threadIdx.x; x < km1 && !sh_ovf; x += TC) single(a.words + ud.word + w0, x, 1u);
        } else {
            // Equal records (reads of one place without errors give equal records but for their ends: two in
            // five at 30x and 1% errors) are counted once, with their number: a hash set of the chunk's
            // records, compared word by word.
            // Words in blocks of four (staged words follow a record's last, or slack), the first one kept.
            uint32_t uniq = (1u << n_in) - 1u;
            uint32_t x[R][4], hash[R];
#pragma unroll
            for (int j = 0; j < R; j++) {
                const uint32_t info = rinfo[threadIdx.x * R + j], w0r = info & C::WMask;
                const uint32_t nw = (uint32_t)j < n_in ? rec_words(info >> C::WBits, k) : 0u;
                uint32_t h = info >> C::WBits;
                auto block = [&](uint32_t i, uint32_t* v) {
#pragma unroll
                    for (uint32_t t = 0; t < 4; t++) v[t] = i + t < nw ? stw[w0r + i + t] : 0u;
#pragma unroll
                    for (int t = 0; t < 4; t++) h = mix_in(h) ^ v[t];
                };
                block(0, x[j]);
                if (nw <= 16u) {
                    uint32_t y[4];
#pragma unroll 1
                    for (uint32_t i = 4; i < nw; i += 4) block(i, y);
                }
                hash[j] = mix(h);
            }
#pragma unroll
            for (int j = 0; j < R; j++) {
                const uint32_t rec = threadIdx.x * R + (uint32_t)j, info = rinfo[rec], w0r = info & C::WMask;
                const uint32_t nw = rec_words(info >> C::WBits, k), h = hash[j];
                if ((uint32_t)j >= n_in || nw > 16u) continue;
                const uint32_t entry = (rec + 1u) | (h << 16);
#pragma unroll 1
                for (uint32_t s = h >> 16, tries = 0; tries < 8u; s++, tries++) {
                    const uint32_t o = atomicCAS(&same[s % C::S], 0u, entry);
                    if (o == 0) break;
                    if ((o ^ entry) >> 16) continue;
                    const uint32_t other = (o & 0xFFFFu) - 1u, oi = rinfo[other];
                    if ((oi ^ info) >> C::WBits) continue;
                    const uint32_t* const q = stw + (oi & C::WMask);
                    uint32_t diff = 0;
#pragma unroll
                    for (uint32_t t = 0; t < 4; t++) diff |= t < nw ? q[t] ^ x[j][t] : 0u;
#pragma unroll 1
                    for (uint32_t i = 4; i < nw; i += 4)
#pragma unroll
                        for (uint32_t t = 0; t < 4; t++) diff |= i + t < nw ? q[i + t] ^ stw[w0r + i + t] : 0u;
                    if (diff) continue;
                    atomicAdd(&rmul[other], 1u);
                    uniq &= ~(1u << j);
                    break;
                }
            }
            __syncthreads();
            // pieces of the records that remain; a record of more than `Long` apart
            {
                uint32_t mine[R], sum = 0;
#pragma unroll
                for (int j = 0; j < R; j++) {
                    const uint32_t np = pieces(rinfo[threadIdx.x * R + j] >> C::WBits);
                    const bool counts = (uniq >> j) & 1u;
                    mine[j] = counts && np <= C::Long ? np : 0u;
                    if (counts && np > C::Long) longs[atomicAdd(&sh_long, 1u)] = (uint16_t)(threadIdx.x * R + j);
                    sum += mine[j];
                }
                const uint32_t incl = wave_incl_scan_u32(sum);
                uint32_t wb = 0;
                if (lane == 63u) wb = atomicAdd(&sh_np, incl);
                uint32_t e = (uint32_t)__builtin_amdgcn_readlane((int)wb, 63) + incl - sum;
#pragma unroll
                for (int j = 0; j < R; j++)
                    for (uint32_t i = 0; i < mine[j]; i++) pmap[e++] = (uint16_t)((threadIdx.x * R + j) | (i << C::RecBits));
            }
            __syncthreads();
            const uint32_t npc = sh_np;
            for (uint32_t x = threadIdx.x; x < npc; x += TC) {
                const uint32_t e = pmap[x], rec = e & ((1u << C::RecBits) - 1u), j = e >> C::RecBits, info = rinfo[rec];
                const uint32_t mul = rmul[rec], c = min(kPiece, (info >> C::WBits) - kPiece * j);
                Window<K> w;
                w.load(stw, (info & C::WMask) * 16u + kPiece * j);
                K key[kPiece];
                uint32_t h[kPiece], valid = (1u << c) - 1u, pend = 0;
#pragma unroll
                for (int t = 0; t < (int)kPiece; t++) {
                    key[t] = w.key(t, k, m);
                    h[t] = KT<K>::hash(key[t]);
                    if (filt) valid &= ~((uint32_t)(slice_of(h[t], ns) != slice) << t);
                    // one at a time: two or four together read no slot sooner (16 waves do) and take 1 and 4% longer
                    pend |= insert_first<1>(tkeys, tcnt, key + t, h + t, valid >> t, mul) << t;
                }
                insert_rest<(int)kPiece>(tkeys, tcnt, key, h, pend, mul, &sh_ovf);
            }
            for (uint32_t q = 0; q < sh_long; q++) {
                const uint32_t info = rinfo[longs[q]], kq = info >> C::WBits, mul = rmul[longs[q]];
                for (uint32_t x = threadIdx.x; x < kq; x += TC) single(stw, (info & C::WMask) * 16u + x, mul);
            }
        }
        __syncthreads();
        const uint32_t ovf = sh_ovf;
        if (!last && !ovf) {
            c0 = c1;
            w0 = w1;
            stage(c0, [] {});
            continue;
        }
        // ---- the sweep ends: its slots to registers, its rows reserved, the next sweep chosen and its first
        // chunk staged, then the rows stored
        Slots<K> sl;
        uint32_t occ, keep;
        sl.take(a, tkeys, tcnt, occ, keep);
        if (lane == 0) wtot[wave] = occ | (keep << 16);
        __syncthreads();
        uint32_t nd, kept, before;
        slot_totals(wtot, wave, nd, kept, before);
        const uint32_t part = ud.part;
        uint64_t row0 = 0;
        if (threadIdx.x == 0) {
            if (ovf) {  // cut: the rest of its records is skipped
                n_retries++;
                cut_sweep(a, ovf, cur, nd, (float)c1 / (float)ud.n_rec, kFill<K>, stack, sh_nstack);
            } else {
                row0 = reserve_rows(a, part, kept, nd);
                n_sweeps++;
                n_distinct += nd;
                seen_i += ud.inst / ns;
                seen_d += nd;
                if (n_sweeps <= 2 || (n_sweeps & 7u) == 0) {
                    atomicAdd(&a.plan_n[kPlanSeenInst], seen_i);
                    atomicAdd(&a.plan_n[kPlanSeenDistinct], seen_d);
                    seen_i = seen_d = 0;
                }
            }
            sh_ovf = 0;
            if (sh_nstack > 0) {
                cur = stack[--sh_nstack];
                sh_next = 0;
            } else if (sh_first < sh_q0) {
                cur = Cut{sh_s0 + sh_first++, sh_ns};
                sh_next = 0;
            } else {
                sh_next = 1;
                if (it + G < it_end) begin(ahead, sh_next_q);
            }
        }
        __syncthreads();
        const bool next_unit = sh_next != 0;
        // what was loaded ahead is the next sweep's, unless this one was cut
        const bool reload = ovf != 0;
        if (next_unit) {
            it += G;
            if (it >= it_end) {
                if (threadIdx.x == 0 && !ovf) sh_row_base = first_row(a, part, row0, kept);
                __syncthreads();
                if (!ovf && sh_row_base != ~0ull) sl.store(a, sh_row_base + before);
                break;
            }
            ud = unit(ahead);
            ahead = fetch(it + G);
            planned = false;
        }
        if (reload) load(ud, 0, 0);
        c0 = w0 = 0;
        stage(0, [&] {
            if (!ovf) sh_row_base = first_row(a, part, row0, kept);
        });
        if (!ovf && sh_row_base != ~0ull) sl.store(a, sh_row_base + before);
    }
    if (threadIdx.x == 0) {
        if (n_sweeps) atomicAdd(&a.stats[0], n_sweeps);
        if (n_retries) atomicAdd(&a.stats[1], n_retries);
        if (n_distinct) atomicAdd(&a.stats[2], n_distinct);
    }
}

// Expanded slices, from their keys.
template <typename K>
__global__ __launch_bounds__(kItemThreads, 4) void k_count_keys(CountArgs a) {
    constexpr int TC = kItemThreads, NW = TC / 64, KB = 4;
    __shared__ __align__(16) K tkeys[KT<K>::H];
    __shared__ uint32_t tcnt[KT<K>::H];
    __shared__ Cut stack[kStack];
    __shared__ uint32_t wtot[NW];
    __shared__ uint64_t sh_row_base;
    __shared__ uint32_t sh_ovf, sh_nstack;
    __shared__ Cut cur;
    const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
    unsigned long long n_sweeps = 0, n_retries = 0, n_distinct = 0;
    for (uint32_t i = threadIdx.x; i < KT<K>::H; i += TC) { tkeys[i] = KT<K>::empty(); tcnt[i] = 0; }
    for (uint64_t it = blockIdx.x; it < a.n_key_items; it += gridDim.x) {
        const KeyItem kd = a.key_desc[it];
        const K* const kreg = (const K*)kd.keys;
        __syncthreads();
        if (threadIdx.x == 0) {
            stack[0] = Cut{kd.slice, kd.q};
            sh_nstack = 1;
        }
        __syncthreads();
        for (;;) {
            if (threadIdx.x == 0) {
                cur.n = 0;
                if (sh_nstack > 0) cur = stack[--sh_nstack];
                sh_ovf = 0;
            }
            __syncthreads();
            const uint32_t slice = cur.slice, ns = cur.n;
            if (ns == 0) break;
            const bool filt = ns != kd.q;  // a region holds exactly its slice: only a finer one filters its keys
            uint32_t scanned = 0;
            K v[KB];
#pragma unroll
            for (int u = 0; u < KB; u++) v[u] = threadIdx.x + (uint32_t)u * TC < kd.n ? kreg[threadIdx.x + (uint32_t)u * TC] : (K)0;
            for (uint32_t x0 = 0; x0 < kd.n; x0 += (uint32_t)(KB * TC)) {
                K key[KB];
                uint32_t h[KB], valid = 0;
#pragma unroll
                for (int u = 0; u < KB; u++) {
                    const uint32_t x = x0 + threadIdx.x + (uint32_t)u * TC, y = x + (uint32_t)(KB * TC);
                    key[u] = v[u];
                    v[u] = y < kd.n ? kreg[y] : (K)0;  // the next batch, in flight while this one is counted
                    h[u] = KT<K>::hash(key[u]);
                    if (x < kd.n && (!filt || slice_of(h[u], ns) == slice)) valid |= 1u << u;
                }
                insert<KB>(tkeys, tcnt, key, h, valid, 1u, &sh_ovf);
                scanned += (uint32_t)(KB * TC);
                if (sh_ovf) break;
            }
            __syncthreads();
            Slots<K> sl;
            uint32_t occ, keep, nd, kept, before;
            sl.take(a, tkeys, tcnt, occ, keep);
            if (lane == 0) wtot[wave] = occ | (keep << 16);
            __syncthreads();
            slot_totals(wtot, wave, nd, kept, before);
            const uint32_t ovf = sh_ovf;
            if (threadIdx.x == 0) {
                if (ovf) {
                    n_retries++;
                    cut_sweep(a, ovf, cur, nd, (float)scanned / (float)kd.n, kFill<K>, stack, sh_nstack);
                } else {
                    sh_row_base = first_row(a, kd.part, reserve_rows(a, kd.part, kept, nd), kept);
                    n_sweeps++;
                    n_distinct += nd;
                }
            }
            __syncthreads();
            if (!ovf && sh_row_base != ~0ull) sl.store(a, sh_row_base + before);
        }
    }
    if (threadIdx.x == 0) {
        if (n_sweeps) atomicAdd(&a.stats[0], n_sweeps);
        if (n_retries) atomicAdd(&a.stats[1], n_retries);
        if (n_distinct) atomicAdd(&a.stats[2], n_distinct);
    }
}

}  // namespace

hipError_t launch_expand(const CountArgs& a, uint64_t n_units, hipStream_t s) {
    if (!n_units) return hipSuccess;
    if (a.k <= 32) hipLaunchKernelGGL((k_expand<uint64_t, false>), dim3((unsigned)n_units), dim3(kExpThreads), 0, s, a);
    else hipLaunchKernelGGL((k_expand<u128, false>), dim3((unsigned)n_units), dim3(kExpThreads), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_ovf_sizes(const CountArgs& a, hipStream_t s) {
    const unsigned nb = (unsigned)((a.n_key_items + 1 + 255) / 256);
    if (a.k <= 32) hipLaunchKernelGGL(k_ovf_sizes<uint64_t>, dim3(nb), dim3(256), 0, s, a);
    else hipLaunchKernelGGL(k_ovf_sizes<u128>, dim3(nb), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_expand_ovf(const CountArgs& a, uint64_t n_units, hipStream_t s) {
    if (!n_units) return hipSuccess;
    if (a.k <= 32) hipLaunchKernelGGL((k_expand<uint64_t, true>), dim3((unsigned)n_units), dim3(kExpThreads), 0, s, a);
    else hipLaunchKernelGGL((k_expand<u128, true>), dim3((unsigned)n_units), dim3(kExpThreads), 0, s, a);
    return hipGetLastError();
}

// one resident workgroup per CU (its table and staging areas take the LDS), looping over units
static unsigned count_grid() {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess || hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
        cus = 256;
    return (unsigned)cus;
}

hipError_t launch_count_units(const CountArgs& a, hipStream_t s) {
    const unsigned grid = count_grid();
    if (a.k <= 32) hipLaunchKernelGGL(k_count_units<uint64_t>, dim3(grid), dim3(kItemThreads), 0, s, a);
    else hipLaunchKernelGGL(k_count_units<u128>, dim3(grid), dim3(kItemThreads), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_count_keys(const CountArgs& a, hipStream_t s) {
    if (!a.n_key_items) return hipSuccess;
    const unsigned pb = (unsigned)((a.n_key_items + 255) / 256);
    const unsigned grid = (unsigned)std::min<uint64_t>(a.n_key_items, count_grid());
    if (a.k <= 32) {
        hipLaunchKernelGGL(k_key_desc<uint64_t>, dim3(pb), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k_count_keys<uint64_t>, dim3(grid), dim3(kItemThreads), 0, s, a);
    } else {
        hipLaunchKernelGGL(k_key_desc<u128>, dim3(pb), dim3(256), 0, s, a);
        hipLaunchKernelGGL(k_count_keys<u128>, dim3(grid), dim3(kItemThreads), 0, s, a);
    }
    return hipGetLastError();
}

}  // namespace rgkc
