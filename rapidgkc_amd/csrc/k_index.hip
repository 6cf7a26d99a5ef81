// Side descriptors for superkmer stores that arrive from the host (e.g. the chunks of an
// SKMStoreNoncon, skmstore.hpp:62-99), which carry only record bytes.
//
// A record starts at byte 0 of a partition and after every "full byte then non-full byte" pair (the
// reference's boundary rule, cpu_funcs.cpp:516-525 / gpu_kmercounting.cu:166-176), so any piece of a
// partition finds its records from its own bytes and the two before it. One workgroup takes one piece of
// kIndexChunk bytes, a thread 32 of them as a bit mask; the piece's starts are listed in LDS and the
// threads take whole records from the list: they follow a record to its last byte (first non-full byte
// after the first), which gives its base count, and in the fill pass compute the minimizer of its first
// k-mer from registers (all k-mers of a superkmer share it) to get the sub-bucket id. Between the two
// passes a scan over the pieces' record counts gives every piece's first record.
// One workgroup per partition, 1024 bytes a step and a byte load per base, took 12.4 ms for 116 MB in 512
// partitions (8 M records).
#include "rgkc_device.h"
#include "rgkc_internal.h"

namespace rgkc {
namespace {

constexpr int T = 256;
constexpr int kBytes = 32;  // bytes of a piece per thread
static_assert(kIndexChunk == (uint64_t)T * kBytes, "one mask per thread");

// Bit b set: byte b of x is full (its two high bits are set).
__device__ __forceinline__ uint32_t full_bits(uint32_t x) {
    const uint32_t t = (x & (x << 1) & 0x80808080u) >> 7;
    return (t & 1u) | ((t >> 7) & 2u) | ((t >> 14) & 4u) | ((t >> 21) & 8u);
}

// Bytes after which a record cannot end with k-mers that a side word holds (18 bits): it is not followed further, so
// that bytes without an end (60 MB of them kept one thread busy for 2.2 s) cost no more than a long record.
constexpr uint64_t kMostBytes = (0x3FFFFu + 64u) / 3u + 4u;

// Record starting at byte i of a partition of n bytes: sets bm3 and bases.
__device__ __forceinline__ void record_shape(const uint8_t* s, uint64_t i, uint64_t n, uint32_t& bm3, uint32_t& L, bool& ok) {
    const uint32_t ind0 = (uint32_t)s[i] >> 6;
    const uint64_t end = min(n, i + kMostBytes);
    uint64_t j = i + 1;
    bool ends = false;
    while (j < end) {  // the store's buffer holds 64 bytes after its last
        const uint32_t f = full_bits(load_u32(s + j));
        if (f != 15u) {
            j += (uint32_t)__builtin_ctz(~f);
            ends = j < n;
            break;
        }
        j += 4;
    }
    ok = ind0 != 0 && ends;
    bm3 = ok ? 3u - ind0 : 0u;
    L = ok ? ind0 + 3u * (uint32_t)(j - i - 1) + ((uint32_t)s[j] >> 6) : 0u;
}

template <bool FILL>
__global__ __launch_bounds__(T) void k_index(IndexArgs a) {
    __shared__ uint16_t starts[kIndexChunk / 2 + 2];  // two starts are at least two bytes apart
    __shared__ uint32_t tmp[T / 64 + 1];
    __shared__ unsigned long long sh_kmers;
    const uint32_t part = a.chunk_part[blockIdx.x];
    const uint64_t b0 = a.part_byte[part], n = a.part_byte[part + 1] - b0;
    const uint64_t c0 = (blockIdx.x - a.part_chunk[part]) * kIndexChunk;
    const uint8_t* const s = a.store + b0;
    const int k = a.k, p = a.p;
    if (threadIdx.x == 0) sh_kmers = 0;
    uint32_t st = 0;
    const uint64_t at = c0 + (uint64_t)threadIdx.x * kBytes;
    if (at < n) {
        uint64_t full = at ? full_bits(load_u16(s + at - 2)) : 0ull;  // bits 0, 1: the two bytes before
#pragma unroll
        for (int q = 0; q < kBytes / 4; q++) full |= (uint64_t)full_bits(load_u32(s + at + 4 * q)) << (2 + 4 * q);
        st = (uint32_t)(full & ~(full >> 1));
        if (at == 0) st |= 1u;
        if (n - at < (uint64_t)kBytes) st &= (1u << (uint32_t)(n - at)) - 1u;
    }
    uint32_t tot;
    uint32_t ex = wg_exscan_u32((uint32_t)__popc(st), tmp, &tot);
    for (; st; st &= st - 1u) starts[ex++] = (uint16_t)(threadIdx.x * kBytes + (uint32_t)__builtin_ctz(st));
    __syncthreads();
    uint64_t kmers = 0;
    for (uint32_t r = threadIdx.x; r < tot; r += T) {
        const uint64_t i = c0 + starts[r];
        uint32_t bm3, L;
        bool ok;
        record_shape(s, i, n, bm3, L, ok);
        if (!ok || L < (uint32_t)k || L - (uint32_t)k + 1u > 0x3FFFFu) {
            raise_err(a.err, RGKC_ERR_BAD_STORE);
            continue;
        }
        const uint32_t km = L - (uint32_t)k + 1u;
        kmers += km;
        if (FILL) {
            // minimizer of the first k-mer: min over its p-mers of the filtered strands
            const uint32_t pmask = (p >= 16) ? 0xFFFFFFFFu : ((1u << (2 * p)) - 1u);
            const uint32_t rsh = 2u * (uint32_t)(p - 1);
            uint32_t f = 0, rv = 0, mm = pmask;
            for (int t0 = 0; t0 < k; t0 += 16) {
                uint32_t w = record_word(s + i, bm3, (uint32_t)t0, L);
                const int te = min(k, t0 + 16);
                for (int t = t0; t < te; t++, w >>= 2) {
                    const uint32_t c = w & 3u;
                    f = ((f << 2) | c) & pmask;
                    rv = (rv >> 2) | ((3u - c) << rsh);
                    if (t >= p - 1) {
                        const uint32_t vf = pmer_valid(f, p) ? f : pmask;
                        const uint32_t vr = pmer_valid(rv, p) ? rv : pmask;
                        const uint32_t v = vf < vr ? vf : vr;
                        mm = v < mm ? v : mm;
                    }
                }
            }
            const uint32_t nmm = ~mm;
            // the store's partition count spreads a partition's minimizers over the
            // sub-buckets; without it, the top bits of a multiplicative hash of them do
            const uint32_t sub = a.parts_total ? (nmm / (uint32_t)a.parts_total) % (uint32_t)kSubIds
                                               : (nmm * 0x9E3779B1u) >> (32 - 12);
            a.side[a.chunk_rec[blockIdx.x] + r] = side_pack(sub, km, bm3);
        }
    }
    if (!FILL) {
        for (int o = 32; o > 0; o >>= 1) kmers += __shfl_down(kmers, o, 64);
        if ((threadIdx.x & 63u) == 0) atomicAdd(&sh_kmers, (unsigned long long)kmers);
        __syncthreads();
        if (threadIdx.x == 0) {
            a.chunk_n[blockIdx.x] = tot;
            if (sh_kmers) atomicAdd((unsigned long long*)&a.rec_count[2 * part + 1], sh_kmers);
        }
    }
}

// records per partition from the pieces' prefix
__global__ void k_index_parts(IndexArgs a) {
    const uint32_t i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < a.n_parts) a.rec_count[2 * i] = a.chunk_rec[a.part_chunk[i + 1]] - a.chunk_rec[a.part_chunk[i]];
}

}  // namespace

// chunk_n receives the records of each piece, rec_count[2 * i + 1] (zeroed) the k-mers of partition i.
hipError_t launch_index_count(const IndexArgs& a, hipStream_t s) {
    if (!a.n_chunks) return hipSuccess;
    hipLaunchKernelGGL(k_index<false>, dim3(a.n_chunks), dim3(T), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_index_parts(const IndexArgs& a, hipStream_t s) {
    hipLaunchKernelGGL(k_index_parts, dim3((a.n_parts + 255) / 256), dim3(256), 0, s, a);
    return hipGetLastError();
}

hipError_t launch_index_fill(const IndexArgs& a, hipStream_t s) {
    if (!a.n_chunks) return hipSuccess;
    hipLaunchKernelGGL(k_index<true>, dim3(a.n_chunks), dim3(T), 0, s, a);
    return hipGetLastError();
}

}  // namespace rgkc
