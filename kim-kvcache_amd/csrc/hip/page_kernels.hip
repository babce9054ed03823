// page_kernels.hip -- append (with fused partial-tail COW), gather, promotion
// and synthetic fill kernels for gfx950.
//
// Reference kernels these replace (semantics only):
//   copyPageTokensKernel / appendTokensKernel  src/cuda/kv/page_kernels.cu:46-127
//   copyLayerTokensKernel / writeLayerTokenKernel
//                                      src/cuda/attention/paged_decode_kernels.cu:29-99
//   promotionKernel                    src/cuda/kv/page_kernels.cu:129-182
//   gatherKernel                       src/cuda/kv/page_kernels.cu:184-242
#include <hip/hip_runtime.h>

#include <type_traits>

#include "device_common.h"
#include "runtime_internal.h"

namespace kimkv {
namespace {

constexpr unsigned kBlock = 256;
constexpr unsigned kTile = 64;   // tokens per gather/fill tile

typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));

struct TokEntry {
    uint16_t* page;
    uint32_t cap;
    uint32_t pt;
};

// x / d and x % d for a d that is uniform over the launch: the reciprocal is
// computed on the host (floor((2^32 - 1) / d)), so the quotient is at most one
// short and one compare corrects it.  Exact for every x < 2^32; an integer
// division by a kernel argument is about 30 instructions, this is 7.
struct Divisor {
    uint32_t d;
    uint32_t m;
};
inline Divisor divisor(uint32_t d) { return Divisor{d, 0xFFFFFFFFu / (d == 0 ? 1u : d)}; }

__device__ inline uint32_t div_mod(uint32_t x, Divisor v, uint32_t* rem)
{
    uint32_t q = __umulhi(x, v.m);
    uint32_t r = x - q * v.d;
    if (r >= v.d) {
        ++q;
        r -= v.d;
    }
    *rem = r;
    return q;
}

// k_offset and v_offset (device_common.h) without their divisions: d < D and
// t < cap, so the column block is a shift or 0, which the compiler cannot
// tell of a width that is 32 or the whole row.  A copy computes two such
// offsets for 16 bytes; the attention kernels, which compute few, are 4%
// slower with this form (a branch per operand load).  In 32 bits, which hold
// every offset of one head's block of 2 cap D elements (cap < 2^16) as long
// as D <= kMaxDim32; in 64 bits the prompts' append and promotion are 1.5%
// slower.  The paths that use them are closed to wider heads, which copy
// element by element at k_offset and v_offset.
constexpr uint32_t kMaxDim32 = 32768;

__device__ inline uint32_t k_at(uint32_t cap, uint32_t D, uint32_t t, uint32_t d)
{
    return D % 32u == 0u ? (d >> 5) * cap * 32u + t * 32u + (d & 31u) : t * D + d;
}

__device__ inline uint32_t v_at(uint32_t cap, uint32_t D, uint32_t t, uint32_t d)
{
    return cap * D + (cap % 32u == 0u ? (t >> 5) * D * 32u + d * 32u + (t & 31u) : d * cap + t);
}

// Whether 16-byte pieces of 8 dims take k_at and v_at.
__device__ inline bool wide_dim(uint32_t D) { return D % 8u == 0u && D <= kMaxDim32; }

// Entries of one wave's table read: lane i holds entry idx + i; token lane of
// the tile is resolved from the entry that covers it.  Returns whether entry
// idx covers t0 (then the following 63 cover everything the tile can reach).
__device__ inline bool resolve_tile_wave(const PoolView& P, const kimkv_block_desc* desc, uint32_t count, uint32_t idx,
                                         uint32_t t0, uint32_t n, bool need_hit, TokEntry* tab)
{
    uint32_t const lane = threadIdx.x & (kWave - 1);
    uint32_t lo = 0;
    uint32_t hi = 0;
    uint32_t begin = 0;
    uint32_t cap = 0;
    uint64_t page = 0;
    bool hit = false;
    if (lane < n && idx + lane < count) {
        kimkv_block_desc const e = desc[idx + lane];
        begin = e.logical_token_begin;
        hit = begin <= t0 && t0 - begin < e.valid_tokens;
        lo = max(begin, t0);
        hi = min(begin + e.valid_tokens, t0 + n);
        cap = e.page_token_capacity;
        if (lo < hi && e.valid_tokens <= cap) {
            page = reinterpret_cast<uint64_t>(page_base(P, e.kind, e.slot, cap));
        }
    }
    bool const found = (__ballot(hit) & 1u) != 0;
    if (need_hit && !found) return false;
    // readlane returns a signed word: made unsigned before it is widened.
    auto from = [](uint32_t v, int j) { return static_cast<uint32_t>(__builtin_amdgcn_readlane(static_cast<int>(v), j)); };
    auto const page_lo = static_cast<uint32_t>(page);
    auto const page_hi = static_cast<uint32_t>(page >> 32);
    TokEntry mine{nullptr, 0, 0};
    for (uint64_t left = __ballot(page != 0); left != 0; left &= left - 1) {
        int const j = __ffsll(static_cast<unsigned long long>(left)) - 1;
        uint32_t const jlo = from(lo, j);
        uint32_t const jhi = from(hi, j);
        uint64_t const jpage = static_cast<uint64_t>(from(page_lo, j)) | static_cast<uint64_t>(from(page_hi, j)) << 32;
        uint32_t const jcap = from(cap, j);
        uint32_t const jbegin = from(begin, j);
        if (t0 + lane >= jlo && t0 + lane < jhi) {
            mine = TokEntry{reinterpret_cast<uint16_t*>(jpage), jcap, t0 + lane - jbegin};
        }
    }
    if (lane < n) tab[lane] = mine;
    return found;
}

// Resolves tokens [t0, t0+n) (n <= 64) of a table into LDS entries.  Tokens
// not covered by a valid descriptor get page == nullptr.  All threads of the
// block must call it.  The first entry is guessed before it is searched for:
// t0 / 64 when every entry before it is a full extent page, t0 / 8 when they
// are full micro pages; each guess is one wave's single read of the table,
// and a guess counts only if its first entry covers t0.
__device__ void build_tile_table(const PoolView& P, const kimkv_block_desc* desc, uint32_t count,
                                 uint32_t t0, uint32_t n, TokEntry* tab, uint32_t* s_hit)
{
    uint32_t const wave = threadIdx.x >> 6;
    if (threadIdx.x == 0) *s_hit = 0;
    __syncthreads();
    if (wave < 2 && resolve_tile_wave(P, desc, count, t0 / (wave == 0 ? 64u : 8u), t0, n, true, tab)) *s_hit = 1;
    __syncthreads();
    if (*s_hit == 0 && wave == 0) {
        uint32_t const idx = find_descriptor_wave(desc, count, t0);
        static_cast<void>(resolve_tile_wave(P, desc, count, idx, t0, n, false, tab));
    }
    __syncthreads();
}

// ---------------------------------------------------------------------------
// Batched append: one block per (job, layer).
// ---------------------------------------------------------------------------
// Stores the first `count` (<= 8) halves of v at a 16-byte aligned address.
__device__ inline void store_prefix(uint16_t* p, u32x4_t v, uint32_t count)
{
    if (count >= 8) {
        *reinterpret_cast<u32x4_t*>(p) = v;
        return;
    }
    uint32_t at = 0;
    if (count & 4u) {
        *reinterpret_cast<uint2*>(p) = make_uint2(v[0], v[1]);
        at = 4;
    }
    if (count & 2u) {
        *reinterpret_cast<uint32_t*>(p + at) = at == 4 ? v[2] : v[0];
        at += 2;
    }
    if (count & 1u) p[at] = static_cast<uint16_t>(at < 4 ? (at == 2 ? v[1] : v[0]) : (at == 6 ? v[3] : v[2]));
}

struct AppendDivisors {
    Divisor hd;        // H * D
    Divisor hd8;       // H * D / 8
    Divisor d;         // D
    Divisor d8;        // D / 8
};

// Copies tokens [0, n) of a page's blocks of one layer to another page, K in
// pieces of 8 dims and V^T in pieces of 8 tokens of one dim, of which the last
// piece stores only the copied tokens (its page may hold others' bytes past
// them).  A thread loads one piece of each before it stores either: more of
// them in flight costs registers that the long appends of this kernel need
// for waves (batches of four: 107 registers, a prompt's append of 5448 tokens
// x 22 layers 57 us instead of 40).  Element by element the copy was seven
// dependent rounds for a 7-token tail of 4 heads x 64; the append of 64 lanes
// x 22 layers, a quarter of the tails copied, went from 12.6 to 7.7 us.
// Both capacities and D are multiples of 8; src and dst are the layer's
// blocks, of fewer than 2^32 elements each.
__device__ inline void copy_tokens_wide(const AppendDivisors& dv, uint32_t n, const uint16_t* src, uint32_t scap,
                                        uint16_t* dst, uint32_t dcap)
{
    uint32_t const D = dv.d.d;
    uint32_t const kchunks = n * dv.hd8.d;
    uint32_t const vchunks = (n + 7) / 8 * dv.hd.d;
    for (uint32_t i = threadIdx.x; i < max(kchunks, vchunks); i += kBlock) {
        uint32_t rem, c, d;
        uint32_t const t = div_mod(i, dv.hd8, &rem);
        uint32_t const kh = div_mod(rem, dv.d8, &c);
        uint32_t const g = div_mod(i, dv.hd, &rem);
        uint32_t const vh = div_mod(rem, dv.d, &d);
        u32x4_t k, v;
        if (i < kchunks) k = *reinterpret_cast<const u32x4_t*>(src + 2 * scap * D * kh + k_at(scap, D, t, c * 8));
        if (i < vchunks) v = *reinterpret_cast<const u32x4_t*>(src + 2 * scap * D * vh + v_at(scap, D, g * 8, d));
        if (i < kchunks) *reinterpret_cast<u32x4_t*>(dst + 2 * dcap * D * kh + k_at(dcap, D, t, c * 8)) = k;
        if (i < vchunks) store_prefix(dst + 2 * dcap * D * vh + v_at(dcap, D, g * 8, d), v, n - g * 8);
    }
}

// kHuge: the layout has offsets past 32 bits (append_huge), so every copy goes
// element by element at 64-bit offsets.  An instance of its own, as the two
// forms of offsets in one kernel cost the 64-lane append 0.15 us of 15.8.
template <bool kHuge>
__global__ __launch_bounds__(kBlock) void append_kernel(PoolView P, const kimkv_append_job* jobs,
                                                        uint32_t job_count, AppendDivisors dv)
{
    if (blockIdx.x >= job_count) return;
    kimkv_append_job const job = jobs[blockIdx.x];
    uint32_t const li = blockIdx.y;
    if (li >= job.layer_count) return;   // a shorter job of a launch sized for the longest
    uint32_t const layer = job.layer_begin + li;
    uint32_t const H = P.heads;
    uint32_t const D = P.dim;
    uint32_t const dcap = pool_tokens(P, job.dst_kind);
    uint16_t* dst = page_base(P, job.dst_kind, job.dst_slot, dcap);
    if (layer >= P.layers || dst == nullptr || static_cast<uint32_t>(job.dst_token) + job.token_count > dcap
        || job.src_key == nullptr || job.src_value == nullptr) {
        report_fault(P, KIMKV_FAULT_APPEND_JOB);
        return;
    }
    uint32_t const tid = threadIdx.x;

    auto k_el = [](uint32_t cap, uint32_t dim, uint32_t t, uint32_t d) -> uint64_t {
        return kHuge ? k_offset(cap, dim, t, d) : k_at(cap, dim, t, d);
    };
    auto v_el = [](uint32_t cap, uint32_t dim, uint32_t t, uint32_t d) -> uint64_t {
        return kHuge ? v_offset(cap, dim, t, d) : v_at(cap, dim, t, d);
    };

    // The copied positions lie below the written ones: neither waits for the other.
    if (job.cow_tokens != 0) {
        uint32_t const scap = pool_tokens(P, job.cow_kind);
        uint16_t const* src = page_base(P, job.cow_kind, job.cow_slot, scap);
        uint32_t const n = job.cow_tokens;
        if (src != nullptr && n <= scap && n <= dcap && n <= job.dst_token) {
            if (!kHuge && ((D | scap | dcap) & 7u) == 0) {
                copy_tokens_wide(dv, n, src + head_block(P, scap, layer, 0), scap, dst + head_block(P, dcap, layer, 0), dcap);
            } else {
                uint32_t const per_head = n * D;
                for (uint32_t i = tid; i < H * per_head; i += kBlock) {
                    uint32_t const h = i / per_head;
                    uint32_t const rem = i - h * per_head;
                    uint32_t const t = rem / D;
                    uint32_t const d = rem - t * D;
                    uint64_t const sh = head_block(P, scap, layer, h);
                    uint64_t const dh = head_block(P, dcap, layer, h);
                    dst[dh + k_el(dcap, D, t, d)] = src[sh + k_el(scap, D, t, d)];
                    dst[dh + v_el(dcap, D, t, d)] = src[sh + v_el(scap, D, t, d)];
                }
            }
        }
    }

    uint32_t const HD = H * D;
    uint32_t const total = job.token_count * HD;
    uint64_t const layer_off = static_cast<uint64_t>(li) * job.src_layer_stride;
    const uint16_t* sk = job.src_key + layer_off;
    const uint16_t* sv = job.src_value + layer_off;
    uint32_t const stride = job.src_token_stride;
    bool const src_aligned = !kHuge && (D & 7u) == 0 && (stride & 7u) == 0
        && ((reinterpret_cast<uintptr_t>(sk) | reinterpret_cast<uintptr_t>(sv)) & 15u) == 0;
    if (src_aligned) {
        // K: 16-byte pieces of 8 dims of one token (contiguous in source and page).
        uint32_t const kchunks = job.token_count * dv.hd8.d;
        for (uint32_t i = tid; i < kchunks; i += kBlock) {
            uint32_t rem, dc;
            uint32_t const t = div_mod(i, dv.hd8, &rem);
            uint32_t const h = div_mod(rem, dv.d8, &dc);
            u32x4_t const v = *reinterpret_cast<const u32x4_t*>(sk + static_cast<uint64_t>(t) * stride + h * D + dc * 8);
            *reinterpret_cast<u32x4_t*>(dst + head_block(P, dcap, layer, h)
                                        + k_at(dcap, D, job.dst_token + t, dc * 8)) = v;
        }
        // V^T: 16-byte pieces of 8 tokens of one dim when the tokens sit in
        // 8-aligned groups of the page, else one element at a time.
        bool const v_groups = (job.token_count & 7u) == 0 && (job.dst_token & 7u) == 0 && (dcap & 7u) == 0;
        if (v_groups) {
            uint32_t const vchunks = (job.token_count / 8) * HD;
            for (uint32_t i = tid; i < vchunks; i += kBlock) {
                uint32_t r, d;
                uint32_t const g = div_mod(i, dv.hd, &r);
                uint32_t const h = div_mod(r, dv.d, &d);
                const uint16_t* src = sv + static_cast<uint64_t>(8 * g) * stride + r;
                u32x4_t w;
#pragma unroll
                for (uint32_t j = 0; j < 4; ++j) {
                    w[j] = static_cast<uint32_t>(src[static_cast<uint64_t>(2 * j) * stride])
                        | (static_cast<uint32_t>(src[static_cast<uint64_t>(2 * j + 1) * stride]) << 16);
                }
                *reinterpret_cast<u32x4_t*>(dst + head_block(P, dcap, layer, h)
                                            + v_at(dcap, D, job.dst_token + 8 * g, d)) = w;
            }
            return;
        }
        for (uint32_t i = tid; i < total; i += kBlock) {
            uint32_t rem, d;
            uint32_t const t = div_mod(i, dv.hd, &rem);
            uint32_t const h = div_mod(rem, dv.d, &d);
            dst[head_block(P, dcap, layer, h) + v_at(dcap, D, job.dst_token + t, d)] =
                sv[static_cast<uint64_t>(t) * stride + rem];
        }
        return;
    }
    for (uint32_t i = tid; i < total; i += kBlock) {
        uint32_t const t = i / HD;
        uint32_t const rem = i - t * HD;
        uint32_t const h = rem / D;
        uint32_t const d = rem - h * D;
        uint64_t const so = layer_off + static_cast<uint64_t>(t) * job.src_token_stride + rem;
        uint64_t const dh = head_block(P, dcap, layer, h);
        uint32_t const pt = job.dst_token + t;
        dst[dh + k_el(dcap, D, pt, d)] = job.src_key[so];
        dst[dh + v_el(dcap, D, pt, d)] = job.src_value[so];
    }
}

// ---------------------------------------------------------------------------
// Gather: block = (64-token tile, group of layers, block of kRows columns of
// the H * D row); output [L][2][T][H][D].  Fast path (every 8-token group of
// the tile sits 8-aligned in one page, D % 8 == 0): a thread issues all its
// 16-byte non-temporal loads, K and V^T, before any store.  K rows are copied
// straight; V^T is transposed through LDS (16-byte chunks of 8 tokens of one
// dim row in, 16-byte chunks of 8 dims of one token out; the chunk column is
// XOR-swizzled by the token's group so the scattered 2-byte writes of one
// instruction spread over the banks).  A tile of fewer than 64 tokens and a
// last block of fewer columns take it too: loads past the edge repeat the
// last token or column, stores past it are left out (the last group's load
// reads the page's own positions past the tile).  Other tiles take the
// element-wise path.  Bound by HBM when the chip is full (5.6 TB/s read and
// written at 16384 tokens x 22 layers), by the chain of table read, load and
// store when it is not (560..2021 tokens x 22 layers, last tile partial: 10
// and 20 us; 42 us with that tile copied 2 bytes at a time).
// ---------------------------------------------------------------------------
typedef const __attribute__((address_space(1))) u32x4_t global_u32x4_t;
typedef __attribute__((address_space(1))) u32x4_t global_u32x4_out_t;

__device__ inline u32x4_t load16_nt(const uint16_t* p)
{
    return __builtin_nontemporal_load((global_u32x4_t*)(p));
}

__device__ inline void store16_nt(uint16_t* p, u32x4_t v)
{
    __builtin_nontemporal_store(v, (global_u32x4_out_t*)(p));
}

__device__ inline uint32_t stage_col(uint32_t t, uint32_t r)
{
    return (((r >> 3) ^ ((t >> 3) & 3u)) << 3) | (r & 7u);
}

// Columns [r0, r0 + kRows) of one (tile, layer).  n tokens, `cols` valid columns.
template <uint32_t kRows, bool kWhole>
__device__ inline void gather_kv_fast(const PoolView& P, const TokEntry* tab, uint32_t layer, uint32_t r0, uint32_t n,
                                      uint32_t cols, Divisor dim, uint16_t* k_base, uint16_t* v_base, uint16_t* stage)
{
    constexpr uint32_t kStageRow = kRows + 8;                 // u16 per staged token row (16-byte multiple)
    constexpr uint32_t per = kTile * kRows / 8 / kBlock;      // 16-byte chunks per thread, each of K and V
    constexpr uint32_t per_token = kRows / 8;
    uint32_t const tid = threadIdx.x;
    uint32_t const D = P.dim;
    uint32_t const HD = P.heads * D;
    u32x4_t kv[per], vv[per];
#pragma unroll
    for (uint32_t k = 0; k < per; ++k) {
        uint32_t const i = k * kBlock + tid;
        uint32_t t = i / per_token;
        uint32_t c = i % per_token * 8;
        if (!kWhole) {
            t = min(t, n - 1);
            c = min(c, cols - 8);
        }
        uint32_t d;
        uint32_t const h = div_mod(r0 + c, dim, &d);
        TokEntry const e = tab[t];
        kv[k] = load16_nt(e.page + head_block(P, e.cap, layer, h) + k_at(e.cap, D, e.pt, d));
    }
    // Chunk q: four consecutive lanes read one 64-byte dim row of a 32-token V^T panel.
#pragma unroll
    for (uint32_t k = 0; k < per; ++k) {
        uint32_t const q = k * kBlock + tid;
        uint32_t rr = (q >> 2) % kRows;
        uint32_t t = 8 * ((q & 3u) + 4u * ((q >> 2) / kRows));
        if (!kWhole) {
            t = min(t, (n - 1) & ~7u);
            rr = min(rr, cols - 1);
        }
        uint32_t d;
        uint32_t const h = div_mod(r0 + rr, dim, &d);
        TokEntry const e = tab[t];
        vv[k] = load16_nt(e.page + head_block(P, e.cap, layer, h) + v_at(e.cap, D, e.pt, d));
    }
#pragma unroll
    for (uint32_t k = 0; k < per; ++k) {
        uint32_t const i = k * kBlock + tid;
        uint32_t const t = i / per_token;
        uint32_t const c = i % per_token * 8;
        if (kWhole || (t < n && c < cols)) store16_nt(k_base + static_cast<uint64_t>(t) * HD + r0 + c, kv[k]);
    }
#pragma unroll
    for (uint32_t k = 0; k < per; ++k) {
        uint32_t const q = k * kBlock + tid;
        uint32_t const rr = (q >> 2) % kRows;
        uint32_t const g = (q & 3u) + 4u * ((q >> 2) / kRows);
#pragma unroll
        for (uint32_t j = 0; j < 8; ++j) {
            uint32_t const t = 8 * g + j;
            uint32_t const word = vv[k][j >> 1];
            stage[t * kStageRow + stage_col(t, rr)] = static_cast<uint16_t>((j & 1u) ? (word >> 16) : (word & 0xFFFFu));
        }
    }
    __syncthreads();
#pragma unroll
    for (uint32_t k = 0; k < per; ++k) {
        uint32_t const i = k * kBlock + tid;
        uint32_t const t = i / per_token;
        uint32_t const c = i % per_token * 8;
        if (kWhole || (t < n && c < cols)) {
            u32x4_t const w = *reinterpret_cast<const u32x4_t*>(&stage[t * kStageRow + stage_col(t, c)]);
            store16_nt(v_base + static_cast<uint64_t>(t) * HD + r0 + c, w);
        }
    }
    __syncthreads();
}

// The tile's page table is resolved once for all the block's layers and both
// components.
template <uint32_t kRows>
__global__ __launch_bounds__(kBlock) void gather_kernel(PoolView P, const kimkv_block_desc* desc,
                                                        uint32_t count, uint32_t T, uint32_t layers_per_block,
                                                        Divisor dim, uint16_t* out)
{
    __shared__ TokEntry tab[kTile];
    __shared__ uint32_t s_hit;
    __shared__ __align__(16) uint16_t stage[kTile * (kRows + 8)];

    uint32_t const t0 = blockIdx.x * kTile;
    uint32_t const n = min(kTile, T - t0);
    build_tile_table(P, desc, count, t0, n, tab, &s_hit);

    uint32_t const D = P.dim;
    uint32_t const HD = P.heads * D;
    uint32_t const tid = threadIdx.x;
    uint32_t const l0 = blockIdx.y * layers_per_block;
    uint32_t const l1 = min(P.layers, l0 + layers_per_block);
    uint32_t const r0 = blockIdx.z * kRows;
    uint32_t const cols = min(kRows, HD - r0);

    int group_ok = 1;
    if (8 * tid < n) {
        uint32_t const last = min(n, 8 * tid + 8) - 1;
        TokEntry const a = tab[8 * tid];
        TokEntry const b = tab[last];
        group_ok = a.page != nullptr && b.page == a.page && (a.pt & 7u) == 0 && b.pt == a.pt + (last - 8 * tid)
            && (a.cap & 7u) == 0;
    }
    // A tile of fewer than 64 tokens stores its rows two bytes at a time into
    // an output off the 16-byte grid (whole tiles have always required it).
    bool const aligned = n == kTile || (reinterpret_cast<uintptr_t>(out) & 15u) == 0;
    bool const fast = __syncthreads_and(group_ok) && wide_dim(D) && aligned;
    bool const whole = n == kTile && cols == kRows;

    for (uint32_t layer = l0; layer < l1; ++layer) {
        uint16_t* k_base = out + (static_cast<uint64_t>(layer * 2) * T + t0) * HD;
        uint16_t* v_base = out + (static_cast<uint64_t>(layer * 2 + 1) * T + t0) * HD;
        if (fast && whole) {
            gather_kv_fast<kRows, true>(P, tab, layer, r0, n, cols, dim, k_base, v_base, stage);
            continue;
        }
        if (fast) {
            gather_kv_fast<kRows, false>(P, tab, layer, r0, n, cols, dim, k_base, v_base, stage);
            continue;
        }
        // Element-wise path: groups across pages or off the 8-token grid, unmapped tokens, outputs off the
        // 16-byte grid, D % 8 != 0.
        for (uint32_t i = tid; i < n * cols; i += kBlock) {
            uint32_t const t = i / cols;
            uint32_t const r = r0 + i - t * cols;
            TokEntry const e = tab[t];
            if (e.page == nullptr) continue;
            uint32_t d;
            uint32_t const h = div_mod(r, dim, &d);
            uint16_t const* hb = e.page + head_block(P, e.cap, layer, h);
            uint64_t const at = static_cast<uint64_t>(t) * HD + r;
            k_base[at] = hb[k_offset(e.cap, D, e.pt, d)];
            v_base[at] = hb[v_offset(e.cap, D, e.pt, d)];
        }
    }
}

// ---------------------------------------------------------------------------
// Batched promotion: block = (job, layer).  Extent token t <- micro page t/8.
// ---------------------------------------------------------------------------
// One workgroup per patch: the range is copied as 32-bit words (a
// descriptor is 5 words), so a one-entry patch is a single wave's loads.
__global__ __launch_bounds__(kBlock) void patch_descriptors_kernel(const kimkv_descriptor_patch* patches,
                                                                   const kimkv_block_desc* descriptors)
{
    static_assert(sizeof(kimkv_block_desc) == 5 * sizeof(uint32_t), "descriptor is five words");
    kimkv_descriptor_patch const p = patches[blockIdx.x];
    uint32_t const words = p.count * 5u;
    auto const* src = reinterpret_cast<const uint32_t*>(descriptors + p.source);
    auto* dst = reinterpret_cast<uint32_t*>(p.table + p.first);
    for (uint32_t w = threadIdx.x; w < words; w += kBlock) dst[w] = src[w];
}

__global__ __launch_bounds__(kBlock) void promote_kernel(PoolView P, const kimkv_promotion_job* jobs,
                                                         uint32_t job_count)
{
    if (blockIdx.x >= job_count) return;
    kimkv_promotion_job const job = jobs[blockIdx.x];
    uint32_t const layer = blockIdx.y;
    uint32_t const mt = P.micro_tokens;
    uint32_t const et = P.extent_tokens;
    uint16_t* dst = page_base(P, KIMKV_PAGE_EXTENT, job.extent_slot, et);
    uint16_t const* src[8];
    bool ok = mt * 8 == et && layer < P.layers && dst != nullptr;
#pragma unroll
    for (int k = 0; k < 8; ++k) {
        src[k] = page_base(P, KIMKV_PAGE_MICRO, job.micro_slots[k], mt);
        ok = ok && src[k] != nullptr;
    }
    if (!ok) {
        report_fault(P, KIMKV_FAULT_PROMOTION_JOB);
        return;
    }
    uint32_t const H = P.heads;
    uint32_t const D = P.dim;
    uint32_t const tid = threadIdx.x;
    if (wide_dim(D) && mt == 8) {
        uint32_t const dchunks = D / 8;
        // K: (h, t, dc) 16-byte chunks.
        uint32_t const kchunks = H * et * dchunks;
        for (uint32_t i = tid; i < kchunks; i += kBlock) {
            uint32_t const h = i / (et * dchunks);
            uint32_t const rem = i - h * et * dchunks;
            uint32_t const t = rem / dchunks;
            uint32_t const dc = rem - t * dchunks;
            uint4 const v = *reinterpret_cast<uint4 const*>(
                src[t >> 3] + head_block(P, mt, layer, h) + k_at(mt, D, t & 7u, dc * 8));
            *reinterpret_cast<uint4*>(dst + head_block(P, et, layer, h) + k_at(et, D, t, dc * 8)) = v;
        }
        // V^T: (h, d, k) -- micro row d (8 tokens, 16 bytes) -> extent row d at 8k.
        uint32_t const vchunks = H * D * 8;
        for (uint32_t i = tid; i < vchunks; i += kBlock) {
            uint32_t const h = i / (D * 8);
            uint32_t const rem = i - h * D * 8;
            uint32_t const d = rem / 8;
            uint32_t const k = rem & 7u;
            uint4 const v = *reinterpret_cast<uint4 const*>(
                src[k] + head_block(P, mt, layer, h) + v_at(mt, D, 0, d));
            *reinterpret_cast<uint4*>(dst + head_block(P, et, layer, h) + v_at(et, D, 8 * k, d)) = v;
        }
        return;
    }
    uint32_t const total = H * et * D;
    for (uint32_t i = tid; i < total; i += kBlock) {
        uint32_t const h = i / (et * D);
        uint32_t const rem = i - h * et * D;
        uint32_t const t = rem / D;
        uint32_t const d = rem - t * D;
        uint16_t const* s = src[t / mt];
        uint32_t const st = t % mt;
        uint64_t const sh = head_block(P, mt, layer, h);
        uint64_t const dh = head_block(P, et, layer, h);
        dst[dh + k_offset(et, D, t, d)] = s[sh + k_offset(mt, D, st, d)];
        dst[dh + v_offset(et, D, t, d)] = s[sh + v_offset(mt, D, st, d)];
    }
}

// ---------------------------------------------------------------------------
// Synthetic fill of a table's pages: block = (64-token tile, layer, component).
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kBlock) void fill_table_kernel(PoolView P, const kimkv_block_desc* desc,
                                                            uint32_t count, uint32_t token_begin,
                                                            uint32_t token_end, uint64_t seed,
                                                            uint32_t stream_id)
{
    __shared__ TokEntry tab[kTile];
    __shared__ uint32_t s_hit;
    uint32_t const t0 = token_begin + blockIdx.x * kTile;
    uint32_t const n = min(kTile, token_end - t0);
    uint32_t const layer = blockIdx.y;
    uint32_t const comp = blockIdx.z;
    build_tile_table(P, desc, count, t0, n, tab, &s_hit);
    uint32_t const D = P.dim;
    uint32_t const HD = P.heads * D;
    uint32_t const tid = threadIdx.x;

    if (comp == 0) {
        for (uint32_t i = tid; i < n * HD; i += kBlock) {
            uint32_t const t = i / HD;
            uint32_t const r = i - t * HD;
            TokEntry const e = tab[t];
            if (e.page == nullptr) continue;
            uint32_t const h = r / D;
            uint32_t const d = r - h * D;
            e.page[head_block(P, e.cap, layer, h) + k_offset(e.cap, D, e.pt, d)] =
                synth_f16(seed, kv_row(stream_id, layer, 0, t0 + t), r);
        }
        return;
    }
    // V^T: thread per (row, token group of 8) with 16-byte stores when aligned.
    uint32_t const groups = (n + 7) / 8;
    for (uint32_t i = tid; i < HD * groups; i += kBlock) {
        uint32_t const r = i / groups;
        uint32_t const g = i - r * groups;
        uint32_t const h = r / D;
        uint32_t const d = r - h * D;
        uint32_t const tb = g * 8;
        uint32_t const te = min(tb + 8, n);
        TokEntry const e = tab[tb];
        bool const vec = te == tb + 8 && e.page != nullptr && (e.pt & 7u) == 0 && (e.cap & 7u) == 0
            && tab[tb + 7].page == e.page && tab[tb + 7].pt == e.pt + 7;
        if (vec) {
            uint32_t w[4];
#pragma unroll
            for (uint32_t j = 0; j < 4; ++j) {
                uint32_t const lo = synth_f16(seed, kv_row(stream_id, layer, 1, t0 + tb + 2 * j), r);
                uint32_t const hi = synth_f16(seed, kv_row(stream_id, layer, 1, t0 + tb + 2 * j + 1), r);
                w[j] = lo | (hi << 16);
            }
            *reinterpret_cast<uint4*>(e.page + head_block(P, e.cap, layer, h) + v_offset(e.cap, D, e.pt, d)) =
                make_uint4(w[0], w[1], w[2], w[3]);
        } else {
            for (uint32_t t = tb; t < te; ++t) {
                TokEntry const f = tab[t];
                if (f.page == nullptr) continue;
                f.page[head_block(P, f.cap, layer, h) + v_offset(f.cap, D, f.pt, d)] =
                    synth_f16(seed, kv_row(stream_id, layer, 1, t0 + t), r);
            }
        }
    }
}

__global__ __launch_bounds__(kBlock) void fill_rows_kernel(uint16_t* out, uint64_t count, uint64_t seed,
                                                           uint64_t row0, uint32_t cols)
{
    uint64_t const stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < count; i += stride) {
        out[i] = synth_f16(seed, row0 + i / cols, static_cast<uint32_t>(i % cols));
    }
}

// Contiguous K/V block [layers][2][tokens][cols]: the row of (l, c, t) is
// kv_row(stream_id, l, c, token0 + t).
__global__ __launch_bounds__(kBlock) void fill_kv_kernel(uint16_t* out, uint32_t layers, uint32_t tokens,
                                                         uint32_t cols, uint64_t seed, uint32_t stream_id,
                                                         uint32_t token0)
{
    uint64_t const per_block = static_cast<uint64_t>(tokens) * cols;
    uint64_t const count = per_block * 2u * layers;
    uint64_t const stride = static_cast<uint64_t>(gridDim.x) * kBlock;
    for (uint64_t i = static_cast<uint64_t>(blockIdx.x) * kBlock + threadIdx.x; i < count; i += stride) {
        uint64_t const lc = i / per_block;
        uint64_t const r = i - lc * per_block;
        uint32_t const t = static_cast<uint32_t>(r / cols);
        uint32_t const col = static_cast<uint32_t>(r - static_cast<uint64_t>(t) * cols);
        out[i] = synth_f16(seed, kv_row(stream_id, static_cast<uint32_t>(lc >> 1), static_cast<uint32_t>(lc & 1u),
                                        token0 + t),
                           col);
    }
}

}  // namespace
}  // namespace kimkv

using namespace kimkv;

namespace {
// Whether a layer's block of some page (from which the copied tails' offsets
// count) or a head's (k_at, v_at) holds more elements than 32 bits count.
bool append_huge(const PoolView& p)
{
    return ((p.micro_slot_elements | p.extent_slot_elements) >> 32) != 0 || p.dim > kMaxDim32;
}

AppendDivisors append_divisors(const kimkv_storage& s)
{
    uint32_t const D = s.layout.head_dim;
    uint32_t const HD = s.layout.kv_heads * D;
    return AppendDivisors{divisor(HD), divisor(HD / 8), divisor(D), divisor(D / 8)};
}
}  // namespace

extern "C" {

kimkv_status kimkv_append_batch(const kimkv_storage* storage, const kimkv_append_job* device_jobs,
                                uint32_t job_count, uint32_t max_layer_count, kimkv_stream_t stream)
{
    if (storage == nullptr || (job_count != 0 && device_jobs == nullptr)) return KIMKV_INVALID_ARGUMENT;
    if (job_count == 0 || max_layer_count == 0) return KIMKV_OK;
    if (max_layer_count > storage->layout.layers || job_count > 0x7FFFFFFFu) return KIMKV_INVALID_ARGUMENT;
    dim3 const grid(job_count, max_layer_count);
    void* start = nullptr;
    kernel_timing_begin(TimedKernel::Append, native(stream), &start);
    PoolView const pv = pool_view(*storage);
    if (append_huge(pv)) {
        append_kernel<true><<<grid, kBlock, 0, native(stream)>>>(pv, device_jobs, job_count, append_divisors(*storage));
    } else {
        append_kernel<false><<<grid, kBlock, 0, native(stream)>>>(pv, device_jobs, job_count, append_divisors(*storage));
    }
    kimkv_status const status = launch_status();
    kernel_timing_end(TimedKernel::Append, native(stream), start);
    return status;
}

kimkv_status kimkv_gather(const kimkv_storage* storage, const kimkv_block_desc* device_descriptors,
                          uint32_t descriptor_count, uint32_t total_tokens, uint16_t* device_output,
                          kimkv_stream_t stream)
{
    if (storage == nullptr || device_descriptors == nullptr || device_output == nullptr
        || descriptor_count == 0 || total_tokens == 0) {
        return KIMKV_INVALID_ARGUMENT;
    }
    uint32_t const tiles = ceil_div(total_tokens, kTile);
    uint32_t const L = storage->layout.layers;
    uint32_t const HD = storage->layout.kv_heads * storage->layout.head_dim;
    Divisor const dim = divisor(storage->layout.head_dim);
    auto launch = [&](auto rows) {
        constexpr uint32_t kRows = decltype(rows)::value;
        uint32_t const columns = ceil_div(HD, kRows);
        // Enough workgroups to fill the chip (~8 per CU) with as few table
        // resolutions as possible: layers are grouped per workgroup.
        uint32_t per = 1;
        while (per < L && static_cast<uint64_t>(tiles) * columns * ceil_div(L, per * 2) >= 2048) per *= 2;
        dim3 const grid(tiles, ceil_div(L, per), columns);
        gather_kernel<kRows><<<grid, kBlock, 0, native(stream)>>>(pool_view(*storage), device_descriptors,
                                                                  descriptor_count, total_tokens, per, dim,
                                                                  device_output);
    };
    // 256 columns a block where that fills the chip twice over (16384 tokens x
    // 22 layers: 128 us, 135 us with 128 columns), narrower blocks where it
    // does not: more of them share the work (560 tokens x 22 layers: 8.4 us).
    if (HD > 128 && static_cast<uint64_t>(tiles) * L * ceil_div(HD, 256) >= 512) {
        launch(std::integral_constant<uint32_t, 256>{});
    } else {
        launch(std::integral_constant<uint32_t, 128>{});
    }
    return launch_status();
}

kimkv_status kimkv_promote_batch(const kimkv_storage* storage, const kimkv_promotion_job* device_jobs,
                                 uint32_t job_count, kimkv_stream_t stream)
{
    if (storage == nullptr || (job_count != 0 && device_jobs == nullptr)) return KIMKV_INVALID_ARGUMENT;
    if (job_count == 0) return KIMKV_OK;
    if (static_cast<uint32_t>(storage->micro_tokens) * 8 != storage->extent_tokens) return KIMKV_INVALID_ARGUMENT;
    dim3 const grid(job_count, storage->layout.layers);
    promote_kernel<<<grid, kBlock, 0, native(stream)>>>(pool_view(*storage), device_jobs, job_count);
    return launch_status();
}

kimkv_status kimkv_patch_descriptors(const kimkv_descriptor_patch* patches, uint32_t patch_count,
                                     const kimkv_block_desc* descriptors, kimkv_stream_t stream)
{
    if (patch_count == 0) return KIMKV_OK;
    if (patches == nullptr || descriptors == nullptr) return KIMKV_INVALID_ARGUMENT;
    patch_descriptors_kernel<<<patch_count, kBlock, 0, native(stream)>>>(patches, descriptors);
    return launch_status();
}

kimkv_status kimkv_fill_table(const kimkv_storage* storage, const kimkv_block_desc* device_descriptors,
                              uint32_t descriptor_count, uint32_t token_begin, uint32_t token_end,
                              uint64_t seed, uint32_t stream_id, kimkv_stream_t stream)
{
    if (storage == nullptr || device_descriptors == nullptr || descriptor_count == 0 || token_end < token_begin) {
        return KIMKV_INVALID_ARGUMENT;
    }
    if (token_end == token_begin) return KIMKV_OK;
    dim3 const grid(ceil_div(token_end - token_begin, kTile), storage->layout.layers, 2);
    fill_table_kernel<<<grid, kBlock, 0, native(stream)>>>(pool_view(*storage), device_descriptors,
                                                           descriptor_count, token_begin, token_end, seed,
                                                           stream_id);
    return launch_status();
}

kimkv_status kimkv_fill_rows(uint16_t* device_out, uint64_t count, uint64_t seed, uint64_t row0,
                             uint32_t cols, kimkv_stream_t stream)
{
    if (device_out == nullptr || cols == 0) return KIMKV_INVALID_ARGUMENT;
    if (count == 0) return KIMKV_OK;
    uint64_t const blocks64 = (count + kBlock - 1) / kBlock;
    unsigned const blocks = static_cast<unsigned>(blocks64 < 65536 ? blocks64 : 65536);
    fill_rows_kernel<<<blocks, kBlock, 0, native(stream)>>>(device_out, count, seed, row0, cols);
    return launch_status();
}

kimkv_status kimkv_fill_kv(uint16_t* device_out, uint32_t layers, uint32_t tokens, uint32_t cols, uint64_t seed,
                           uint32_t stream_id, uint32_t token0, kimkv_stream_t stream)
{
    if (device_out == nullptr || cols == 0 || static_cast<uint64_t>(token0) + tokens > (1ull << 32)) {
        return KIMKV_INVALID_ARGUMENT;
    }
    uint64_t const count = static_cast<uint64_t>(layers) * 2u * tokens * cols;
    if (count == 0) return KIMKV_OK;
    uint64_t const blocks64 = (count + kBlock - 1) / kBlock;
    unsigned const blocks = static_cast<unsigned>(blocks64 < 65536 ? blocks64 : 65536);
    fill_kv_kernel<<<blocks, kBlock, 0, native(stream)>>>(device_out, layers, tokens, cols, seed, stream_id, token0);
    return launch_status();
}

}  // extern "C"
