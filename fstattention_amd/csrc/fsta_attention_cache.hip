// Tree attention behind a shared prefix (the KV cache of a decoding step) for gfx950: bf16 / fp16 queries, K and V in
// the same type or as 8-bit floats, head_dim 64 / 128.
//
// A workgroup owns 32 query rows of one (batch, head) slice and a run of keys: prefix tiles of 32 keys first (they need
// no metadata, so the first requests leave with the first instructions), then the block's ancestor tiles and the rows'
// own keys (reference fstattention.py:61-136 in another order; the tree part belongs to the last run).  Its eight waves
// deal the tiles out among themselves, each with a ring of its own in LDS that only it fills and reads: no barrier between
// the first tile and the last, a wave waits for nothing but its own transfers.  A tile stays in LDS only until its
// fragments are in registers, one tile ahead of their use, so that the ring is nearly always on its way to memory.  Each
// wave keeps a running softmax of its own; the waves' results are joined in LDS at the end.  Several runs (few slices in
// front of a long prefix) write normalised float32 parts that a second launch joins.
//
// 32x32x16 products in transposed form (lane = 32*h + i): A holds row i, k = 8h .. 8h+7; B holds k = 8h .. 8h+7 of
// column i; C register r holds row 8*(r/4) + 4h + r%4 of column i.  S^T = K.Q^T: the column is the query, a lane has 16
// of a tile's 32 keys for one query, and registers 8kk .. 8kk+7 are its k-slots of O^T += V^T.P^T over keys 16kk ..
// 16kk+15, in the order {4h .. 4h+3, 8+4h .. 8+4h+3}, which the transposing reads of V follow.
#include <type_traits>

#include "fsta_mfma_common.h"

namespace fsta {
namespace {

using namespace mfma;

constexpr int kRows = 32;      // query rows per workgroup

// LDS of one half (K or V) of a ring slot
template <int D, bool KV8> constexpr int half_bytes() { return kTileN * D * (KV8 ? 1 : 2); }
// The rings take 128 (head_dim 128) or 64 KB of the CU's 160: one workgroup per CU, or two.
template <int D> constexpr int ring_bytes_per_wave() { return D == 128 ? 16384 : 8192; }
template <int D, bool KV8> constexpr int ring_slots() { return ring_bytes_per_wave<D>() / (2 * half_bytes<D, KV8>()); }
// (the waves' float32 results, joined at the end where the rings were, are exactly as large)
template <int D, int NW> constexpr int front_bytes() { return NW * ring_bytes_per_wave<D>(); }
static_assert(ring_bytes_per_wave<128>() == 32 * 128 * 4 && ring_bytes_per_wave<64>() == 32 * 64 * 4, "rings and results share LDS");

template <int D, int NW> size_t cache_lds_bytes(int max_anc) {
    return (size_t)front_bytes<D, NW>() + (size_t)kRows * D * 2 + (size_t)NW * 2 * kRows * 4 + (size_t)plan_layout(kRows, max_anc).block_words * 4;
}

// 16-byte chunk positions of an 8-bit V row for the transposing read: one instruction touches keys {4h .. 4h+3,
// 8+4h .. +3} x 32 bytes per half-wave; the XOR spreads these eight rows over all banks.
template <int D> __device__ __forceinline__ int v8_chunk(int row, int c) {
    const int f = D == 128 ? ((row >> 1) & 1) | (((row >> 3) & 1) << 1) : (row >> 3) & 1;
    return c ^ (f << 1);
}

struct CacheGrid {
    int32_t total, per_xcd;      // workgroups, and how many of them an XCD takes
    int32_t chunks, runs;        // groups of 32 query rows, runs of prefix tiles
    int32_t run_tiles;           // prefix tiles per run
    uint32_t chunks_inv, runs_inv;   // ceil(2^32 / chunks), ceil(2^32 / runs): quotients by one multiplication (0 for a divisor of 1)
    int32_t block_shift;         // log2 of the caller's block size
};

// ONCE: the keys of a run are read by one workgroup only (non-temporal transfers)
template <bool BF16, int D, bool KV8, int NW, bool SPLIT, bool ONCE>
__global__ __launch_bounds__(NW * 64, 2) void attn_cache_kernel(AttnParams p, CacheGrid gr) {
    using MM = Mma<BF16>;
    using T = typename MM::elem;
    using Frag = typename MM::frag;
    constexpr int kWaves = NW;
    constexpr int kRowBytes = KV8 ? D : 2 * D;          // a K/V row in memory
    constexpr int kCpr = kRowBytes / 16;                // 16-byte chunks per K/V row
    constexpr int kHalf = half_bytes<D, KV8>();
    constexpr int kDma = kHalf / 1024;                  // transfers per half tile
    constexpr int kRowsPerDma = kTileN / kDma;
    constexpr int kSlots = ring_slots<D, KV8>();
    constexpr int kAux = ONCE ? 2 : 0;
    constexpr int kSteps = D / 16;                      // products per S^T tile
    constexpr int kDTiles = D / 32;                     // 32-row tiles of O^T
    constexpr int kQChunks = D / 8;                     // 16-byte chunks per Q row
    constexpr int kQDma = kRows * D * 2 / 1024;
    constexpr float kTrustedSum = BF16 ? 16777216.f : 32768.f;

    extern __shared__ __attribute__((aligned(16))) unsigned char smem[];
    unsigned char* q_s = smem + front_bytes<D, NW>();
    float* ml_s = reinterpret_cast<float*>(q_s + kRows * D * 2);         // [wave][m of 32 rows | l of 32 rows]
    uint32_t* plan_s = reinterpret_cast<uint32_t*>(ml_s + kWaves * 2 * kRows);
    const int anc_cap = anc_tile_capacity(p.max_anc);
    const int common_words = kPlanHeaderWords + anc_cap * kTileN;
    const int group_words = kTileN * (1 + anc_cap);

    // all kernel arguments by one batch of scalar loads (see the tree kernel)
    asm volatile("" ::"s"(p.q), "s"(p.k), "s"(p.v), "s"(p.o), "s"(p.lse), "s"(p.plan), "s"(p.key_shift), "s"(p.nq), "s"(p.nk),
                 "s"(p.prefix), "s"(p.max_anc), "s"(p.heads_total), "s"(p.out_f32), "s"(p.scale_log2e),
                 "s"(p.part_o), "s"(p.part_lse), "s"(gr.total), "s"(gr.per_xcd), "s"(gr.chunks), "s"(gr.runs), "s"(gr.run_tiles), "s"(gr.chunks_inv), "s"(gr.runs_inv), "s"(gr.block_shift));

    // Workgroup -> (slice, run, row chunk): workgroups go to the XCDs round-robin, and each XCD gets a contiguous piece of
    // the list in which the chunks of a run of a slice stand next to each other: they read the same keys at the same time
    // and find them in their XCD's L2.  (Pieces of the list, not whole slices: no XCD is left with less work.)
    const uint32_t work = (blockIdx.x % kXcds) * (uint32_t)gr.per_xcd + blockIdx.x / kXcds;
    if (work >= (uint32_t)gr.total) return;
    const uint32_t rest = gr.chunks_inv ? __umulhi(work, gr.chunks_inv) : work;
    const int chunk = (int)(work - rest * (uint32_t)gr.chunks);
    const int hz = (int)(gr.runs_inv ? __umulhi(rest, gr.runs_inv) : rest);
    const int run = (int)(rest - (uint32_t)hz * (uint32_t)gr.runs);
    const int row_base = chunk * kRows;

    const int tid = threadIdx.x;
    const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
    const int lane = tid & 63;
    const int ql = lane & 31, h = lane >> 5;

    const char* kb = static_cast<const char*>(p.k) + (size_t)hz * p.nk * kRowBytes;
    const char* vb = static_cast<const char*>(p.v) + (size_t)hz * p.nk * kRowBytes;
    const bool tree = run == gr.runs - 1;
    const int first_tile = run * gr.run_tiles;
    const int all_tiles = (p.prefix + kTileN - 1) / kTileN;
    const int n_pfx = min(gr.run_tiles, all_tiles - first_tile);     // prefix tiles of this run

    // ---- metadata and Q rows first, then this wave's first prefix tiles --------------------------------------------
    const int block = row_base >> gr.block_shift;
    const int group = (row_base >> 5) & ((1 << (gr.block_shift - 5)) - 1);           // of 32 rows in the block
    uint32_t* const group_s = plan_s + common_words;
    if (tree) {
        const char* rec = reinterpret_cast<const char*>(p.plan) +
                          (size_t)block * (size_t)(common_words + (group_words << (gr.block_shift - 5))) * 4;
        const int common_chunks = common_words / 4;
        const int chunks = common_chunks + group_words / 4;
        const uint32_t group_skip = (uint32_t)(group * group_words * 4);
        for (int piece = wave; piece * 64 < chunks; piece += kWaves) {
            const int c = piece * 64 + lane;
            if (c < chunks)
                __builtin_amdgcn_global_load_lds(
                    (const void __attribute__((address_space(1)))*)(rec + (size_t)((uint32_t)c * 16u + (c >= common_chunks ? group_skip : 0u))),
                    (void __attribute__((address_space(3)))*)(reinterpret_cast<char*>(plan_s) + piece * 1024), 16, 0, 0);
        }
    }
    {
        constexpr int kQRowsPerDma = 64 / kQChunks;
        const char* qb = static_cast<const char*>(p.q) + (size_t)hz * p.nq * (D * 2);
        for (int i = wave; i < kQDma; i += kWaves) {
            const int r = i * kQRowsPerDma + lane / kQChunks;
            const uint32_t off = (uint32_t)min(row_base + r, p.nq - 1) * (uint32_t)(D * 2) + (uint32_t)k_chunk<D>(r, lane % kQChunks) * 16u;
            __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)(qb + (size_t)off),
                                             (void __attribute__((address_space(3)))*)(q_s + i * 1024), 16, 0, 0);
        }
    }

    // ---- this wave's ring: slot = [K half | V half]; transfer i of a half moves kRowsPerDma rows, lane l landing in row
    // l / kCpr, chunk slot l % kCpr of them, and fetching the chunk the swizzle puts there
    unsigned char* ring = smem + wave * kSlots * 2 * kHalf;
    const int dma_row = lane / kCpr, dma_slot = lane % kCpr;
    auto k_swz = [](int row, int c) { return KV8 ? k_chunk<D / 2>(row, c) : k_chunk<D>(row, c); };
    auto v_swz = [](int row, int c) { return KV8 ? v8_chunk<D>(row, c) : v_chunk<D>(row, c); };
    uint32_t k_off[kDma], v_off[kDma];       // row and chunk of this lane's piece, in bytes from the transfer's first row
#pragma unroll
    for (int i = 0; i < kDma; ++i) {
        const int r = (i * kRowsPerDma) % 16 + dma_row;      // (the swizzles repeat after 16 rows at most)
        k_off[i] = (uint32_t)dma_row * kRowBytes + (uint32_t)k_swz(r, dma_slot) * 16u;
        v_off[i] = (uint32_t)dma_row * kRowBytes + (uint32_t)v_swz(r, dma_slot) * 16u;
    }
    constexpr int kRawBuffer = 0x00020000;   // descriptor word 3: raw 32-bit data
    const int slice_bytes = (int)((uint32_t)p.nk * (uint32_t)kRowBytes);
    const __amdgpu_buffer_rsrc_t k_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(kb), 0, slice_bytes, kRawBuffer);
    const __amdgpu_buffer_rsrc_t v_rsrc = __builtin_amdgcn_make_buffer_rsrc(const_cast<char*>(vb), 0, slice_bytes, kRawBuffer);
    // Row groups that walk a run in step ask for the same keys at the same time: 256 workgroups of eight groups have 4 MB of
    // distinct bytes on their way, which at 2 us to HBM and back is 2.1 TB/s (a probe with nothing but such transfers; pairs:
    // 5.5).  So every other group takes the rounds of a run (a tile per wave) two by two in the other order: twice the bytes on
    // their way, and what one group fetched from memory its neighbour finds in L2 a round later.  Measured with K and V in HBM,
    // as a step through a model's layers finds them (32 slices, bf16, D 128): 256 rows behind 600, 1100, 6000 keys 12.0 ->
    // 10.3, 16.3 -> 14.6, 54.0 -> 51.7 us, 130 rows, 1100 keys 16.0 -> 14.4; 1506 launches of 8-32 slices behind 64-4096 keys:
    // 0.90-1.00 of the time in every class of slices and bytes, the smallest (8 slices, under 2.5 MB) 0.98-0.99.  With K and V
    // in the Infinity Cache, where the way is short, 0.96-1.02, 1.02-1.05 above 15 MB at D 64: no line in the bytes would win
    // more than it gives.  Two to four groups have enough on their way (128 rows, 2000 keys: 4 % slower, 61 rows: 7 %); whole
    // runs or four rounds in other orders bring more at once and overfill the L2; 8-bit tiles are half as large and their
    // arithmetic is longer than the way (no gain).
    const bool swapped = !KV8 && gr.chunks >= 5 && (chunk & 1);
    const int pairs_end = n_pfx / (2 * kWaves) * (2 * kWaves);
    auto prefix_tile = [&](int t) { return first_tile + (swapped && t < pairs_end ? t ^ kWaves : t); };
    int n_anc_tiles = 0;                     // the list is [prefix tiles | ancestor tiles | the rows' own keys]
    auto issue = [&](int t, int slot) {
        unsigned char* dst = ring + slot * 2 * kHalf;
        const int pt = prefix_tile(t);
        if (t < n_pfx && (pt + 1) * kTileN <= p.prefix) {
            // 32 consecutive rows: one uniform offset, lane offsets that never change.  Buffer addressing takes both as they
            // are (a flat address is 64-bit vector arithmetic per transfer: 8192 keys in 8 bits 35.3 us, 33.9 this way).
            const uint32_t tile_off = (uint32_t)pt * (uint32_t)kHalf;
#pragma unroll
            for (int i = 0; i < 2 * kDma; ++i)
                __builtin_amdgcn_raw_ptr_buffer_load_lds(i < kDma ? k_rsrc : v_rsrc, (void __attribute__((address_space(3)))*)(dst + i * 1024), 16,
                                                         (int)(i < kDma ? k_off[i % kDma] : v_off[i % kDma]), (int)(tile_off + (i % kDma) * 1024), 0, kAux);
        } else {
            // the partial tile at the end of the prefix, ancestor tiles, then the tile of the rows' own keys
            int rows[kDma];
            if (t < n_pfx) {
#pragma unroll
                for (int i = 0; i < kDma; ++i) rows[i] = min(pt * kTileN + i * kRowsPerDma + dma_row, p.prefix - 1);
            } else {
                const int ta = t - n_pfx;
                const uint32_t keys = lds_addr(ta < n_anc_tiles ? plan_s + kPlanHeaderWords + ta * kTileN : group_s) + dma_row * 4;
                uint32_t key[kDma];          // (all requested at once: one LDS round trip)
#pragma unroll
                for (int i = 0; i < kDma; ++i) key[i] = lds_read_b32(keys + i * kRowsPerDma * 4);
                lds_wait();
#pragma unroll
                for (int i = 0; i < kDma; ++i) {
                    lds_tie(key[i]);
                    rows[i] = min((int)key[i] + p.key_shift, p.nk - 1);
                }
            }
#pragma unroll
            for (int i = 0; i < 2 * kDma; ++i) {
                const uint32_t off = (uint32_t)(rows[i % kDma] - dma_row) * (uint32_t)kRowBytes + (i < kDma ? k_off[i % kDma] : v_off[i % kDma]);
                __builtin_amdgcn_global_load_lds((const void __attribute__((address_space(1)))*)((i < kDma ? kb : vb) + (size_t)off),
                                                 (void __attribute__((address_space(3)))*)(dst + i * 1024), 16, 0, 0);
            }
        }
    };
    // tiles of this wave that may stay outstanding
    auto wait_tiles = [&](int tiles) {
        switch (tiles) {
            case 0: wait_vmcnt<0>(); break;
            case 1: wait_vmcnt<2 * kDma>(); break;
            default: wait_vmcnt<4 * kDma>(); break;
        }
    };
    // (Tiles are dealt out in turn, not as the waves ask for them: the sums would be formed in another order in every launch.)
    static_assert(kSlots <= 2, "at most two tiles of a wave are outstanding");
    int issued = 0;                          // tiles of this wave that have been requested
#pragma unroll
    for (int i = 0; i < kSlots; ++i)
        if (wave + i * kWaves < n_pfx) {
            issue(wave + i * kWaves, i);
            ++issued;
        }
    wait_tiles(issued);                      // plan and Q have landed
    ring_barrier();                          // .. for every wave

    uint32_t leaf_word = 0u;                 // this row's own key, if it has one
    if (tree) {
        uint32_t head = lds_read_b32(lds_addr(plan_s));
        uint32_t valid = lds_read_b32(lds_addr(plan_s + kPlanLeafValid + group));
        lds_wait();
        lds_tie(head);
        lds_tie(valid);
        const int n_anc = min(max(__builtin_amdgcn_readfirstlane((int)head), 0), p.max_anc);
        n_anc_tiles = (n_anc + kTileN - 1) / kTileN;
        leaf_word = valid & (1u << ql);
    }
    const int total = n_pfx + (tree ? n_anc_tiles + 1 : 0);
    const bool own_here = tree && (total - 1) % kWaves == wave;      // the rows' own keys are this wave's last tile
    const int mine = wave < total ? (total - wave + kWaves - 1) / kWaves : 0;      // tiles wave, wave + 8, ...
    const int mine_shared = mine - (own_here ? 1 : 0);      // those whose keys the rows share
#pragma unroll
    for (int i = 0; i < kSlots; ++i)
        if (i >= issued && i < mine) issue(wave + i * kWaves, i);
    issued = min(mine, kSlots);
    Frag qf[kSteps];
    {
        u32x4 raw[kSteps];
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            // k-slots of product s: head dims 16s + 8h .. +7; with 8-bit K, whose rows are read 16 bytes (two products) at
            // a time, 32(s/2) + 16h + 8(s%2) .. +7
            const int c = KV8 ? 4 * (s / 2) + 2 * h + (s & 1) : 2 * s + h;
            raw[s] = lds_read_b128(lds_addr(q_s + ql * D * 2 + k_chunk<D>(ql, c) * 16));
        }
        lds_wait();
#pragma unroll
        for (int s = 0; s < kSteps; ++s) {
            lds_tie(raw[s]);
            qf[s] = __builtin_bit_cast(Frag, raw[s]);
        }
    }

    float m_i = -INFINITY, l_i = 0.f;
    f32x16 o[kDTiles];
#pragma unroll
    for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
        for (int r = 0; r < 16; ++r) o[dt][r] = 0.f;
    float sc = p.scale_log2e;
    if (KV8 && p.k_scale) sc *= p.k_scale[hz];

    // ---- fragments: K as read row by row (16-bit: one product each, 8-bit: two), V through the transposing reads.  Lane
    // offsets; product s / head-dim tile dt enter by XOR, rows further down by an immediate.
    const uint32_t k_lane0 = (uint32_t)(ql * kRowBytes + k_swz(ql, h) * 16);
    uint32_t v_lane0;
    if constexpr (KV8) {
        const int jr = (lane & 15) >> 1;
        const int row = jr < 4 ? 4 * h + jr : 8 + 4 * h + jr - 4;
        v_lane0 = (uint32_t)(row * kRowBytes + v8_chunk<D>(row, (lane >> 4) & 1) * 16 + 8 * (lane & 1));
    } else {
        const int row = 4 * h + ((lane & 15) >> 2), col = 16 * ((lane >> 4) & 1) + 4 * (lane & 3);
        v_lane0 = (uint32_t)(row * kRowBytes + v_chunk<D>(row, col >> 3) * 16 + (col & 7) * 2);
    }
    constexpr int kKReads = KV8 ? kSteps / 2 : kSteps;
    constexpr int kVRegs = KV8 ? 1 : 2;      // transposing reads per V fragment
    u32x4 kf[kKReads];
    u32x2 vf[2][kDTiles][kVRegs];
    auto read_k = [&](int slot) {
        const uint32_t a = lds_addr(ring + slot * 2 * kHalf) + k_lane0;
#pragma unroll
        for (int u = 0; u < kKReads; ++u) kf[u] = lds_read_b128(a ^ (uint32_t)(u << 5));
    };
    auto read_v = [&](int slot) {
        const uint32_t a = lds_addr(ring + slot * 2 * kHalf) + kHalf + v_lane0;
#pragma unroll
        for (int dt = 0; dt < kDTiles; ++dt) {
            if constexpr (KV8) {
                const uint32_t ad = a ^ (uint32_t)(dt << 5);
                asm volatile("ds_read_b64_tr_b8 %0, %1" : "=v"(vf[0][dt][0]) : "v"(ad) : "memory");
                asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(vf[1][dt][0]) : "v"(ad), "n"(16 * kRowBytes) : "memory");
            } else {
                const uint32_t ad = a ^ (uint32_t)(dt << 6);
                vf[0][dt][0] = __builtin_bit_cast(u32x2, lds_read_tr16(ad));
                vf[0][dt][kVRegs - 1] = __builtin_bit_cast(u32x2, lds_read_tr16_at<8 * kRowBytes>(ad));
                vf[1][dt][0] = __builtin_bit_cast(u32x2, lds_read_tr16_at<16 * kRowBytes>(ad));
                vf[1][dt][kVRegs - 1] = __builtin_bit_cast(u32x2, lds_read_tr16_at<24 * kRowBytes>(ad));
            }
        }
    };
    auto tie_all = [&]() {
        lds_wait();
#pragma unroll
        for (int u = 0; u < kKReads; ++u) lds_tie(kf[u]);
#pragma unroll
        for (int kk = 0; kk < 2; ++kk)
#pragma unroll
            for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
                for (int w = 0; w < kVRegs; ++w) lds_tie(vf[kk][dt][w]);
    };
    auto widen = [](uint32_t lo, uint32_t hi) -> Frag {      // eight 8-bit floats -> eight values of the 16-bit type, exactly
        u32x4 w;
        if constexpr (BF16) {
            w[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, false));
            w[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 1.0f, true));
            w[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, false));
            w[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 1.0f, true));
        } else {
            w[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, false));
            w[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, true));
            w[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, false));
            w[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, true));
        }
        return __builtin_bit_cast(Frag, w);
    };
    auto v_frag = [&](int kk, int dt) -> Frag {
        const uint32_t a = vf[kk][dt][0][0], b = vf[kk][dt][0][1];
        if constexpr (KV8) {
            return widen(a, b);
        } else {
            const uint32_t c = vf[kk][dt][kVRegs - 1][0], d = vf[kk][dt][kVRegs - 1][1];
            const u32x4 w = {a, b, c, d};
            return __builtin_bit_cast(Frag, w);
        }
    };

    // One tile ahead: at the top of iteration i the fragments of tile i are in registers, tiles behind it are on their way.
    // (The rows' own keys come behind the loop, K fragments read as any tile's, V from the ring as it is needed there.)
    if (mine > 0) {
        wait_tiles(issued - 1);
        read_k(0);
        if (mine_shared > 0) read_v(0);
        tie_all();
        if (mine > kSlots) issue(wave + kSlots * kWaves, 0);
    }
    auto scores = [&]() {                    // S^T = K_tile . Q^T of the tile whose fragments are in registers
        f32x16 s;
#pragma unroll
        for (int r = 0; r < 16; ++r) s[r] = 0.f;
#pragma unroll
        for (int u = 0; u < kKReads; ++u) {
            if constexpr (KV8) {
                const uint32_t r0 = kf[u][0], r1 = kf[u][1], r2 = kf[u][2], r3 = kf[u][3];
                s = MM::mfma(widen(r0, r1), qf[2 * u], s);
                s = MM::mfma(widen(r2, r3), qf[2 * u + 1], s);
            } else {
                s = MM::mfma(__builtin_bit_cast(Frag, kf[u]), qf[u], s);
            }
        }
        return s;
    };
    int slot = 0;                            // ring slot of tile i
    for (int i = 0; i < mine_shared; ++i) {
        const int t = wave + i * kWaves;
        const int next_slot = slot + 1 == kSlots ? 0 : slot + 1;

        f32x16 s = scores();
        // mask: none for whole prefix tiles (uniform branch)
        uint32_t word = 0xffffffffu;
        const int pt = prefix_tile(t);
        if (t >= n_pfx || (pt + 1) * kTileN > p.prefix) {
            if (t < n_pfx) word = (1u << (p.prefix - pt * kTileN)) - 1u;
            else word = group_s[kTileN + (t - n_pfx) * kTileN + ql];
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                const uint32_t keep = (uint32_t)__builtin_amdgcn_sbfe((int)(word >> (4 * h)), 8 * (r / 4) + r % 4, 1);
                const float score = s[r];
                const uint32_t bits = __builtin_bit_cast(uint32_t, score);
                s[r] = __builtin_bit_cast(float, (bits & keep) | (0xff800000u & ~keep));
            }
        }
        // weights against the running maximum as it stands; the full update only where a row has none yet or a weight
        // gets large (exact: a power of two on a row's weights cancels in O / l)
        float pw[16], rowsum;
        auto weights = [&]() {
            const float neg_m = m_i == -INFINITY ? 0.f : -m_i;
            float part[2] = {0.f, 0.f};
#pragma unroll
            for (int r = 0; r < 16; ++r) {
                pw[r] = __builtin_amdgcn_exp2f(__builtin_fmaf(s[r], sc, neg_m));
                part[r & 1] += pw[r];
            }
            rowsum = part[0] + part[1];
        };
        const bool first = i == 0;
        bool redo = first;
        if (!first) {
            weights();
            redo = __ballot(!(rowsum <= kTrustedSum) || (m_i == -INFINITY && word != 0u)) != 0ull;
        }
        if (redo) {
            float mx_raw = s[0];
#pragma unroll
            for (int r = 1; r < 16; ++r) mx_raw = fmaxf(mx_raw, s[r]);
            float a, b;
            swap_halves(mx_raw, false, a, b);
            const float mx = fmaxf(a, b) * sc;      // the scale is positive here
            const bool raise = mx > m_i + kRescaleSlack || (m_i == -INFINITY && mx > -INFINITY);
            const float alpha = raise ? __builtin_amdgcn_exp2f(m_i - mx) : 1.f;   // exp2(-inf) = 0
            if (raise) m_i = mx;
            if (!first) {
                l_i *= alpha;
#pragma unroll
                for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
                    for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
            }
            weights();
        }
        l_i += rowsum;

        // the next tile has landed (with one slot: its K half; V is waited for below)
        if constexpr (kSlots == 1) wait_vmcnt<kDma>();
        else wait_tiles(min(kSlots - 1, max(mine - 2 - i, 0)));
        // O^T += V_tile^T . P^T.  The K fragments of the next tile are requested in front of the products, its V fragments
        // behind them, and the second half of the weights is packed while the matrix pipeline works on the first.
        read_k(next_slot);
        Frag ph[2], pl[2];
        auto pack = [&](int kk) {
            u32x4 hi4, lo4;
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const float a = pw[8 * kk + 2 * e], b = pw[8 * kk + 2 * e + 1];
                const uint32_t hi = MM::pack(a, b);
                hi4[e] = hi;
                if (SPLIT) lo4[e] = MM::pack(a - MM::low(hi), b - MM::high(hi));
            }
            ph[kk] = __builtin_bit_cast(Frag, hi4);
            if (SPLIT) pl[kk] = __builtin_bit_cast(Frag, lo4);
        };
        auto products = [&](int kk) {
            Frag f[kDTiles];
#pragma unroll
            for (int dt = 0; dt < kDTiles; ++dt) {
                f[dt] = v_frag(kk, dt);
                o[dt] = MM::mfma(f[dt], ph[kk], o[dt]);
            }
            if (SPLIT) {
#pragma unroll
                for (int dt = 0; dt < kDTiles; ++dt) o[dt] = MM::mfma(f[dt], pl[kk], o[dt]);
            }
        };
        pack(0);
        products(0);
        pack(1);
        products(1);
        if (kSlots == 1) wait_vmcnt<0>();
        if (i + 1 < mine_shared) read_v(next_slot);
        tie_all();
        if (i + 1 + kSlots < mine) issue(t + (1 + kSlots) * kWaves, next_slot);
        slot = next_slot;
    }

    if (own_here) {
        // The rows' own keys: one score and the V row of that query alone, by the vector ALU.  As products under 31 zero
        // weights an infinity or a NaN in one row's V would reach the whole group (reference fstattention.py:104-107 takes
        // the row's own V by itself, too).
        typedef typename std::conditional<KV8, uint32_t, u32x2>::type Raw;
        Raw raw[kDTiles][4];                 // head dims 32 dt + 8 q4 + 4 h .. +3
        const uint32_t v_row = lds_addr(ring + slot * 2 * kHalf) + kHalf + (uint32_t)(ql * kRowBytes);
#pragma unroll
        for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                if constexpr (KV8) raw[dt][q4] = lds_read_b32(v_row + (uint32_t)(v_swz(ql, 2 * dt + (q4 >> 1)) * 16 + 8 * (q4 & 1) + 4 * h));
                else raw[dt][q4] = lds_read_b64(v_row + (uint32_t)(v_swz(ql, 4 * dt + q4) * 16 + 8 * h));
            }
        const f32x16 s = scores();
        uint32_t bits = 0u;                  // key ql's score: one of the registers of one half
        const uint32_t own_bit = (1u << ql) >> (4 * h);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
            const float score = s[r];
            bits |= __builtin_bit_cast(uint32_t, score) & (uint32_t)__builtin_amdgcn_sbfe((int)own_bit, 8 * (r / 4) + r % 4, 1);
        }
        const u32x2 both = __builtin_amdgcn_permlane32_swap(bits, bits, false, false);
        const uint32_t b0 = both[0], b1 = both[1];
        const float score = __builtin_bit_cast(float, b0 | b1) * sc;
        // (the maximum is raised as above)
        const bool raise = leaf_word != 0u && (score > m_i + kRescaleSlack || (m_i == -INFINITY && score > -INFINITY));
        if (__ballot(raise) != 0ull) {
            const float alpha = raise ? __builtin_amdgcn_exp2f(m_i - score) : 1.f;      // exp2(-inf) = 0
            if (raise) m_i = score;
            l_i *= alpha;
#pragma unroll
            for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
                for (int r = 0; r < 16; ++r) o[dt][r] *= alpha;
        }
        const float w = __builtin_amdgcn_exp2f(score - (m_i == -INFINITY ? 0.f : m_i));
        lds_wait();
#pragma unroll
        for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) lds_tie(raw[dt][q4]);
        if (leaf_word != 0u) {
            if (h == 0) l_i += w;
#pragma unroll
            for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
                for (int q4 = 0; q4 < 4; ++q4) {
                    float x[4];
                    if constexpr (KV8) {
                        const f32x2 lo = __builtin_amdgcn_cvt_pk_f32_fp8((int)raw[dt][q4], false);
                        const f32x2 hi = __builtin_amdgcn_cvt_pk_f32_fp8((int)raw[dt][q4], true);
                        x[0] = lo[0], x[1] = lo[1], x[2] = hi[0], x[3] = hi[1];
                    } else {
                        const uint32_t lo = raw[dt][q4][0], hi = raw[dt][q4][1];
                        x[0] = MM::low(lo), x[1] = MM::high(lo), x[2] = MM::low(hi), x[3] = MM::high(hi);
                    }
#pragma unroll
                    for (int e = 0; e < 4; ++e) o[dt][4 * q4 + e] = __builtin_fmaf(x[e], w, o[dt][4 * q4 + e]);
                }
        }
    }

    // ---- join the waves: results to LDS (16-byte pieces swizzled by the row), then every thread sums 4 * kPieces head dims
    // of one row over the waves (one that had no tile brings zeros under a maximum of -inf)
    __syncthreads();                         // every wave is done with its ring
    {
        float a, b;
        swap_halves(l_i, false, a, b);
        if (h == 0) {
            ml_s[wave * 64 + ql] = m_i;
            ml_s[wave * 64 + 32 + ql] = a + b;
        }
        float* mine_s = reinterpret_cast<float*>(smem) + (wave * 32 + ql) * D;
#pragma unroll
        for (int dt = 0; dt < kDTiles; ++dt)
#pragma unroll
            for (int q4 = 0; q4 < 4; ++q4) {
                const int c = 8 * dt + 2 * q4 + h;       // head dims 4c .. 4c+3
                const f32x4 val = {o[dt][4 * q4], o[dt][4 * q4 + 1], o[dt][4 * q4 + 2], o[dt][4 * q4 + 3]};
                *reinterpret_cast<f32x4*>(mine_s + ((c ^ ql) % (D / 4)) * 4) = val;
            }
    }
    __syncthreads();
    constexpr int kThreadsPerRow = kWaves * 64 / kRows;      // 16
    constexpr int kPieces = D / 4 / kThreadsPerRow;          // 16-byte pieces per thread
    static_assert(kPieces >= 1 && kPieces * kThreadsPerRow * 4 == D, "threads of a row share its head dims");
    const int row = tid / kThreadsPerRow, piece0 = (tid % kThreadsPerRow) * kPieces;
    float ms[kWaves], ls[kWaves];
    f32x4 x[kWaves][kPieces];
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        ms[w] = ml_s[w * 64 + row];
        ls[w] = ml_s[w * 64 + 32 + row];
        const float* src = reinterpret_cast<const float*>(smem) + (w * 32 + row) * D;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) x[w][i] = *reinterpret_cast<const f32x4*>(src + (((piece0 + i) ^ row) % (D / 4)) * 4);
    }
    float m_all = ms[0];
#pragma unroll
    for (int w = 1; w < kWaves; ++w) m_all = fmaxf(m_all, ms[w]);
    const float m_safe = m_all == -INFINITY ? 0.f : m_all;
    float l_tot = 0.f;
    f32x4 acc[kPieces];
#pragma unroll
    for (int i = 0; i < kPieces; ++i) acc[i] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const float wt = __builtin_amdgcn_exp2f(ms[w] - m_safe);      // exp2(-inf) = 0
        l_tot = __builtin_fmaf(ls[w], wt, l_tot);
#pragma unroll
        for (int i = 0; i < kPieces; ++i)
#pragma unroll
            for (int e = 0; e < 4; ++e) acc[i][e] = __builtin_fmaf(x[w][i][e], wt, acc[i][e]);
    }
    float inv = l_tot > 0.f ? 1.f / l_tot : 0.f;
    if (KV8 && p.v_scale) inv *= p.v_scale[hz];
    const int grow = row_base + row;
    if (grow >= p.nq) return;
    const bool partial = gr.runs > 1;
    const size_t out_row = ((size_t)(partial ? run * p.heads_total + hz : hz)) * p.nq + grow;
    float* lse_out = partial ? p.part_lse : p.lse;
    if (lse_out && tid % kThreadsPerRow == 0) lse_out[out_row] = l_tot > 0.f ? m_all + log2f(l_tot) : -INFINITY;
#pragma unroll
    for (int i = 0; i < kPieces; ++i)
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[i][e] *= inv;
    if (partial || p.out_f32) {
        float* dst = static_cast<float*>(partial ? static_cast<void*>(p.part_o) : p.o) + out_row * D + piece0 * 4;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) *reinterpret_cast<f32x4*>(dst + 4 * i) = acc[i];
    } else {
        T* dst = static_cast<T*>(p.o) + out_row * D + piece0 * 4;
#pragma unroll
        for (int i = 0; i < kPieces; ++i) {
            const u32x2 packed = {MM::pack_out(acc[i][0], acc[i][1]), MM::pack_out(acc[i][2], acc[i][3])};
            *reinterpret_cast<u32x2*>(dst + 4 * i) = packed;
        }
    }
}

template <bool BF16, int D, bool KV8, int NW, bool SPLIT>
int launch_waves(const AttnParams& p, const CachePlan& plan, hipStream_t stream) {
    const size_t lds = cache_lds_bytes<D, NW>(p.max_anc);
    CacheGrid g;
    g.chunks = (p.nq + kRows - 1) / kRows;
    g.runs = plan.runs;
    g.run_tiles = plan.run_tiles;
    const int64_t total = (int64_t)p.heads_total * g.chunks * g.runs;
    g.total = (int32_t)total;
    g.per_xcd = (int32_t)((total + kXcds - 1) / kXcds);
    g.chunks_inv = g.chunks > 1 ? (uint32_t)((0x100000000ull + g.chunks - 1) / g.chunks) : 0u;
    g.runs_inv = g.runs > 1 ? (uint32_t)((0x100000000ull + g.runs - 1) / g.runs) : 0u;
    g.block_shift = p.block_m == 32 ? 5 : p.block_m == 64 ? 6 : 7;
    const dim3 grid((unsigned)(kXcds * g.per_xcd)), block(NW * 64);
    // One group of rows: nobody reads the keys again, they go past the caches (30 rows, 256 slices x 4000 keys, bf16: 93 ->
    // 82 us, 5.7 -> 6.5 TB/s).  With two groups the second reader would miss (61 rows: 58 -> 64 us).
    if (g.chunks == 1) {
        const int rc = allow_full_lds<&attn_cache_kernel<BF16, D, KV8, NW, SPLIT, true>>();
        if (rc != FSTA_OK) return rc;
        hipLaunchKernelGGL((attn_cache_kernel<BF16, D, KV8, NW, SPLIT, true>), grid, block, lds, stream, p, g);
    } else {
        const int rc = allow_full_lds<&attn_cache_kernel<BF16, D, KV8, NW, SPLIT, false>>();
        if (rc != FSTA_OK) return rc;
        hipLaunchKernelGGL((attn_cache_kernel<BF16, D, KV8, NW, SPLIT, false>), grid, block, lds, stream, p, g);
    }
    FSTA_HIP_OK(hipGetLastError());
    note_launch({"attn_cache_kernel", BF16 ? "true" : "false", {D, KV8 ? 1 : 0, NW, SPLIT ? 1 : 0, g.chunks == 1 ? 1 : 0, 0}, 5, 0x1au, 0, 0});
    return FSTA_OK;
}

template <bool BF16, int D, bool KV8, bool SPLIT>
int launch_split(const AttnParams& p, const CachePlan& plan, hipStream_t stream) {
    return plan.waves == 4 ? launch_waves<BF16, D, KV8, 4, SPLIT>(p, plan, stream) : launch_waves<BF16, D, KV8, 8, SPLIT>(p, plan, stream);
}

template <bool BF16, bool KV8, bool SPLIT>
int launch_dim(const AttnParams& p, int head_dim, const CachePlan& plan, hipStream_t stream) {
    return head_dim == 64 ? launch_split<BF16, 64, KV8, SPLIT>(p, plan, stream) : launch_split<BF16, 128, KV8, SPLIT>(p, plan, stream);
}

}  // namespace

bool cache_kernel_supported(int dtype, int head_dim, int block_m) {
    return (dtype == FSTA_F16 || dtype == FSTA_BF16) && (head_dim == 64 || head_dim == 128) && plan_block_size_ok(block_m);
}

bool cache_kernel_takes(int64_t slices, int nq, int nk, int head_dim, bool kv8, int max_anc, const CachePlan& plan) {
    if ((uint64_t)nk * (uint64_t)head_dim * (kv8 ? 1u : 2u) > 0xffffffffull) return false;      // 32-bit byte offsets in a slice
    const size_t lds = head_dim == 64 ? (plan.waves == 4 ? cache_lds_bytes<64, 4>(max_anc) : cache_lds_bytes<64, 8>(max_anc))
                                      : (plan.waves == 4 ? cache_lds_bytes<128, 4>(max_anc) : cache_lds_bytes<128, 8>(max_anc));
    if (lds > 160 * 1024) return false;
    const int64_t chunks = (nq + kRows - 1) / kRows, total = slices * chunks * plan.runs;
    // (a launch's quotients by multiplication are exact while dividend * divisor < 2^32)
    return total <= 0x7fffff00 && (uint64_t)(total + kXcds) * (uint64_t)(chunks > plan.runs ? chunks : plan.runs) < 0xffffffffull;
}

int launch_attention_cache(const AttnParams& p, int dtype, int head_dim, bool kv8, bool fast_pv, const CachePlan& plan,
                           hipStream_t stream) {
    if (!p.plan || !cache_kernel_takes(p.heads_total, p.nq, p.nk, head_dim, kv8, p.max_anc, plan)) return FSTA_EUNSUPPORTED;
    const bool split = dtype == FSTA_BF16 && !fast_pv;
    if (dtype == FSTA_F16)
        return kv8 ? launch_dim<false, true, false>(p, head_dim, plan, stream) : launch_dim<false, false, false>(p, head_dim, plan, stream);
    if (kv8) return launch_dim<true, true, true>(p, head_dim, plan, stream);
    return split ? launch_dim<true, false, true>(p, head_dim, plan, stream) : launch_dim<true, false, false>(p, head_dim, plan, stream);
}

}  // namespace fsta
