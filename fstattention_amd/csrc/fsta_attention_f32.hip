// Tree attention in float32 for gfx950 (head_dim 64 / 128): the products on the matrix cores' float32 form, operands
// straight from memory into the registers the products take them from.
//
// What bounds it: float32 trees are small (tens to hundreds of rows, a few heads), so a launch is a chain of latencies:
// launch, lists, K/V rows, one tile of arithmetic, store.  Hence the split: a workgroup owns 16 query rows of one
// (batch, head) slice, and its waves take 16 keys each -- ancestors, then the shared prefix -- so that all K/V rows of a
// block are on their way after the first round trip, wherever they are used.  Nothing is staged in LDS; the waves' running
// softmaxes are joined there at the end.  (64 rows of 16 ancestors, 8 heads, head_dim 64: 7.4 us with the scalar kernel's
// workgroup of 64 rows that walks its keys in tiles of 32.)  Sums, maxima and the row that empty slots repeat go from lane to
// lane by register moves: a permute is a round trip through the LDS unit in the chain (in a graph 3.81 -> 3.69 us for that shape,
// 256 rows, 12 heads 5.14 -> 5.00; the rows' V keys by sixteen such moves instead of four permutes: no change).
//
// 16x16x4 products: A holds row i = lane % 16, k = g = lane / 16; B column i, k = g; C register r row 4g + r of column i.
//   S^T = K.Q^T   row: key, column: query.  The product over dims is split as 16 j + 4 g + e: product (j, e) takes dim
//                 16 j + 4 g + e from lane group g, so a lane loads 16 bytes (e = 0 .. 3) and four lanes 64 in a row.
//   O^T += V^T.P  register r of S^T is the B operand for keys 4g + r as it stands; V is loaded as 16 bytes per lane, dims
//                 64 b + 4 i + e of key 4g + r, which makes O^T tile (b, e) rows i: a lane ends with dims 64 b + 16 g .. +15.
// A row's own key (reference fstattention.py:86-91) needs no product: its wave starts from score, weight 1 and V row.
#include "fsta_mfma_common.h"

namespace fsta {
namespace {

typedef float f32x4 __attribute__((ext_vector_type(4)));

constexpr int kRows = 16;
constexpr int kKeys = 16;     // per tile

template <int D, int NW>
__global__ __launch_bounds__(NW * 64, NW == 8 ? 2 : 1) void attn_f32_kernel(AttnParams p) {
    constexpr int kQLoads = D / 16;          // 16-byte loads of a lane's part of a Q or K row
    constexpr int kVb = D / 64;              // 16-byte loads of a lane's part of a V row
    constexpr int kPitch = D + 4;            // floats per row of a wave's result (rows start in different banks)
    __shared__ __attribute__((aligned(16))) float out_s[NW][kRows * kPitch];
    __shared__ float m_s[NW][kRows], l_s[NW][kRows];

    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int i = lane & 15, g = lane >> 4;
    const int row0 = blockIdx.x * kRows;
    const int hz = blockIdx.y;
    const int j = row0 / p.block_m;          // (block sizes are multiples of 16)
    const int in_block = row0 - j * p.block_m + i;
    const float* qb = static_cast<const float*>(p.q) + (size_t)hz * p.nq * D;
    const float* kb = static_cast<const float*>(p.k) + (size_t)hz * p.nk * D;
    const float* vb = static_cast<const float*>(p.v) + (size_t)hz * p.nk * D;
    const int64_t* list = p.ancestor_idx + (size_t)j * p.max_anc;
    const uint32_t* words = p.mask_bits + (size_t)j * p.mask_words * p.block_m + in_block;

    // the wave's first list entries, their mask word, the count, the own key: one round trip
    auto list_entry = [&](int t) -> int64_t {
        const int c = t * kKeys + i;
        return c < p.max_anc ? list[c] : -1;
    };
    auto mask_word = [&](int t) -> uint32_t { return (t >> 1) < p.mask_words ? words[(size_t)(t >> 1) * p.block_m] : 0u; };
    int64_t entry = list_entry(wave);
    uint32_t word = mask_word(wave);
    const bool own_wave = wave == NW - 1;
    int64_t own = own_wave ? p.leaf_idx[(size_t)j * p.block_m + in_block] : -1;
    int n_anc = p.anc_count ? p.anc_count[j] : p.max_anc;
    const float* q_row = qb + (size_t)min(row0 + i, p.nq - 1) * D + 4 * g;
    f32x4 q[kQLoads];
#pragma unroll
    for (int s = 0; s < kQLoads; ++s) q[s] = *reinterpret_cast<const f32x4*>(q_row + 16 * s);

    n_anc = min(max(__builtin_amdgcn_readfirstlane(n_anc), 0), p.max_anc);
    const int anc_tiles = (n_anc + kKeys - 1) / kKeys;
    const int total = anc_tiles + (p.prefix + kKeys - 1) / kKeys;

    float m_i = -INFINITY, l_i = 0.f;        // m_i: of the query, l_i: this lane's keys only
    f32x4 o[kVb][4];
#pragma unroll
    for (int b = 0; b < kVb; ++b)
#pragma unroll
        for (int e = 0; e < 4; ++e) o[b][e] = f32x4{0.f, 0.f, 0.f, 0.f};

    f32x4 k[kQLoads], v[4][kVb];
    // bit r: key 4g + r of the tile exists and query i attends to it; bit 16 + c: slot c of the tile has no key
    uint32_t ok = 0u;
    auto request = [&](int t, int64_t id, uint32_t w) {
        int key;
        if (t < anc_tiles) {
            const bool there = t * kKeys + i < n_anc && id >= 0 && id < p.nk;
            const uint32_t exists = (uint32_t)__ballot(there) & 0xffffu;        // (the four lane groups hold the same entries)
            const int first = exists ? __builtin_ctz(exists) : 0;
            // an empty slot repeats the tile's first row: no row outside the list is read
            key = there ? (int)id : -1;
            const int repeat = __builtin_amdgcn_readlane(key, first);
            if (key < 0) key = max(repeat, 0);
            ok = ((((w >> (kKeys * (t & 1))) & exists) >> (4 * g)) & 0xfu) | (~exists << 16);
        } else {
            const int c = (t - anc_tiles) * kKeys;
            key = min(c + i, p.prefix - 1);
            const int left = p.prefix - c - 4 * g;
            ok = left >= 4 ? 0xfu : left > 0 ? (1u << left) - 1u : 0u;
            if (p.prefix - c < kKeys) ok |= 0xffffffffu << (16 + p.prefix - c);
        }
        const float* k_row = kb + (size_t)key * D + 4 * g;
#pragma unroll
        for (int s = 0; s < kQLoads; ++s) k[s] = *reinterpret_cast<const f32x4*>(k_row + 16 * s);
        return key;
    };
    auto request_v = [&](int key) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            const float* v_row = vb + (size_t)__shfl(key, 4 * g + r) * D + 4 * i;
#pragma unroll
            for (int b = 0; b < kVb; ++b) v[r][b] = *reinterpret_cast<const f32x4*>(v_row + 64 * b);
        }
    };
    int key = 0;
    if (wave < total) {
        key = request(wave, entry, word);
        request_v(key);
    }
    if (own_wave) {
        const bool there = own >= 0 && own < p.nk;
        const int own_key = there ? (int)own : 0;
        const float* k_row = kb + (size_t)own_key * D + 4 * g;
        const float* v_row = vb + (size_t)own_key * D + 16 * g;
        f32x4 ko[kQLoads], vo[kVb][4];
#pragma unroll
        for (int s = 0; s < kQLoads; ++s) ko[s] = *reinterpret_cast<const f32x4*>(k_row + 16 * s);
#pragma unroll
        for (int b = 0; b < kVb; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r) vo[b][r] = *reinterpret_cast<const f32x4*>(v_row + 64 * b + 4 * r);
        float dot[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int s = 0; s < kQLoads; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) dot[e] = __builtin_fmaf(q[s][e], ko[s][e], dot[e]);
        float score = (dot[0] + dot[1]) + (dot[2] + dot[3]);
        score = mfma::sum_quarters(score);
        if (there) {
            m_i = score * p.scale_log2e;
            l_i = g == 0 ? 1.f : 0.f;
#pragma unroll
            for (int b = 0; b < kVb; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e)
#pragma unroll
                    for (int r = 0; r < 4; ++r) o[b][e][r] = vo[b][r][e];
        }
    }
    for (int t = wave; t < total; t += NW) {
        const bool more = t + NW < total;
        const uint32_t mine = ok, empty = __builtin_amdgcn_readfirstlane(ok >> 16);
        if (more) {                          // (entries of the next tile: on their way under this tile's products)
            entry = list_entry(t + NW);
            word = mask_word(t + NW);
        }
        f32x4 s2[2] = {f32x4{0.f, 0.f, 0.f, 0.f}, f32x4{0.f, 0.f, 0.f, 0.f}};
#pragma unroll
        for (int s = 0; s < kQLoads; ++s)
#pragma unroll
            for (int e = 0; e < 4; ++e) s2[e & 1] = __builtin_amdgcn_mfma_f32_16x16x4f32(k[s][e], q[s][e], s2[e & 1], 0, 0, 0);
        if (more) key = request(t + NW, entry, word);
        float sv[4], mx = -INFINITY;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            sv[r] = (mine >> r) & 1u ? (s2[0][r] + s2[1][r]) * p.scale_log2e : -INFINITY;
            mx = fmaxf(mx, sv[r]);
        }
        mx = mfma::max_quarters(mx);
        const float m_new = fmaxf(m_i, mx);
        const float base = m_new == -INFINITY ? 0.f : m_new;
        const float alpha = __builtin_amdgcn_exp2f(m_i - base);       // exp2(-inf) = 0
        m_i = m_new;
        l_i *= alpha;
        float w[4];
#pragma unroll
        for (int r = 0; r < 4; ++r) {
            w[r] = __builtin_amdgcn_exp2f(sv[r] - base);
            l_i += w[r];
        }
#pragma unroll
        for (int b = 0; b < kVb; ++b)
#pragma unroll
            for (int e = 0; e < 4; ++e) o[b][e] *= alpha;
        if (empty) {
            // slots without a key repeat a row under weight 0: nothing of it may come through, not even as 0 * infinity
#pragma unroll
            for (int r = 0; r < 4; ++r)
                if ((empty >> (4 * g + r)) & 1u)
#pragma unroll
                    for (int b = 0; b < kVb; ++b) v[r][b] = f32x4{0.f, 0.f, 0.f, 0.f};
        }
#pragma unroll
        for (int r = 0; r < 4; ++r)
#pragma unroll
            for (int b = 0; b < kVb; ++b)
#pragma unroll
                for (int e = 0; e < 4; ++e) o[b][e] = __builtin_amdgcn_mfma_f32_16x16x4f32(v[r][b][e], w[r], o[b][e], 0, 0, 0);
        if (more) request_v(key);
    }

    // ---- join the waves that had keys
    const int busy = min(total, NW);
    if (wave < busy || own_wave) {
        l_i = mfma::sum_quarters(l_i);
        if (g == 0) {
            m_s[wave][i] = m_i;
            l_s[wave][i] = l_i;
        }
#pragma unroll
        for (int b = 0; b < kVb; ++b)
#pragma unroll
            for (int r = 0; r < 4; ++r)
                *reinterpret_cast<f32x4*>(&out_s[wave][i * kPitch + 64 * b + 16 * g + 4 * r]) = f32x4{o[b][0][r], o[b][1][r], o[b][2][r], o[b][3][r]};
    }
    __syncthreads();
    constexpr int kPieces = kRows * D / 4;
#pragma unroll
    for (int e = threadIdx.x; e < kPieces; e += NW * 64) {
        const int row = e / (D / 4), d = (e % (D / 4)) * 4;
        if (row0 + row >= p.nq) break;       // (rows ascend with e)
        float m_all = m_s[NW - 1][row];
#pragma unroll
        for (int w = 0; w < NW - 1; ++w) m_all = fmaxf(m_all, w < busy ? m_s[w][row] : -INFINITY);
        const float base = m_all == -INFINITY ? 0.f : m_all;
        float l = 0.f;
        f32x4 acc = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int w = 0; w < NW; ++w) {
            if (w >= busy && w != NW - 1) continue;
            const float wt = __builtin_amdgcn_exp2f(m_s[w][row] - base);
            l = __builtin_fmaf(l_s[w][row], wt, l);
            acc += wt * *reinterpret_cast<const f32x4*>(&out_s[w][row * kPitch + d]);
        }
        const size_t out_row = (size_t)hz * p.nq + row0 + row;
        if (p.lse && d == 0) p.lse[out_row] = l > 0.f ? m_all + log2f(l) : -INFINITY;
        const f32x4 val = l > 0.f ? acc / l : f32x4{0.f, 0.f, 0.f, 0.f};
        __builtin_nontemporal_store(val, reinterpret_cast<f32x4*>(static_cast<float*>(p.o) + out_row * D + d));
    }
}

template <int D, int NW>
int launch_one(const AttnParams& p, hipStream_t stream) {
    const unsigned groups = (unsigned)((p.nq + kRows - 1) / kRows);
    hipLaunchKernelGGL((attn_f32_kernel<D, NW>), dim3(groups, p.heads_total), dim3(NW * 64), 0, stream, p);
    FSTA_HIP_OK(hipGetLastError());
    note_launch({"attn_f32_kernel", D == 64 ? "64" : "128", {NW, 0, 0, 0, 0, 0}, 1, 0u, 0, 0});
    return FSTA_OK;
}

}  // namespace

int launch_attention_f32(const AttnParams& p, int head_dim, hipStream_t stream) {
    if (head_dim != 64 && head_dim != 128) return FSTA_EUNSUPPORTED;
    // Four waves, so that several workgroups share a CU and one's arithmetic lies under another's round trips, also where a
    // wave then takes two or three tiles (eight waves for up to 8 tiles, 512 rows, 16 heads, head_dim 128: 18.6 us, four:
    // 14.6; 4096 rows, 32 heads: 412, 310); eight once every wave of four would walk ten tiles (long prefixes).
    const int tiles = (p.max_anc + kKeys - 1) / kKeys + (p.prefix + kKeys - 1) / kKeys;
    if (head_dim == 64) return tiles < 40 ? launch_one<64, 4>(p, stream) : launch_one<64, 8>(p, stream);
    return tiles < 40 ? launch_one<128, 4>(p, stream) : launch_one<128, 8>(p, stream);
}

}  // namespace fsta
