// extern "C" surface of libfsta: argument validation, error text, kernel dispatch.
#include <cstdarg>
#include <cstdio>

#include "fsta_common.h"

namespace fsta {

static thread_local char g_error[512] = "";

int fail(int code, const char* fmt, ...) {
    va_list ap;
    va_start(ap, fmt);
    vsnprintf(g_error, sizeof(g_error), fmt, ap);
    va_end(ap);
    return code;
}

static thread_local LaunchNote g_note = {nullptr, "", {0, 0, 0, 0, 0, 0}, 0, 0u, 0, 0};
static thread_local char g_note_text[192] = "";

void note_launch(const LaunchNote& note) { g_note = note; }

}  // namespace fsta

using namespace fsta;

extern "C" const char* fsta_last_attention_kernel(void) {
    if (!g_note.kernel) return "";
    int len = snprintf(g_note_text, sizeof(g_note_text), "%s<%s", g_note.kernel, g_note.first);
    for (int i = 0; i < g_note.n_args && len < (int)sizeof(g_note_text); ++i)
        len += (g_note.bool_args >> i) & 1u
                   ? snprintf(g_note_text + len, sizeof(g_note_text) - len, ", %s", g_note.args[i] ? "true" : "false")
                   : snprintf(g_note_text + len, sizeof(g_note_text) - len, ", %d", g_note.args[i]);
    if (len < (int)sizeof(g_note_text))
        snprintf(g_note_text + len, sizeof(g_note_text) - len, ">%s%s", g_note.half_blocks ? " half-blocks" : "",
                 g_note.early_start ? " early-start" : "");
    return g_note_text;
}

extern "C" int fsta_abi_version(void) { return FSTA_ABI_VERSION; }

extern "C" const char* fsta_last_error(void) { return g_error; }

namespace {

constexpr int kKeyTile = 32;        // keys per tile of the attention kernels
constexpr int kMinRunTiles = 8;     // shortest run of prefix tiles worth a workgroup of its own
constexpr int kTargetGroups = 512;  // two workgroups per CU
constexpr int kDenseMinRunTiles = 16;   // the same for the dense prefix kernel, whose partial results the tree part's launch reads back
                                        // (2048 keys: 4 runs 33.7 us, 8 runs 38.1; 4096 keys: 4 and 8 runs alike)

// How the shared prefix is cut for a launch of the narrow matrix-core kernel: number of runs
// (1 = no split) and prefix tiles per run.  Depends on the shape and flags only, so that the
// workspace query and the launch agree.
int plan_key_splits(int64_t slices, int nq, int nk, int head_dim, int dtype, int block_m, float sm_scale,
                    uint32_t flags, int* split_tiles) {
    const int tiles = (nk - nq + kKeyTile - 1) / kKeyTile;
    *split_tiles = tiles;
    if (tiles < 2 || slices <= 0 || nq <= 0) return 1;
    if ((flags & (FSTA_FLAG_GENERIC | FSTA_FLAG_WIDE_WAVES)) || !(sm_scale > 0.f) ||
        !mfma_supported(dtype, head_dim, block_m))
        return 1;
    const int forced = (int)((flags >> 8) & 0xffu);
    int64_t want = forced;
    if (!forced) {
        const int64_t groups = ((slices + 7) / 8) * 8 * ((nq + block_m - 1) / block_m);
        want = (kTargetGroups + groups - 1) / groups;
        if (want > tiles / kMinRunTiles) want = tiles / kMinRunTiles;
    }
    if (want > tiles) want = tiles;
    if (want > 255) want = 255;
    if (want <= 1) return 1;
    const int per = (int)((tiles + want - 1) / want);
    *split_tiles = per;
    return (tiles + per - 1) / per;
}

size_t key_split_bytes(int splits, int64_t slices, int nq, int head_dim) {
    return (size_t)splits * (size_t)slices * (size_t)nq * (size_t)(head_dim + 1) * sizeof(float);
}

constexpr int kDenseMinKeys = 2048;   // shortest prefix handed to the dense prefix kernel (below: two more launches cost more than they save)
constexpr int kDenseRows = 128;       // query rows per workgroup of that kernel

// Whether (and how) the prefix goes to the dense prefix kernel: number of key runs (0 = not at all) and
// prefix tiles per run.  The tree part then takes one more workspace slot.  Shape and flags only.
int plan_dense_prefix(int64_t slices, int nq, int nk, int head_dim, int dtype, int block_m, float sm_scale,
                      uint32_t flags, int* split_tiles) {
    const int prefix = nk - nq;
    if (slices <= 0 || nq <= 0 || prefix < kDenseMinKeys) return 0;
    if ((flags & (FSTA_FLAG_GENERIC | FSTA_FLAG_WIDE_WAVES)) || !(sm_scale > 0.f) ||
        !mfma_supported(dtype, head_dim, block_m) || !prefix_kernel_supported(dtype, head_dim))
        return 0;
    const int forced = (int)((flags >> 8) & 0xffu);
    if (forced == 1) return 0;        // "never split": the prefix stays in the tree kernel's own loop
    const int tiles = (prefix + kKeyTile - 1) / kKeyTile;
    int64_t want = forced;
    if (!forced) {
        const int64_t groups = ((slices + 7) / 8) * 8 * ((nq + kDenseRows - 1) / kDenseRows);
        want = (kTargetGroups + groups - 1) / groups;
        if (want > tiles / kDenseMinRunTiles) want = tiles / kDenseMinRunTiles;
        if (want < 1) want = 1;
    }
    if (want > tiles) want = tiles;
    if (want > 254) want = 254;
    const int per = (int)((tiles + want - 1) / want);
    *split_tiles = per;
    return (tiles + per - 1) / per;
}

// How the cache kernel (32 query rows per workgroup, tree and prefix in one launch) takes a launch: waves per workgroup
// and runs of prefix tiles (runs = 0: not at all).  Shape and flags only.
//
// The number of runs is the one with the shortest predicted time.  The constants are those that choose best, not those that
// predict best, over 28199 shapes (8-512 rows, 8-bit K/V up to 4096; 1-512 slices; 64-32768 keys), every candidate timed with K
// and V from HBM, as a step through a model's layers finds them, and from the Infinity Cache; HBM counts more.  They cost 0.9 to
// 1.2 % over the best candidate on average, 3 to 4 % at the ninetieth percentile, 47 % at worst (8790 shapes of another
// day: 0.9-1.3, 3-5, 33 %).  Constants fitted to K and V of three calls in turn, mostly from the Infinity Cache, took too few
// runs where fewer workgroups than CUs leave HBM idle (32 slices of 87 rows behind 2829 keys, D 128: 23.2 us in two runs, 22.4 in
// five; of 12513 shapes at head_dim 128 in 16 bits 129 were more than 4 % slower from HBM than under the constants before
// those, 48 are now); constants without `cu_rate`, fitted to the times, cost 1.7-2.3, 6-7 and 66 %.
//   1.6 (launch) + rounds of workgroups * start_end + the larger of
//     workgroups on the fullest CU * tiles * tile   (a CU's matrix cores, L2 and LDS)      [us]
//     rounds * tiles per wave * wave_tile           (one wave's chain)
//       both times f16 for float16, which needs no second weight half,
//   but no less than start_end + the prefix read once at `tb1` or, with several row groups, `tb` TB/s (rereading by the other
//   groups: a fraction `again` each), and no faster than `cu_rate` B/ns for each CU that has a workgroup,
//   + for more than one run `join` and the float32 parts, written and read once at `join_tb` TB/s.
// Several runs are taken only where they are predicted at less than `several` of one run's time.
struct CacheCost {
    float start_end8, start_end4, tile, wave_tile, f16, join, join_tb, tb1, tb, again, cu_rate, several;
};
constexpr CacheCost kCost16[2] = {{2.06f, 1.71f, 0.273f, 1.5f, 0.932f, 4.11f, 1.0f, 5.4f, 4.24f, 0.193f, 29.7f, 1.0f},         // head_dim 64
                                  {3.65f, 1.23f, 0.5f, 1.39f, 1.0f, 3.26f, 1.71f, 6.01f, 7.0f, 0.61f, 35.6f, 0.956f}};         // head_dim 128
constexpr CacheCost kCost8[2] = {{2.42f, 3.46f, 0.112f, 0.602f, 1.01f, 2.39f, 16.8f, 6.09f, 4.28f, 0.08f, 33.7f, 0.92f},        // the same on 8-bit K/V
                                 {1.78f, 1.26f, 0.436f, 0.45f, 0.961f, 2.68f, 1.22f, 3.25f, 3.96f, 0.8f, 67.9f, 0.931f}};
// Prefixes of at most 7 MB, 32 layers of which the Infinity Cache holds: constants searched on K and V of three calls in turn.  What
// those above gain from HBM there (7 % where they choose otherwise, nearly always more runs) they lose from the cache at head_dim
// 128 (9 %; 24 layers of 8 slices, 165 rows behind 744 keys: 261 us a step, 221 this way), and calls that short wait for the
// host, for which a second launch is half a call more (24 layers of 8 slices, 63 rows behind 1290 keys, head_dim 64: 204 to 247 us
// a step on three hosts in six runs, 213 in one).
constexpr CacheCost kFew16[2] = {{2.71f, 2.42f, 0.0481f, 1.1f, 1.06f, 2.84f, 2.83f, 9.67f, 8.05f, 0.34f, 50.2f, 0.92f},
                                 {4.11f, 0.236f, 0.346f, 0.555f, 1.04f, 1.56f, 1.27f, 9.0f, 11.5f, 0.64f, 46.3f, 1.0f}};
constexpr CacheCost kFew8[2] = {{2.42f, 3.46f, 0.112f, 0.602f, 1.01f, 2.39f, 16.8f, 6.09f, 4.28f, 0.08f, 33.7f, 0.92f},
                                {2.76f, 5.56f, 0.208f, 0.628f, 1.16f, 3.14f, 15.4f, 8.89f, 6.05f, 0.412f, 66.8f, 0.92f}};
constexpr double kFewBytes = 7.0;      // MB of K and V
// Longer trees: 16-bit K/V go to the dense prefix kernel and the tree kernel, which read the prefix once per 128 and 64
// rows; a workgroup of the cache kernel reads it for 32 rows.
constexpr int kCacheMaxRows = 512;
// 8-bit K/V have no other kernel with runs of keys: a workgroup of the tree kernel walks the whole prefix for one block.  It
// is the faster one only where workgroups fill the GPU more than twice and the prefix is too short to pay for reading it once
// per 32 rows instead of once per block (bf16, 64 slices, us, tree and cache kernel: 2048 rows in blocks of 128, head_dim
// 128, behind 100 keys 65.3, 67.9, 700 keys 130, 126; 4096 shallow rows in blocks of 64, head_dim 64, behind 1 key 31.4, 35.6,
// 100 keys 46.2, 44.7; blocks of 32: 1.0 to 4 times in favour of the cache kernel from one key on.  Elsewhere: 513 rows, 32
// slices, 8192 keys, head_dim 128: 419, 153).
constexpr int short_prefix8(int block_m) { return block_m == 128 ? 700 : block_m == 64 ? 100 : 0; }
constexpr int kGpuCus = 256;

CachePlan plan_cache(int64_t slices, int nq, int nk, int head_dim, int dtype, int block_m, int max_anc, float sm_scale,
                     uint32_t flags, bool kv8) {
    CachePlan c = {8, 0, 0};
    const int prefix = nk - nq;
    if (slices <= 0 || nq <= 0 || prefix <= 0 || (nq > kCacheMaxRows && !kv8)) return c;
    if ((flags & (FSTA_FLAG_GENERIC | FSTA_FLAG_WIDE_WAVES | FSTA_FLAG_STREAM | FSTA_FLAG_SHARE_TILES)) || !(sm_scale > 0.f) ||
        !cache_kernel_supported(dtype, head_dim, block_m))
        return c;
    const int tiles = (prefix + kKeyTile - 1) / kKeyTile;
    const int64_t groups = (nq + 31) / 32, wgs1 = slices * groups;
    if (kv8 && nq > kCacheMaxRows && wgs1 > 2 * kGpuCus && prefix < short_prefix8(block_m)) return c;
    if (!kv8) {
        // Enough rows and keys to be bound by the matrix cores: the dense prefix kernel, which shares every tile among 128
        // rows (256 rows, 32 slices, 16384 keys, bf16: 119 us against 139; 8192 keys: 76 against 74).
        const double dense_tiles = (double)((nq + kDenseRows - 1) / kDenseRows) * (double)slices * tiles / kGpuCus;
        if (nq >= 96 && prefix >= kDenseMinKeys && dense_tiles >= (head_dim == 128 ? 64.0 : 110.0)) return c;
        // Many workgroups with little to do each: the tree kernel, whose workgroups of 64 rows read half as much and start
        // faster (97 rows, 154 slices, 283 keys: 16.5 against 17.7 us; 119 rows, 396 slices, 1487 keys: 90 against 106).
        if (head_dim == 128 && wgs1 > 512 && (prefix < 600 || (wgs1 > 1200 && nq > 96 && prefix < kDenseMinKeys))) return c;
    }
    const int forced = (int)((flags >> 8) & 0xffu);
    const double bytes = (double)slices * prefix * head_dim * (kv8 ? 2.0 : 4.0) * 1e-6;      // prefix K and V, MB
    const CacheCost& k = (bytes <= kFewBytes ? (kv8 ? kFew8 : kFew16) : (kv8 ? kCost8 : kCost16))[head_dim == 128 ? 1 : 0];
    const double product = dtype == FSTA_F16 ? k.f16 : 1.0;
    double best = 0.0, one = 0.0;
    // candidates: one run, the counts that fill the CUs once, twice, .., and those whose runs are one, two, .. tiles for
    // each of eight waves, if they promise a tenth (few slices: 46 rows, 8 slices, 1955 keys fill
    // 16 CUs in one run, 15.0 us, 9.3 in eight); a run has work for half of a workgroup's waves
    for (int i = 0; i <= 8; ++i) {
        const int64_t fill = i == 0 ? 1 : i <= 4 ? (int64_t)kGpuCus * i / wgs1 : (tiles + 8 * (i - 4) - 1) / (8 * (i - 4));
        const int want = forced ? forced : (int)(fill > 64 ? 64 : fill);
        if (i > 0 && (forced || want <= 1 || tiles / want < 4)) continue;
        const int per = (tiles + want - 1) / want;
        const int runs = (tiles + per - 1) / per;
        const int64_t wgs = wgs1 * runs;
        // more workgroups than CUs: four waves each, so that one workgroup's start and end lie under another's tiles
        const int waves = wgs > kGpuCus ? 4 : 8;
        // Half of the CUs busy with one or two row groups in one run, at most three tiles a wave in two: K and V from HBM up to
        // 8 % faster, from the Infinity Cache 15 % slower (64 slices of 37 and 46 rows behind 1310 keys, bf16; fp16, without the
        // second weight half, 10-16 % faster and 2-9 % slower: two runs).
        if (i > 0 && !forced && !kv8 && head_dim == 128 && dtype == FSTA_BF16 && groups <= 2 && waves == 8 && 2 * wgs1 >= kGpuCus &&
            per <= 3 * waves)
            continue;
        const double on_cu = (double)((wgs + kGpuCus - 1) / kGpuCus);
        const int at_once = (head_dim == 128 ? 1 : 2) * (waves == 4 ? 2 : 1);
        const double rounds = (double)(((int64_t)on_cu + at_once - 1) / at_once);
        const double t_tiles = per + 3.0;                        // (a few ancestor tiles and the own rows)
        const double chain = rounds * (double)((per + 3 + waves - 1) / waves) * k.wave_tile;
        const double work = on_cu * t_tiles * k.tile;
        double t = 1.6 + rounds * (waves == 8 ? k.start_end8 : k.start_end4) + (chain > work ? chain : work) * product;
        const double cus = wgs < kGpuCus ? (double)wgs : (double)kGpuCus;
        const double together = (1.0 + k.again * (double)(groups - 1)) / (groups == 1 ? k.tb1 : k.tb);
        const double each = (double)groups / (cus * k.cu_rate * 1e-3);
        const double mem = 1.6 + k.start_end8 + bytes * (together > each ? together : each);
        if (mem > t) t = mem;
        if (runs > 1) t += k.join + 2.0 * runs * (double)slices * nq * head_dim * 4e-6 / k.join_tb;
        if (i == 0) one = t;
        if (c.runs == 0 || (t < (i <= 4 ? best : 0.9 * best) && t < k.several * one)) {
            best = t;
            c.waves = waves;
            c.runs = runs;
            c.run_tiles = per;
        }
    }
    // (what the kernel would refuse is not planned for it: the workspace queries have to know)
    if (!cache_kernel_takes(slices, nq, nk, head_dim, kv8, max_anc, c)) c.runs = 0;
    return c;
}

// launches it; FSTA_EUNSUPPORTED where the plan says no
int launch_cache(AttnParams p, int dtype, int out_dtype, int head_dim, bool kv8, bool fast_pv, CachePlan c, void* workspace,
                 size_t workspace_bytes, size_t wanted_bytes, hipStream_t s) {
    if (c.runs < 1) return FSTA_EUNSUPPORTED;
    const int64_t slices = p.heads_total;
    if (c.runs > 1 && (!workspace || workspace_bytes < wanted_bytes)) {      // (too small a workspace: no runs, as documented)
        c.waves = slices * ((p.nq + 31) / 32) > kGpuCus ? 4 : 8;
        c.runs = 1;
        c.run_tiles = (p.prefix + kKeyTile - 1) / kKeyTile;
    }
    if (c.runs > 1 && reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
        return fail(FSTA_EINVAL, "fsta_attention_fwd_ws: workspace must be 16-byte aligned");
    if (c.runs > 1) {
        p.part_o = static_cast<float*>(workspace);
        p.part_lse = p.part_o + (size_t)c.runs * slices * p.nq * head_dim;
    }
    const int rc = launch_attention_cache(p, dtype, head_dim, kv8, fast_pv, c, s);
    if (rc != FSTA_OK || c.runs == 1) return rc;
    return launch_merge_splits(p.part_o, p.part_lse, c.runs, slices * p.nq, head_dim, p.o, out_dtype, p.lse, s);
}

}  // namespace

// Runs the cache kernel would take this problem in, 0 where it would not: what tests pin the choice by.  Not part of the interface.
extern "C" int fsta_internal_cache_runs(int64_t slices, int32_t nq, int32_t nk, int32_t head_dim, int32_t dtype, int32_t block_m,
                                        int32_t max_ancestors, int32_t kv8) {
    return plan_cache(slices, nq, nk, head_dim, dtype, block_m, max_ancestors, 0.1f, 0u, kv8 != 0).runs;
}

extern "C" size_t fsta_attention_workspace_bytes(int32_t batch, int32_t heads, int32_t nq, int32_t nk,
                                                 int32_t head_dim, int32_t dtype, int32_t block_m,
                                                 int32_t max_ancestors, float sm_scale, uint32_t flags) {
    if (batch <= 0 || heads <= 0 || nq <= 0 || nk <= nq || block_m <= 0) return 0;
    int split_tiles = 0;
    const int64_t slices = (int64_t)batch * heads;
    const int runs = plan_dense_prefix(slices, nq, nk, head_dim, dtype, block_m, sm_scale, flags, &split_tiles);
    size_t bytes = runs > 0 ? key_split_bytes(runs + 1, slices, nq, head_dim) : 0;
    if (runs == 0) {
        const int splits = plan_key_splits(slices, nq, nk, head_dim, dtype, block_m, sm_scale, flags, &split_tiles);
        if (splits > 1) bytes = key_split_bytes(splits, slices, nq, head_dim);
    }
    const CachePlan c = plan_cache(slices, nq, nk, head_dim, dtype, block_m, max_ancestors, sm_scale, flags, false);
    if (c.runs > 1 && key_split_bytes(c.runs, slices, nq, head_dim) > bytes) bytes = key_split_bytes(c.runs, slices, nq, head_dim);
    return bytes;
}

extern "C" int fsta_attention_uses_workspace(int32_t batch, int32_t heads, int32_t nq, int32_t nk, int32_t head_dim,
                                             int32_t dtype, int32_t block_m, int32_t max_ancestors, float sm_scale,
                                             uint32_t flags) {
    if (fsta_attention_workspace_bytes(batch, heads, nq, nk, head_dim, dtype, block_m, max_ancestors, sm_scale, flags) == 0) return 0;
    const CachePlan c = plan_cache((int64_t)batch * heads, nq, nk, head_dim, dtype, block_m, max_ancestors, sm_scale, flags, false);
    return c.runs == 1 ? 0 : 1;
}

extern "C" int fsta_attention_fwd(const void* q, const void* k, const void* v, void* o, float* lse,
                                  const int64_t* ancestor_idx, const uint32_t* mask_bits,
                                  const int32_t* anc_count, const int64_t* leaf_idx,
                                  const uint32_t* block_plan, int32_t plan_key_shift,
                                  int32_t batch, int32_t heads, int32_t nq, int32_t nk,
                                  int32_t head_dim, int32_t dtype, int32_t out_dtype,
                                  int32_t block_m, int32_t max_ancestors, int32_t num_blocks,
                                  float sm_scale, uint32_t flags, void* stream) {
    return fsta_attention_fwd_ws(q, k, v, o, lse, ancestor_idx, mask_bits, anc_count, leaf_idx, block_plan,
                                 plan_key_shift, batch, heads, nq,
                                 nk, head_dim, dtype, out_dtype, block_m, max_ancestors, num_blocks, sm_scale,
                                 flags, nullptr, 0, stream);
}

extern "C" int fsta_attention_fwd_ws(const void* q, const void* k, const void* v, void* o, float* lse,
                                     const int64_t* ancestor_idx, const uint32_t* mask_bits,
                                     const int32_t* anc_count, const int64_t* leaf_idx,
                                     const uint32_t* block_plan, int32_t plan_key_shift,
                                     int32_t batch, int32_t heads, int32_t nq, int32_t nk,
                                     int32_t head_dim, int32_t dtype, int32_t out_dtype,
                                     int32_t block_m, int32_t max_ancestors, int32_t num_blocks,
                                     float sm_scale, uint32_t flags, void* workspace, size_t workspace_bytes,
                                     void* stream) {
    if (batch < 0 || heads < 0 || nq < 0 || nk < nq)
        return fail(FSTA_EINVAL, "fsta_attention_fwd: batch=%d heads=%d nq=%d nk=%d (need nk >= nq >= 0)",
                    batch, heads, nq, nk);
    if (dtype != FSTA_F32 && dtype != FSTA_F16 && dtype != FSTA_BF16)
        return fail(FSTA_EINVAL, "fsta_attention_fwd: dtype=%d", dtype);
    if (out_dtype != dtype && out_dtype != FSTA_F32)
        return fail(FSTA_EINVAL, "fsta_attention_fwd: out_dtype=%d must equal dtype=%d or be float32",
                    out_dtype, dtype);
    if (head_dim != 16 && head_dim != 32 && head_dim != 64 && head_dim != 128)
        return fail(FSTA_EUNSUPPORTED, "fsta_attention_fwd: head_dim=%d (supported: 16, 32, 64, 128)", head_dim);
    if (block_m != 16 && block_m != 32 && block_m != 64 && block_m != 128)
        return fail(FSTA_EUNSUPPORTED, "fsta_attention_fwd: block_m=%d (supported: 16, 32, 64, 128)", block_m);
    if (max_ancestors < 1)
        return fail(FSTA_EINVAL, "fsta_attention_fwd: max_ancestors=%d", max_ancestors);
    if (num_blocks != (nq + block_m - 1) / block_m)
        return fail(FSTA_EINVAL, "fsta_attention_fwd: num_blocks=%d but ceil(nq=%d / block_m=%d) = %d",
                    num_blocks, nq, block_m, (nq + block_m - 1) / block_m);
    const int64_t slices = (int64_t)batch * heads;
    if (slices > 65535)
        return fail(FSTA_EUNSUPPORTED, "fsta_attention_fwd: batch*heads=%lld > 65535", (long long)slices);
    if (slices == 0 || nq == 0) return FSTA_OK;
    if (!q || !k || !v || !o || !ancestor_idx || !mask_bits || !leaf_idx)
        return fail(FSTA_EINVAL, "fsta_attention_fwd: null pointer");
    // rows and plan records are moved 16 bytes at a time, list entries 8, mask words and counts 4
    if (misaligned(q, 16) || misaligned(k, 16) || misaligned(v, 16) || misaligned(o, 16))
        return fail(FSTA_EINVAL, "fsta_attention_fwd: q, k, v and o must be 16-byte aligned");
    if (misaligned(block_plan, 16))
        return fail(FSTA_EINVAL, "fsta_attention_fwd: block_plan must be 16-byte aligned");
    if (misaligned(ancestor_idx, 8) || misaligned(leaf_idx, 8))
        return fail(FSTA_EINVAL, "fsta_attention_fwd: ancestor_idx and leaf_idx must be 8-byte aligned");
    if (misaligned(mask_bits, 4) || misaligned(anc_count, 4) || misaligned(lse, 4))
        return fail(FSTA_EINVAL, "fsta_attention_fwd: mask_bits, anc_count and lse must be 4-byte aligned");
    if (block_plan && (plan_key_shift < 0 || plan_key_shift > nk))
        return fail(FSTA_EINVAL, "fsta_attention_fwd: plan_key_shift=%d outside [0, nk=%d]", plan_key_shift, nk);

    AttnParams p;
    p.q = q; p.k = k; p.v = v; p.o = o; p.lse = lse;
    p.ancestor_idx = ancestor_idx; p.mask_bits = mask_bits; p.anc_count = anc_count;
    p.leaf_idx = leaf_idx;
    p.plan = plan_block_size_ok(block_m) ? block_plan : nullptr;
    p.key_shift = plan_key_shift;
    p.nq = nq; p.nk = nk; p.prefix = nk - nq;
    p.block_m = block_m; p.max_anc = max_ancestors; p.mask_words = fsta_mask_words(max_ancestors);
    p.nb = num_blocks;
    p.heads_total = (int32_t)slices;
    p.out_f32 = (out_dtype == FSTA_F32) ? 1 : 0;
    p.scale_log2e = sm_scale * kLog2e;
    p.key_splits = 1; p.split_tiles = 0; p.part_o = nullptr; p.part_lse = nullptr;
    p.share_tiles = (flags & FSTA_FLAG_SHARE_TILES) ? 1 : 0;
    p.k_scale = nullptr; p.v_scale = nullptr;
    p.merge_parts = 0; p.dry_run = 0;
    p.stream_mode = (flags & FSTA_FLAG_STREAM) ? 1 : 0;

    hipStream_t s = static_cast<hipStream_t>(stream);
    if (p.plan) {
        const CachePlan c = plan_cache(slices, nq, nk, head_dim, dtype, block_m, max_ancestors, sm_scale, flags, false);
        const size_t wanted = c.runs > 1 ? fsta_attention_workspace_bytes(batch, heads, nq, nk, head_dim, dtype, block_m, max_ancestors,
                                                                          sm_scale, flags) : 0;
        const int rc = launch_cache(p, dtype, out_dtype, head_dim, false, (flags & FSTA_FLAG_FAST_PV) != 0, c, workspace, workspace_bytes,
                                    wanted, s);
        if (rc != FSTA_EUNSUPPORTED) return rc;
    }
    if (workspace && p.plan) {
        // a long prefix goes to the dense prefix kernel, run by run (slots 1 .. runs of the workspace); the tree
        // kernel then does the tree part and, in its epilogue, joins it with those partial results into o / lse
        int run_tiles = 0;
        const int runs = plan_dense_prefix(slices, nq, nk, head_dim, dtype, block_m, sm_scale, flags, &run_tiles);
        if (runs > 0 && workspace_bytes >= key_split_bytes(runs + 1, slices, nq, head_dim)) {
            if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
                return fail(FSTA_EINVAL, "fsta_attention_fwd_ws: workspace must be 16-byte aligned");
            const bool fast_pv = (flags & FSTA_FLAG_FAST_PV) != 0;
            AttnParams pt = p;
            pt.part_o = static_cast<float*>(workspace);
            pt.part_lse = pt.part_o + (size_t)(runs + 1) * slices * nq * head_dim;
            pt.key_splits = 1;
            pt.split_tiles = 0;        // no prefix tile for the tree kernel
            pt.merge_parts = runs;
            pt.dry_run = 1;            // (would the tree kernel take this shape? asked before anything is launched)
            int rc = launch_attention_mfma16(pt, dtype, head_dim, fast_pv, s);
            if (rc == FSTA_OK) {
                AttnParams pp = pt;
                pp.dry_run = 0;
                pp.merge_parts = 0;
                pp.key_splits = runs;
                pp.split_tiles = run_tiles;
                rc = launch_attention_prefix(pp, dtype, head_dim, fast_pv, s);
                if (rc != FSTA_OK) return rc;
                pt.dry_run = 0;
                return launch_attention_mfma16(pt, dtype, head_dim, fast_pv, s);
            }
            if (rc != FSTA_EUNSUPPORTED) return rc;
            // (ancestor lists too long for the kernel with key runs: the launches below)
        }
        int split_tiles = 0;
        // (a workspace too small for what fsta_attention_workspace_bytes asked for: no split of any kind)
        const int splits = runs > 0 ? 1 : plan_key_splits(slices, nq, nk, head_dim, dtype, block_m, sm_scale, flags, &split_tiles);
        if (splits > 1 && workspace_bytes >= key_split_bytes(splits, slices, nq, head_dim)) {
            if (reinterpret_cast<uintptr_t>(workspace) % 16 != 0)
                return fail(FSTA_EINVAL, "fsta_attention_fwd_ws: workspace must be 16-byte aligned");
            AttnParams ps = p;
            ps.key_splits = splits;
            ps.split_tiles = split_tiles;
            ps.part_o = static_cast<float*>(workspace);
            ps.part_lse = ps.part_o + (size_t)splits * slices * nq * head_dim;
            const int rc = launch_attention_mfma16(ps, dtype, head_dim, (flags & FSTA_FLAG_FAST_PV) != 0, s);
            if (rc == FSTA_OK)
                return launch_merge_splits(ps.part_o, ps.part_lse, splits, slices * nq, head_dim, o, out_dtype, lse, s);
            // (this shape cannot take the narrow kernel: one launch without key splits below)
            if (rc != FSTA_EUNSUPPORTED) return rc;
        }
    }
    // the matrix-core kernel takes row maxima before scaling, which needs a positive scale
    if (!(flags & FSTA_FLAG_GENERIC) && sm_scale > 0.f && mfma_supported(dtype, head_dim, block_m)) {
        const bool fast_pv = (flags & FSTA_FLAG_FAST_PV) != 0;
        // (the kernel with 16 rows per wave reads the block plan only; it hands launches it cannot
        // take on to the other matrix-core kernel itself)
        int rc = FSTA_EUNSUPPORTED;
        if (!(flags & FSTA_FLAG_WIDE_WAVES)) rc = launch_attention_stream(p, dtype, head_dim, fast_pv, s);
        if (rc == FSTA_EUNSUPPORTED)
            rc = (flags & FSTA_FLAG_WIDE_WAVES) || !p.plan ? launch_attention_mfma(p, dtype, head_dim, fast_pv, s)
                                                           : launch_attention_mfma16(p, dtype, head_dim, fast_pv, s);
        // ancestor lists too long for the LDS-resident lists of these kernels: the scalar kernel
        // streams them and takes any length
        if (rc != FSTA_EUNSUPPORTED) return rc;
    }
    if (dtype == FSTA_F32 && !(flags & FSTA_FLAG_GENERIC)) {
        const int rc = launch_attention_f32(p, head_dim, s);
        if (rc != FSTA_EUNSUPPORTED) return rc;
    }
    return launch_attention_generic(p, dtype, head_dim, s);
}

extern "C" int fsta_attention_fwd_kv8(const void* q, const void* k8, const void* v8, const float* k_scale,
                                      const float* v_scale, void* o, float* lse, const uint32_t* block_plan,
                                      int32_t plan_key_shift, int32_t batch, int32_t heads, int32_t nq, int32_t nk,
                                      int32_t head_dim, int32_t dtype, int32_t out_dtype, int32_t block_m,
                                      int32_t max_ancestors, int32_t num_blocks, float sm_scale, void* stream) {
    return fsta_attention_fwd_kv8_ws(q, k8, v8, k_scale, v_scale, o, lse, block_plan, plan_key_shift, batch, heads, nq, nk,
                                     head_dim, dtype, out_dtype, block_m, max_ancestors, num_blocks, sm_scale, nullptr, 0, stream);
}

extern "C" size_t fsta_attention_kv8_workspace_bytes(int32_t batch, int32_t heads, int32_t nq, int32_t nk, int32_t head_dim,
                                                     int32_t dtype, int32_t block_m, int32_t max_ancestors, float sm_scale) {
    if (batch <= 0 || heads <= 0 || nq <= 0 || nk <= nq || block_m <= 0) return 0;
    const int64_t slices = (int64_t)batch * heads;
    const CachePlan c = plan_cache(slices, nq, nk, head_dim, dtype, block_m, max_ancestors, sm_scale, 0, true);
    return c.runs > 1 ? key_split_bytes(c.runs, slices, nq, head_dim) : 0;
}

extern "C" int fsta_attention_fwd_kv8_ws(const void* q, const void* k8, const void* v8, const float* k_scale,
                                         const float* v_scale, void* o, float* lse, const uint32_t* block_plan,
                                         int32_t plan_key_shift, int32_t batch, int32_t heads, int32_t nq, int32_t nk,
                                         int32_t head_dim, int32_t dtype, int32_t out_dtype, int32_t block_m,
                                         int32_t max_ancestors, int32_t num_blocks, float sm_scale, void* workspace,
                                         size_t workspace_bytes, void* stream) {
    if (batch < 0 || heads < 0 || nq < 0 || nk < nq)
        return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: batch=%d heads=%d nq=%d nk=%d (need nk >= nq >= 0)", batch,
                    heads, nq, nk);
    if (dtype != FSTA_F16 && dtype != FSTA_BF16)
        return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: dtype=%d (q must be float16 or bfloat16)", dtype);
    if (out_dtype != dtype && out_dtype != FSTA_F32)
        return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: out_dtype=%d must equal dtype=%d or be float32", out_dtype, dtype);
    if (head_dim != 64 && head_dim != 128)
        return fail(FSTA_EUNSUPPORTED, "fsta_attention_fwd_kv8: head_dim=%d (supported: 64, 128)", head_dim);
    if (!plan_block_size_ok(block_m))
        return fail(FSTA_EUNSUPPORTED, "fsta_attention_fwd_kv8: block_m=%d (supported: 32, 64, 128)", block_m);
    if (max_ancestors < 1) return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: max_ancestors=%d", max_ancestors);
    if (num_blocks != (nq + block_m - 1) / block_m)
        return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: num_blocks=%d but ceil(nq=%d / block_m=%d) = %d", num_blocks, nq,
                    block_m, (nq + block_m - 1) / block_m);
    if (!(sm_scale > 0.f)) return fail(FSTA_EUNSUPPORTED, "fsta_attention_fwd_kv8: sm_scale must be positive");
    const int64_t slices = (int64_t)batch * heads;
    if (slices > 65535) return fail(FSTA_EUNSUPPORTED, "fsta_attention_fwd_kv8: batch*heads=%lld > 65535", (long long)slices);
    if (slices == 0 || nq == 0) return FSTA_OK;
    if (!q || !k8 || !v8 || !o || !block_plan) return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: null pointer");
    if (misaligned(q, 16) || misaligned(k8, 16) || misaligned(v8, 16) || misaligned(o, 16) || misaligned(block_plan, 16))
        return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: q, k8, v8, o and block_plan must be 16-byte aligned");
    if (misaligned(k_scale, 4) || misaligned(v_scale, 4) || misaligned(lse, 4))
        return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: k_scale, v_scale and lse must be 4-byte aligned");
    if (plan_key_shift < 0 || plan_key_shift > nk)
        return fail(FSTA_EINVAL, "fsta_attention_fwd_kv8: plan_key_shift=%d outside [0, nk=%d]", plan_key_shift, nk);
    AttnParams p;
    p.q = q; p.k = k8; p.v = v8; p.o = o; p.lse = lse;
    p.ancestor_idx = nullptr; p.mask_bits = nullptr; p.anc_count = nullptr; p.leaf_idx = nullptr;
    p.plan = block_plan; p.key_shift = plan_key_shift;
    p.nq = nq; p.nk = nk; p.prefix = nk - nq;
    p.block_m = block_m; p.max_anc = max_ancestors; p.mask_words = fsta_mask_words(max_ancestors);
    p.nb = num_blocks;
    p.heads_total = (int32_t)slices;
    p.out_f32 = (out_dtype == FSTA_F32) ? 1 : 0;
    p.scale_log2e = sm_scale * kLog2e;
    p.key_splits = 1; p.split_tiles = 0; p.part_o = nullptr; p.part_lse = nullptr;
    p.share_tiles = 0;
    p.k_scale = k_scale; p.v_scale = v_scale;
    p.merge_parts = 0; p.dry_run = 0; p.stream_mode = 0;
    const hipStream_t s = static_cast<hipStream_t>(stream);
    const CachePlan c = plan_cache(slices, nq, nk, head_dim, dtype, block_m, max_ancestors, sm_scale, 0, true);
    const int rc = launch_cache(p, dtype, out_dtype, head_dim, true, false, c, workspace, workspace_bytes,
                                c.runs > 1 ? key_split_bytes(c.runs, slices, nq, head_dim) : 0, s);
    if (rc != FSTA_EUNSUPPORTED) return rc;
    return launch_attention_mfma16_kv8(p, dtype, head_dim, s);
}
