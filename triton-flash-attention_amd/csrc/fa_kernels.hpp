// fa_kernels.hpp — argument blocks and launcher registry shared by the
// kernel translation units and the C ABI (fa_capi.hip).
#pragma once

#include <hip/hip_runtime.h>
#include <stddef.h>
#include <stdint.h>

namespace fa {

typedef _Float16 half_t;

// 1 / ln(2): converts natural-log scores to the base-2 domain (attention.py:20).
constexpr float kLog2e = 1.4426950408889634f;

// A persistent causal forward's job plan (the launch takes it by value): the
// grid has ngroups * nbin work-groups; work-group s serves head group
// s % ngroups and runs the jobs job[start[b] .. start[b + 1]) of bin
// b = s / ngroups in order. A job is hoff * kTileLimit + qtile: query tile
// qtile of the head at tile-row position ngroups * hoff + s % ngroups.
struct FwdJobs {
  static constexpr int kMaxBins = 64;
  static constexpr int kMaxJobs = 256;
  static constexpr int kTileLimit = 1 << 16;
  int ngroups;
  int nbin;
  int start[kMaxBins + 1];
  int job[kMaxJobs];
};

// How input tensors [B, H, N, columns] lie in memory: the columns of a row are
// consecutive; batches lie `sb` elements apart, heads 8 * `sh8` and rows `row`
// (all multiples of 8, row >= columns: the kernels move 16-byte chunks). The two
// tensors that a kernel reads side by side (k and v, q and dO) have one layout, so
// that they share a work-group's address arithmetic and, in the loop, an offset
// register; the head stride is held in 32 bits. Each work-group does this
// arithmetic before its first load: with a layout and 64-bit strides for each of the
// four tensors the dK/dV launch of B2 H16, 64 queries against 16384 keys (D = 64),
// 4096 work-groups of two units each, took 76.8 us instead of 72.3, and with two
// offset registers its bf16 causal build spilled.
struct Layout {
  int64_t sb;
  uint32_t sh8;
  int row;

  // Elements from the tensor's first to the first of head h of batch b.
  __host__ __device__ uint64_t head(uint32_t b, uint32_t h) const {
    return (uint64_t)b * (uint64_t)sb + ((uint64_t)h * sh8 << 3);
  }
  // Bytes from a head's first element past its last one, of n rows of `cols`
  // columns: a buffer of that size reads zeros for rows >= n.
  __host__ __device__ uint32_t slab_bytes(int n, int cols) const {
    return ((uint32_t)(n - 1) * (uint32_t)row + (uint32_t)cols) * 2u;
  }
};

// Arguments of one forward launch (the values _attn_fwd receives at
// attention.py:690-718). The kernel of width D serves any head size d <= D that
// is a multiple of 8: columns past it read as zeros (their 16-byte chunks take
// an out-of-range offset) and are not stored.
// The fields are ordered so that the first ones a kernel reads (num_tiles, BH, pack)
// touch both 64-byte lines of the arguments at once: read one after the other, each
// line is a miss of the scalar cache in the prologue of a new launch.
struct FwdArgs {
  int num_tiles;   // filled in by the launcher
  int N;           // query sequence length
  int Nkv;         // key/value sequence length (== N for self-attention)
  int Hq, Hkv;     // query heads, key/value heads
  int group;       // Hq / Hkv
  int d;           // columns of q, k, v and o
  float c;         // scale * log2(e)
  const half_t* q;
  const half_t* k;
  const half_t* v;
  float* lse;
  // --- second line ---
  int BH;          // B * Hq
  // Query heads per work-group. 1: a work-group serves 32 * NW query rows of
  // one head. pack > 1 (GQA, pack dividing both the group and NW): it serves
  // 32 * NW / pack rows of `pack` consecutive query heads of one key/value
  // head, wave w taking head w % pack and rows 32 * (w / pack) onward, so the
  // heads share each K/V tile the work-group streams.
  int pack;
  // Split-KV mode (nsplit > 1): work-group split s covers keys
  // [s * split_keys, (s + 1) * split_keys) and writes its fp32 partial O
  // ([nsplit, BH, N, D], normalised by its own row sums) and base-2 LSE
  // ([nsplit, BH, N], -inf where it saw no key) to `part`;
  // launch_fwd_combine merges them. The ranges together cover the keys some
  // query sees (visible_kv: all Nkv, or min(N, Nkv) under the causal mask).
  // nsplit = 1: split_keys >= Nkv, part unused.
  int nsplit;
  int split_keys;  // a multiple of 128
  Layout ql;       // of q
  Layout kl;       // of k and v
  half_t* o;       // contiguous [B, Hq, N, d]
  float* part;
  // Host-side plan of the persistent forward variant (kJobs); its launcher
  // passes *jobs to the kernel by value. Unused by the other variants.
  const FwdJobs* jobs = nullptr;
};
static_assert(offsetof(FwdArgs, BH) == 64 && offsetof(FwdArgs, jobs) == 128, "two lines");

// Arguments of the backward launches (attention.py:736-770).
// Ordered as FwdArgs: num_tiles and BH or BHkv touch the first two lines; the third is
// for the epilogues and the fused Delta.
struct BwdArgs {
  int num_tiles;   // filled in by the launcher
  int N;           // query sequence length
  int Nkv;         // key/value sequence length (== N for self-attention)
  int Hq, Hkv, group;
  int d;           // columns of every tensor (see FwdArgs)
  // dK/dV split mode (nsplit > 1): work-group (tile, head, split) covers one
  // contiguous chunk of its key tile's (query head, query tile) steps and
  // writes fp32 partials part[split][B*Hkv][N][D] (dK then dV planes).
  int nsplit;
  const half_t* q;
  const half_t* k;
  const half_t* v;
  const half_t* dO;
  // --- second line ---
  int BH;          // B * Hq
  int BHkv;        // B * Hkv
  // dQ split mode (nsplit > 1 in a dQ launch): work-group split s covers keys
  // [s * split_keys, (s + 1) * split_keys) and writes its fp32 partial dQ
  // (scaled) to part[split][B*Hq][N][D]; launch_split_sum adds them. The
  // ranges cover visible_kv keys; with nsplit = 1, split_keys >= Nkv. Unused
  // by the dK/dV launches.
  int split_keys;
  float c;         // scale * log2(e)
  Layout ql;       // of q and dO
  Layout kl;       // of k and v
  const float* lse;
  const float* delta;
  // --- third line ---
  // Fused Delta (dQ kernels whose variant has kFusesDelta): when o is set the
  // kernel computes Delta = rowsum(O * dO) itself and writes it to delta_out
  // instead of reading delta. o is contiguous [B, Hq, N, d].
  const half_t* o;
  float* delta_out;
  half_t* dq;      // contiguous [B, Hq, N, d]
  half_t* dk;      // contiguous [B, Hkv, Nkv, d]
  half_t* dv;      // contiguous [B, Hkv, Nkv, d]
  float* part;
  float scale;
};
static_assert(offsetof(BwdArgs, BH) == 64 && offsetof(BwdArgs, o) == 128, "lines");

// Keys some query can see, which a split launch's key ranges must cover: all
// Nkv, or under the top-left causal mask the first min(N, Nkv) (query i sees
// keys j <= i; the keys after them are masked for every query).
template <bool CAUSAL, class Args>
inline int64_t visible_kv(const Args& a) {
  return CAUSAL && a.N < a.Nkv ? a.N : a.Nkv;
}

enum KernelKind { kFwd = 0, kDkdv = 1, kDq = 2, kNumKinds = 3 };

typedef hipError_t (*fwd_launch_fn)(const FwdArgs&, hipStream_t);
typedef hipError_t (*bwd_launch_fn)(const BwdArgs&, hipStream_t);

// One compiled tiling of a kernel, for every (D, causal).
// rows = rows owned by a work-group (queries for fwd/dq, keys for dkdv),
// tile = length of the streamed tile (keys for fwd/dq, queries for dkdv).
struct Variant {
  int waves;
  int rows;
  int tile;
  void* fn[2][3][2];  // [element type: fp16, bf16][D index: 32, 64, 128][causal]; null = not compiled
  int flags;          // kFusesDelta, kSplitsKv, kPairs, kKeyGroups, kJobs, kFewSplits, kLateSplit
  int per_cu = 0;     // kJobs: work-groups resident per CU (the plan's slots per CU)
};

// Element type index of Variant::fn.
enum DType { kF16 = 0, kBF16 = 1 };

// The six launchers (D = 32, 64, 128; bidirectional, causal) of one tiling
// ENTRY<D, causal, args..., E>(), and an empty table.
#define FA_ENTRIES(ENTRY, E, ...)                                              \
  {{ENTRY<32, false, __VA_ARGS__, E>(), ENTRY<32, true, __VA_ARGS__, E>()},    \
   {ENTRY<64, false, __VA_ARGS__, E>(), ENTRY<64, true, __VA_ARGS__, E>()},    \
   {ENTRY<128, false, __VA_ARGS__, E>(), ENTRY<128, true, __VA_ARGS__, E>()}}
#define FA_NO_ENTRIES {{nullptr, nullptr}, {nullptr, nullptr}, {nullptr, nullptr}}

// The dQ variant can compute Delta itself (BwdArgs::o / delta_out).
constexpr int kFusesDelta = 1;
// The forward variant has the split-KV mode (FwdArgs::nsplit > 1).
constexpr int kSplitsKv = 2;
// The backward variant (pipelined dK/dV or dQ, D <= 64) also runs in the
// combined launch of bwd_pair_launcher.
constexpr int kPairs = 4;
// The forward variant splits each work-group's keys over two wave groups
// (one query head per work-group: no packed GQA).
constexpr int kKeyGroups = 8;
// The forward variant runs a causal one-pass launch as a persistent grid when
// the host attaches a job plan (FwdArgs::jobs), else as the grid form.
constexpr int kJobs = 16;
// The forward variant's split-KV launches at D >= 64 aim at one work-group per
// CU (fewer, longer key ranges) instead of three.
constexpr int kFewSplits = 32;
// The forward variant splits its keys into ranges only up to 256 work-groups
// (at D = 128 and without the mask); the others below 512.
constexpr int kLateSplit = 64;

// Most key ranges a split-KV forward uses; its merge holds one partial per
// range in registers.
constexpr int kMaxFwdSplitKv = 32;

// Registries defined in the kernel translation units.
const Variant* fwd_variants(int* count);
const Variant* dkdv_variants(int* count);
const Variant* dq_variants(int* count);

// Combined dK/dV + dQ launch (fa_bwd_pair.hip): `dkdv` as for the pipelined
// dK/dV launch (split mode allowed), `dq` as for the pipelined dQ launch in one
// pass that reads Delta (o == nullptr). Null for head sizes other than 32, 64.
typedef hipError_t (*bwd_pair_launch_fn)(const BwdArgs& dkdv, const BwdArgs& dq, hipStream_t);
bwd_pair_launch_fn bwd_pair_launcher(int dtype, int di, int causal);
// Waves per work-group of the combined launch (both kinds' tiling).
int bwd_pair_waves();

// Sum of the nsplit fp32 partial planes (`rows` rows of D values each for dK, then
// dV) into 16-bit dK, dV of d columns (fixed order).
// dtype: kF16 or kBF16 (the element type of the 16-bit tensors).
hipError_t launch_split_reduce(const float* part, half_t* dk, half_t* dv, int64_t rows, int D,
                               int d, int nsplit, int dtype, hipStream_t stream);

// Delta of o (contiguous) and dO, B x H heads of N rows of cols columns, by the
// kernel of width D.
hipError_t launch_preprocess(const half_t* o, const half_t* dO, const Layout& dol, float* delta,
                             int64_t B, int64_t H, int64_t N, int D, int cols, int dtype,
                             hipStream_t stream);

// Sum of nsplit fp32 partial planes of `rows` rows of D values into 16-bit `out` of
// `cols` columns.
hipError_t launch_split_sum(const float* part, half_t* out, int64_t rows, int D, int cols,
                            int nsplit, int dtype, hipStream_t stream);

// The forward for launches whose query rows per key/value head (group x N) are at
// most kDecodeRows, without the mask (fa_fwd_decode.hip); pack is unused.
constexpr int kDecodeRows = 16;
hipError_t launch_fwd_decode(const FwdArgs& a, int D, int dtype, hipStream_t stream);

// Columns that the pipelined bodies of width 128 work on where the head size is at
// most that: the last 32, which hold zeros, take no MFMAs, LDS reads or accumulators
// (a quarter of each; the LDS layout and the DMA stay those of 128). The results are
// the same bit for bit. MI355X, B4 H16 N1025 D80 bf16 bidirectional, a training step:
// 234.9 -> 201.5 us. Between 97 and 128 all four 32-column blocks hold columns; a
// 64-wide call has no whole block to leave out between 33 and 64.
constexpr int kUsed96 = 96;

// Merge of the forward's nsplit partials (FwdArgs::part) into O (16-bit) and
// base-2 LSE, rows = B * Hq * N: O = sum_s w_s O_s / sum_s w_s with
// w_s = exp2(lse_s - max_s lse_s), LSE = max + log2(sum_s w_s).
// The partials have D columns, o the first `cols` of them.
hipError_t launch_fwd_combine(const float* part, half_t* o, float* lse, int64_t rows, int D,
                              int cols, int nsplit, int dtype, hipStream_t stream);

inline int log2_of(int x) {
  int s = 0;
  while ((1 << s) < x) ++s;
  return s;
}

inline int head_dim_index(int64_t D) {
  return D == 32 ? 0 : D == 64 ? 1 : D == 128 ? 2 : -1;
}

}  // namespace fa
