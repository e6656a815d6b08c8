// fa_fwd_decode.hip — the forward for decoding: all query rows that read one
// key/value head (query heads of its GQA group x queries) fit one 16-row MFMA
// block (gfx950).
//
// Such a launch reads K and V once and computes next to nothing, so what bounds
// it is the bytes in flight on as many CUs as the key ranges reach. In the
// general tilings the four waves of a work-group own different query rows and
// all walk the same keys, one barrier per 32-key unit: with 16 rows or fewer
// three of them repeat the first one's K and V reads for rows that do not
// exist, and a range moves at one unit per barrier step (0.33 us). Here the rows
// of the whole group are packed into one block and the waves split the keys
// instead: wave w takes every fourth unit of the range through a DMA ring of its
// own, so no barrier runs before the end, where the four partial results are
// merged through LDS. Four units are in work at once and a short range of keys
// ends sooner: B2 Hq32 Hkv8, one query against 3001 keys (D = 128) 23.8 -> 15.4 us
// with its call from Python, B1 Hkv8 2000 keys 26.4 -> 13.6. Large launches read K and
// V at the rate of HBM either way (B8 Hkv8 8192 keys, 268 MB, 44 us).
//
// Layouts as in fwd_pipe16_body (16x16x32 MFMAs, lane l, c16 = l % 16, G = l / 16):
//   S^T block kb: lane holds row c16 and keys 16 kb + 4 gq + j of the unit;
//   O^T block dd: lane holds row c16, d = 16 dd + 4 G + j.
// Row r of the block is query r / P of query head r % P of the group (P heads).
// The softmax is the general one's (fp32, base 2, lazily moved reference max).
#include "fa_common.hpp"
#include "fa_kernels.hpp"

namespace fa {

template <int D>
struct DecodeTile {
  static constexpr int NW = 4;
  static constexpr int KT = 32;              // keys of a unit
  static constexpr int TILE = KT * D;        // halves of its K (or V) rows
  static constexpr int STAGE = 2 * TILE;
  // Ring slots of a wave: 16 KiB units (D = 128) leave room for two; four of 8 KiB
  // at D = 64 are no faster than two and a second work-group on the CU.
  static constexpr int NSTAGE = D == 32 ? 4 : 2;
  static constexpr int LDS_HALVES = NW * NSTAGE * STAGE;  // 128 KiB at D = 128, else 64
  static constexpr int ROWS = kDecodeRows;
  static_assert(ROWS == 16, "one row block");
};

// A row's probabilities are taken against a reference max that moves only when
// their sum over a unit exceeds this (see fwd_kernel's kSumLimit in fa_fwd.hip).
constexpr float kDecodeSumLimit = 256.0f;

template <int D, class E>
__global__ __launch_bounds__(256) void fwd_decode_kernel(FwdArgs a) {
  using T = DecodeTile<D>;
  using Dma = DmaStager<D, T::KT, 1>;
  constexpr int NS = T::NSTAGE;
  constexpr int IPU = 2 * Dma::PER_WAVE;  // a wave's DMA instructions per unit
  constexpr int KD = D / 32, DD = D / 16;
  static_assert((NS - 1) * IPU < 64, "vmcnt range");
  __shared__ __attribute__((aligned(16))) half_t lds[T::LDS_HALVES];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int c16 = lane & 15;
  const int G = lane >> 4;
  const int sg = (4 - G) & 3;   // d chunk order of the k-slots (conflict-free row reads)
  const int gq = quad16<D>(G);  // key quad (of 16) of the lane's result rows

  const int P = a.group;
  const int kv_heads = a.BH / P;
  const int split = blockIdx.x / kv_heads;
  const int kvh = blockIdx.x - split * kv_heads;
  const int b = kvh / a.Hkv;
  const int hkv = kvh - b * a.Hkv;
  const int Nkv = a.Nkv;
  const int4v r_k = make_rsrc_words(a.k + a.kl.head(b, hkv), a.kl.slab_bytes(Nkv, a.d));
  const int4v r_v = make_rsrc_words(a.v + a.kl.head(b, hkv), a.kl.slab_bytes(Nkv, a.d));

  // The lane's row: query n of query head kvh * P + h.
  const bool row_ok = c16 < P * a.N;
  const int n = c16 / P;
  const int h = c16 - n * P;

  // Q^T operand fragments: column = row c16, d = 32 kd + 8 sg .. +7.
  half8 qf[KD];
  {
    const half_t* q = a.q + a.ql.head(b, hkv * P + h) + (int64_t)n * a.ql.row;
#pragma unroll
    for (int kd = 0; kd < KD; ++kd) {
      u32x4 v = {0u, 0u, 0u, 0u};
      const int col = 32 * kd + 8 * sg;
      if (row_ok && col < a.d) v = *reinterpret_cast<const u32x4*>(q + col);
      qf[kd] = __builtin_bit_cast(half8, v);
    }
  }
  wait_all_vm();

  const int kv_lo = split * a.split_keys;
  const int kv_hi = min(Nkv, kv_lo + a.split_keys);
  const int units = kv_hi > kv_lo ? (kv_hi - kv_lo + T::KT - 1) / T::KT : 0;
  const int n_w = units > wave ? (units - wave + T::NW - 1) / T::NW : 0;

  Dma dma;
  dma.init(0, lane, a.kl.row, a.d);
  half_t* const ring = lds + wave * (NS * T::STAGE);
  // Unit i of the wave -> slot i % NS (past its last: rows that read zeros).
  auto issue = [&](int i) __attribute__((always_inline)) {
    const int row0 = i < n_w ? kv_lo + (T::NW * i + wave) * T::KT : Nkv;
    half_t* slot = ring + (i % NS) * T::STAGE;
    dma.issue(r_k, row0, slot, 0);
    dma.issue(r_v, row0, slot + T::TILE, 0);
  };

  // LDS offsets as in fwd_pipe16_body (rows 16 apart differ by a constant).
  int k_off[KD], v_off[DD];
#pragma unroll
  for (int kd = 0; kd < KD; ++kd) k_off[kd] = swz_offset<D>(rows16<D>(c16), 4 * kd + sg);
#pragma unroll
  for (int dd = 0; dd < DD; ++dd) {
    const int row = 4 * gq + (c16 >> 2);
    const int col = 16 * dd + 4 * (c16 & 3);
    v_off[dd] = row * D + 8 * swz_chunk<D>(row, col >> 3) + (col & 7);
  }

  float4v o[DD];
#pragma unroll
  for (int dd = 0; dd < DD; ++dd) o[dd] = {0.f, 0.f, 0.f, 0.f};
  float m = -INFINITY;
  float l = 0.f;
  const float c = a.c;

#pragma unroll
  for (int i = 0; i < NS - 1; ++i) issue(i);
  for (int i = 0; i < n_w; ++i) {
    // The slot of the previous unit is free once its reads have returned.
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    issue(i + NS - 1);
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"((NS - 1) * IPU) : "memory");
    const half_t* Ks = ring + (i % NS) * T::STAGE;
    const half_t* Vs = Ks + T::TILE;
    const int ka = kv_lo + (T::NW * i + wave) * T::KT;

    float4v s[2];
#pragma unroll
    for (int kb = 0; kb < 2; ++kb) {
      s[kb] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
      for (int kd = 0; kd < KD; ++kd)
        s[kb] = mma16<E>(*reinterpret_cast<const half8*>(Ks + 16 * kb * D + k_off[kd]), qf[kd],
                         s[kb]);
    }
    // V^T operands, read ahead of the softmax.
    half8 va[DD];
#pragma unroll
    for (int dd = 0; dd < DD; ++dd) {
      const half4 lo = __builtin_bit_cast(
          half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(Vs + v_off[dd])));
      const half4 hi = __builtin_bit_cast(
          half4, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4*)(Vs + v_off[dd] + 16 * D)));
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        va[dd][e] = lo[e];
        va[dd][4 + e] = hi[e];
      }
    }
    if (ka + T::KT > kv_hi) {
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (ka + 16 * kb + 4 * gq + j >= kv_hi) s[kb][j] = -INFINITY;
    }
    half8 pa;
    auto probs = [&](float ref) {
      float sum = 0.f;
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const float p = exp2_fast(fmaf(s[kb][j], c, -ref));
          sum += p;
          pa[4 * kb + j] = to_elem<E>(p);
        }
      return sum;
    };
    float l_u = probs(m);
    if (__builtin_amdgcn_ballot_w64(!(l_u <= kDecodeSumLimit)) != 0) {
      float mt = s[0][0];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int j = 0; j < 4; ++j) mt = __builtin_fmaxf(mt, s[kb][j]);
      mt = quarters_max(mt) * c;
      const float m_new = __builtin_fmaxf(m, mt);
      const float ref = exp_reference(m_new);
      const float alpha = exp2_fast(m - ref);
      l *= alpha;
#pragma unroll
      for (int dd = 0; dd < DD; ++dd) o[dd] *= alpha;
      m = m_new;
      l_u = probs(ref);
    }
    l += l_u;
#pragma unroll
    for (int dd = 0; dd < DD; ++dd) o[dd] = mma16<E>(va[dd], pa, o[dd]);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // Merge of the waves' results: O, and per row m and l, through the rings.
  __syncthreads();
  float* const xo = reinterpret_cast<float*>(lds);  // [wave][dd][lane][4]
  float* const xm = xo + T::NW * DD * 256;          // [wave][row], m then l
  static_assert(T::NW * DD * 256 + 2 * T::NW * T::ROWS <= T::LDS_HALVES / 2, "exchange fits");
  const float lw = quarters_sum(l);
#pragma unroll
  for (int dd = 0; dd < DD; ++dd)
    *reinterpret_cast<float4v*>(xo + ((wave * DD + dd) * 64 + lane) * 4) = o[dd];
  if (G == 0) {
    xm[wave * T::ROWS + c16] = m;
    xm[(T::NW + wave) * T::ROWS + c16] = lw;
  }
  __syncthreads();
  float mt = -INFINITY;
#pragma unroll
  for (int w = 0; w < T::NW; ++w) mt = __builtin_fmaxf(mt, xm[w * T::ROWS + c16]);
  float wt[T::NW], lt = 0.f;
#pragma unroll
  for (int w = 0; w < T::NW; ++w) {
    const float mw = xm[w * T::ROWS + c16];
    wt[w] = mw == -INFINITY ? 0.f : exp2_fast(mw - mt);  // a wave that saw no key weighs 0
    lt += wt[w] * xm[(T::NW + w) * T::ROWS + c16];
  }
  // A range in which every score is -inf is a partial of weight 0; a row of them is
  // 0 / 0, as in the combine.
  const bool split_mode = a.nsplit > 1;
  const float inv = lt > 0.f || !split_mode ? 1.0f / lt : 0.f;
  const int64_t row = (int64_t)(kvh * P + h) * a.N + n;  // of [B * Hq, N]
  const int64_t prow = (int64_t)split * a.BH * a.N + row;
#pragma unroll
  for (int dd = wave; dd < DD; dd += T::NW) {
    float4v v = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int w = 0; w < T::NW; ++w)
      v += *reinterpret_cast<const float4v*>(xo + ((w * DD + dd) * 64 + lane) * 4) * wt[w];
    v *= inv;
    const int col = 16 * dd + 4 * G;
    if (row_ok) {
      if (split_mode) *reinterpret_cast<float4v*>(a.part + prow * D + col) = v;
      else if (col < a.d)
        *reinterpret_cast<u32x2*>(a.o + row * a.d + col) = pack4<E>(v[0], v[1], v[2], v[3]);
    }
  }
  if (wave == 0 && G == 0 && row_ok) {
    const float lse = lt > 0.f ? mt + log2_fast(lt) : -INFINITY;
    if (split_mode) a.part[(int64_t)a.nsplit * a.BH * a.N * D + prow] = lse;
    else a.lse[row] = lse;
  }
}

template <int D, class E>
hipError_t fwd_decode_launch(const FwdArgs& a, hipStream_t stream) {
  if (a.N < 1 || (int64_t)a.N * a.group > DecodeTile<D>::ROWS || a.nsplit < 1 || (a.nsplit > 1 && a.part == nullptr) || a.split_keys % 128 != 0 ||
      (int64_t)a.nsplit * a.split_keys < a.Nkv)
    return hipErrorInvalidValue;
  const int64_t blocks = (int64_t)(a.BH / a.group) * a.nsplit;
  if (blocks <= 0 || blocks > 0x7fffffff) return hipErrorInvalidConfiguration;
  hipLaunchKernelGGL((fwd_decode_kernel<D, E>), dim3((unsigned)blocks), dim3(256), 0, stream, a);
  return hipGetLastError();
}

hipError_t launch_fwd_decode(const FwdArgs& a, int D, int dtype, hipStream_t stream) {
  const bool bf = dtype == kBF16;
  switch (D) {
    case 32: return bf ? fwd_decode_launch<32, BF16>(a, stream) : fwd_decode_launch<32, F16>(a, stream);
    case 64: return bf ? fwd_decode_launch<64, BF16>(a, stream) : fwd_decode_launch<64, F16>(a, stream);
    case 128: return bf ? fwd_decode_launch<128, BF16>(a, stream) : fwd_decode_launch<128, F16>(a, stream);
    default: return hipErrorInvalidValue;
  }
}

}  // namespace fa
