// Forward pass of the attention chain, rows of any length in one sweep: o = softmax(q . k^T * scale + key padding) . v over
// the tiles of a line, with a running maximum and sum per row; stores o and, for the backward pass, one float per row.
// Replaces the three operators sdd, softmax, dsd of the reference's modules (deepspeedsparseselfattention.py:152-157;
// attention.py:190-202).
//
// The running maximum moves only when a lane's exponentials of a step, taken relative to the old one, add up to more than
// 8192: until then each of them is at most that, well inside the 16-bit types and with the same relative precision.  So a
// step normally looks for no maximum, exchanges nothing between lanes and leaves the accumulators alone.  Per score: half
// a rounding, one fma, one exponential, an addition, half a conversion.
#include "attention_quad.h"

namespace bsp {
namespace {

template <typename T, int D, bool KPM>
__global__ void __launch_bounds__(128, D == 64 ? 4 : 3) k_attn_fwd(QuadArgs a) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  typedef Quad<D> Q;
  constexpr int MT = D / 32;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  unsigned char *kraw = smem + Q::RING;                 // the stage's 32 key-padding values, 256 bytes a stage
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int64_t wg = xcd_remap(blockIdx.x, (int64_t)a.Z * a.H * a.R);
  int line, zh;
  line_of(wg, a, line, zh);
  const int h = zh % a.H, z = zh / a.H;
  const table_ptr lut = as_table(a.lut);
  const int steps = lut[2 * (h * a.R + line)] * 2;            // halves of tiles
  const table_ptr core = lut + lut[2 * (h * a.R + line) + 1];
  const int64_t row = (int64_t)line * 64 + 32 * wave + l32;
  f32x16 o[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[mt][i] = 0.f;
  float m = -INFINITY, l = 0.f;
  int rows_seen = 0;                                    // bits 0 .. 3: the first sixteen rows have a block, bits 4 .. 7: the others have one

  if (steps > 0) {
    frag_t xq[D / 16];
    load_operand<T, D>(xq, reinterpret_cast<const T *>(a.q) + z * a.q_sz + h * a.q_sh + row * a.q_ld + 8 * half);
    if (a.scale < 0.f) negate<T>(xq);
    const float sc = logit_scale(a.scale);
    const char *pk = reinterpret_cast<const char *>(reinterpret_cast<const T *>(a.k) + z * a.k_sz + h * a.k_sh);
    const char *pv = reinterpret_cast<const char *>(reinterpret_cast<const T *>(a.v) + z * a.v_sz + h * a.v_sh);
    const char *pkpm = reinterpret_cast<const char *>(reinterpret_cast<const T *>(a.kpm) + z * a.kpm_sz);
    GroupLoad<D> gk, gv;
    gk.init(a.k_ld, lane);
    gv.init(a.v_ld, lane);
    // each wavefront loads one of the two groups of sixteen rows of each piece
    auto issue = [&](int stage_no, Groups groups) {
      const uint32_t st = lds_address(smem) + stage_no * Q::STAGE + wave * (32 * D), pos = wave ? groups.hi : groups.lo;
      gk.issue(pk, pos, (uint32_t)a.k_ld * 2u, st);
      gv.issue(pv, pos, (uint32_t)a.v_ld * 2u, st + Q::PIECE);
      if constexpr (KPM) {
        if (wave == 0)                                  // two values a lane; lanes from 16 on fetch them again
          load_to_lds<4>(pkpm, (uint32_t)((lane & 8 ? groups.hi : groups.lo) + 2 * (lane & 7)) * 2u, 0, lds_address(kraw) + stage_no * 256);
      }
    };
    issue(0, half_groups(core, 0));
    // the table runs ahead of the loads: the groups of the next half, the pieces of this one
    Groups groups_next = half_groups(core, 1);
    int bits = core[4];
    RowReads<D, false> rows_k;
    TrReads<D, false> tr_v;
    rows_k.init(0, lane);
    tr_v.init(lds_address(smem), 0, lane);
    // the lane's place among the key-padding values: value i of the lane comes from lane i of each sixteen
    const T *kp_lane = reinterpret_cast<const T *>(kraw) + 16 * ((lane >> 3) & 1) + 8 * half + (lane & 7);

    auto step = [&](auto stage_no, int n) {
      constexpr int S = decltype(stage_no)::value;
      quad_barrier();
      if (n + 1 < steps) issue(1 - S, groups_next);
      Scores<T> raw;
      raw.set(row_product<T, D, S * Q::STAGE>(smem, rows_k, xq));
      const int here = bits >> (8 * wave + 2 * S);      // bit column group, + 4 for the second sixteen rows (S is also the half of the tile)
      // the table a step ahead, behind the product's LDS reads (which would otherwise wait for it)
      bits = half_bits(core, n + 1 < steps ? n + 1 : n);
      groups_next = half_groups(core, n + 2 < steps ? n + 2 : steps - 1);
      rows_seen |= here & 0x33;
      if ((here & 0x33) != 0x33) {                      // pieces without a block take no part in the row
        const int mine = here >> ((lane >> 4) & 1) * 4;
        raw.keep_if(0, mine & 1);
        raw.keep_if(1, mine & 2);
      }
      const float kp = KPM ? kpm_term(kp_lane[S * 128], a.kpm_mul) : 0.f;
      if (KPM && __builtin_amdgcn_ballot_w64(far_padding<T>(kp))) raw.settle(sc, [&](auto ic) { return row_bcast<decltype(ic)::value>(kp); });
      // the exponentials relative to the running maximum as it stands: nearly always it still serves
      float e[16], sum;
      auto exponentials = [&]() {
        const float ms = m == -INFINITY ? 0.f : m;      // (nothing but -inf so far: exp(-inf - 0) = 0)
        sum = 0.f;
        for_16<0>([&](auto ic) {
          constexpr int i = decltype(ic)::value;
          e[i] = __builtin_amdgcn_exp2f(fmaf(raw[i], sc, KPM ? row_bcast<i>(kp) - ms : -ms));
          sum += e[i];
        });
      };
      exponentials();
      if (__builtin_amdgcn_ballot_w64(sum > 8192.f || m == -INFINITY)) {
        float top = -INFINITY;
        for_16<0>([&](auto ic) { top = fmaxf(top, fmaf(raw[decltype(ic)::value], sc, KPM ? row_bcast<decltype(ic)::value>(kp) : 0.f)); });
        const float mn = fmaxf(m, fmaxf(top, swap32(top)));
        const float f = __builtin_amdgcn_exp2f(m - (mn == -INFINITY ? 0.f : mn));
        l *= f;
#pragma unroll
        for (int mt = 0; mt < MT; mt++)
#pragma unroll
          for (int i = 0; i < 16; i++) o[mt][i] *= f;
        m = mn;
        exponentials();
      }
      l += sum;
      frag_t pf[2];
#pragma unroll
      for (int ks = 0; ks < 2; ks++) pf[ks] = pack8<T>(reinterpret_cast<const float (&)[8]>(e[8 * ks]));
      tr_product<T, D, S * Q::STAGE + Q::PIECE>(o, tr_v, pf);
    };
    for (int n = 0; n < steps; n += 2) {
      step(Const<0>{}, n);
      step(Const<1>{}, n + 1);
    }
  }

  l += swap32(l);
  const bool any_block = (rows_seen >> 4 * ((lane >> 4) & 1)) & 15;
  const float inv = any_block ? 1.f / l : 0.f;          // masked everywhere: 0 * inf = NaN, as the softmax operator gives; no block at all: zeros
  if (a.lse != nullptr && half == 0) {
    const float log_l = __builtin_amdgcn_logf(l), lse = m + log_l;
    float *to = a.lse + ((int64_t)z * a.H + h) * a.row_sh + row;
    *to = any_block ? lse : INFINITY;                   // (... and a share of 0 in the backward pass)
    if (a.rest) to[a.rest] = any_block ? row_rest(m, log_l, lse) : 0.f;
  }
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[mt][i] *= inv;
  quad_barrier();                                       // the ring is free
  T *po = reinterpret_cast<T *>(a.o) + z * a.o_sz + h * a.o_sh + ((int64_t)line * 64 + 32 * wave) * a.o_ld;
  store_32_rows<T, D>(reinterpret_cast<T *>(smem) + wave * 32 * (D + 8), po, po + 16 * a.o_ld, a.o_ld, o, lane);
}

template <typename T, int D, bool KPM> int launch_fwd(const QuadArgs &a, hipStream_t st) {
  constexpr int LDS = Quad<D>::RING + (KPM ? 2 * 256 : 0);
  hipLaunchKernelGGL((k_attn_fwd<T, D, KPM>), dim3((unsigned)((int64_t)a.Z * a.H * a.R)), dim3(128), LDS, st, a);
  return BSP_OK;
}

template <typename T> int launch_fwd_t(const QuadArgs &a, int D, hipStream_t st) {
  if (D == 64) return a.kpm ? launch_fwd<T, 64, true>(a, st) : launch_fwd<T, 64, false>(a, st);
  return a.kpm ? launch_fwd<T, 128, true>(a, st) : launch_fwd<T, 128, false>(a, st);
}

}  // namespace
}  // namespace bsp

using namespace bsp;

extern "C" int bsp_attention_rows_fwd(int dtype, const void *q, const void *k, const void *v, void *o, float *lse, int Z, int H, int R, int64_t keys, int D,
                                      int64_t q_stride_z, int64_t q_stride_h, int64_t ldq, int64_t k_stride_z, int64_t k_stride_h, int64_t ldk,
                                      int64_t v_stride_z, int64_t v_stride_h, int64_t ldv, int64_t o_stride_z, int64_t o_stride_h, int64_t ldo,
                                      int64_t lse_stride_h, float scale, const int32_t *d_lut, const void *kpm, int64_t kpm_stride_z, int kpm_mul,
                                      void *stream) {
  const int rest = dtype & BSP_ROWS_WITH_REST ? R * 64 : 0;
  dtype &= ~BSP_ROWS_WITH_REST;
  const void *ptrs[] = {q, k, v, o, kpm};
  const int64_t strides[] = {q_stride_z, q_stride_h, ldq, k_stride_z, k_stride_h, ldk, v_stride_z, v_stride_h, ldv, o_stride_z, o_stride_h, ldo, kpm_stride_z};
  const int64_t lds[] = {ldk, ldv, ldq, ldo};
  if (!q || !k || !v || !o || !d_lut || Z <= 0 || H <= 0 || R <= 0 || (lse && (lse_stride_h < (int64_t)R * 64 + rest || (reinterpret_cast<uintptr_t>(lse) & 15)))) return BSP_ERR_ARG;
  const int rc = quad_check(dtype, D, ptrs, 5, strides, 13, lds, 4, 2, keys, (int64_t)Z * H * R);
  if (rc != BSP_OK) return rc;
  QuadArgs a{};
  a.q = q; a.k = k; a.v = v; a.o = o; a.lse = lse; a.row_sh = lse_stride_h;
  a.rest = rest;
  a.q_sz = q_stride_z; a.q_sh = q_stride_h; a.q_ld = ldq;
  a.k_sz = k_stride_z; a.k_sh = k_stride_h; a.k_ld = ldk;
  a.v_sz = v_stride_z; a.v_sh = v_stride_h; a.v_ld = ldv;
  a.o_sz = o_stride_z; a.o_sh = o_stride_h; a.o_ld = ldo;
  a.scale = scale; a.lut = d_lut;
  a.kpm = kpm; a.kpm_sz = kpm_stride_z; a.kpm_mul = kpm_mul;
  a.Z = Z; a.H = H; a.R = R;
  const int rl = dtype == BSP_F16 ? launch_fwd_t<f16>(a, D, as_stream(stream)) : launch_fwd_t<bf16>(a, D, as_stream(stream));
  if (rl != BSP_OK) return rl;
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}
