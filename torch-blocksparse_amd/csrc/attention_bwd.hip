// Backward pass of the attention chain without any sparse tensor: p = exp2(logit - lse) is computed again from q, k and
// the row's lse (its rounding: row_rest), the softmax gradient from it, dp = do . v^T and delta = sum_d do_d o_d (= sum_j p_j dp_j, because o = p . v
// and dp = do . v^T; softmax.py:189, matmul.py:587-606):
//     ds = p * (dp - delta) * scale,   dq = ds . k,   dk = ds^T . q,   dv = p^T . do.
// A scale of at most 1 is applied to the sums dq and dk: as an operand p (dp - delta) stays below half of the largest |dp| (it is
// at most p (1 - p) times the difference of two dp), so it fits the storage type wherever dp itself does.  (Larger: scale_place.)
//   row kernel    : a line of tiles per workgroup -> dq and delta
//   column kernel : a column of tiles (or a part of a long one) per workgroup -> dk and dv
// The two together read q, k, v, do twice and o once; a stored p would be written once and read twice, and is larger
// than all of them from five tiles a row on at head dimension 64.
#include "attention_quad.h"

namespace bsp {
namespace {

template <typename T, int D, bool KPM>
__global__ void __launch_bounds__(128, D == 64 ? 4 : 2) k_attn_bwd_rows(QuadArgs a) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  typedef Quad<D> Q;
  constexpr int MT = D / 32;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  unsigned char *kraw = smem + Q::RING;
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int64_t wg = xcd_remap(blockIdx.x, (int64_t)a.Z * a.H * a.R);
  int line, zh;
  line_of(wg, a, line, zh);
  const int h = zh % a.H, z = zh / a.H;   // as in the forward kernel
  const table_ptr lut = as_table(a.lut);
  const int steps = lut[2 * (h * a.R + line)] * 2;            // halves of tiles
  const table_ptr core = lut + lut[2 * (h * a.R + line) + 1];
  const int64_t row = (int64_t)line * 64 + 32 * wave + l32;
  f32x16 dq[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) dq[mt][i] = 0.f;

  frag_t xo[D / 16];
  load_operand<T, D>(xo, reinterpret_cast<const T *>(a.d_o) + z * a.do_sz + h * a.do_sh + row * a.do_ld + 8 * half);
  float delta = 0.f;
  {
    frag_t of[D / 16];
    load_operand<T, D>(of, reinterpret_cast<const T *>(a.o_in) + z * a.oin_sz + h * a.oin_sh + row * a.oin_ld + 8 * half);
#pragma unroll
    for (int s = 0; s < D / 16; s++)
#pragma unroll
      for (int i = 0; i < 8; i++) delta = fmaf(to_float(xo[s][i]), to_float(of[s][i]), delta);
    delta += swap32(delta);
  }
  if (a.delta != nullptr && half == 0) a.delta[((int64_t)z * a.H + h) * a.row_sh + row] = -delta;   // (its negative: where the column kernel's dp starts from)

  if (steps > 0) {
    frag_t xq[D / 16];
    load_operand<T, D>(xq, reinterpret_cast<const T *>(a.q) + z * a.q_sz + h * a.q_sh + row * a.q_ld + 8 * half);
    if (a.scale < 0.f) negate<T>(xq);
    const bool shifted = __is_same(T, f16) && a.ds_shift != 0.f;
    const float shift = __builtin_amdgcn_exp2f(a.ds_shift);
    const float sc = logit_scale(a.scale), lse = a.lse[((int64_t)z * a.H + h) * a.row_sh + row];
    const char *pk = reinterpret_cast<const char *>(reinterpret_cast<const T *>(a.k) + z * a.k_sz + h * a.k_sh);
    const char *pv = reinterpret_cast<const char *>(reinterpret_cast<const T *>(a.v) + z * a.v_sz + h * a.v_sh);
    const char *pkpm = reinterpret_cast<const char *>(reinterpret_cast<const T *>(a.kpm) + z * a.kpm_sz);
    GroupLoad<D> gk, gv;
    gk.init(a.k_ld, lane);
    gv.init(a.v_ld, lane);
    auto issue = [&](int stage_no, Groups groups) {
      const uint32_t st = lds_address(smem) + stage_no * Q::STAGE + wave * (32 * D), pos = wave ? groups.hi : groups.lo;
      gk.issue(pk, pos, (uint32_t)a.k_ld * 2u, st);
      gv.issue(pv, pos, (uint32_t)a.v_ld * 2u, st + Q::PIECE);
      if constexpr (KPM) {
        if (wave == 0)
          load_to_lds<4>(pkpm, (uint32_t)((lane & 8 ? groups.hi : groups.lo) + 2 * (lane & 7)) * 2u, 0, lds_address(kraw) + stage_no * 256);
      }
    };
    issue(0, half_groups(core, 0));
    Groups groups_next = half_groups(core, 1);
    int bits = core[4];
    RowReads<D, false> rows;                            // the same for the k and the v piece
    TrReads<D, false> tr;
    rows.init(0, lane);
    tr.init(lds_address(smem), 0, lane);
    const T *kp_lane = reinterpret_cast<const T *>(kraw) + 16 * ((lane >> 3) & 1) + 8 * half + (lane & 7);

    auto step = [&](auto stage_no, int n) {
      constexpr int S = decltype(stage_no)::value;
      quad_barrier();
      if (n + 1 < steps) issue(1 - S, groups_next);
      Scores<T> raw;
      raw.set(row_product<T, D, S * Q::STAGE>(smem, rows, xq));
      const f32x16 dp = row_product<T, D, S * Q::STAGE + Q::PIECE>(smem, rows, xo);
      const int here = bits >> (8 * wave + 2 * S);
      bits = half_bits(core, n + 1 < steps ? n + 1 : n);
      groups_next = half_groups(core, n + 2 < steps ? n + 2 : steps - 1);
      if ((here & 0x33) != 0x33) {                      // pieces without a block take no part in the row
        const int mine = here >> ((lane >> 4) & 1) * 4;
        raw.keep_if(0, mine & 1);
        raw.keep_if(1, mine & 2);
      }
      const float kp = KPM ? kpm_term(kp_lane[S * 128], a.kpm_mul) : 0.f;
      if (KPM && __builtin_amdgcn_ballot_w64(far_padding<T>(kp))) raw.settle(sc, [&](auto ic) { return row_bcast<decltype(ic)::value>(kp); });
      float e[16];
      for_16<0>([&](auto ic) {
        constexpr int i = decltype(ic)::value;
        const float p = __builtin_amdgcn_exp2f(fmaf(raw[i], sc, KPM ? row_bcast<i>(kp) - lse : -lse));
        e[i] = p * (dp[i] - delta);
      });
      if (shifted)                                      // (the rest of the scale comes last, on dq)
#pragma unroll
        for (int i = 0; i < 16; i++) e[i] *= shift;
      frag_t df[2];
#pragma unroll
      for (int ks = 0; ks < 2; ks++) df[ks] = pack8<T>(reinterpret_cast<const float (&)[8]>(e[8 * ks]));
      tr_product<T, D, S * Q::STAGE>(dq, tr, df);
    };
    for (int n = 0; n < steps; n += 2) {
      step(Const<0>{}, n);
      step(Const<1>{}, n + 1);
    }
  }
  const float last = a.rest ? a.sum_scale * __builtin_amdgcn_exp2f(-a.lse[((int64_t)z * a.H + h) * a.row_sh + a.rest + row]) : a.sum_scale;
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) dq[mt][i] *= last;
  quad_barrier();                                       // the ring is free
  T *po = reinterpret_cast<T *>(a.o) + z * a.o_sz + h * a.o_sh + ((int64_t)line * 64 + 32 * wave) * a.o_ld;
  store_32_rows<T, D>(reinterpret_cast<T *>(smem) + wave * 32 * (D + 8), po, po + 16 * a.o_ld, a.o_ld, dq, lane);
}

// Columns.  A work item is a column of tiles (64 keys: four groups of sixteen) or a part of a long one: twelve ints (tiles,
// offset of their entries, head, column, slot of its partial sums or -1, ., ., ., the positions of the four groups of
// keys); an entry names the four groups of rows.  A wavefront owns 32 of the keys; its k and v rows stay in registers.
template <typename T, int D, bool KPM>
__global__ void __launch_bounds__(128, D == 64 ? 3 : 2) k_attn_bwd_cols(QuadArgs a) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  typedef Quad<D> Q;
  constexpr int MT = D / 32;
  constexpr bool LEAN = D == 128;                       // dk, dv, k and v alone take 192 registers there
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  unsigned char *rowvals = smem + Q::RING;              // per stage, 128 bytes each: lse of its rows, their rests, their deltas, unused
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5;
  const int64_t wg = xcd_remap(blockIdx.x, (int64_t)a.Z * a.R);
  const int item = (int)(wg % a.R), z = (int)(wg / a.R);
  const table_ptr lut = as_table(a.lut), head = lut + 12 * item;
  const int steps = head[0] * 2, h = head[2], slot = head[4];
  const table_ptr core = lut + head[1];
  const int64_t key_lo = head[8 + 2 * wave], key_hi = head[8 + 2 * wave + 1];
  const bool shifted = __is_same(T, f16) && a.ds_shift != 0.f;
  const float shift = __builtin_amdgcn_exp2f(a.ds_shift), unshift = __builtin_amdgcn_exp2f(-a.ds_shift);
  f32x16 dk[MT], dv[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) dk[mt][i] = dv[mt][i] = 0.f;

  if (steps > 0) {
    const int64_t key = (l32 < 16 ? key_lo : key_hi) + (l32 & 15);
    frag_t xk[D / 16], xv[D / 16];
    load_operand<T, D>(xk, reinterpret_cast<const T *>(a.k) + z * a.k_sz + h * a.k_sh + key * a.k_ld + 8 * half);
    load_operand<T, D>(xv, reinterpret_cast<const T *>(a.v) + z * a.v_sz + h * a.v_sh + key * a.v_ld + 8 * half);
    if (a.scale < 0.f) negate<T>(xk);
    const float sc = logit_scale(a.scale);
    float kp = 0.f;
    if constexpr (KPM) kp = kpm_term((reinterpret_cast<const T *>(a.kpm) + z * a.kpm_sz)[key], a.kpm_mul);
    const char *pq = reinterpret_cast<const char *>(reinterpret_cast<const T *>(a.q) + z * a.q_sz + h * a.q_sh);
    const char *pdo = reinterpret_cast<const char *>(reinterpret_cast<const T *>(a.d_o) + z * a.do_sz + h * a.do_sh);
    const char *prow = reinterpret_cast<const char *>((wave == 0 ? a.lse : a.delta) + ((int64_t)z * a.H + h) * a.row_sh);
    const bool far = KPM && __builtin_amdgcn_ballot_w64(far_padding<T>(kp));
    const uint32_t to_rest = wave == 0 && half ? (uint32_t)a.rest * 4u : 0u;
    GroupLoad<D, LEAN> gq, gdo;
    gq.init(a.q_ld, lane);
    gdo.init(a.do_ld, lane);
    auto issue = [&](int stage_no, Groups groups) {
      const uint32_t st = lds_address(smem) + stage_no * Q::STAGE + wave * (32 * D), pos = wave ? groups.hi : groups.lo;
      gq.issue(pq, pos, (uint32_t)a.q_ld * 2u, st);
      gdo.issue(pdo, pos, (uint32_t)a.do_ld * 2u, st + Q::PIECE);
      // one wavefront the lse of the stage's 32 rows and (the upper lanes) their rests, one their -delta (twice)
      load_to_lds<4>(prow, (uint32_t)((lane & 16 ? groups.hi : groups.lo) + (lane & 15)) * 4u + to_rest, 0, lds_address(rowvals) + stage_no * 512 + wave * 256);
    };
    issue(0, half_groups(core, 0));
    Groups groups_next = half_groups(core, 1);
    int bits = core[4];
    RowReads<D, LEAN> rows;                             // the same for the q and the do piece
    TrReads<D, LEAN> tr;
    rows.init(0, lane);
    tr.init(lds_address(smem), 0, lane);
    const float *rv_half = reinterpret_cast<const float *>(rowvals) + 8 * half;   // the lane's rows: 8 half .., 16 + 8 half ..

    auto step = [&](auto stage_no, int n) {
      constexpr int S = decltype(stage_no)::value, Q0 = S * Q::STAGE, O0 = Q0 + Q::PIECE;
      quad_barrier();
      if (n + 1 < steps) issue(1 - S, groups_next);
      const bool some_rest = a.rest && __builtin_amdgcn_ballot_w64(reinterpret_cast<const float *>(rowvals)[S * 128 + 32 + l32] != 0.f);   // (of row l32 of the stage's 32)
      Scores<T> raw;
      raw.set(row_product<T, D, Q0>(smem, rows, xk));
      if (far) raw.settle(sc, [&](auto) { return kp; });
      const int here = bits >> (2 * wave + 8 * S);      // bit 4 * row group + column group; the wavefront's column groups are 2 wave, 2 wave + 1
      bits = half_bits(core, n + 1 < steps ? n + 1 : n);
      groups_next = half_groups(core, n + 2 < steps ? n + 2 : steps - 1);
      // Pieces without a block: their shares and softmax gradients are set to zero once they are operands.  (A score of -inf
      // is not enough: in a row that is masked everywhere lse or delta is not a number, and the keys of such a piece, which
      // the row does not attend to, would take it up.)
      const bool holes = (here & 0x33) != 0x33;
      // The rows' values are read into as many registers as there are scores (two addresses a read, which costs the LDS
      // little): lse is what the scaled scores are added to, -delta where the product dp starts.
      const float *rv = rv_half + S * 128;
      float p[16], e[16];
      frag_t pf[2], df[2];
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x4 lse = *reinterpret_cast<const f32x4 *>(rv + 16 * (g >> 1) + 4 * (g & 1));
#pragma unroll
        for (int i = 0; i < 4; i++) p[4 * g + i] = __builtin_amdgcn_exp2f(fmaf(raw[4 * g + i], sc, KPM ? kp - lse[i] : -lse[i]));
      }
      if (some_rest) {
#pragma unroll
        for (int g = 0; g < 4; g++) {
          const f32x4 rest = *reinterpret_cast<const f32x4 *>(rv + 32 + 16 * (g >> 1) + 4 * (g & 1));
#pragma unroll
          for (int i = 0; i < 4; i++) p[4 * g + i] *= __builtin_amdgcn_exp2f(-rest[i]);
        }
      }
      if (shifted)                                      // (dv is scaled back at the end)
#pragma unroll
        for (int i = 0; i < 16; i++) p[i] *= shift;
#pragma unroll
      for (int ks = 0; ks < 2; ks++) pf[ks] = pack8<T>(reinterpret_cast<const float (&)[8]>(p[8 * ks]));
      if (holes) {
        zero_unless(pf[0], here);
        zero_unless(pf[1], here >> 4);
      }
      tr_product<T, D, O0>(dv, tr, pf);
      f32x16 dp;
#pragma unroll
      for (int g = 0; g < 4; g++) {
        const f32x4 nd = *reinterpret_cast<const f32x4 *>(rv + 64 + 16 * (g >> 1) + 4 * (g & 1));
#pragma unroll
        for (int i = 0; i < 4; i++) dp[4 * g + i] = nd[i];
      }
      dp = row_product<T, D, O0>(smem, rows, xv, dp);
#pragma unroll
      for (int i = 0; i < 16; i++) e[i] = p[i] * dp[i]; // (the rest of the scale comes last, on dk)
#pragma unroll
      for (int ks = 0; ks < 2; ks++) df[ks] = pack8<T>(reinterpret_cast<const float (&)[8]>(e[8 * ks]));
      if (LEAN || holes) {                              // (a branch here costs registers that the wide head does not have)
        zero_unless(df[0], here);
        zero_unless(df[1], here >> 4);
      }
      tr_product<T, D, Q0>(dk, tr, df);
    };
    for (int n = 0; n < steps; n += 2) {
      step(Const<0>{}, n);
      step(Const<1>{}, n + 1);
    }
  }

#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) {
      dk[mt][i] *= a.sum_scale;
      if constexpr (__is_same(T, f16)) dv[mt][i] *= unshift;
    }
  if (slot >= 0) {                                      // a part of a long column: fp32 sums to its slot [dk, dv][64 keys][D]
    float *ws = a.partial + ((int64_t)z * a.n_slots + slot) * (2 * 64 * D) + (32 * wave + l32) * D + 4 * half;
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        *reinterpret_cast<f32x4 *>(ws + 32 * j + 8 * g) = f32x4{dk[j][4 * g], dk[j][4 * g + 1], dk[j][4 * g + 2], dk[j][4 * g + 3]};
        *reinterpret_cast<f32x4 *>(ws + 64 * D + 32 * j + 8 * g) = f32x4{dv[j][4 * g], dv[j][4 * g + 1], dv[j][4 * g + 2], dv[j][4 * g + 3]};
      }
    return;
  }
  quad_barrier();                                       // the ring is free
  T *stage = reinterpret_cast<T *>(smem) + wave * 32 * (D + 8);
  T *pdk = reinterpret_cast<T *>(a.o) + z * a.o_sz + h * a.o_sh, *pdv = reinterpret_cast<T *>(a.o2) + z * a.o2_sz + h * a.o2_sh;
  store_32_rows<T, D>(stage, pdk + key_lo * a.o_ld, pdk + key_hi * a.o_ld, a.o_ld, dk, lane);
  store_32_rows<T, D>(stage, pdv + key_lo * a.o2_ld, pdv + key_hi * a.o2_ld, a.o2_ld, dv, lane);
}

// dk and dv of the columns computed in parts: the sum of the parts' slots in order.  split_lut: per such column eight ints
// (head, column, first slot, parts, the positions of its four groups of keys).
template <typename T, int D> __global__ void __launch_bounds__(256) k_attn_bwd_cols_sum(QuadArgs a) {
  constexpr int PER = 64 * D / 4, WGS = 2 * PER / 512;   // four values a thread, two of them per thread
  const int piece = blockIdx.x % WGS, col = (blockIdx.x / WGS) % a.n_split, z = (blockIdx.x / WGS) / a.n_split;
  const table_ptr lut = as_table(a.split_lut) + 8 * col;
  const int h = lut[0], first = lut[2], parts = lut[3];
  const float *ws = a.partial + ((int64_t)z * a.n_slots + first) * (2 * 64 * D);
#pragma unroll
  for (int t = 0; t < 2; t++) {
    const int g = (piece * 2 + t) * 256 + threadIdx.x, which = g / PER, rem = g % PER, key = rem / (D / 4), d4 = rem % (D / 4);
    f32x4 sum = *reinterpret_cast<const f32x4 *>(ws + 4 * g);
    for (int part = 1; part < parts; part++) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>(ws + (int64_t)part * (2 * 64 * D) + 4 * g);
#pragma unroll
      for (int e = 0; e < 4; e++) sum[e] += v[e];
    }
    union { u32x2 raw; T e[4]; } pk;
#pragma unroll
    for (int e = 0; e < 4; e++) pk.e[e] = from_float<T>(sum[e]);
    const int64_t pos = (key < 32 ? (key < 16 ? lut[4] : lut[5]) : (key < 48 ? lut[6] : lut[7])) + (key & 15);
    T *dst = which ? reinterpret_cast<T *>(a.o2) + z * a.o2_sz + h * a.o2_sh + pos * a.o2_ld
                   : reinterpret_cast<T *>(a.o) + z * a.o_sz + h * a.o_sh + pos * a.o_ld;
    *reinterpret_cast<u32x2 *>(dst + 4 * d4) = pk.raw;
  }
}

template <typename T, int D, bool KPM> int launch_rows(const QuadArgs &a, hipStream_t st) {
  constexpr int LDS = Quad<D>::RING + (KPM ? 2 * 256 : 0);
  hipLaunchKernelGGL((k_attn_bwd_rows<T, D, KPM>), dim3((unsigned)((int64_t)a.Z * a.H * a.R)), dim3(128), LDS, st, a);
  return BSP_OK;
}

template <typename T, int D, bool KPM> int launch_cols(const QuadArgs &a, hipStream_t st) {
  constexpr int LDS = Quad<D>::RING + 2 * 512;
  hipLaunchKernelGGL((k_attn_bwd_cols<T, D, KPM>), dim3((unsigned)((int64_t)a.Z * a.R)), dim3(128), LDS, st, a);
  if (a.n_split > 0)
    hipLaunchKernelGGL((k_attn_bwd_cols_sum<T, D>), dim3((unsigned)((int64_t)a.Z * a.n_split * (2 * 64 * D / 4 / 512))), dim3(256), 0, st, a);
  return BSP_OK;
}

template <typename T> int launch_t(const QuadArgs &a, int D, bool cols, hipStream_t st) {
  if (D == 64) return cols ? (a.kpm ? launch_cols<T, 64, true>(a, st) : launch_cols<T, 64, false>(a, st))
                           : (a.kpm ? launch_rows<T, 64, true>(a, st) : launch_rows<T, 64, false>(a, st));
  return cols ? (a.kpm ? launch_cols<T, 128, true>(a, st) : launch_cols<T, 128, false>(a, st))
              : (a.kpm ? launch_rows<T, 128, true>(a, st) : launch_rows<T, 128, false>(a, st));
}

}  // namespace
}  // namespace bsp

using namespace bsp;

extern "C" int bsp_attention_rows_bwd(int dtype, const void *d_o, const void *q, const void *k, const void *v, const void *o, const float *lse,
                                      void *dq, float *neg_delta, int Z, int H, int R, int64_t keys, int D, int64_t do_stride_z, int64_t do_stride_h, int64_t lddo,
                                      int64_t q_stride_z, int64_t q_stride_h, int64_t ldq, int64_t k_stride_z, int64_t k_stride_h, int64_t ldk,
                                      int64_t v_stride_z, int64_t v_stride_h, int64_t ldv, int64_t o_stride_z, int64_t o_stride_h, int64_t ldo,
                                      int64_t dq_stride_z, int64_t dq_stride_h, int64_t lddq, int64_t row_stride_h, float scale,
                                      const int32_t *d_lut, const void *kpm, int64_t kpm_stride_z, int kpm_mul, void *stream) {
  const int rest = dtype & BSP_ROWS_WITH_REST ? R * 64 : 0;
  dtype &= ~BSP_ROWS_WITH_REST;
  const void *ptrs[] = {d_o, q, k, v, o, dq, kpm, lse, neg_delta};
  const int64_t strides[] = {do_stride_z, do_stride_h, lddo, q_stride_z, q_stride_h, ldq, k_stride_z, k_stride_h, ldk, v_stride_z, v_stride_h, ldv,
                             o_stride_z, o_stride_h, ldo, dq_stride_z, dq_stride_h, lddq, kpm_stride_z};
  const int64_t lds[] = {ldk, ldv, lddo, ldq, ldo, lddq};
  if (!d_o || !q || !k || !v || !o || !lse || !dq || !d_lut || Z <= 0 || H <= 0 || R <= 0 || row_stride_h < (int64_t)R * 64 + rest) return BSP_ERR_ARG;
  const int rc = quad_check(dtype, D, ptrs, 9, strides, 19, lds, 6, 2, keys, (int64_t)Z * H * R);
  if (rc != BSP_OK) return rc;
  QuadArgs a{};
  a.d_o = d_o; a.q = q; a.k = k; a.v = v; a.o_in = o; a.o = dq;
  a.lse = const_cast<float *>(lse); a.delta = neg_delta; a.row_sh = row_stride_h;
  a.rest = rest;
  a.do_sz = do_stride_z; a.do_sh = do_stride_h; a.do_ld = lddo;
  a.q_sz = q_stride_z; a.q_sh = q_stride_h; a.q_ld = ldq;
  a.k_sz = k_stride_z; a.k_sh = k_stride_h; a.k_ld = ldk;
  a.v_sz = v_stride_z; a.v_sh = v_stride_h; a.v_ld = ldv;
  a.oin_sz = o_stride_z; a.oin_sh = o_stride_h; a.oin_ld = ldo;
  a.o_sz = dq_stride_z; a.o_sh = dq_stride_h; a.o_ld = lddq;
  a.scale = scale; a.lut = d_lut;
  scale_place(a, dtype);
  a.kpm = kpm; a.kpm_sz = kpm_stride_z; a.kpm_mul = kpm_mul;
  a.Z = Z; a.H = H; a.R = R;
  const int rl = dtype == BSP_F16 ? launch_t<f16>(a, D, false, as_stream(stream)) : launch_t<bf16>(a, D, false, as_stream(stream));
  if (rl != BSP_OK) return rl;
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}

extern "C" int bsp_attention_cols_bwd(int dtype, const void *d_o, const void *q, const void *k, const void *v, const float *lse, const float *neg_delta,
                                      void *dk, void *dv, int Z, int H, int C, int64_t rows, int D, int64_t do_stride_z, int64_t do_stride_h, int64_t lddo,
                                      int64_t q_stride_z, int64_t q_stride_h, int64_t ldq, int64_t k_stride_z, int64_t k_stride_h, int64_t ldk,
                                      int64_t v_stride_z, int64_t v_stride_h, int64_t ldv, int64_t dk_stride_z, int64_t dk_stride_h, int64_t lddk,
                                      int64_t dv_stride_z, int64_t dv_stride_h, int64_t lddv, int64_t row_stride_h, float scale,
                                      const int32_t *d_items, int n_items, float *partial, int n_slots, const int32_t *d_split, int n_split,
                                      const void *kpm, int64_t kpm_stride_z, int kpm_mul, void *stream) {
  const int64_t rest = dtype & BSP_ROWS_WITH_REST ? rows : 0;
  dtype &= ~BSP_ROWS_WITH_REST;
  const void *ptrs[] = {d_o, q, k, v, dk, dv, kpm, lse, neg_delta, partial};
  const int64_t strides[] = {do_stride_z, do_stride_h, lddo, q_stride_z, q_stride_h, ldq, k_stride_z, k_stride_h, ldk, v_stride_z, v_stride_h, ldv,
                             dk_stride_z, dk_stride_h, lddk, dv_stride_z, dv_stride_h, lddv, kpm_stride_z};
  const int64_t lds[] = {lddo, ldq, ldk, ldv, lddk, lddv};
  if (!d_o || !q || !k || !v || !lse || !neg_delta || !dk || !dv || !d_items || Z <= 0 || H <= 0 || C <= 0 || n_items < H * C) return BSP_ERR_ARG;
  if (n_slots < 0 || n_split < 0 || (n_slots > 0) != (n_split > 0) || (n_slots > 0 && (!partial || !d_split)) || n_items > H * C + n_slots) return BSP_ERR_ARG;
  if (row_stride_h < rows + rest) return BSP_ERR_ARG;
  const int rc = quad_check(dtype, D, ptrs, 10, strides, 19, lds, 6, 2, rows, (int64_t)Z * n_items + (int64_t)Z * n_split * 16);
  if (rc != BSP_OK) return rc;
  QuadArgs a{};
  a.d_o = d_o; a.q = q; a.k = k; a.v = v; a.o = dk; a.o2 = dv;
  a.lse = const_cast<float *>(lse); a.delta = const_cast<float *>(neg_delta); a.row_sh = row_stride_h;
  a.rest = rest;
  a.do_sz = do_stride_z; a.do_sh = do_stride_h; a.do_ld = lddo;
  a.q_sz = q_stride_z; a.q_sh = q_stride_h; a.q_ld = ldq;
  a.k_sz = k_stride_z; a.k_sh = k_stride_h; a.k_ld = ldk;
  a.v_sz = v_stride_z; a.v_sh = v_stride_h; a.v_ld = ldv;
  a.o_sz = dk_stride_z; a.o_sh = dk_stride_h; a.o_ld = lddk;
  a.o2_sz = dv_stride_z; a.o2_sh = dv_stride_h; a.o2_ld = lddv;
  a.scale = scale; scale_place(a, dtype);
  a.lut = d_items; a.partial = partial; a.n_slots = n_slots; a.split_lut = d_split; a.n_split = n_split;
  a.kpm = kpm; a.kpm_sz = kpm_stride_z; a.kpm_mul = kpm_mul;
  a.Z = Z; a.H = H; a.R = n_items;
  const int rl = dtype == BSP_F16 ? launch_t<f16>(a, D, true, as_stream(stream)) : launch_t<bf16>(a, D, true, as_stream(stream));
  if (rl != BSP_OK) return rl;
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}
