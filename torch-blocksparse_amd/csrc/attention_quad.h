// Shared pieces of the attention kernels that keep no sparse tensor between the passes (attention_fwd.hip,
// attention_bwd.hip): scores and softmax of a 64 x 64 tile are computed where they are needed, from q, k and one float
// per row (the logarithm of the row's sum of exponentials), so the [Z, nnz, block, block] tensors of the chain never
// exist in memory.
//
// Tiles.  A tile is 64 rows by 64 columns of the score matrix, each side made of four groups of sixteen consecutive
// positions that may lie anywhere: blocks of 64 give four neighbouring groups, blocks of 32 pairs, blocks of 16 gather
// four block-columns (or block-rows).  A tile's table entry is eight ints: the positions of the four groups, the bits
// 4 * row group + column group of the 16 x 16 pieces that exist, and three unused; one kernel serves every block size.
//
// Work split.  A workgroup is two wavefronts, each with 32 of the 64 rows of its line (keys of its column), which walk the
// tiles of the line (column) in halves of 32 columns (rows), MFMA 32x32x16: nothing is exchanged between the wavefronts at
// the end and a barrier joins two of them.  What these kernels wait for is the vector unit: on the self-attention module's
// default configuration it computes in 58 / 51 / 42 % of the cycles (forward / rows / columns), the matrix cores in
// 31 / 38 / 38 %, the LDS in 18 / 21 / 32 % (counters: profiles/attention_units.txt).  So what counts is instructions per score
// and wavefronts to hide their latencies: with 16 KiB of LDS a workgroup at head dimension 64 the registers decide, four
// wavefronts per SIMD (three in the column kernel).  Measured on that configuration (block 16, stride 64, 8 x 16 heads x
// 4096, forward / rows / columns): 124 / 161 / 262 us; whole tiles per stage, so 32 KiB and 2.5 wavefronts per SIMD:
// 148 / 177 / 284; four wavefronts with a 32 x 32 quadrant of the tile each, which add partial results up at the end:
// 155 / 190 / 288.
//
// LDS.  Two stages of two operand pieces (32 rows of k and v; of q and do), filled by direct global -> LDS loads one stage
// ahead, one barrier per stage.  Rows lie unpadded; 16-byte chunk c of row r is found at slot c ^ quad_swz(r).  A piece is
// read two ways: along its rows (16 bytes per lane, sixteen consecutive rows served together) and transposed (a 16-lane
// group takes 32 bytes of four consecutive rows, two groups with neighbouring 32 bytes are served together); the swizzle
// spreads both over all banks.
#ifndef BSP_ATTENTION_QUAD_H
#define BSP_ATTENTION_QUAD_H
#include "attention_common.h"
#include <cmath>

namespace bsp {

struct QuadArgs {
  const void *q, *k, *v;
  const void *d_o, *o_in;          // backward: do, and the forward result (row kernel)
  void *o, *o2;                    // forward: o; row kernel: dq; column kernel: dk and dv
  float *lse, *delta;              // per row, [Z][H] rows row_sh apart
  int64_t row_sh, rest;            // rest: floats from a row's lse to what its rounding left out (row_rest); 0: not kept
  int64_t q_sz, q_sh, q_ld, k_sz, k_sh, k_ld, v_sz, v_sh, v_ld, do_sz, do_sh, do_ld, oin_sz, oin_sh, oin_ld;
  int64_t o_sz, o_sh, o_ld, o2_sz, o2_sh, o2_ld;
  float scale;
  float ds_shift, sum_scale;       // the scale's place in the backward pass, 2^ds_shift in ds and the rest on its sums: scale_place
  const int32_t *lut;
  const void *kpm; int64_t kpm_sz; int kpm_mul;
  float *partial;                  // column kernel: slots of the parts of long columns, [Z][n_slots][dk, dv][64][D]
  const int32_t *split_lut;
  int n_slots, n_split;
  int Z, H, R;                     // R: lines of tiles per head (column kernel: work items)
};

namespace {

constexpr int kEntry = 8;          // ints per tile
template <int D> struct Quad {
  static constexpr int PIECE = 32 * D * 2;             // bytes of an operand piece
  static constexpr int STAGE = 2 * PIECE, RING = 2 * STAGE;
};

template <int D> __device__ __forceinline__ int quad_swz(int r) {
  return D == 64 ? ((((r >> 1) & 1) << 2) | ((r >> 2) & 3)) : (((r & 3) << 2) | ((r >> 2) & 3));
}
template <int D> __device__ __forceinline__ int quad_offset(int r, int chunk) { return r * (2 * D) + ((chunk ^ quad_swz<D>(r)) << 4); }

// The first product deals the 32 tile rows of its A operand to the result rows of the MFMA so that a lane's sixteen
// values are rows 16 (i / 8) + 8 (lane / 32) + i % 8: two runs of eight, which is what the next product wants as its
// operand for two steps of sixteen.
__device__ __forceinline__ int deal_row(int m) { return (m & 16) | ((m & 4) << 1) | ((m & 8) >> 1) | (m & 3); }

template <int N> struct Const { static constexpr int value = N; };

// value of lane I of each row of sixteen lanes, in all lanes of the row
template <int I> __device__ __forceinline__ float row_bcast(float v) {
  return __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), 0x150 + I, 0xf, 0xf, true));
}
template <int I, class F> __device__ __forceinline__ void for_16(F &&f) {
  if constexpr (I < 16) {
    f(Const<I>{});
    for_16<I + 1>(f);
  }
}

__device__ __forceinline__ float swap32(float v) { return __shfl_xor(v, 32); }

// Finite padding values so large that fp32 cannot hold them and the scores together (bf16 only: -1e9, say): the softmax operator
// adds the two and rounds, which leaves little or nothing of the score, so that a row of such keys gets equal shares.  These
// kernels take the maximum off the padding value first and would bring the scores back; where a padding value is this
// large they are first reduced to what the rounding leaves of them (Scores::settle).  Below it the rounding is worth
// 2^-4 in the exponent at most and is left out.
constexpr float kFarPadding = 2097152.f;
template <typename T> __device__ __forceinline__ bool far_padding(float kp) {
  return !__is_same(T, f16) && fabsf(kp) >= kFarPadding && kp != -INFINITY;
}

// The scores of a quadrant rounded to the storage type, as the sdd operator would have stored them (the chain then gives what
// the three operators give, up to the order of its sums); the conversion back is part of the multiply-add that uses them.
template <typename T> struct Scores {
  typedef T t2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  t2 pair[8];
  __device__ __forceinline__ void set(const f32x16 &s) {
#pragma unroll
    for (int i = 0; i < 8; i++) pair[i] = __builtin_convertvector((f32x2{s[2 * i], s[2 * i + 1]}), t2);
  }
  __device__ __forceinline__ float operator[](int i) const { return (float)pair[i >> 1][i & 1]; }
  // values 8 k .. 8 k + 7 take no part in the row unless `here`
  __device__ __forceinline__ void keep_if(int k, bool here) {
    const uint32_t none = sizeof(T) == 2 && __is_same(T, f16) ? 0xfc00fc00u : 0xff80ff80u;   // two times -inf
#pragma unroll
    for (int i = 4 * k; i < 4 * k + 4; i++) pair[i] = here ? pair[i] : __builtin_bit_cast(t2, none);
  }
  // value i, scaled by sc, to what is left of it beside the padding value kp(i) (see far_padding)
  template <class F> __device__ __forceinline__ void settle(float sc, F &&kp) {
    for_16<0>([&](auto ic) {
      constexpr int i = decltype(ic)::value;
      const float pad = kp(ic), left = (fmaf((*this)[i], sc, pad) - pad) * __builtin_amdgcn_rcpf(sc);
      pair[i >> 1][i & 1] = far_padding<T>(pad) ? (T)left : pair[i >> 1][i & 1];
    });
  }
  __device__ __forceinline__ float top() const {
    if constexpr (__is_same(T, f16)) {
      t2 m = pair[0];
#pragma unroll
      for (int i = 1; i < 8; i++) m = __builtin_elementwise_max(m, pair[i]);
      return fmaxf((float)m[0], (float)m[1]);
    } else {
      float m = (*this)[0];
#pragma unroll
      for (int i = 1; i < 16; i++) m = fmaxf(m, (*this)[i]);
      return m;
    }
  }
};

// eight values rounded to the storage type, as an MFMA operand
template <typename T> __device__ __forceinline__ typename Mma<T, 32>::frag_t pack8(const float (&v)[8]) {
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  typedef T t2 __attribute__((ext_vector_type(2)));
  union { t2 p[4]; typename Mma<T, 32>::frag_t f; } u;
#pragma unroll
  for (int i = 0; i < 4; i++) u.p[i] = __builtin_convertvector((f32x2{v[2 * i], v[2 * i + 1]}), t2);
  return u.f;
}

// The eight values of an operand that belong to a piece without a block: zero, whatever came out for them.  pieces: bit 0 the
// lanes 0 .. 15 and 32 .. 47 have one, bit 1 the others (made a lane mask by scalar instructions: no vector register holds it)
template <typename F> __device__ __forceinline__ void zero_unless(F &f, int pieces) {
  const bool here = __builtin_amdgcn_inverse_ballot_w64((pieces & 1 ? 0x0000ffff0000ffffull : 0) | (pieces & 2 ? 0xffff0000ffff0000ull : 0));
  u32x4 r = __builtin_bit_cast(u32x4, f);
#pragma unroll
  for (int i = 0; i < 4; i++) r[i] = here ? r[i] : 0u;
  f = __builtin_bit_cast(F, r);
}

// An operand fragment through the transposing LDS read: rows 0 .. 3 of the lane's column at the first address, 4 .. 7 at the second
template <typename T> __device__ __forceinline__ typename Mma<T, 32>::frag_t tr_fragment(uint32_t lo, uint32_t hi) {
  typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
  const s16x4 a = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(uintptr_t)lo), b = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(uintptr_t)hi);
  typedef short s16x8 __attribute__((ext_vector_type(8)));
  return __builtin_bit_cast(typename Mma<T, 32>::frag_t, (s16x8)__builtin_shufflevector(a, b, 0, 1, 2, 3, 4, 5, 6, 7));
}

// Line and (batch, head) of a workgroup of the forward and the row kernel: four heads at a time (their k and v fit the L2 of
// the XCD that works on them), the last lines first, which in a causal layout are the longest.  One head at a time leaves
// long lines to the end of the launch: 82 -> 71 us for the forward pass over 64 lines of 4 to 7 tiles in 128 heads; eight
// heads at a time gain nothing more there.
constexpr int kHeadsTogether = 4;
__device__ __forceinline__ void line_of(int64_t wg, const QuadArgs &a, int &line, int &zh) {
  const int per = kHeadsTogether * a.R, first = (int)(wg / per) * kHeadsTogether, j = (int)(wg % per);
  const int heads = a.Z * a.H - first < kHeadsTogether ? a.Z * a.H - first : kHeadsTogether;
  line = a.R - 1 - j / heads;
  zh = first + j % heads;
}

// The lane's part of the LDS addresses of its reads of 32 rows of a tile: held in registers, or (LEAN, where registers are
// what limits the kernel) one register each, the others an exclusive-or away (a chunk number that is a power of two
// further is a bit of the address, the swizzle being an exclusive-or itself; the empty assembly keeps the compiler from
// computing them once and holding them).
template <int D, bool LEAN> struct RowReads {             // along the rows: chunk 2 s + lane / 32 of the dealt row
  uint32_t a[LEAN ? 1 : D / 16];
  __device__ __forceinline__ void init(int r0, int lane) {
    const int r = r0 + deal_row(lane & 31);
#pragma unroll
    for (int s = 0; s < (LEAN ? 1 : D / 16); s++) a[s] = quad_offset<D>(r, 2 * s + (lane >> 5));
  }
  __device__ __forceinline__ void get(uint32_t (&out)[D / 16]) const {
    if constexpr (LEAN) {
      uint32_t base = a[0];
      asm volatile("" : "+v"(base));
#pragma unroll
      for (int s = 0; s < D / 16; s++) out[s] = base ^ (uint32_t)(s << 5);
    } else {
#pragma unroll
      for (int s = 0; s < D / 16; s++) out[s] = a[s];
    }
  }
};
template <int D, bool LEAN> struct TrReads {              // transposed: rows 8 (lane / 32) + (lane % 16) / 4 (+ 4, + 16), columns 32 mt + 16 (lane / 16 % 2) + 4 (lane % 4)
  uint32_t lo[LEAN ? 1 : D / 32], hi[LEAN ? 1 : D / 32];   // (LEAN: hi is not used; four rows further the swizzle differs in its lowest bit)
  __device__ __forceinline__ void init(uint32_t base, int r0, int lane) {
    const int i = lane & 15, r = r0 + 8 * (lane >> 5) + (i >> 2), col = 16 * ((lane >> 4) & 1) + 4 * (i & 3);
#pragma unroll
    for (int mt = 0; mt < (LEAN ? 1 : D / 32); mt++) {
      const int c = 32 * mt + col;
      lo[mt] = base + quad_offset<D>(r, c >> 3) + ((c & 7) << 1);
      if constexpr (!LEAN) hi[mt] = base + quad_offset<D>(r + 4, c >> 3) + ((c & 7) << 1);
    }
  }
  __device__ __forceinline__ void get(uint32_t (&l)[D / 32], uint32_t (&h)[D / 32]) const {
    if constexpr (LEAN) {
      uint32_t base = lo[0];
      asm volatile("" : "+v"(base));
#pragma unroll
      for (int mt = 0; mt < D / 32; mt++) l[mt] = base ^ (uint32_t)(mt << 6), h[mt] = base ^ (uint32_t)((mt << 6) | 16);
    } else {
#pragma unroll
      for (int mt = 0; mt < D / 32; mt++) l[mt] = lo[mt], h[mt] = hi[mt];
    }
  }
};

// acc[mt] += (32 tile rows, transposed)[column 32 mt ..][row] . b[row]: the tile at LDS byte OFF
template <typename T, int D, int OFF, bool LEAN>
__device__ __forceinline__ void tr_product(f32x16 (&acc)[D / 32], const TrReads<D, LEAN> &reads, const typename Mma<T, 32>::frag_t (&b)[2]) {
  typedef Mma<T, 32> M;
  uint32_t lo[D / 32], hi[D / 32];
  reads.get(lo, hi);
#pragma unroll
  for (int mt = 0; mt < D / 32; mt += 2) {
    constexpr int HI = LEAN ? 4 * 2 * D : 0;
    typename M::frag_t f[4];
#pragma unroll
    for (int i = 0; i < 4; i++) f[i] = tr_fragment<T>(lo[mt + (i & 1)] + OFF + (i >> 1) * (16 * 2 * D), hi[mt + (i & 1)] + OFF + HI + (i >> 1) * (16 * 2 * D));
#pragma unroll
    for (int i = 0; i < 4; i++) acc[mt + (i & 1)] = M::run(f[i], b[i >> 1], acc[mt + (i & 1)]);
  }
}

// (32 tile rows, dealt by deal_row) . b: acc[i] = result row 16 (i / 8) + 8 (lane / 32) + i % 8, column lane % 32
template <typename T, int D, int OFF, bool LEAN>
__device__ __forceinline__ f32x16 row_product(const unsigned char *smem, const RowReads<D, LEAN> &reads, const typename Mma<T, 32>::frag_t (&b)[D / 16], f32x16 acc) {
  typedef Mma<T, 32> M;
  uint32_t addr[D / 16];
  reads.get(addr);
  typename M::frag_t f[D / 16];
#pragma unroll
  for (int s = 0; s < D / 16; s++) f[s] = *reinterpret_cast<const typename M::frag_t *>(smem + OFF + addr[s]);
#pragma unroll
  for (int s = 0; s < D / 16; s++) acc = M::run(f[s], b[s], acc);
  return acc;
}
template <typename T, int D, int OFF, bool LEAN>
__device__ __forceinline__ f32x16 row_product(const unsigned char *smem, const RowReads<D, LEAN> &reads, const typename Mma<T, 32>::frag_t (&b)[D / 16]) {
  f32x16 zero;
#pragma unroll
  for (int i = 0; i < 16; i++) zero[i] = 0.f;
  return row_product<T, D, OFF, LEAN>(smem, reads, b, zero);
}

// BYTES (4 or 16) a lane from base + add (the same in all lanes) + off straight to LDS byte dst + BYTES * lane.  As assembly,
// because the compiler cannot tell which stage such a load fills: before every LDS read behind it, it would wait for the
// load to land.  The only wait is the one in front of a stage's barrier (quad_barrier).
template <int BYTES> __device__ __forceinline__ void load_to_lds(const char *base, uint32_t off, uint32_t add, uint32_t dst) {
  uint32_t at;                                            // (the addition also is the instruction that must lie between m0 and its use)
  if constexpr (BYTES == 16) asm volatile("s_mov_b32 m0, %4\n\tv_add_u32 %0, %2, %1\n\tglobal_load_lds_dwordx4 %0, %3" : "=&v"(at) : "v"(off), "s"(add), "s"(base), "s"(dst) : "m0", "memory");
  else asm volatile("s_mov_b32 m0, %4\n\tv_add_u32 %0, %2, %1\n\tglobal_load_lds_dword %0, %3" : "=&v"(at) : "v"(off), "s"(add), "s"(base), "s"(dst) : "m0", "memory");
}
// the positions of the two groups of half n of a line's (column's) tiles
struct Groups { int lo, hi; };
__device__ __forceinline__ Groups half_groups(table_ptr core, int n) {
  const table_ptr e = core + kEntry * (n >> 1) + 2 * (n & 1);
  return Groups{e[0], e[1]};
}
__device__ __forceinline__ int half_bits(table_ptr core, int n) { return core[kEntry * (n >> 1) + 4]; }
__device__ __forceinline__ uint32_t lds_address(const void *p) { return (uint32_t)(uintptr_t)BSP_LDS_PTR(p); }

// The wavefront's sixteen rows (one group) of a tile, global -> LDS: per lane byte offsets from the group's first row, and
// the loads themselves
template <int D, bool LEAN = false> struct GroupLoad {
  static constexpr int CPR = D / 8, RPL = 64 / CPR, LW = 16 / RPL;
  uint32_t off[LEAN ? 1 : LW];
  uint32_t chunk;                                         // LEAN: the chunk of the first load; off[0]: its row
  __device__ __forceinline__ void init(int64_t ld, int lane) {
    if constexpr (LEAN) {
      chunk = (uint32_t)((lane % CPR) ^ quad_swz<D>(lane / CPR));
      off[0] = (uint32_t)((lane / CPR) * ld) * 2u;
    } else {
#pragma unroll
      for (int i = 0; i < LW; i++) {
        const int r = i * RPL + lane / CPR;
        off[i] = (uint32_t)(r * ld + ((lane % CPR) ^ quad_swz<D>(r)) * 8) * 2u;
      }
    }
  }
  // pos, row_bytes: the group's first row and the distance of rows in bytes
  __device__ __forceinline__ void issue(const char *base, uint32_t pos, uint32_t row_bytes, uint32_t lds) const {
    if constexpr (LEAN) {
      uint32_t c = chunk;
      asm volatile("" : "+v"(c));
#pragma unroll
      for (int i = 0; i < LW; i++)
        load_to_lds<16>(base + (pos + i * RPL) * row_bytes, off[0] + ((c ^ (uint32_t)quad_swz<D>(i * RPL)) << 4), 0, lds + i * 1024);
    } else {
#pragma unroll
      for (int i = 0; i < LW; i++) load_to_lds<16>(base, off[i], pos * row_bytes, lds + i * 1024);
    }
  }
};

// sixteen bytes a lane, D / 16 of them: the lane's row of a 32-row operand that stays in registers (row lane % 32,
// elements 16 s + 8 (lane / 32) ..)
template <typename T, int D> __device__ __forceinline__ void load_operand(typename Mma<T, 32>::frag_t (&f)[D / 16], const T *row) {
#pragma unroll
  for (int s = 0; s < D / 16; s++) f[s] = *reinterpret_cast<const typename Mma<T, 32>::frag_t *>(row + 16 * s);
}
// ... with the sign of every element changed: exact, so that the kernels may take |scale| and look for maxima only
template <typename T, int N> __device__ __forceinline__ void negate(typename Mma<T, 32>::frag_t (&f)[N]) {
#pragma unroll
  for (int s = 0; s < N; s++) {
    u32x4 r = __builtin_bit_cast(u32x4, f[s]);
#pragma unroll
    for (int i = 0; i < 4; i++) r[i] ^= 0x80008000u;
    f[s] = __builtin_bit_cast(typename Mma<T, 32>::frag_t, r);
  }
}

// |scale| in the log2 domain; not zero, so that -inf stays -inf; what is not a number stays that
__device__ __forceinline__ float logit_scale(float scale) {
  const float s = fabsf(scale) * kLog2e;
  return s < 1e-30f ? 1e-30f : s;
}

// A row's lse = m + log2 l has the precision of m: where the maximum is far from zero (finite padding values of -10000 or
// -65504 on every key that the row sees, large scores) the sum rounds log2 l away, and exp2(logit - lse) would not add up to
// one: by 0.3 % at -65504, by the number of keys at -1e9.  From a maximum of kRestFrom on (below it the sum loses 2^-18 at
// most) the forward kernel keeps what was lost as a second float; the backward kernels multiply by exp2(-rest), the row
// kernel its sums at the end, the column kernel the shares of a step in which a row has one.
constexpr float kRestFrom = 64.f;
__device__ __forceinline__ float row_rest(float m, float log_l, float lse) { return fabsf(m) >= kRestFrom ? log_l - (lse - m) : 0.f; }

// key-padding value -> addend in the log2 domain (softmax.py:104-106, 122-124)
template <typename T> __device__ __forceinline__ float kpm_term(T v, int mul) {
  const float m = to_float(v);
  return mul ? (m == 0.f ? -INFINITY : 0.f) : m * kLog2e;
}

// All loads of this wavefront have landed and its LDS reads have returned; then everybody's
__device__ __forceinline__ void quad_barrier() {
  BSP_WAIT_VM(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// acc[mt][4g + e] = out[row][32 mt + 8 g + 4 (lane / 32) + e], row = lane % 32 of the wavefront's 32 rows, which start at
// lo (rows 0 .. 15) and hi (16 .. 31): through the wavefront's piece of LDS (rows of D + 8) to stores of whole rows
template <typename T, int D> __device__ __forceinline__ void store_32_rows(T *stage, T *lo, T *hi, int64_t ld, const f32x16 (&acc)[D / 32], int lane) {
#pragma unroll
  for (int mt = 0; mt < D / 32; mt++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      union { u32x2 raw; T e[4]; } pk;
#pragma unroll
      for (int e = 0; e < 4; e++) pk.e[e] = from_float<T>(acc[mt][4 * g + e]);
      *reinterpret_cast<u32x2 *>(stage + (lane & 31) * (D + 8) + 32 * mt + 8 * g + 4 * (lane >> 5)) = pk.raw;
    }
  __builtin_amdgcn_wave_barrier();   // LDS operations of one wavefront complete in order; this only pins the code order
  constexpr int CPR = D / 8, RPS = 64 / CPR;           // rows per store
#pragma unroll
  for (int i = 0; i < 32 / RPS; i++) {
    const int r = i * RPS + lane / CPR, ch = lane % CPR;
    T *dst = (i * RPS < 16 ? lo + (int64_t)r * ld : hi + (int64_t)(r - 16) * ld) + 8 * ch;
    __builtin_nontemporal_store(*reinterpret_cast<const u32x4 *>(stage + r * (D + 8) + 8 * ch), reinterpret_cast<u32x4 *>(dst));
  }
  __builtin_amdgcn_wave_barrier();
}

// ds = p (dp - delta) scale is rounded to the storage type.  Up to 1 the scale is left to the sums dq and dk: without it ds has
// the range of dp.  Above, ds without it could fall into the subnormals where with it, as the operators round it, it does not:
// its power of two goes in first (with p: exact, and no more than 2^14 of it, which fp16 holds).  bf16 has no such values.
inline void scale_place(QuadArgs &a, int dtype) {
  const float s = fabsf(a.scale);
  const int shift = dtype == BSP_F16 && s >= 2.f ? (s < 16384.f ? ilogbf(s) : 14) : 0;
  a.ds_shift = (float)shift;
  a.sum_scale = ldexpf(a.scale, -shift);
}

// What the launchers check: types and sizes, 16-byte alignment of every pointer (NULL is aligned) and stride, and that the
// `loaded` first of the row strides lds, which belong to operands of `positions` rows that are fetched tile by tile, keep
// the byte offsets of those rows within 32 bits
inline int quad_check(int dtype, int D, const void *const *ptrs, int n_ptrs, const int64_t *strides, int n_strides, const int64_t *lds, int n_lds, int loaded,
                      int64_t positions, int64_t n_wg) {
  if ((dtype != BSP_F16 && dtype != BSP_BF16) || (D != 64 && D != 128) || n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  for (int i = 0; i < n_ptrs; i++)
    if (reinterpret_cast<uintptr_t>(ptrs[i]) & 15) return BSP_ERR_ARG;
  for (int i = 0; i < n_strides; i++)
    if (strides[i] % 8) return BSP_ERR_ARG;
  for (int i = 0; i < n_lds; i++)
    if (lds[i] < D || (i < loaded && (positions <= 0 || lds[i] > (((int64_t)1 << 32) - 1) / (2 * positions)))) return BSP_ERR_ARG;
  return BSP_OK;
}

}  // namespace
}  // namespace bsp
#endif
