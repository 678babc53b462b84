// The attention chain without sparse tensors in fp32 (head dimension 64 or 128; calls without relative position embedding and attention
// mask): what attention_fwd.hip and attention_bwd.hip do for 16-bit tensors, in single precision and on the bfloat16 matrix units.
//
// Products.  A number of 24 bits is the sum of three bfloat16 numbers, each rounded to nearest: x = x0 + x1 + x2, exactly down
// to 2^-110.  The parts are those of 2^16 x, so of every number that fp32 has, and the sums are scaled back where they are used (powers of
// two, in factors that are there).  A product is the sum of the six products of such parts that count in 24 bits, smallest first, in one fp32
// accumulator: x2 y0 + x1 y1 + x0 y2 + x1 y0 + x0 y1 + x0 y0 (the three left out are 2^-27 of it and less).  Six MFMAs of bfloat16 do in 6 x 32 cycles what eight of fp32 do in
// 8 x 64, and round less often (once a step of sixteen instead of two).  Error against 64 bits of 32 x 32 products of N(0, 1) operands, relative 2-norm, this /
// fp32 MFMA: 64 terms 1.1e-7 / 1.5e-7, 512 terms 3.4e-7 / 4.0e-7, 4096 terms 9.9e-7 / 1.15e-6; uniform operands 0.9e-7 / 1.2e-7, 2.4e-7 /
// 2.9e-7, 5.2e-7 / 8.3e-7.  (Parts cut off instead of rounded: 1e-5 for 4096 uniform terms, their sums being one-sided.)
// Infinities have no such parts, and their products with zero parts would be NaN: where a head's operands hold a value of 2^20 or
// more, an infinity or a NaN (a flag per 64 rows, made beside the parts), the kernels compute its products from the whole
// values on the fp32 units, as the operators do.  Below 2^20 no sum of products of parts overflows.  Where every head has such a value the pass
// takes 512 us where the operators take 287 and parts 196 (training, 2 x 8 heads of 2048 positions, head dimension 64).
//
// Softmax.  The same logits as the operator's, in the natural domain and rounded once, and delta from the same products in the same order as
// dp (delta_of), so that over a tensor the error to 64 bits is 0.6 to 1.0 of the operators': N(0, 1) operands o / dq / dk / dv 2.2 / 2.4 / 2.5 / 2.3e-7
// against 3.6 / 3.7 / 3.9 / 3.8e-7, logits up to some hundreds 0.65-0.97 of theirs, keys of a sequence all padded with -100 ... -65504 1.0.
//
// Launches.  k_attn32_planes writes the three parts of q, k and v (backward: do) as planes, [row][part][D], so that the other
// kernels fetch them tile by tile straight into LDS.  Those walk the same tables and 64 x 64 tiles as the 16-bit kernels; a
// workgroup is four wavefronts, one per 32 x 32 quadrant, since a line is few tiles and 64 rows with two wavefronts would leave
// half of the SIMDs of a launch of a few hundred lines without any.  The quadrants of the same rows add up at the end through LDS.
// A tile's operands come in two pieces (k, v; columns: q, do) of 64 rows x 3 parts, 24 KiB at head dimension 64; the ring has
// three slots of a piece, so two workgroups share a CU (one at 128): while a piece is used the next is on its way, and the one after that
// where a slot is free.
#include "attention_quad.h"

// (a multiplication and the addition behind it stay two roundings, as in the operators)
#pragma clang fp contract(off)

namespace bsp {
namespace {

struct F32Args : QuadArgs {            // k, v: the planes; q: forward q itself, backward the planes; d_o: row kernel do itself, column kernel
                                       // the planes; lse: per row the reference m of its exponentials, rest floats on kUp / l
  const int32_t *fq, *fk, *fv, *fdo;   // flags [Z][H][pieces of 64 rows]; fq (forward) and fdo (row kernel) NULL: not there, no other kernel follows
  int64_t rows, keys;
  int sub;                             // column kernel: pieces that a part of a long column is cut into
};

typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float f32x2 __attribute__((ext_vector_type(2)));
struct Parts { bf16x8 p[3]; };
constexpr float kLargest = 1048576.f;                  // 2^20
constexpr float kUp = 65536.f, kDown = 1.f / kUp, kDown2 = kDown * kDown;   // parts are those of kUp x
constexpr float kReversed = 1267650600228229401496703205376.f;              // 2^100
// Where products are of whole values, those may be as large as fp32 holds.  The operators multiply shares, which add up to one; the kernels
// then take every exponential against the row's maximum and 2^-16 of it (a row has fewer keys), p and not its numerator in the
// row kernel, and the scale with ds instead of with its sums, so that no sum overflows which theirs do not.
constexpr float kWholeShare = 1.f / 65536.f;

// the parts of eight values
__device__ __forceinline__ Parts split8(const float (&v)[8]) {
  union { bf16x2 two[4]; bf16x8 all; } h, m, l;
#pragma unroll
  for (int i = 0; i < 4; i++) {
    const f32x2 x = {v[2 * i], v[2 * i + 1]};
    h.two[i] = __builtin_convertvector(x, bf16x2);
    const f32x2 r = x - __builtin_convertvector(h.two[i], f32x2);
    m.two[i] = __builtin_convertvector(r, bf16x2);
    l.two[i] = __builtin_convertvector(r - __builtin_convertvector(m.two[i], f32x2), bf16x2);
  }
  Parts s;
  s.p[0] = h.all; s.p[1] = m.all; s.p[2] = l.all;
  return s;
}
// ... of an operand's, scaled up.  What fp32 does not hold then is kept as it is, for `whole` to find: from 2^100 on with the smallest part first,
// infinities and NaN in the first part alone.
__device__ __forceinline__ Parts split_operand(const float (&v)[8]) {
  float x[8];
#pragma unroll
  for (int i = 0; i < 8; i++) x[i] = v[i] * kUp;
  Parts s = split8(x);
#pragma unroll
  for (int i = 0; i < 8; i++)
    if (!(fabsf(v[i]) < kReversed)) {
      const bool finite = fabsf(v[i]) < INFINITY;
      const float a = finite ? __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, v[i]) & 0xffff0000u) : 0.f, r = finite ? v[i] - a : 0.f;
      const float b = __builtin_bit_cast(float, __builtin_bit_cast(uint32_t, r) & 0xffff0000u);
      s.p[0][i] = finite ? (bf16)(r - b) : (bf16)v[i]; s.p[1][i] = (bf16)b; s.p[2][i] = (bf16)a;
    }
  return s;
}

__device__ __forceinline__ f32x16 mma(const bf16x8 &a, const bf16x8 &b, const f32x16 &c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
// value i of eight that are held as parts (split_operand)
__device__ __forceinline__ float whole(const u32x4 (&v)[3], int i) {
  auto part = [&](int p) { return __builtin_bit_cast(float, i & 1 ? v[p][i >> 1] & 0xffff0000u : v[p][i >> 1] << 16); };
  const float a = part(0), c = part(2), sum = a + part(1) + c;
  return fabsf(c) > fabsf(a) ? sum : sum * kDown;
}
// acc += a . b over sixteen indices from the whole values, on the fp32 units.  (The empty assembly keeps whole values from being held
// beside the parts, the barrier keeps the next operands from being fetched ahead: this way is about registers, not time.)
template <class F> __device__ __forceinline__ f32x16 whole_product(const Parts &a, F &&b, f32x16 acc) {
  u32x4 x[3];
#pragma unroll
  for (int p = 0; p < 3; p++) {
    x[p] = __builtin_bit_cast(u32x4, a.p[p]);
    asm volatile("" : "+v"(x[p]));
  }
#pragma unroll
  for (int i = 0; i < 8; i++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(whole(x, i), b(i), acc, 0, 0, 0);
  __builtin_amdgcn_sched_barrier(0);
  return acc;
}
__device__ __forceinline__ f32x16 whole_parts_product(const Parts &a, const Parts &b, f32x16 acc) {
  u32x4 y[3];
#pragma unroll
  for (int p = 0; p < 3; p++) {
    y[p] = __builtin_bit_cast(u32x4, b.p[p]);
    asm volatile("" : "+v"(y[p]));
  }
  return whole_product(a, [&](int i) { return whole(y, i); }, acc);
}

// the same of parts, in the order of the parts' sizes; SWAP: those of b count as the first factor's
template <bool SWAP> __device__ __forceinline__ f32x16 parts_product(const Parts &a, const Parts &b, f32x16 acc) {
  const Parts &x = SWAP ? b : a, &y = SWAP ? a : b;
  auto term = [&](int i, int j) { acc = SWAP ? mma(y.p[j], x.p[i], acc) : mma(x.p[i], y.p[j], acc); };
  term(2, 0); term(0, 2); term(1, 1); term(0, 1); term(1, 0); term(0, 0);
  return acc;
}

// a sum of products of parts -> what it stands for, times scale (in the order in which nothing that fp32 holds is lost on the way)
struct ScaledDown {
  float first, then;
  __device__ __forceinline__ explicit ScaledDown(float scale) : first(fabsf(scale) < 1.f ? scale : scale * kDown2), then(fabsf(scale) < 1.f ? kDown2 : 1.f) {}
  __device__ __forceinline__ float operator()(float sum) const { return sum * first * then; }
};

template <int D> struct Ring {
  static constexpr int PLANE = 64 * D * 2, PIECE = 3 * PLANE, SIDE = 4 * 512;   // SIDE: two words a lane for each wavefront, beside a piece
  static constexpr int BYTES = 3 * (PIECE + SIDE);
};

// acc[i] += (32 rows of the piece, dealt by deal_row) . b, as in attention_quad.h
// The sums come out the same, bit for bit, with either factor's rows in LDS (SWAP: the parts of b are taken as the first factor's): the
// backward pass has the forward pass's probabilities however large the scores are, and dp minus delta is zero where it is (see delta_of).
// (FETCH: b is fetched again for each product, from its planes or as it is, which leaves its registers to the fp32 units' way of working;
// by_parts: the product is made of parts all the same, which only planes can be)
template <bool FETCH, bool SWAP, int D, typename S>
__device__ __forceinline__ f32x16 rows_times(const unsigned char *piece, const RowReads<D, true> &reads, const Parts (&b)[D / 16], const S *b_row, bool by_parts, f32x16 acc) {
  uint32_t at[D / 16];
  reads.get(at);
#pragma unroll
  for (int s = 0; s < D / 16; s++) {
    Parts f;
#pragma unroll
    for (int p = 0; p < 3; p++) f.p[p] = *reinterpret_cast<const bf16x8 *>(piece + p * Ring<D>::PLANE + at[s]);
    auto terms = [&](const Parts &own) { acc = parts_product<SWAP>(f, own, acc); };
    if constexpr (FETCH) {
      asm volatile("" : "+v"(b_row));
      if constexpr (sizeof(S) == 4) {
        const f32x4 lo = *reinterpret_cast<const f32x4 *>(b_row + 16 * s), hi = *reinterpret_cast<const f32x4 *>(b_row + 16 * s + 4);
        acc = whole_product(f, [&](int i) { return i < 4 ? lo[i & 3] : hi[i & 3]; }, acc);
      } else {
        Parts mine;
#pragma unroll
        for (int p = 0; p < 3; p++) mine.p[p] = *reinterpret_cast<const bf16x8 *>(b_row + p * D + 16 * s);
        if (by_parts) {
          terms(mine);
          __builtin_amdgcn_sched_barrier(0);
        } else {
          acc = whole_parts_product(f, mine, acc);
        }
      }
    } else {
      terms(b[s]);
    }
  }
  return acc;
}
// acc[mt] += (32 rows of the piece, transposed) . b; WHOLE: only where here0 / here1, the first / second sixteen rows have a block (nothing of the
// rows of a block that does not exist may reach the sums, and an infinity among them would).  Two chains of products at a time: two groups
// of columns, each step's 32 terms added up first; TIGHT (where registers are short): one group, the smaller products of a step and the others.
template <bool WHOLE, bool TIGHT, int D>
__device__ __forceinline__ void columns_times(f32x16 (&acc)[D / 32], uint32_t piece, const TrReads<D, true> &reads, const float (&e)[16], bool here0, bool here1) {
  Parts b[2];
  if constexpr (!WHOLE) {                               // (e is kUp times what it stands for)
    b[0] = split8(reinterpret_cast<const float (&)[8]>(e[0]));
    b[1] = split8(reinterpret_cast<const float (&)[8]>(e[8]));
  }
  uint32_t lo[D / 32], hi[D / 32];
  reads.get(lo, hi);
  auto fetch = [&](int mt, int ks) {
    Parts f;
#pragma unroll
    for (int p = 0; p < 3; p++)
      f.p[p] = tr_fragment<bf16>(lo[mt] + piece + p * Ring<D>::PLANE + ks * (16 * 2 * D), hi[mt] + piece + p * Ring<D>::PLANE + ks * (16 * 2 * D) + 4 * 2 * D);
    return f;
  };
  auto none = [] {
    f32x16 v;
#pragma unroll
    for (int i = 0; i < 16; i++) v[i] = 0.f;
    return v;
  };
  if constexpr (WHOLE) {
#pragma unroll
    for (int mt = 0; mt < D / 32; mt++)
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        const f32x16 sum = whole_product(fetch(mt, ks), [&](int i) { return e[8 * ks + i]; }, acc[mt]);
#pragma unroll
        for (int i = 0; i < 16; i++) acc[mt][i] = (ks ? here1 : here0) ? sum[i] : acc[mt][i];
        __builtin_amdgcn_sched_barrier(0);
      }
  } else if constexpr (TIGHT) {
#pragma unroll
    for (int mt = 0; mt < D / 32; mt++) {
      f32x16 small = none();
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        const Parts f = fetch(mt, ks);
        small = mma(f.p[2], b[ks].p[0], small);
        acc[mt] = mma(f.p[0], b[ks].p[1], acc[mt]);
        small = mma(f.p[1], b[ks].p[1], small);
        acc[mt] = mma(f.p[0], b[ks].p[0], acc[mt]);
        small = mma(f.p[0], b[ks].p[2], small);
        small = mma(f.p[1], b[ks].p[0], small);
        __builtin_amdgcn_sched_barrier(0);              // (nothing is fetched further ahead)
      }
#pragma unroll
      for (int i = 0; i < 16; i++) acc[mt][i] += small[i];
    }
  } else {
#pragma unroll
    for (int mt = 0; mt < D / 32; mt += 2) {
      f32x16 sum[2] = {none(), none()};
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        const Parts f[2] = {fetch(mt, ks), fetch(mt + 1, ks)};
#pragma unroll
        for (int t = 0; t < 6; t++)
#pragma unroll
          for (int j = 0; j < 2; j++) sum[j] = mma(f[j].p[t == 0 ? 2 : t == 1 || t == 3 ? 1 : 0], b[ks].p[t == 1 || t == 4 ? 1 : t == 2 ? 2 : 0], sum[j]);
      }
#pragma unroll
      for (int j = 0; j < 2; j++)
#pragma unroll
        for (int i = 0; i < 16; i++) acc[mt + j][i] += sum[j][i];
    }
  }
}

// Logits are what the softmax operator forms in fp32, in the natural domain and rounded once: score * scale + mask.
// key-padding value -> mask (softmax.py:104-106, 122-124)
__device__ __forceinline__ float pad_term(float v, int mul) { return mul ? (v == 0.f ? -INFINITY : 0.f) : v; }

// e^y for y up to some ten.  v_exp_f32 of the rounded product y log2 e, times one plus what its rounding left out: within two units in the last
// place for every y, where the product alone is off by |y| / 2 of them.  (Below -87 zero.  WHOLE: the library's, whose tiny values
// make infinities of infinities as the operators' do.)
template <bool WHOLE> __device__ __forceinline__ float exp_of(float y) {
  if constexpr (WHOLE) return expf(y);
  constexpr double kLn2 = 0.69314718055994530942;
  constexpr float hi = (float)kLn2, lo = (float)(kLn2 - (double)hi);
  y = __builtin_elementwise_maximum(y, -110.f);         // (NaN stays; minus infinity would become it)
  const float product = y * kLog2e, left = fmaf(product, -lo, fmaf(product, -hi, y)), e = __builtin_amdgcn_exp2f(product);
  return fmaf(e, left, e);
}

// The work of a workgroup.  The tables have the long lines (columns) of four heads at a time first; from eight such groups on each XCD takes
// its own ones, so that their rows meet in its L2.  Fewer groups would leave the XCDs that begin in the middle of one with its short lines alone: they
// are dealt in turn.
__device__ __forceinline__ int64_t place(const F32Args &a, int64_t n) {
  return a.Z * a.H >= 8 * kHeadsTogether ? xcd_remap(blockIdx.x, n) : (int64_t)blockIdx.x;
}

// the flags of a head: is one of n set?  (in this lane; its first one is fetched before any is looked at)
__device__ __forceinline__ int32_t flags_of(const int32_t *f, int64_t zh, int64_t n, int lane) {
  int32_t set = f[zh * n + (lane < n ? lane : 0)];
  for (int64_t i = lane + 64; i < n; i += 64) set |= f[zh * n + i];
  return set;
}

// The way of a product is the head's (n_rows: pieces of 64 rows of q): the scores' that of the forward pass, which knows q, k and v, so that the
// backward kernels have its probabilities also where only do is flagged.
__device__ __forceinline__ int32_t forward_flags(const F32Args &a, int64_t zh, int64_t n_rows, int lane) {
  return flags_of(a.fq, zh, n_rows, lane) | flags_of(a.fk, zh, a.keys / 64, lane) | flags_of(a.fv, zh, a.keys / 64, lane);
}

// the wavefront's sixteen rows of a piece (its group), three planes
template <int D> struct PieceLoad {
  static constexpr int COUNT = 3 * GroupLoad<D>::LW;
  GroupLoad<D> g;
  __device__ __forceinline__ void init(int lane) { g.init(3 * D, lane); }
  __device__ __forceinline__ void issue(const char *planes, int pos, uint32_t lds, int wave) const {
#pragma unroll
    for (int p = 0; p < 3; p++) g.issue(planes + p * (D * 2), (uint32_t)pos, 3 * D * 2, lds + p * Ring<D>::PLANE + wave * (16 * D * 2));
  }
};

template <int N> __device__ __forceinline__ void wait_barrier() {
  BSP_WAIT_VM(N);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
}

// The walk over the tiles of a line.  Each tile is two pieces, used one after the other: first(slot, n) with x in LDS, then second(slot, n) with
// y.  Piece after piece goes round the three slots, so that two are on their way while one is used.  issue_x / issue_y(n, slot) ask for them
// (NX / NY vector-memory operations a wavefront); those of the first tile (slots 0 and 1) are on their way when the walk begins.
template <int NX, int NY, class IX, class IY, class F1, class F2> __device__ __forceinline__ void walk(int tiles, IX &&issue_x, IY &&issue_y, F1 &&first, F2 &&second) {
  int a = 0, b = 1, c = 2;                              // the slots of this piece, the next and the one after it
  for (int n = 0; n < tiles; n++) {
    wait_barrier<NY>();                                 // x is here, and everybody is done with the piece before it
    if (n + 1 < tiles) issue_x(n + 1, c);
    first(a, n);
    if (n + 1 < tiles) wait_barrier<NX>();
    else wait_barrier<0>();
    if (n + 1 < tiles) issue_y(n + 1, a);
    second(b, n);
    const int was = b;
    b = a; a = c; c = was;
  }
}
// ... where x is used again beside y: y can only be asked for when its tile begins (and only x of the first tile is on its way)
template <int NX, class IX, class IY, class F1, class F2> __device__ __forceinline__ void walk_x_twice(int tiles, IX &&issue_x, IY &&issue_y, F1 &&first, F2 &&second) {
  int x = 0, y = 1, free = 2;
  for (int n = 0; n < tiles; n++) {
    wait_barrier<0>();                                  // x of this tile is here; everybody is done with the tile before
    issue_y(n, y);
    if (n + 1 < tiles) issue_x(n + 1, free);
    first(x, n);
    if (n + 1 < tiles) wait_barrier<NX>();
    else wait_barrier<0>();
    second(x, y, n);
    const int was = x;
    x = free; free = y; y = was;
  }
}

// 32 rows of D sums (as store_32_rows) to LDS rows of D + 4 and from there to whole rows in memory, the first sixteen from lo on, the others from hi
template <int D> __device__ __forceinline__ void store_32_f32(float *stage, float *lo, float *hi, int64_t ld, const f32x16 (&acc)[D / 32], int lane) {
#pragma unroll
  for (int mt = 0; mt < D / 32; mt++)
#pragma unroll
    for (int g = 0; g < 4; g++)
      *reinterpret_cast<f32x4 *>(stage + (lane & 31) * (D + 4) + 32 * mt + 8 * g + 4 * (lane >> 5)) = f32x4{acc[mt][4 * g], acc[mt][4 * g + 1], acc[mt][4 * g + 2], acc[mt][4 * g + 3]};
  __builtin_amdgcn_wave_barrier();                      // (the LDS operations of one wavefront complete in order)
  constexpr int CPR = D / 4, RPS = 64 / CPR;
#pragma unroll
  for (int i = 0; i < 32 / RPS; i++) {
    const int r = i * RPS + lane / CPR, c = 4 * (lane % CPR);
    float *dst = (i * RPS < 16 ? lo + (int64_t)r * ld : hi + (int64_t)(r - 16) * ld) + c;
    *reinterpret_cast<f32x4 *>(dst) = *reinterpret_cast<const f32x4 *>(stage + r * (D + 4) + c);
  }
  __builtin_amdgcn_wave_barrier();
}
// sums of one wavefront to another through LDS: lane by lane
template <int D> __device__ __forceinline__ void put_sums(float *to, const f32x16 (&acc)[D / 32], int lane) {
#pragma unroll
  for (int mt = 0; mt < D / 32; mt++)
#pragma unroll
    for (int g = 0; g < 4; g++)
      *reinterpret_cast<f32x4 *>(to + ((mt * 4 + g) * 64 + lane) * 4) = f32x4{acc[mt][4 * g], acc[mt][4 * g + 1], acc[mt][4 * g + 2], acc[mt][4 * g + 3]};
}
template <int D, class F> __device__ __forceinline__ void take_sums(const float *from, f32x16 (&acc)[D / 32], int lane, F &&add) {
#pragma unroll
  for (int mt = 0; mt < D / 32; mt++)
#pragma unroll
    for (int g = 0; g < 4; g++) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>(from + ((mt * 4 + g) * 64 + lane) * 4);
#pragma unroll
      for (int e = 0; e < 4; e++) acc[mt][4 * g + e] = add(acc[mt][4 * g + e], v[e]);
    }
}

// the lane's row of an operand that stays in registers, from the planes
template <int D> __device__ __forceinline__ void load_parts(Parts (&f)[D / 16], const bf16 *row) {
#pragma unroll
  for (int s = 0; s < D / 16; s++)
#pragma unroll
    for (int p = 0; p < 3; p++) f[s].p[p] = *reinterpret_cast<const bf16x8 *>(row + p * D + 16 * s);
}

// ... from a piece in LDS: its row r
template <int D> __device__ __forceinline__ void own_parts(Parts (&f)[D / 16], const unsigned char *piece, int r, int half) {
#pragma unroll
  for (int s = 0; s < D / 16; s++)
#pragma unroll
    for (int p = 0; p < 3; p++) f[s].p[p] = *reinterpret_cast<const bf16x8 *>(piece + p * Ring<D>::PLANE + quad_offset<D>(r, 2 * s + half));
}
// ... from the operand itself, fp32
template <int D> __device__ __forceinline__ void fetch_row(f32x4 (&v)[D / 8], const float *row) {
#pragma unroll
  for (int s = 0; s < D / 16; s++)
#pragma unroll
    for (int j = 0; j < 2; j++) v[2 * s + j] = *reinterpret_cast<const f32x4 *>(row + 16 * s + 4 * j);
}
// its parts.  -> does it (in this lane) hold a value that is not below kLargest?
template <int D> __device__ __forceinline__ int take_parts(Parts (&f)[D / 16], const f32x4 (&v)[D / 8]) {
  int large = 0;
#pragma unroll
  for (int s = 0; s < D / 16; s++) {
    float e[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      e[j] = v[2 * s + (j >> 2)][j & 3];
      large |= !(fabsf(e[j]) < kLargest);
    }
    f[s] = split_operand(e);
  }
  return large;
}

// delta = sum_d do . o of the lane's row.  ds = p (dp - delta), so in a row whose share is one key's delta has to be that key's dp to the last bit
// (what is left of the two, 1e-7 of |do| |v|, would be multiplied by rows of q and k that may be of any size): o is that key's v there, and
// the sum is taken from the same unit's products in the same order as dp, off the diagonal of do . o^T.
// (do with an infinity: sums of infinities of both signs in the operators, so NaN)
template <bool WHOLE, int D> __device__ __forceinline__ float delta_of(const f32x4 (&o)[D / 8], const Parts (&do_parts)[D / 16], const f32x4 (&d_o)[D / 8], int lane) {
  f32x16 acc;
#pragma unroll
  for (int i = 0; i < 16; i++) acc[i] = 0.f;
#pragma unroll
  for (int s = 0; s < D / 16; s++) {
    if constexpr (WHOLE) {
#pragma unroll
      for (int i = 0; i < 8; i++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(o[2 * s + (i >> 2)][i & 3], d_o[2 * s + (i >> 2)][i & 3], acc, 0, 0, 0);
    } else {
      float e[8];
#pragma unroll
      for (int i = 0; i < 8; i++) e[i] = o[2 * s + (i >> 2)][i & 3];
      acc = parts_product<false>(split_operand(e), do_parts[s], acc);
    }
  }
  const int r = lane & 31, at = 4 * (r >> 3) + (r & 3);  // acc[i]: row 8 (i / 4) + 4 (lane / 32) + i % 4 of o, column r of do
  float own = 0.f;
#pragma unroll
  for (int i = 0; i < 16; i++) own = at == i ? acc[i] : own;
  const float other = swap32(own), delta = ((r >> 2) & 1) == (lane >> 5) ? own : other;
  return !WHOLE ? delta * kDown2 : fabsf(delta) < INFINITY ? delta : NAN;
}

// ---- planes ----
struct PlaneArgs {
  struct Tensor {
    const float *x;
    bf16 *planes;
    int32_t *flags;
    int64_t sz, sh, ld;
    uint32_t chunks, end;              // pieces of 64 rows of a head; the first workgroup behind the tensor's
  } t[3];
  int H;                               // heads of a batch
};
template <int D> __global__ void __launch_bounds__(256) k_attn32_planes(PlaneArgs a) {
  const int t = blockIdx.x < a.t[0].end ? 0 : blockIdx.x < a.t[1].end ? 1 : 2;
  const PlaneArgs::Tensor &own = a.t[t];
  const uint32_t wg = blockIdx.x - (t ? a.t[t - 1].end : 0u);
  const Quotient head(wg, own.chunks), zh(head.q, a.H);
  const float *x = own.x + zh.q * own.sz + zh.r * own.sh + (int64_t)head.r * 64 * own.ld;
  bf16 *to = own.planes + (int64_t)wg * (64 * 3 * D);
  int large = 0;
  constexpr int PER = 64 * D / 8 / 256;
  f32x4 v[PER][2];
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int c = threadIdx.x + 256 * i, row = c / (D / 8), col = 8 * (c % (D / 8));
    const f32x4 *src = reinterpret_cast<const f32x4 *>(x + row * own.ld + col);
    v[i][0] = src[0]; v[i][1] = src[1];
  }
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int c = threadIdx.x + 256 * i, row = c / (D / 8), col = 8 * (c % (D / 8));
    float e[8];
#pragma unroll
    for (int j = 0; j < 8; j++) {
      e[j] = v[i][j >> 2][j & 3];
      large |= !(fabsf(e[j]) < kLargest);
    }
    const Parts s = split_operand(e);
#pragma unroll
    for (int p = 0; p < 3; p++) *reinterpret_cast<bf16x8 *>(to + row * (3 * D) + p * D + col) = s.p[p];
  }
  const int any = __syncthreads_or(large);
  if (threadIdx.x == 0) own.flags[wg] = any;
}

// ---- forward ----
template <int D, bool KPM> __global__ void __launch_bounds__(256, D == 64 ? 2 : 1) k_attn32_fwd(F32Args a) {
  typedef Ring<D> R;
  constexpr int MT = D / 32, NK = PieceLoad<D>::COUNT + (KPM ? 1 : 0);
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float *side = reinterpret_cast<float *>(smem + 3 * R::PIECE);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5, rh = wave & 1, kh = wave >> 1;       // the wavefront's rows and columns of a tile
  const int64_t wg = place(a, (int64_t)a.Z * a.H * a.R);
  int line, zh;
  line_of(wg, a, line, zh);
  const int h = zh % a.H, z = zh / a.H;
  const table_ptr lut = as_table(a.lut);
  const int tiles = lut[2 * (h * a.R + line)];
  const table_ptr core = lut + lut[2 * (h * a.R + line) + 1];
  const int64_t row = (int64_t)line * 64 + 32 * rh + l32;
  f32x16 o[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) o[mt][i] = 0.f;
  float m = -INFINITY, l = 0.f, share = 1.f, down = 1.f;   // l and o are `share` times what they stand for; down: takes the scale of v off o
  int rows_seen = 0;

  if (tiles > 0) {
    Parts xq[D / 16];
    const float *q_row = reinterpret_cast<const float *>(a.q) + z * a.q_sz + h * a.q_sh + row * a.q_ld + 8 * half;
    float sc = a.scale * kDown2;
    const char *pk = reinterpret_cast<const char *>(reinterpret_cast<const bf16 *>(a.k) + zh * a.keys * (3 * D));
    const char *pv = reinterpret_cast<const char *>(reinterpret_cast<const bf16 *>(a.v) + zh * a.keys * (3 * D));
    const char *pkpm = reinterpret_cast<const char *>(reinterpret_cast<const float *>(a.kpm) + z * a.kpm_sz);
    PieceLoad<D> load;
    load.init(lane);
    RowReads<D, true> rows_k;
    TrReads<D, true> tr_v;
    rows_k.init(32 * kh, lane);
    tr_v.init(lds_address(smem), 32 * kh, lane);
    const float *kp_lane = side + (2 * kh + ((lane >> 3) & 1)) * 128 + 8 * half + (lane & 7);   // value i of the lane comes from lane i of each sixteen
    // the table runs a tile ahead of the loads
    int pos_next = core[wave], pos = 0, bits_next = 0;
    auto issue_k = [&](int n, int slot) {
      pos = pos_next;
      load.issue(pk, pos, lds_address(smem) + slot * R::PIECE, wave);
      if constexpr (KPM) load_to_lds<4>(pkpm, (uint32_t)(pos + (lane & 15)) * 4u, 0, lds_address(side) + slot * R::SIDE + wave * 512);
      pos_next = core[kEntry * (n + 1 < tiles ? n + 1 : n) + wave];
    };
    auto issue_v = [&](int n, int slot) {
      load.issue(pv, pos, lds_address(smem) + slot * R::PIECE, wave);
      bits_next = core[kEntry * n + 4];
    };
    float e[16];
    auto run = [&](auto whole) {
      constexpr bool W = decltype(whole)::value;
      share = W ? kWholeShare : kUp;
      down = W ? 1.f : kDown;
      if constexpr (W) sc = a.scale;
      int here = 0;
      walk<NK, PieceLoad<D>::COUNT>(tiles, issue_k, issue_v,
        [&](int x, int) {
          f32x16 s;
#pragma unroll
          for (int i = 0; i < 16; i++) s[i] = 0.f;
          s = rows_times<W, false, D>(smem + x * R::PIECE, rows_k, xq, q_row, false, s);
          here = bits_next >> (8 * rh + 2 * kh);
          rows_seen |= here & 0x33;
          const float kp = KPM ? pad_term(kp_lane[x * (R::SIDE / 4)], a.kpm_mul) : 0.f;
          const int mine = here >> ((lane >> 4) & 1) * 4;
          const bool here0 = mine & 1, here1 = mine & 2;        // pieces without a block take no part in the row
          for_16<0>([&](auto ic) { s[decltype(ic)::value] = KPM ? fmaf(s[decltype(ic)::value], sc, row_bcast<decltype(ic)::value>(kp)) : s[decltype(ic)::value] * sc; });
          float sum, top = -INFINITY;
          auto highest = [&]() {
#pragma unroll
            for (int i = 0; i < 16; i++) top = fmaxf(top, (i < 8 ? here0 : here1) ? s[i] : -INFINITY);
          };
          auto exponentials = [&]() {
            const float ms = m == -INFINITY ? 0.f : m;
#pragma unroll
            for (int i = 0; i < 16; i++) e[i] = exp_of<W>(s[i] - ms) * (W ? kWholeShare : kUp);
            if ((here & 0x33) != 0x33) {                // (whatever the logits came out as there: a mask may hold NaN or an infinity, the scale may make one)
#pragma unroll
              for (int i = 0; i < 16; i++) e[i] = (i < 8 ? here0 : here1) ? e[i] : 0.f;
            }
            sum = 0.f;
#pragma unroll
            for (int i = 0; i < 16; i++) sum += e[i];
          };
          if constexpr (W) highest();
          else exponentials();
          if (__builtin_amdgcn_ballot_w64(W ? top > m || m == -INFINITY : !(sum <= 8192.f * kUp) || m == -INFINITY)) {      // (also where an exponential overflowed)
            if constexpr (!W) highest();
            const float mn = fmaxf(m, fmaxf(top, swap32(top))), f = exp_of<W>(m - (mn == -INFINITY ? 0.f : mn));
            l *= f;
#pragma unroll
            for (int mt = 0; mt < MT; mt++)
#pragma unroll
              for (int i = 0; i < 16; i++) o[mt][i] *= f;
            m = mn;
            if constexpr (!W) exponentials();
          }
          if constexpr (W) exponentials();
          l += sum;
        },
        [&](int y, int) {
          const int mine = here >> ((lane >> 4) & 1) * 4;
          columns_times<W, false, D>(o, y * R::PIECE, tr_v, e, mine & 1, mine & 2);
        });
    };
    issue_k(0, 0);
    issue_v(0, 1);
    f32x4 q[D / 8];
    fetch_row<D>(q, q_row);
    int large = flags_of(a.fk, zh, a.keys / 64, lane) | flags_of(a.fv, zh, a.keys / 64, lane);
    const int mine = take_parts<D>(xq, q);
    large |= a.fq ? flags_of(a.fq, zh, a.R, lane) : mine;
    if (__builtin_amdgcn_ballot_w64(large != 0)) run(Const<1>{});
    else run(Const<0>{});
  }

  // the two halves of the columns, each with its own reference m
  l += swap32(l);
  float *other = reinterpret_cast<float *>(smem) + rh * (16 * MT * 64 + 256);
  wait_barrier<0>();                                    // the ring is free
  if (kh) {
    put_sums<D>(other, o, lane);
    other[16 * MT * 64 + lane] = m;
    other[16 * MT * 64 + 64 + lane] = l;
    reinterpret_cast<int *>(other)[16 * MT * 64 + 128 + lane] = rows_seen;
  }
  wait_barrier<0>();
  if (!kh) {
    const float m1 = other[16 * MT * 64 + lane], l1 = other[16 * MT * 64 + 64 + lane];
    rows_seen |= reinterpret_cast<const int *>(other)[16 * MT * 64 + 128 + lane];
    const float top = fmaxf(m, m1), ms = top == -INFINITY ? 0.f : top, f0 = exp_of<false>(m - ms), f1 = exp_of<false>(m1 - ms);
    const float sum = l * f0 + l1 * f1;
    const bool any_block = (rows_seen >> 4 * ((lane >> 4) & 1)) & 15;
    const float inv = any_block ? 1.f / sum : 0.f;      // masked everywhere: 0 * inf = NaN, as the softmax operator gives; no block at all: zeros
    const float last = inv * down;
    take_sums<D>(other, o, lane, [&](float a0, float a1) { return (a0 * f0 + a1 * f1) * last; });
    if (a.lse != nullptr && half == 0) {
      float *to = a.lse + zh * a.row_sh + row;
      to[0] = ms;
      to[a.rest] = inv * share * kUp;
    }
  }
  wait_barrier<0>();
  if (!kh) {
    float *po = reinterpret_cast<float *>(a.o) + z * a.o_sz + h * a.o_sh + ((int64_t)line * 64 + 32 * rh) * a.o_ld;
    float *stage = reinterpret_cast<float *>(smem) + rh * 32 * (D + 4);
    store_32_f32<D>(stage, po, po + 16 * a.o_ld, a.o_ld, o, lane);
    if (a.o2 != nullptr) {
      float *copy = reinterpret_cast<float *>(a.o2) + (zh * a.rows + (int64_t)line * 64 + 32 * rh) * D;
      store_32_f32<D>(stage, copy, copy + 16 * D, D, o, lane);
    }
  }
}

// ---- backward, rows: dq and -delta ----
template <int D, bool KPM> __global__ void __launch_bounds__(256, D == 64 ? 2 : 1) k_attn32_bwd_rows(F32Args a) {
  typedef Ring<D> R;
  constexpr int MT = D / 32, NK = PieceLoad<D>::COUNT + (KPM ? 1 : 0);
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float *side = reinterpret_cast<float *>(smem + 3 * R::PIECE);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5, rh = wave & 1, kh = wave >> 1;
  const int64_t wg = place(a, (int64_t)a.Z * a.H * a.R);
  int line, zh;
  line_of(wg, a, line, zh);
  const int h = zh % a.H, z = zh / a.H;
  const table_ptr lut = as_table(a.lut);
  const int tiles = lut[2 * (h * a.R + line)];
  const table_ptr core = lut + lut[2 * (h * a.R + line) + 1];
  const int64_t row = (int64_t)line * 64 + 32 * rh + l32;
  float last = 1.f;
  bool parts = false;
  f32x16 dq[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) dq[mt][i] = 0.f;
  // the rows' do, and delta
  const float *do_row = reinterpret_cast<const float *>(a.d_o) + z * a.do_sz + h * a.do_sh + row * a.do_ld + 8 * half;
  const float *o_row = reinterpret_cast<const float *>(a.o_in) + z * a.oin_sz + h * a.oin_sh + row * a.oin_ld + 8 * half;
  if (tiles > 0) {
    Parts xq[D / 16], xo[D / 16];
    const bf16 *q_row = reinterpret_cast<const bf16 *>(a.q) + (zh * a.rows + row) * (3 * D) + 8 * half;
    const float m = a.lse[zh * a.row_sh + row], inv = a.lse[zh * a.row_sh + a.rest + row];
    const char *pk = reinterpret_cast<const char *>(reinterpret_cast<const bf16 *>(a.k) + zh * a.keys * (3 * D));
    const char *pv = reinterpret_cast<const char *>(reinterpret_cast<const bf16 *>(a.v) + zh * a.keys * (3 * D));
    const char *pkpm = reinterpret_cast<const char *>(reinterpret_cast<const float *>(a.kpm) + z * a.kpm_sz);
    PieceLoad<D> load;
    load.init(lane);
    RowReads<D, true> rows;
    TrReads<D, true> tr;
    rows.init(32 * kh, lane);
    tr.init(lds_address(smem), 32 * kh, lane);
    const float *kp_lane = side + (2 * kh + ((lane >> 3) & 1)) * 128 + 8 * half + (lane & 7);
    int pos_next = core[wave], pos = 0, bits_next = 0;   // (as in the forward kernel)
    auto issue_v = [&](int n, int slot) {
      pos = pos_next;
      load.issue(pv, pos, lds_address(smem) + slot * R::PIECE, wave);
      pos_next = core[kEntry * (n + 1 < tiles ? n + 1 : n) + wave];
    };
    auto issue_k = [&](int n, int slot) {
      load.issue(pk, pos, lds_address(smem) + slot * R::PIECE, wave);
      if constexpr (KPM) load_to_lds<4>(pkpm, (uint32_t)(pos + (lane & 15)) * 4u, 0, lds_address(side) + slot * R::SIDE + wave * 512);
      bits_next = core[kEntry * n + 4];
    };
    issue_v(0, 0);
    issue_k(0, 1);
    f32x4 g[D / 8], o[D / 8];
    fetch_row<D>(g, do_row);
    fetch_row<D>(o, o_row);
    int large = forward_flags(a, zh, a.R, lane);
    const bool by_parts = !__builtin_amdgcn_ballot_w64(large != 0);   // the scores, as in the forward pass
    const float sc = by_parts ? a.scale * kDown2 : a.scale;
    const int mine = take_parts<D>(xo, g);
    large |= a.fdo ? flags_of(a.fdo, zh, a.R, lane) : mine;
    f32x16 dp;
    auto run = [&](auto whole) {
      constexpr bool W = decltype(whole)::value;
      const float delta = delta_of<W, D>(o, xo, g, lane);
      const float up = delta * -kUp;
      parts = !W;
      last = inv * kDown;
      if (a.delta != nullptr && half == 0 && kh == 0) a.delta[zh * a.rows + row] = -delta;
      __builtin_amdgcn_sched_barrier(0);                // (q takes the registers of o and do)
      if constexpr (!W) load_parts<D>(xq, q_row);
      int here = 0;
      walk<PieceLoad<D>::COUNT, NK>(tiles, issue_v, issue_k,
        [&](int x, int) {
          here = bits_next >> (8 * rh + 2 * kh);
#pragma unroll
          for (int i = 0; i < 16; i++) dp[i] = 0.f;
          dp = rows_times<W, false, D>(smem + x * R::PIECE, rows, xo, do_row, false, dp);
        },
        [&](int y, int) {
          f32x16 s;
#pragma unroll
          for (int i = 0; i < 16; i++) s[i] = 0.f;
          s = rows_times<W, false, D>(smem + y * R::PIECE, rows, xq, q_row, by_parts, s);
          const float kp = KPM ? pad_term(kp_lane[y * (R::SIDE / 4)], a.kpm_mul) : 0.f;
          const int mine = here >> ((lane >> 4) & 1) * 4;
          float e[16];                                  // (1 / l of the row and the scale come last, on dq, unless W)
          for_16<0>([&](auto ic) {
            constexpr int i = decltype(ic)::value;
            const float x = exp_of<W>((KPM ? fmaf(s[i], sc, row_bcast<i>(kp)) : s[i] * sc) - m);
            e[i] = W ? x * (inv * kDown) * (dp[i] - delta) * a.scale : x * fmaf(dp[i], kDown, up);
          });
          if ((here & 0x33) != 0x33) {                  // pieces without a block
#pragma unroll
            for (int i = 0; i < 16; i++) e[i] = mine >> (i >> 3) & 1 ? e[i] : 0.f;
          }
          columns_times<W, false, D>(dq, y * R::PIECE, tr, e, mine & 1, mine & 2);
        });
    };
    if (__builtin_amdgcn_ballot_w64(large != 0)) run(Const<1>{});
    else run(Const<0>{});
  }
  float *other = reinterpret_cast<float *>(smem) + rh * (16 * MT * 64);
  wait_barrier<0>();
  if (kh) put_sums<D>(other, dq, lane);
  wait_barrier<0>();
  if (!kh) {
    const ScaledDown scaled(a.scale);
    take_sums<D>(other, dq, lane, [&](float a0, float a1) { return parts ? scaled((a0 + a1) * last) : a0 + a1; });
  }
  wait_barrier<0>();
  if (!kh) {
    float *po = reinterpret_cast<float *>(a.o) + z * a.o_sz + h * a.o_sh + ((int64_t)line * 64 + 32 * rh) * a.o_ld;
    store_32_f32<D>(reinterpret_cast<float *>(smem) + rh * 32 * (D + 4), po, po + 16 * a.o_ld, a.o_ld, dq, lane);
  }
}

// ---- backward, columns: dk and dv (work items as in attention_bwd.hip) ----
template <int D, bool KPM> __global__ void __launch_bounds__(256, D == 64 ? 2 : 1) k_attn32_bwd_cols(F32Args a) {
  typedef Ring<D> R;
  constexpr int MT = D / 32, NX = PieceLoad<D>::COUNT + 2;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  float *side = reinterpret_cast<float *>(smem + 3 * R::PIECE);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31, half = lane >> 5, kh = wave & 1, rh = wave >> 1;       // the wavefront's keys and rows of a tile
  const int64_t work = place(a, (int64_t)a.Z * a.R * a.sub), wg = work / a.sub;     // the pieces of an item side by side
  const bool in_turn = a.Z * a.H < 8 * kHeadsTogether;  // (then the long items of all batches come first)
  const int item = (int)(in_turn ? wg / a.Z : wg % a.R), z = (int)(in_turn ? wg % a.Z : wg / a.R);
  const table_ptr lut = as_table(a.lut), head = lut + 12 * item;
  int tiles = head[0], slot_no = head[4];
  const int h = head[2];
  table_ptr core = lut + head[1];
  if (a.sub > 1) {
    const int piece = (int)(work % a.sub);
    if (slot_no < 0) {                                  // not a part of a long column: one piece
      if (piece) return;
    } else {
      const int from = (int)((int64_t)tiles * piece / a.sub), upto = (int)((int64_t)tiles * (piece + 1) / a.sub);
      core += kEntry * from;
      tiles = upto - from;
      slot_no = slot_no * a.sub + piece;
    }
  }
  const int64_t key_lo = head[8 + 2 * kh], key_hi = head[8 + 2 * kh + 1], zh = (int64_t)z * a.H + h;
  bool parts = false;
  f32x16 dk[MT], dv[MT];
#pragma unroll
  for (int mt = 0; mt < MT; mt++)
#pragma unroll
    for (int i = 0; i < 16; i++) dk[mt][i] = dv[mt][i] = 0.f;

  if (tiles > 0) {
    const int64_t key = (l32 < 16 ? key_lo : key_hi) + (l32 & 15);
    Parts xk[D / 16], xv[D / 16];
    const bf16 *k_row = reinterpret_cast<const bf16 *>(a.k) + (zh * a.keys + key) * (3 * D) + 8 * half;
    const bf16 *v_row = reinterpret_cast<const bf16 *>(a.v) + (zh * a.keys + key) * (3 * D) + 8 * half;
    const float kp = KPM ? pad_term((reinterpret_cast<const float *>(a.kpm) + z * a.kpm_sz)[key], a.kpm_mul) : 0.f;
    const char *pq = reinterpret_cast<const char *>(reinterpret_cast<const bf16 *>(a.q) + zh * a.rows * (3 * D));
    const char *pdo = reinterpret_cast<const char *>(reinterpret_cast<const bf16 *>(a.d_o) + zh * a.rows * (3 * D));
    const char *pstat = reinterpret_cast<const char *>(a.lse + zh * a.row_sh), *pdelta = reinterpret_cast<const char *>(a.delta + zh * a.rows);
    const uint32_t to_inv = lane & 16 ? (uint32_t)a.rest * 4u : 0u;
    PieceLoad<D> load;
    load.init(lane);
    RowReads<D, true> rows;
    TrReads<D, true> tr;
    rows.init(32 * rh, lane);
    tr.init(lds_address(smem), 32 * rh, lane);
    const float *rv = side + 2 * rh * 128 + 8 * half;   // per group of sixteen rows: m (16 floats), 1 / l (16), 32 more; -delta
    int pos_next = core[wave], pos = 0, bits = 0, bits_next = core[4];
    auto issue_q = [&](int n, int slot) {
      pos = pos_next;
      load.issue(pq, pos, lds_address(smem) + slot * R::PIECE, wave);
      const uint32_t at = (uint32_t)(pos + (lane & 15)) * 4u, to = lds_address(side) + slot * R::SIDE + wave * 512;
      load_to_lds<4>(pstat, at + to_inv, 0, to);
      load_to_lds<4>(pdelta, at, 0, to + 256);
      pos_next = core[kEntry * (n + 1 < tiles ? n + 1 : n) + wave];
    };
    auto issue_do = [&](int n, int slot) {              // (pos is still that of tile n: the next tile's q is asked for after it)
      load.issue(pdo, pos, lds_address(smem) + slot * R::PIECE, wave);
      bits = bits_next;
      bits_next = core[kEntry * (n + 1 < tiles ? n + 1 : n) + 4];
    };
    float p[16];
    bool by_parts;
    auto run = [&](auto whole) {
      constexpr bool W = decltype(whole)::value;
      parts = !W;
      const float sc = by_parts ? a.scale * kDown2 : a.scale;
      if constexpr (!W) {
        own_parts<D>(xk, smem + R::PIECE, 32 * kh + l32, half);
        own_parts<D>(xv, smem + 2 * R::PIECE, 32 * kh + l32, half);
      }
      int here = 0;
      walk_x_twice<NX>(tiles, issue_q, issue_do,
        [&](int x, int) {
          f32x16 s;
#pragma unroll
          for (int i = 0; i < 16; i++) s[i] = 0.f;
          s = rows_times<W, true, D>(smem + x * R::PIECE, rows, xk, k_row, by_parts, s);
          here = bits >> (2 * kh + 8 * rh);
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const float *at = rv + x * (R::SIDE / 4) + (g >> 1) * 128 + 4 * (g & 1);
            const f32x4 m = *reinterpret_cast<const f32x4 *>(at), inv = *reinterpret_cast<const f32x4 *>(at + 16);
#pragma unroll
            for (int i = 0; i < 4; i++) p[4 * g + i] = exp_of<W>((KPM ? fmaf(s[4 * g + i], sc, kp) : s[4 * g + i] * sc) - m[i]) * (W ? inv[i] * kDown : inv[i]);
          }
          if ((here & 0x33) != 0x33) {                  // pieces without a block (a row that is masked everywhere has NaN here, which its other keys must not take up)
            const int mine = here >> ((lane >> 4) & 1);
#pragma unroll
            for (int i = 0; i < 16; i++) p[i] = mine >> 4 * (i >> 3) & 1 ? p[i] : 0.f;
          }
        },
        [&](int x, int y, int) {
          const int mine = here >> ((lane >> 4) & 1);
          f32x16 dp;
#pragma unroll
          for (int i = 0; i < 16; i++) dp[i] = 0.f;
          dp = rows_times<W, true, D>(smem + y * R::PIECE, rows, xv, v_row, false, dp);
          float e[16];
#pragma unroll
          for (int g = 0; g < 4; g++) {
            const f32x4 nd = *reinterpret_cast<const f32x4 *>(rv + x * (R::SIDE / 4) + (g >> 1) * 128 + 4 * (g & 1) + 64);
#pragma unroll
            for (int i = 0; i < 4; i++) e[4 * g + i] = W ? p[4 * g + i] * (dp[4 * g + i] + nd[i]) * a.scale : p[4 * g + i] * fmaf(dp[4 * g + i], kDown2, nd[i]);
          }
          if ((here & 0x33) != 0x33)
#pragma unroll
            for (int i = 0; i < 16; i++) e[i] = mine >> 4 * (i >> 3) & 1 ? e[i] : 0.f;
          columns_times<W, true, D>(dv, y * R::PIECE, tr, p, mine & 1, mine & 16);
          columns_times<W, true, D>(dk, x * R::PIECE, tr, e, mine & 1, mine & 16);
        });
    };
    issue_q(0, 0);
    // the column's own rows through the slots that are free yet: fetched by whole lines
    load.issue(reinterpret_cast<const char *>(reinterpret_cast<const bf16 *>(a.k) + zh * a.keys * (3 * D)), head[8 + wave], lds_address(smem) + R::PIECE, wave);
    load.issue(reinterpret_cast<const char *>(reinterpret_cast<const bf16 *>(a.v) + zh * a.keys * (3 * D)), head[8 + wave], lds_address(smem) + 2 * R::PIECE, wave);
    int large = forward_flags(a, zh, a.rows / 64, lane);
    by_parts = !__builtin_amdgcn_ballot_w64(large != 0);
    large |= flags_of(a.fdo, zh, a.rows / 64, lane);
    wait_barrier<0>();
    if (__builtin_amdgcn_ballot_w64(large != 0)) run(Const<1>{});
    else run(Const<0>{});
  }
  float *other = reinterpret_cast<float *>(smem) + kh * (2 * 16 * MT * 64);
  wait_barrier<0>();
  if (rh) {
    put_sums<D>(other, dk, lane);
    put_sums<D>(other + 16 * MT * 64, dv, lane);
  }
  wait_barrier<0>();
  if (!rh) {
    const ScaledDown scaled(a.scale);
    take_sums<D>(other, dk, lane, [&](float a0, float a1) { return parts ? scaled(a0 + a1) : a0 + a1; });
    take_sums<D>(other + 16 * MT * 64, dv, lane, [&](float a0, float a1) { return parts ? (a0 + a1) * kDown2 : a0 + a1; });
  }
  wait_barrier<0>();
  if (rh) return;
  if (slot_no >= 0) {                                   // a part of a long column: its sums to its slot [dk, dv][64 keys][D]
    float *ws = a.partial + ((int64_t)z * a.n_slots * a.sub + slot_no) * (2 * 64 * D) + (32 * kh + l32) * D + 4 * half;
#pragma unroll
    for (int j = 0; j < MT; j++)
#pragma unroll
      for (int g = 0; g < 4; g++) {
        *reinterpret_cast<f32x4 *>(ws + 32 * j + 8 * g) = f32x4{dk[j][4 * g], dk[j][4 * g + 1], dk[j][4 * g + 2], dk[j][4 * g + 3]};
        *reinterpret_cast<f32x4 *>(ws + 64 * D + 32 * j + 8 * g) = f32x4{dv[j][4 * g], dv[j][4 * g + 1], dv[j][4 * g + 2], dv[j][4 * g + 3]};
      }
    return;
  }
  float *stage = reinterpret_cast<float *>(smem) + kh * 32 * (D + 4);
  float *pdk = reinterpret_cast<float *>(a.o) + z * a.o_sz + h * a.o_sh, *pdv = reinterpret_cast<float *>(a.o2) + z * a.o2_sz + h * a.o2_sh;
  store_32_f32<D>(stage, pdk + key_lo * a.o_ld, pdk + key_hi * a.o_ld, a.o_ld, dk, lane);
  store_32_f32<D>(stage, pdv + key_lo * a.o2_ld, pdv + key_hi * a.o2_ld, a.o2_ld, dv, lane);
}

// dk and dv of the columns computed in parts: the slots of a column in order (split_lut as in attention_bwd.hip)
template <int D> __global__ void __launch_bounds__(256) k_attn32_cols_sum(F32Args a) {
  constexpr int WGS = 2 * 64 * D / 4 / 256;            // four values a thread
  const int piece = blockIdx.x % WGS, col = (blockIdx.x / WGS) % a.n_split, z = (blockIdx.x / WGS) / a.n_split;
  const table_ptr lut = as_table(a.split_lut) + 8 * col;
  const int h = lut[0], first = lut[2] * a.sub, parts = lut[3] * a.sub;
  const float *ws = a.partial + ((int64_t)z * a.n_slots * a.sub + first) * (2 * 64 * D);
  const int g = piece * 256 + threadIdx.x, which = g / (16 * D), rem = g % (16 * D), key = rem / (D / 4), d4 = rem % (D / 4);
  f32x4 sum = *reinterpret_cast<const f32x4 *>(ws + 4 * g);
  for (int part = 1; part < parts; part++) {
    const f32x4 v = *reinterpret_cast<const f32x4 *>(ws + (int64_t)part * (2 * 64 * D) + 4 * g);
#pragma unroll
    for (int e = 0; e < 4; e++) sum[e] += v[e];
  }
  const int64_t pos = (key < 32 ? (key < 16 ? lut[4] : lut[5]) : (key < 48 ? lut[6] : lut[7])) + (key & 15);
  float *dst = which ? reinterpret_cast<float *>(a.o2) + z * a.o2_sz + h * a.o2_sh + pos * a.o2_ld
                     : reinterpret_cast<float *>(a.o) + z * a.o_sz + h * a.o_sh + pos * a.o_ld;
  *reinterpret_cast<f32x4 *>(dst + 4 * d4) = sum;
}

template <int D, bool KPM, int WHICH> int launch(const F32Args &a, unsigned n_wg, hipStream_t st) {
  static std::atomic<uint64_t> done{0};
  void (*kernel)(F32Args) = WHICH == 0 ? k_attn32_fwd<D, KPM> : WHICH == 1 ? k_attn32_bwd_rows<D, KPM> : k_attn32_bwd_cols<D, KPM>;
  if (!raise_lds_limit(reinterpret_cast<const void *>(kernel), Ring<D>::BYTES, done)) return BSP_ERR_HIP;
  hipLaunchKernelGGL(kernel, dim3(n_wg), dim3(256), Ring<D>::BYTES, st, a);
  return BSP_OK;
}
template <int WHICH> int launch_d(const F32Args &a, int D, int64_t n_wg, hipStream_t st) {
  if (D == 64) return a.kpm ? launch<64, true, WHICH>(a, (unsigned)n_wg, st) : launch<64, false, WHICH>(a, (unsigned)n_wg, st);
  return a.kpm ? launch<128, true, WHICH>(a, (unsigned)n_wg, st) : launch<128, false, WHICH>(a, (unsigned)n_wg, st);
}

// planes of a tensor of n rows in all: [n][3][D] bf16, then its flags, an int for 64 rows; a multiple of 16 bytes
inline int64_t plane_bytes(int64_t n, int D) { return n * 3 * D * 2 + (n / 64 * 4 + 15) / 16 * 16; }
inline int32_t *flags_in(void *planes, int64_t n, int D) { return reinterpret_cast<int32_t *>(reinterpret_cast<char *>(planes) + n * 3 * D * 2); }

// sizes, 16-byte alignment of pointers (NULL is aligned) and strides (n tensors: batch, head, row; multiples of 4 floats), rows that hold D
int f32_check(const bsp_attention_f32_call &c, const void *const *ptrs, int n_ptrs, int n) {
  if (c.Z <= 0 || c.H <= 0 || c.R <= 0 || c.keys <= 0 || c.keys % 64 || !c.planes) return BSP_ERR_ARG;
  if (c.D != 64 && c.D != 128) return BSP_ERR_UNSUPPORTED;
  for (int i = 0; i < n_ptrs; i++)
    if (reinterpret_cast<uintptr_t>(ptrs[i]) & 15) return BSP_ERR_ARG;
  for (int i = 0; i < 3 * n; i++)
    if (c.strides[i] % 4 || (i % 3 == 2 && c.strides[i] < c.D)) return BSP_ERR_ARG;
  const int64_t most = c.keys > (int64_t)c.R * 64 ? c.keys : (int64_t)c.R * 64;
  // workgroups of a launch, and byte offsets within a head's planes, in 32 bits
  return (int64_t)c.Z * c.H * c.R >= ((int64_t)1 << 31) || most * 3 * c.D * 2 >= ((int64_t)1 << 32) ? BSP_ERR_UNSUPPORTED : BSP_OK;
}

// what both directions take from the call: sizes, masks, the parts of the buffer of k, v and q
F32Args f32_args(const bsp_attention_f32_call &c) {
  F32Args a{};
  a.Z = c.Z; a.H = c.H; a.R = c.R;
  a.rows = (int64_t)c.R * 64; a.keys = c.keys;
  a.lse = c.stats; a.rest = a.rows; a.row_sh = 2 * a.rows;
  a.scale = c.scale;
  a.kpm = c.kpm; a.kpm_sz = c.kpm_stride_z; a.kpm_mul = c.kpm_mul;
  const int64_t n = (int64_t)c.Z * c.H * c.keys;
  char *p = reinterpret_cast<char *>(c.planes);
  a.k = p; a.fk = flags_in(p, n, c.D);
  p += plane_bytes(n, c.D);
  a.v = p; a.fv = flags_in(p, n, c.D);
  p += plane_bytes(n, c.D);
  a.q = p; a.fq = flags_in(p, (int64_t)c.Z * c.H * a.rows, c.D);
  return a;
}
void take_strides(const int64_t *s, int64_t &z, int64_t &h, int64_t &row) { z = s[0]; h = s[1]; row = s[2]; }

// the planes of up to three tensors of rows rows a head and their flags (no planes: left out)
struct ToPlanes { const float *x; const void *planes; const int64_t *strides; int64_t rows; };
int launch_planes(const bsp_attention_f32_call &c, const ToPlanes (&tensors)[3], hipStream_t st) {
  const int64_t heads = (int64_t)c.Z * c.H;
  PlaneArgs pl{};
  pl.H = c.H;
  int64_t end = 0;
  for (int i = 0; i < 3; i++) {
    const ToPlanes &from = tensors[i];
    PlaneArgs::Tensor &t = pl.t[i];
    if (from.planes) {
      t.x = from.x;
      t.planes = reinterpret_cast<bf16 *>(const_cast<void *>(from.planes));
      t.flags = flags_in(t.planes, heads * from.rows, c.D);
      take_strides(from.strides, t.sz, t.sh, t.ld);
      t.chunks = (uint32_t)(from.rows / 64);
      end += heads * t.chunks;
    }
    if (end >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
    t.end = (uint32_t)end;
  }
  if (c.D == 64) hipLaunchKernelGGL(k_attn32_planes<64>, dim3((unsigned)end), dim3(256), 0, st, pl);
  else hipLaunchKernelGGL(k_attn32_planes<128>, dim3((unsigned)end), dim3(256), 0, st, pl);
  return BSP_OK;
}

// Pieces of the parts of long columns.  A part is up to sixteen tiles, eight times as long as the short columns of the layouts that have
// any: a launch of few parts ends with them alone and does better on halves, as long as every half has a compute unit of its own; each half costs
// a workgroup's first loads and a slot written and read once more.  Backward pass in 1 / 2 pieces, us: head dimension 64, 128 parts 100.6 / 92.9,
// 192 parts 157 / 176 and (columns of 128 keys' blocks) 278 / 269, 256 parts 155 / 155, 384 parts 197 / 204, 512 parts 233 / 248; 128, whose workgroups
// have a compute unit each: 128 parts 183 / 171, 192 parts 340 / 400, 256 parts 283 / 328, 512 parts 569 / 656.
int pieces(int64_t parts) { return parts > 0 && parts <= 128 ? 2 : 1; }

}  // namespace
}  // namespace bsp

using namespace bsp;

extern "C" int64_t bsp_attention_f32_bytes(int Z, int H, int64_t rows, int64_t keys, int D) {
  const int64_t heads = (int64_t)Z * H;
  return plane_bytes(heads * rows, D) + (keys ? 2 * plane_bytes(heads * keys, D) : 0);
}
extern "C" int64_t bsp_attention_f32_slots(int Z, int n_slots) { return (int64_t)Z * n_slots * pieces((int64_t)Z * n_slots); }

extern "C" int bsp_attention_f32_fwd(const bsp_attention_f32_call *c, const float *q, const float *k, const float *v, float *o, void *stream) {
  if (!c || !q || !k || !v || !o || !c->d_rows) return BSP_ERR_ARG;
  const void *ptrs[] = {q, k, v, o, c->planes, c->stats, c->kpm, c->o_copy};
  const int rc = f32_check(*c, ptrs, 8, 4);
  if (rc != BSP_OK) return rc;
  F32Args a = f32_args(*c);
  const int64_t heads = (int64_t)a.Z * a.H;
  hipStream_t st = as_stream(stream);
  const int rp = launch_planes(*c, {{k, a.k, c->strides + 3, a.keys}, {v, a.v, c->strides + 6, a.keys}, {q, c->stats ? a.q : nullptr, c->strides, a.rows}}, st);
  if (rp != BSP_OK) return rp;
  if (!c->stats) a.fq = nullptr;
  a.q = q;
  take_strides(c->strides, a.q_sz, a.q_sh, a.q_ld);
  a.o = o; a.o2 = c->o_copy;
  take_strides(c->strides + 9, a.o_sz, a.o_sh, a.o_ld);
  a.lut = c->d_rows;
  const int rl = launch_d<0>(a, c->D, heads * a.R, st);
  if (rl != BSP_OK) return rl;
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}

extern "C" int bsp_attention_f32_bwd(const bsp_attention_f32_call *c, const float *d_o, const float *o, float *dq, float *dk, float *dv, void *do_planes, float *neg_delta,
                                     const int32_t *d_items, int n_items, float *partial, int n_slots, const int32_t *d_split, int n_split, void *stream) {
  if (!c || !d_o || !o || !dq || !c->stats || !c->d_rows || (dk == nullptr) != (dv == nullptr) || (dk && (!do_planes || !neg_delta || !d_items))) return BSP_ERR_ARG;
  if (n_slots < 0 || n_split < 0 || (n_slots > 0) != (n_split > 0) || (dk && n_slots > 0 && (!partial || !d_split))) return BSP_ERR_ARG;
  const void *ptrs[] = {d_o, o, dq, dk, dv, do_planes, c->planes, c->stats, neg_delta, partial, c->kpm};
  const int rc = f32_check(*c, ptrs, 11, dk ? 5 : 3);
  if (rc != BSP_OK) return rc;
  F32Args a = f32_args(*c);
  a.sub = pieces((int64_t)a.Z * n_slots);
  if (dk && (n_items < (int64_t)a.H * (a.keys / 64) || n_items > (int64_t)a.H * (a.keys / 64) + n_slots || (int64_t)a.Z * n_items * a.sub >= ((int64_t)1 << 31) ||
             (int64_t)a.Z * n_split * 16 >= ((int64_t)1 << 31))) return BSP_ERR_ARG;
  hipStream_t st = as_stream(stream);
  a.d_o = d_o; a.o_in = o;
  if (dk) {
    const int rp = launch_planes(*c, {{d_o, do_planes, c->strides, a.rows}}, st);
    if (rp != BSP_OK) return rp;
    a.fdo = flags_in(do_planes, (int64_t)a.Z * a.H * a.rows, c->D);
    a.delta = neg_delta;
  }
  take_strides(c->strides, a.do_sz, a.do_sh, a.do_ld);
  take_strides(c->strides + 3, a.oin_sz, a.oin_sh, a.oin_ld);
  take_strides(c->strides + 6, a.o_sz, a.o_sh, a.o_ld);
  a.o = dq; a.lut = c->d_rows;
  int rl = launch_d<1>(a, c->D, (int64_t)a.Z * a.H * a.R, st);
  if (rl != BSP_OK) return rl;
  if (dk) {
    a.d_o = do_planes;
    take_strides(c->strides + 9, a.o_sz, a.o_sh, a.o_ld);
    take_strides(c->strides + 12, a.o2_sz, a.o2_sh, a.o2_ld);
    a.o = dk; a.o2 = dv; a.lut = d_items; a.R = n_items;
    a.partial = partial; a.n_slots = n_slots; a.split_lut = d_split; a.n_split = n_split;
    rl = launch_d<2>(a, c->D, (int64_t)a.Z * n_items * a.sub, st);
    if (rl != BSP_OK) return rl;
    if (n_split > 0) {
      const unsigned n_wg = (unsigned)((int64_t)a.Z * n_split * (2 * 64 * c->D / 4 / 256));
      if (c->D == 64) hipLaunchKernelGGL(k_attn32_cols_sum<64>, dim3(n_wg), dim3(256), 0, st, a);
      else hipLaunchKernelGGL(k_attn32_cols_sum<128>, dim3(n_wg), dim3(256), 0, st, a);
    }
  }
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}
