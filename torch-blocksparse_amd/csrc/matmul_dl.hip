// dsd / dds for a wide free dimension (a few hundred dense rows or more), blocks of 64 and 128, fp16 / bf16: the
// products that are bound by the matrix cores and by how fast tiles travel from L2 into the CUs, not by HBM
// (a block-sparse linear layer: 8192 tokens against a 4096 x 4096 weight in blocks of 128).
//
// Same work decomposition as the general kernel k_xsd (one workgroup per table segment and 256-wide tile of the free
// dimension, tables and semantics of the reference's DSD / DDS branches, matmul.py:56-99), other pipeline:
//   * operand tiles go from global memory straight into LDS (global_load_lds_dwordx4: 16 bytes per lane, 1 KiB of
//     consecutive LDS per wavefront-level load): no staging registers, no LDS store instructions, and the only wait
//     for memory is the one in front of the barrier of a reduction step;
//   * a ring of three LDS stages, loads two reduction steps (of 32) ahead of their use, one barrier per step;
//   * conflict-free LDS reads through an XOR swizzle of the 16-byte chunks, applied by choosing which global chunk
//     each lane fetches (the data lands where the swizzled layout wants it);
//   * all eight orientations (sparse operand as stored / transposed, dense operand with the reduction contiguous or
//     strided, result written along either index): a tile whose reduction index is strided in memory is kept as it
//     lies and read with the transposing LDS load.
//   * the ring is walked in rounds of three steps, so that a stage is a constant: LDS addresses are registers made before the
//     loop plus immediates, and a load is a scalar base plus a 32-bit register.  With the stage a run-time value a step
//     spent some 250 instructions per wavefront on addresses and bookkeeping and was bound by issuing them: fp16, 8 products
//     of 2048^3 at a quarter of the blocks, dsd at block 32 107 -> 85 us, 64 87-90 -> 74-89, 128 91 -> 82; sdd at
//     block 32 127 -> 105-108 (125 with both reductions contiguous); the block-16 sdd over a hidden size of 512 131 -> 116.
//     (Measured slower: reduction steps of 64, full 128-byte lines, eight wavefronts a CU: sdd 129 -> 152; six stages and
//     one workgroup per CU, at any launch size: dsd at block 32 25 -> 37 us for 1024^3.)
// A standalone dense probe of this pipeline (128 x 256 x 32 tiles) reaches 0.9 PFLOP/s on an 8192 x 4096 x 4096
// product where the register-staged general kernel reaches 0.75.
#include "matmul_generic.h"
#include <algorithm>
#include <vector>

namespace bsp {
namespace {

constexpr int kTK = 32;          // reduction step (elements)
constexpr int kTN = 256;         // tile of the dense free dimension
constexpr int kStages = 3;

// Sixteen bytes per lane from base (the same in all lanes) + off to LDS byte dst + 16 * lane (dst the same in all lanes).  As
// assembly and not as the builtin: the compiler cannot tell which stage of the ring a load fills, and in front of every
// transposing LDS read it would wait for all loads in flight (s_waitcnt vmcnt(0) once or several times per reduction
// step), which leaves nothing of the prefetch.  The waits are the counted ones of BSP_WAIT_VM alone.  The scalar no-op
// is the wait state between the write of m0 and its use.  Measured against the builtin, fp16, 4 x 8 products of 2048^3 at a
// quarter of the blocks: dsd with the dense operand's reduction strided 286 -> 247 us at block 64 and 228 -> 199 at 128, sdd of
// 2 x 4 such products with a strided operand 153-162 -> 121-133 at block 32; kernels that read both tiles along the
// reduction are as fast as before.  dsd with the sparse operand transposed and the dense reduction contiguous comes here for the
// same reason: 299 us in the general kernel, 270 here at block 64, 231 and 210 at 128.
__device__ __forceinline__ void load_lds16(const void *base, uint32_t off, const unsigned char *dst) {
  const uint32_t at = (uint32_t)(uintptr_t)((const void __attribute__((address_space(3))) *)dst);
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "s"(at) : "m0", "memory");
}
template <int N> struct Const { static constexpr int value = N; };
// step(stage, s) for s = 0 .. n - 1, the stage (s modulo the ring's length) a compile-time constant: the LDS addresses of a
// stage are then immediates of its reads
template <int S = 0, class F> __device__ __forceinline__ void ring_round(int s, int n, F &&step) {
  step(Const<S>{}, s + S);
  if constexpr (S + 1 < kStages)
    if (s + S + 1 < n) ring_round<S + 1>(s, n, step);
}
// Wait until at most n vector-memory operations of this wavefront are outstanding and all of its LDS reads have
// returned.  It stands before the barrier of a reduction step, behind which other wavefronts start the direct-to-LDS
// loads that overwrite the stage read last: a read still in flight then could return the new bytes.  (In these
// kernels the matrix instructions that consume a step's reads come before the barrier in the compiled code, so the
// reads have returned anyway; the explicit wait does not leave that to the instruction scheduler.)
#define BSP_WAIT_VM(n) __builtin_amdgcn_s_waitcnt(((n) & 0xF) | (((n) >> 4) << 14) | (0x7 << 4) | (0x0 << 8))

// ---- LDS tile layouts (byte offsets) ------------------------------------------------------------------------
// Reduction contiguous: [row][4 chunks of 16 bytes]; chunk c of row r sits at chunk slot c ^ ((r >> 2) & 3).  A 128-bit
// read is served sixteen lanes (rows) per clock from 64 banks: rows r, r + 4, r + 8, r + 12 start in the same bank and
// get four different slots.  (Measured: with the slot c ^ ((r >> 1) & 3), which suits 32 banks, half of the LDS-active
// cycles were bank conflicts; with this one 7-17 %.)
__device__ __forceinline__ int kc_swz(int row) { return (row >> 2) & 3; }
__device__ __forceinline__ int kc_offset(int row, int chunk) { return row * 64 + ((chunk ^ kc_swz(row)) << 4); }
// Reduction strided: [32 reduction indices][R elements], as in memory.  The transposing read of a 16-lane group takes
// 32 contiguous bytes (a pair of chunks) from each of four consecutive reduction rows, and two such groups (neighbouring
// pairs p, p + 1 of the same four rows) are served together: eight pieces of 32 bytes that should cover the 64 banks
// once.  R >= 128 (a row is a multiple of 256 bytes: every row starts in bank 0): pair p of row k sits at pair slot
// p ^ 2 (k & 3), so the even pair lands on the four even slots and the odd pair on the four odd ones (with p ^ (k & 3)
// the two groups met in the same four slots: half of the LDS cycles of the kernels that read both operands this way
// were bank conflicts).  R = 64 (128-byte rows: two rows per bank period): p ^ (k & 3).  R = 32 (a row is 2 pairs,
// rows k and k + 2 start in the same bank): p ^ ((k >> 1) & 1).
template <int R> __device__ __forceinline__ int ks_swz(int k) { return R >= 128 ? ((k & 3) << 1) : R >= 64 ? (k & 3) : ((k >> 1) & 1); }
template <int R> __device__ __forceinline__ int ks_offset(int k, int col) {   // col in elements, multiple of 4
  const int chunk = col >> 3, pair = (chunk >> 1) ^ ks_swz<R>(k);
  return k * (R * 2) + (((pair << 1) | (chunk & 1)) << 4) + ((col & 7) << 1);
}

// One operand tile of a stage: ROWS rows of the tile index (m or n) by kTK reduction indices.
template <typename T, int ROWS, bool KCONTIG> struct DlTile {
  static constexpr int BYTES = ROWS * kTK * 2;
  static constexpr int LOADS = BYTES / 1024;          // wavefront-level loads per stage
  static_assert(KCONTIG || ROWS >= 32, "a reduction row holds at least two pairs of chunks");
  // Global byte offset (relative to the tile's origin) of the chunk that lane `lane` of load `ld` fetches, as
  // (row index, reduction index): rows advance by `row_stride` elements, reduction indices by `k_stride`.
  __device__ __forceinline__ static uint32_t lane_offset(int ld, int lane, int64_t row_stride, int64_t k_stride) {
    if constexpr (KCONTIG) {
      const int row = ld * 16 + (lane >> 2), slot = lane & 3;
      const int chunk = slot ^ kc_swz(row);      // the global chunk that belongs into this LDS slot
      return (uint32_t)(row * row_stride + chunk * 8 * k_stride) * 2u;
    } else {
      constexpr int CPR = ROWS / 8;                    // chunks per reduction row
      const int j = ld * 64 + lane, k = j / CPR, slot = j % CPR;
      const int pair = (slot >> 1) ^ ks_swz<ROWS>(k);
      return (uint32_t)(k * k_stride + (((pair << 1) | (slot & 1)) * 8) * row_stride) * 2u;
    }
  }
  // MFMA operand (32 x 16 slice): rows row0 .. row0 + 31 of the tile, reduction indices 16 * kk ..; lane l supplies row
  // l % 32, indices 8 * (l / 32) .. + 7
  __device__ __forceinline__ static typename Mma<T, 32>::frag_t frag(const unsigned char *tile, int row0, int kk, int lane) {
    typedef typename Mma<T, 32>::frag_t frag_t;
    if constexpr (KCONTIG) {
      return *reinterpret_cast<const frag_t *>(tile + kc_offset(row0 + (lane & 31), kk * 2 + (lane >> 5)));
    } else {
      typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
      const int t = lane & 15, gi = lane >> 4;
      const int k = kk * 16 + 8 * (gi >> 1) + (t >> 2), col = row0 + 16 * (gi & 1) + 4 * (t & 3);
      s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + ks_offset<ROWS>(k, col)));
      s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(tile + ks_offset<ROWS>(k + 4, col)));
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      return __builtin_bit_cast(frag_t, v);
    }
  }
};

// N consecutive ints per entry of a table, read by the whole wavefront: lane l holds entry 64 w + l of the window w in use, and
// an entry of the window is N readlanes.  A reduction step that reads its entry from memory (scalar loads share their
// counter with the LDS reads, and return in any order) waits for that read before its first matrix instruction.
template <int N> struct TableWindow {
  const int32_t *first;
  int entries, at;                                    // entries of the table; first entry of the window, -1: none yet
  int v[N];
  __device__ __forceinline__ TableWindow(const int32_t *first_, int entries_) : first(first_), entries(entries_), at(-1) {}
  __device__ __forceinline__ void get(int e, int lane, int (&out)[N]) {   // e (the same in all lanes) below `entries`
    if ((e & ~63) != at) {
      at = e & ~63;
      const int mine = at + lane < entries ? at + lane : entries - 1;
#pragma unroll
      for (int i = 0; i < N; i++) v[i] = first[(int64_t)N * mine + i];
#pragma unroll
      for (int i = 0; i < N; i++) asm volatile("" : "+v"(v[i]));          // (wait for them here, not at every use)
    }
#pragma unroll
    for (int i = 0; i < N; i++) out[i] = __builtin_amdgcn_readlane(v[i], e & 63);
  }
};

template <typename T, int BLOCK, bool SP_TRANS, bool DN_KC, bool OUT_NC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) k_xsd_dl(XsdArgs g) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  typedef DlTile<T, BLOCK, !SP_TRANS> XT;             // sparse block: rows m
  typedef DlTile<T, kTN, DN_KC> YT;                   // dense tile: rows n
  constexpr int STAGE = XT::BYTES + YT::BYTES;
  constexpr int WGM = BLOCK >= 128 ? 2 : 1, WGN = 4 / WGM;          // wavefronts along m and n
  constexpr int RM = BLOCK / (32 * WGM), RN = kTN / (32 * WGN);     // 32 x 32 MFMA tiles per wavefront
  constexpr int XL = XT::LOADS / 4, YL = YT::LOADS / 4, L = XL + YL; // loads per wavefront and stage
  static_assert(XT::LOADS % 4 == 0 && YT::LOADS % 4 == 0, "the loads of a stage divide evenly among four wavefronts");
  constexpr int SPB = BLOCK / kTK;                    // reduction steps per block
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / WGN, wn = wave % WGN;

  const int n_tiles = (g.NF + kTN - 1) / kTN;
  int z, nt, seg0;
  xsd_work_item(g, n_tiles, blockIdx.x, z, nt, seg0);
  const int seg = g.order ? as_table(g.order)[seg0] : seg0;
  const table_ptr hd = as_table(g.lut) + 6 * (int64_t)seg;
  const int offset = hd[0], seglen = hd[1], column = hd[2], depth = hd[3];
  const int nblk = seglen / BLOCK;
  // a zero-length segment that follows a real one of the same line must not touch the output; one that stands alone
  // is an empty line and zero-fills its tile (as in k_xsd)
  if (nblk == 0 && seg > 0 && hd[-6 + 2] == column && hd[-6 + 3] == depth) return;
  TableWindow<2> plan(g.plan + 2 * (int64_t)((offset - 6 * g.width) / g.div2), nblk);
  const int n0 = nt * kTN, NF = g.NF;
  const int64_t ldd = g.ldd, ldo = g.ldo;
  const T *sp = reinterpret_cast<const T *>(g.sp) + z * g.sp_sz;
  const T *dn = reinterpret_cast<const T *>(g.dn) + z * g.dn_sz + depth * g.dn_sh + (DN_KC ? n0 * ldd : n0);
  T *oz = reinterpret_cast<T *>(g.out) + z * g.out_sz + depth * g.out_sh;

  // Per-lane part of every load address, computed once.  Sparse block element (m, k): stored [m][k] or, transposed,
  // [k][m], rows of BLOCK elements.  Dense element (n, k): [n][k] (reduction contiguous) or [k][n], rows of ldd; dense
  // rows past the free dimension read row NF - 1 instead (their results are not stored).
  uint32_t xoff[XL], yoff[YL];
#pragma unroll
  for (int i = 0; i < XL; i++)
    xoff[i] = SP_TRANS ? XT::lane_offset(wave * XL + i, lane, 1, BLOCK) : XT::lane_offset(wave * XL + i, lane, BLOCK, 1);
#pragma unroll
  for (int i = 0; i < YL; i++) {
    if constexpr (DN_KC) {
      const int ld = wave * YL + i, row = ld * 16 + (lane >> 2), chunk = (lane & 3) ^ kc_swz(row);
      const int n = n0 + row < NF ? row : NF - 1 - n0;
      yoff[i] = (uint32_t)(n * ldd + chunk * 8) * 2u;
    } else {
      constexpr int CPR = kTN / 8;
      const int j = (wave * YL + i) * 64 + lane, k = j / CPR, slot = j % CPR;
      const int chunk = (((slot >> 1) ^ ks_swz<kTN>(k)) << 1) | (slot & 1);
      const int n = n0 + chunk * 8 < NF ? chunk * 8 : NF - 8 - n0;   // whole chunks: NF is a multiple of 8
      yoff[i] = (uint32_t)(k * ldd + n) * 2u;
    }
  }
  typename M::acc_t acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; i++)
#pragma unroll
    for (int j = 0; j < RN; j++)
#pragma unroll
      for (int v = 0; v < M::NACC; v++) acc[i][j][v] = 0.f;

  const int ksteps = nblk * SPB;
  // loads of step s into stage st
  auto issue = [&](int s, unsigned char *st) {
    int e[2];                                          // position of the step's block in the dense operand, storage index of the block
    plan.get(s / SPB, lane, e);
    const int kin = (s % SPB) * kTK;
    const T *xb = sp + (int64_t)e[1] * (BLOCK * BLOCK) + (SP_TRANS ? kin * BLOCK : kin);
    const T *yb = dn + (DN_KC ? (int64_t)e[0] + kin : ((int64_t)e[0] + kin) * ldd);
#pragma unroll
    for (int i = 0; i < XL; i++)
      load_lds16(xb, xoff[i], st + (wave * XL + i) * 1024);
#pragma unroll
    for (int i = 0; i < YL; i++)
      load_lds16(yb, yoff[i], st + XT::BYTES + (wave * YL + i) * 1024);
  };
  if (nblk > 0) {
    static_assert(kStages == 3 && SPB >= 2, "the first two steps exist");
    issue(0, smem);
    issue(1, smem + STAGE);
    auto step = [&](auto stage, int s) {
      constexpr int S = decltype(stage)::value;
      // this wavefront's loads of step s have landed: all but those of the one step issued after them, or, at the
      // last step, all (no load is issued for steps past the end)
      if (s + 1 < ksteps) BSP_WAIT_VM(L * (kStages - 2));
      else BSP_WAIT_VM(0);
      asm volatile("" ::: "memory");                   // (the compiler must not move LDS accesses across the barrier)
      __builtin_amdgcn_s_barrier();                    // everybody's have, and everybody is done reading step s - 1
      asm volatile("" ::: "memory");
      if (s + 2 < ksteps) issue(s + 2, smem + (S + 2) % kStages * STAGE);   // into the stage that step s - 1 used
      const unsigned char *st = smem + S * STAGE;
      // operands of the second half of the step are fetched from LDS before the matrix instructions of the first
      frag_t xf[kTK / 16][RM], yf[kTK / 16][RN];
#pragma unroll
      for (int kk = 0; kk < kTK / 16; kk++) {
#pragma unroll
        for (int i = 0; i < RM; i++) xf[kk][i] = XT::frag(st, (wm * RM + i) * 32, kk, lane);
#pragma unroll
        for (int j = 0; j < RN; j++) yf[kk][j] = YT::frag(st + XT::BYTES, (wn * RN + j) * 32, kk, lane);
      }
#pragma unroll
      for (int kk = 0; kk < kTK / 16; kk++)
#pragma unroll
        for (int i = 0; i < RM; i++)
#pragma unroll
          for (int j = 0; j < RN; j++) {
            if constexpr (OUT_NC) acc[i][j] = M::run(yf[kk][j], xf[kk][i], acc[i][j]);   // 4 consecutive values run along n
            else acc[i][j] = M::run(xf[kk][i], yf[kk][j], acc[i][j]);                    // ... along m
          }
    };
    for (int s = 0; s < ksteps; s += kStages) ring_round(s, ksteps, step);
    BSP_WAIT_VM(0);                                    // (nothing is in flight any more unless the segment had a single step)
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // Epilogue: the whole tile through LDS (the ring is free now), then 16-byte stores along the output's contiguous
  // index, consecutive lanes on consecutive chunks.  Staged as [row][CW + 8] with CW = the contiguous extent: 256 (n)
  // or BLOCK (m).  acc[i][j][4g + e]: the A operand's row 8g + 4 * (lane / 32) + e, the B operand's row lane % 32.
  constexpr int CW = OUT_NC ? kTN : BLOCK, NR = OUT_NC ? BLOCK : kTN, LDR = CW + 8;
  static_assert(NR * LDR * 2 <= kStages * STAGE, "the staged tile fits into the ring");
  T *stage = reinterpret_cast<T *>(smem);
#pragma unroll
  for (int i = 0; i < RM; i++)
#pragma unroll
    for (int j = 0; j < RN; j++)
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++) {
        const int m0 = (wm * RM + i) * 32, nn0 = (wn * RN + j) * 32;
        const int fast = 8 * g4 + 4 * (lane >> 5), slow = lane & 31;
        const int row = OUT_NC ? m0 + slow : nn0 + slow, col = OUT_NC ? nn0 + fast : m0 + fast;
        union { u32x2 raw; T e[4]; } u;
#pragma unroll
        for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(acc[i][j][4 * g4 + e]);
        *reinterpret_cast<u32x2 *>(stage + row * LDR + col) = u.raw;
      }
  __syncthreads();
  constexpr int CHUNKS = NR * CW / 8;
#pragma unroll 4
  for (int c = tid; c < CHUNKS; c += 256) {
    const int row = c / (CW / 8), col = (c % (CW / 8)) * 8;
    const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + row * LDR + col);
    if constexpr (OUT_NC) {
      if (n0 + col < NF) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(oz + ((int64_t)column * BLOCK + row) * ldo + n0 + col));
    } else {
      if (n0 + row < NF) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(oz + (int64_t)(n0 + row) * ldo + column * BLOCK + col));
    }
  }
}

// ---------------------------------------------------------------------------------------------------------
// Blocks of 32 with a wide free dimension.  A 32-row line is too little work per byte fetched: with one line per
// workgroup every dense tile (32 reduction rows x 256 columns, 16 KiB) serves 32 output rows, and the launch is bound
// by the feed from L2 at a seventh of the matrix peak.  Here a workgroup owns a group of BSP_GROUP consecutive lines
// (the group plan of bsp_group_plan_build) and walks the union of their blocks: per entry one dense tile, fetched
// once, serves every member that has a block there.  Each wavefront owns 64 of the tile's 256 columns for all four
// members (its dense operands are read from LDS once per entry and used by up to four blocks) and loads one member's
// block; absent members load block 0 instead (a fixed number of loads per stage keeps the waits exact).
// Chains of the plan (long lines taken out of their groups) are groups with a single member here.
// ---------------------------------------------------------------------------------------------------------
template <typename T, bool SP_TRANS, bool DN_KC, bool OUT_NC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) k_xsd_rg_dl(XsdArgs g) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  constexpr int B = 32, G = BSP_GROUP;
  static_assert(G == 4, "one member block per wavefront");
  typedef DlTile<T, B, !SP_TRANS> XT;                 // a member's block: 2 KiB
  typedef DlTile<T, kTN, DN_KC> YT;                   // dense tile: 16 KiB
  constexpr int STAGE = G * XT::BYTES + YT::BYTES;
  constexpr int XL = XT::LOADS, YL = YT::LOADS / 4, L = XL + YL;   // loads per wavefront and stage
  constexpr int RN = kTN / (32 * 4);                  // 32-column tiles per wavefront
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n_tiles = (g.NF + kTN - 1) / kTN;
  const int64_t per_z = (int64_t)g.n_pgroups * n_tiles;
  const int64_t w = xcd_remap(blockIdx.x, per_z * g.Z);
  const int z = (int)(w / per_z);
  const int nt = (int)((w % per_z) / g.n_pgroups);
  const table_ptr hd = as_table(g.gplan) + 4 * ((w % per_z) % g.n_pgroups);
  const int e0 = hd[0], ne = hd[1], depth = hd[2], code = hd[3];
  const int32_t *entries = g.gplan + 4 * (int64_t)g.n_pgroups + (int64_t)(G + 1) * e0;
  const bool chain = code < 0;
  const int line0 = chain ? -(code + 1) : (code & 0xffffff) * G;
  const int absent = chain ? 0xe : ((code >> 24) & 0xf);            // members that are not this group's to compute
  const int n0 = nt * kTN, NF = g.NF;
  const int64_t ldd = g.ldd, ldo = g.ldo;
  const T *sp = reinterpret_cast<const T *>(g.sp) + z * g.sp_sz;
  const T *dn = reinterpret_cast<const T *>(g.dn) + z * g.dn_sz + depth * g.dn_sh + (DN_KC ? n0 * ldd : n0);
  T *oz = reinterpret_cast<T *>(g.out) + z * g.out_sz + depth * g.out_sh;

  uint32_t xoff[XL], yoff[YL];
#pragma unroll
  for (int i = 0; i < XL; i++) xoff[i] = SP_TRANS ? XT::lane_offset(i, lane, 1, B) : XT::lane_offset(i, lane, B, 1);
#pragma unroll
  for (int i = 0; i < YL; i++) {
    if constexpr (DN_KC) {
      const int ld = wave * YL + i, row = ld * 16 + (lane >> 2), chunk = (lane & 3) ^ kc_swz(row);
      const int n = n0 + row < NF ? row : NF - 1 - n0;
      yoff[i] = (uint32_t)(n * ldd + chunk * 8) * 2u;
    } else {
      constexpr int CPR = kTN / 8;
      const int j = (wave * YL + i) * 64 + lane, k = j / CPR, slot = j % CPR;
      const int chunk = (((slot >> 1) ^ ks_swz<kTN>(k)) << 1) | (slot & 1);
      const int n = n0 + chunk * 8 < NF ? chunk * 8 : NF - 8 - n0;   // whole chunks: NF is a multiple of 8
      yoff[i] = (uint32_t)(k * ldd + n) * 2u;
    }
  }
  typename M::acc_t acc[G][RN];
#pragma unroll
  for (int m = 0; m < G; m++)
#pragma unroll
    for (int j = 0; j < RN; j++)
#pragma unroll
      for (int v = 0; v < M::NACC; v++) acc[m][j][v] = 0.f;

  // The entries of the plan (position of the reduction block, block id of each member or -1) in windows of 64, lane l holding
  // entry l of the window: its position, this wavefront's member's block (-1: none), and a bit per member that has a block.
  // A step reads its own with readlanes.  (Read from memory step by step, with scalar loads, which share their counter with
  // the LDS reads and return in any order, an entry was waited for before the step's first matrix instruction.)
  int window = -1, w_pos = 0, w_bid = 0, w_has = 0;
  auto issue = [&](int e, unsigned char *st) -> unsigned {
    if ((e & ~63) != window) {
      window = e & ~63;
      const int32_t *mine = entries + (int64_t)(G + 1) * (window + lane < ne ? window + lane : ne - 1);
      w_pos = mine[0];
      w_has = 0;
#pragma unroll
      for (int m = 0; m < G; m++) {
        const int id = (absent >> m) & 1 ? -1 : mine[1 + m];
        w_has |= id >= 0 ? 1 << m : 0;
        w_bid = wave == m ? id : w_bid;
      }
      asm volatile("" : "+v"(w_pos), "+v"(w_bid), "+v"(w_has));   // (wait for them here, not at every use)
    }
    const int pos = __builtin_amdgcn_readlane(w_pos, e & 63), bid = __builtin_amdgcn_readlane(w_bid, e & 63);
    // an absent member still issues its loads (the count per stage is fixed), but all lanes fetch one and the same
    // chunk: a single cache line instead of sixteen
    const T *xb = sp + (int64_t)(bid > 0 ? bid : 0) * (B * B);
    const T *yb = dn + (DN_KC ? (int64_t)pos * B : (int64_t)pos * B * ldd);
#pragma unroll
    for (int i = 0; i < XL; i++)
      load_lds16(xb, bid >= 0 ? xoff[i] : 0u, st + wave * XT::BYTES + i * 1024);
#pragma unroll
    for (int i = 0; i < YL; i++)
      load_lds16(yb, yoff[i], st + G * XT::BYTES + (wave * YL + i) * 1024);
    return __builtin_amdgcn_readlane(w_has, e & 63);
  };
  if (ne > 0) {
    unsigned cur = issue(0, smem), next = ne > 1 ? issue(1, smem + STAGE) : 0;   // members with a block in entries s, s + 1
    auto step = [&](auto stage, int s) {
      constexpr int S = decltype(stage)::value;
      if (s + 1 < ne) BSP_WAIT_VM(L * (kStages - 2));
      else BSP_WAIT_VM(0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      const unsigned here = cur;
      cur = next;
      if (s + 2 < ne) next = issue(s + 2, smem + (S + 2) % kStages * STAGE);
      const unsigned char *st = smem + S * STAGE;
      // all operands of the step first, then its products: the latency of the LDS is waited for once and not per member
      frag_t xf[G][kTK / 16] = {}, yf[kTK / 16][RN];
#pragma unroll
      for (int kk = 0; kk < kTK / 16; kk++)
#pragma unroll
        for (int j = 0; j < RN; j++) yf[kk][j] = YT::frag(st + G * XT::BYTES, (wave * RN + j) * 32, kk, lane);
#pragma unroll
      for (int m = 0; m < G; m++)
        if ((here >> m) & 1)
#pragma unroll
          for (int kk = 0; kk < kTK / 16; kk++) xf[m][kk] = XT::frag(st + m * XT::BYTES, 0, kk, lane);
#pragma unroll
      for (int m = 0; m < G; m++)
        if ((here >> m) & 1)
#pragma unroll
          for (int kk = 0; kk < kTK / 16; kk++)
#pragma unroll
            for (int j = 0; j < RN; j++) {
              if constexpr (OUT_NC) acc[m][j] = M::run(yf[kk][j], xf[m][kk], acc[m][j]);
              else acc[m][j] = M::run(xf[m][kk], yf[kk][j], acc[m][j]);
            }
    };
    for (int s = 0; s < ne; s += kStages) ring_round(s, ne, step);
    BSP_WAIT_VM(0);
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // epilogue: the 128 x 256 tile of the group through LDS, then 16-byte stores along the contiguous output index
  constexpr int TM = G * B;
  constexpr int CW = OUT_NC ? kTN : TM, NR = OUT_NC ? TM : kTN, LDR = CW + 8;
  static_assert(NR * LDR * 2 <= kStages * STAGE, "the staged tile fits into the ring");
  T *stage = reinterpret_cast<T *>(smem);
#pragma unroll
  for (int m = 0; m < G; m++)
#pragma unroll
    for (int j = 0; j < RN; j++)
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++) {
        const int m0 = m * 32, nn0 = (wave * RN + j) * 32;
        const int fast = 8 * g4 + 4 * (lane >> 5), slow = lane & 31;
        const int row = OUT_NC ? m0 + slow : nn0 + slow, col = OUT_NC ? nn0 + fast : m0 + fast;
        union { u32x2 raw; T e[4]; } u;
#pragma unroll
        for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(acc[m][j][4 * g4 + e]);
        *reinterpret_cast<u32x2 *>(stage + row * LDR + col) = u.raw;
      }
  __syncthreads();
  // lines of this group that exist and are its own (a line that became a chain is written by that chain)
  int own = 0;
#pragma unroll
  for (int m = 0; m < G; m++) own |= (line0 + m < g.lines && !((absent >> m) & 1)) ? 1 << m : 0;
  constexpr int CHUNKS = NR * CW / 8;
#pragma unroll 4
  for (int c = tid; c < CHUNKS; c += 256) {
    const int row = c / (CW / 8), col = (c % (CW / 8)) * 8;
    const u32x4 v = *reinterpret_cast<const u32x4 *>(stage + row * LDR + col);
    if constexpr (OUT_NC) {   // row = m (member row / 32), col = n
      if (((own >> (row >> 5)) & 1) && n0 + col < NF)
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(oz + ((int64_t)line0 * B + row) * ldo + n0 + col));
    } else {                  // row = n, col = m: a chunk of 8 lies inside one member
      if (((own >> (col >> 5)) & 1) && n0 + row < NF)
        __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(oz + (int64_t)(n0 + row) * ldo + line0 * B + col));
    }
  }
}

template <typename T> int launch_rg_dl(const XsdArgs &g, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st) {
  const int64_t n_wg = (int64_t)g.n_pgroups * ((g.NF + kTN - 1) / kTN) * g.Z;
  if (n_wg <= 0) return BSP_OK;
  if (n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  constexpr int SMEM = kStages * (BSP_GROUP * 32 + kTN) * kTK * 2;
  dim3 grid((unsigned)n_wg), wg(256);
#define BSP_RG_LAUNCH(ST, DK, ON)                                                                                       \
  do {                                                                                                                  \
    static std::atomic<uint64_t> done{0};                                                                               \
    if (!raise_lds_limit((const void *)k_xsd_rg_dl<T, ST, DK, ON>, SMEM, done)) return BSP_ERR_HIP;                     \
    hipLaunchKernelGGL((k_xsd_rg_dl<T, ST, DK, ON>), grid, wg, SMEM, st, g);                                           \
  } while (0)
  const int key = (sp_trans ? 4 : 0) | (dn_kc ? 2 : 0) | (out_nc ? 1 : 0);
  switch (key) {
    case 0: BSP_RG_LAUNCH(false, false, false); break;
    case 1: BSP_RG_LAUNCH(false, false, true); break;
    case 2: BSP_RG_LAUNCH(false, true, false); break;
    case 3: BSP_RG_LAUNCH(false, true, true); break;
    case 4: BSP_RG_LAUNCH(true, false, false); break;
    case 5: BSP_RG_LAUNCH(true, false, true); break;
    case 6: BSP_RG_LAUNCH(true, true, false); break;
    default: BSP_RG_LAUNCH(true, true, true); break;
  }
#undef BSP_RG_LAUNCH
  return BSP_OK;
}

// ---------------------------------------------------------------------------------------------------------
// ... and from chunks with lists of blocks: a workgroup of eight wavefronts takes sixteen consecutive lines and 128 columns of the free
// dimension (512 x 128 of the result, 128 accumulators a lane) and walks chunks of up to four reduction blocks in which the lines have
// at most 24 blocks together.  k_xsd_rg_dl feeds 16 KiB of the dense operand for the 1.5 blocks that four lines have in a reduction
// block at a quarter density, 40 flops a byte, and the feed from L2 bounds it; here 8 KiB serve the four of sixteen lines: 64 flops a
// byte.  A wavefront has 32 columns and eight of the lines, so the two wavefronts of a SIMD share the lines of the same columns and
// every SIMD has all the blocks of a chunk to multiply, however they fall.  The dense operands of a chunk stay in registers
// for all of its lines; a block is 2 LDS reads and 2 matrix instructions behind a bit of the chunk's mask.  Two stages of 80 KiB: one
// workgroup a compute unit, which stays for many tiles, so that the next chunk is in flight while this one is multiplied, also where it
// is the first of the next tile, during this one's stores.  What bounds it now is the chunk's loads, of which one chunk's are in flight:
// 1060 us take 700 without them and 1000 without the products (matrix units busy 22 % of the cycles, LDS 20 %, 8 TB/s into LDS where
// whole lines from L2 reach 35).  Touching the lines of the chunk after next, so that they are in L2 by then: 1200.
// 16 heads of 64 x 64 blocks, a quarter of them there, batch 8, free dimension 2048, fp16: 1175 -> 1054 us (519 TFLOP/s), with the dense
// operand's reduction contiguous 1500 -> 1045.  A workgroup a tile with the whole tile staged in LDS at its end: 1277; the results
// stored from registers: 1105.
// Chunk records (bsp_xsd_chunks_build), kChunkInts ints: reduction blocks n, blocks m, the mask (two ints, bit 4 line + block of the
// chunk), the n positions, the m ids in the order of the mask's bits.  Before them per group: head, first line, first chunk, chunks (a
// group without blocks has a chunk without any).
// ---------------------------------------------------------------------------------------------------------
constexpr int kChunkLines = 16, kChunkCols = 4, kChunkBlocks = 24, kChunkInts = 8 + kChunkBlocks, kChunkN = 128;

// Tiles lo, lo + stride ... below hi of a workgroup: the tiles are dealt to the XCDs in contiguous ranges, and an XCD's to its workgroups
struct TileRange { uint32_t at, end, stride; };
__device__ __forceinline__ TileRange tile_range(uint32_t n) {
  const uint32_t v = (uint32_t)xcd_remap(blockIdx.x, gridDim.x);
  if (gridDim.x % 8) return {v, n, gridDim.x};
  const uint32_t per = gridDim.x / 8, x = v / per;
  return {(uint32_t)((uint64_t)n * x / 8) + v % per, (uint32_t)((uint64_t)n * (x + 1) / 8), per};
}

template <typename T, bool SP_TRANS, bool DN_KC, bool OUT_NC>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) k_xsd_list_dl(XsdArgs g) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  constexpr int B = 32, HALF = kChunkLines / 2;
  typedef DlTile<T, B, !SP_TRANS> XT;                 // a block: 2 KiB
  typedef DlTile<T, kChunkN, DN_KC> YT;               // 32 reduction indices of the dense tile: 8 KiB
  static_assert(YT::LOADS == 8 && XT::LOADS == 2 && kChunkCols == 4 && kChunkBlocks % 8 == 0, "two wavefronts load a dense tile, each every eighth block");
  constexpr int XBYTES = kChunkBlocks * XT::BYTES, STAGE = XBYTES + kChunkCols * YT::BYTES;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int half = wave >> 2, wn = wave & 3;          // wavefronts w and w + 4 run on one SIMD
  // tiles in the order batch, head, columns, group: neighbours share the dense operand and the blocks in L2
  const uint32_t n_tiles = (g.NF + kChunkN - 1) / kChunkN, per_head = (g.lines + kChunkLines - 1) / kChunkLines, heads = g.n_pgroups / per_head;
  const TileRange tiles = tile_range((uint32_t)g.n_pgroups * n_tiles * (uint32_t)g.Z);
  if (tiles.at >= tiles.end) return;
  const int NF = g.NF;
  const int64_t ldd = g.ldd, ldo = g.ldo;
  const int32_t *records = g.gplan + 4 * (int64_t)g.n_pgroups;
  struct Place { uint32_t group, nt, z; };             // of a tile: group of lines (of all heads), columns, batch
  auto place = [&](uint32_t w) {
    const uint32_t a = w / per_head, b = a / n_tiles, z = b / heads;
    return Place{(b - z * heads) * per_head + (w - a * per_head), a - b * n_tiles, z};
  };

  // the tile being loaded
  const int ycol = wave >> 1;                         // the wavefront loads one half of the dense tile of this reduction block
  uint32_t xoff[2], yoff[4];
  const T *sp = nullptr, *dn = nullptr;
#pragma unroll
  for (int i = 0; i < 2; i++) xoff[i] = SP_TRANS ? XT::lane_offset(i, lane, 1, B) : XT::lane_offset(i, lane, B, 1);
  auto load_from = [&](Place p, int depth) {
    const int n0 = (int)p.nt * kChunkN;
    sp = reinterpret_cast<const T *>(g.sp) + p.z * g.sp_sz;
    dn = reinterpret_cast<const T *>(g.dn) + p.z * g.dn_sz + depth * g.dn_sh + (DN_KC ? n0 * ldd : n0);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int ld = (wave & 1) * 4 + i;
      if constexpr (DN_KC) {
        const int row = ld * 16 + (lane >> 2), chunk = (lane & 3) ^ kc_swz(row);
        const int n = n0 + row < NF ? row : NF - 1 - n0;
        yoff[i] = (uint32_t)(n * ldd + chunk * 8) * 2u;
      } else {
        constexpr int CPR = kChunkN / 8;
        const int j = ld * 64 + lane, k = j / CPR, slot = j % CPR;
        const int chunk = (((slot >> 1) ^ ks_swz<kChunkN>(k)) << 1) | (slot & 1);
        const int n = n0 + chunk * 8 < NF ? chunk * 8 : NF - 8 - n0;   // whole chunks: NF is a multiple of 8
        yoff[i] = (uint32_t)(k * ldd + n) * 2u;
      }
    }
  };
  auto issue = [&](int rec, unsigned char *st) {       // rec: the chunk's record, int l in lane l
    const int cols = __builtin_amdgcn_readlane(rec, 0), blocks = __builtin_amdgcn_readlane(rec, 1);
    if (ycol < cols) {
      const int64_t pos = (int64_t)__builtin_amdgcn_readlane(rec, 4 + ycol) * B;
      const T *yb = dn + (DN_KC ? pos : pos * ldd);
#pragma unroll
      for (int i = 0; i < 4; i++) load_lds16(yb, yoff[i], st + XBYTES + ycol * YT::BYTES + ((wave & 1) * 4 + i) * 1024);
    }
#pragma unroll
    for (int b0 = 0; b0 < kChunkBlocks; b0 += 8) {
      const int b = b0 + wave;
      if (b < blocks) {
        const T *xb = sp + (int64_t)__builtin_amdgcn_readlane(rec, 8 + b) * (B * B);
#pragma unroll
        for (int i = 0; i < 2; i++) load_lds16(xb, xoff[i], st + b * XT::BYTES + i * 1024);
      }
    }
  };
  typename M::acc_t acc[HALF];
#pragma unroll
  for (int m = 0; m < HALF; m++)
#pragma unroll
    for (int v = 0; v < M::NACC; v++) acc[m][v] = 0.f;

  const int at = lane & (kChunkInts - 1);
  uint32_t w = tiles.at;
  Place here = place(w);
  int depth, line0, chunk0, chunks;                    // of the tile at w, then of the one after it
  auto header = [&](uint32_t group) {
    const table_ptr hd = as_table(g.gplan) + 4 * (int64_t)group;
    depth = hd[0]; line0 = hd[1]; chunk0 = hd[2]; chunks = hd[3];
  };
  header(here.group);
  int rec = records[(int64_t)kChunkInts * chunk0 + at], next = records[(int64_t)kChunkInts * (chunk0 + (chunks > 1)) + at];
  load_from(here, depth);
  asm volatile("" : "+v"(rec), "+v"(next));
  unsigned stage = 0;
  issue(rec, smem);
  BSP_WAIT_VM(0);
  for (;;) {
    const bool more = w + tiles.stride < tiles.end;
    const int depth_here = depth, line_here = line0, chunk_here = chunk0, n_chunks = chunks;
    Place then = here;
    // the next tile's place and first records
    int rec_after = 0, next_after = 0;
    if (more) {
      then = place(w + tiles.stride);
      header(then.group);
      rec_after = records[(int64_t)kChunkInts * chunk0 + at];
      next_after = records[(int64_t)kChunkInts * (chunk0 + (chunks > 1)) + at];
    }
    for (int s = 0;; s++) {
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();                    // everybody's loads of the chunk have landed, and everybody is done reading the one before
      asm volatile("" ::: "memory");
      const unsigned low = __builtin_amdgcn_readlane(rec, 2), mask = half ? __builtin_amdgcn_readlane(rec, 3) : low;
      const unsigned char *st = smem + stage * STAGE;
      stage ^= 1;
      if (s + 1 < n_chunks) {
        issue(next, smem + stage * STAGE);
        rec = next;
        if (s + 2 < n_chunks) next = records[(int64_t)kChunkInts * (chunk_here + s + 2) + at];
      } else if (more) {
        load_from(then, depth);
        issue(rec_after, smem + stage * STAGE);
        rec = rec_after;
        next = next_after;
      }
      const unsigned char *xs = st + (half ? __builtin_popcount(low) : 0) * XT::BYTES;
      frag_t yf[kChunkCols][kTK / 16];
#pragma unroll
      for (int c = 0; c < kChunkCols; c++)
#pragma unroll
        for (int kk = 0; kk < kTK / 16; kk++) yf[c][kk] = YT::frag(st + XBYTES + c * YT::BYTES, wn * 32, kk, lane);   // (past the chunk's reduction blocks: never used)
#pragma unroll
      for (int m = 0; m < HALF; m++)
#pragma unroll
        for (int c = 0; c < kChunkCols; c++)
          if ((mask >> (m * kChunkCols + c)) & 1) {
            // (their latency is the other wavefront's time: read a block ahead, which takes moving them, the kernel was 2 % slower)
            frag_t xf[kTK / 16];
#pragma unroll
            for (int kk = 0; kk < kTK / 16; kk++) xf[kk] = XT::frag(xs, 0, kk, lane);
#pragma unroll
            for (int kk = 0; kk < kTK / 16; kk++) {
              if constexpr (OUT_NC) acc[m] = M::run(yf[c][kk], xf[kk], acc[m]);
              else acc[m] = M::run(xf[kk], yf[c][kk], acc[m]);
            }
            xs += XT::BYTES;
          }
      if (s + 1 >= n_chunks) break;
      BSP_WAIT_VM(0);                                  // this wavefront's loads of the next chunk, and the record after it
      asm volatile("" : "+v"(next), "+v"(rec_after), "+v"(next_after) : : "memory");
    }
    // the results, one half of the lines at a time, through the stage just read (the next tile's first chunk is on its way to the other
    // one), so that whole rows of them are stored: from registers it would be 64 bytes of a row at a time
    const int n0 = (int)here.nt * kChunkN;
    T *oz = reinterpret_cast<T *>(g.out) + here.z * g.out_sz + depth_here * g.out_sh;
    constexpr int TM = HALF * B, CW = OUT_NC ? kChunkN : TM, NR = OUT_NC ? TM : kChunkN, LDR = CW + 8;
    static_assert(NR * LDR * 2 <= STAGE && NR * CW / 8 == 512 * HALF, "half a tile fits into a stage, eight stores a lane");
    T *buf = reinterpret_cast<T *>(smem + (stage ^ 1) * STAGE);
    auto store = [&](auto whole) {
#pragma unroll
      for (int hh = 0; hh < 2; hh++) {
        BSP_WAIT_VM(63);                               // (LDS only)
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        if (half == hh) {
#pragma unroll
          for (int m = 0; m < HALF; m++)
#pragma unroll
            for (int g4 = 0; g4 < 4; g4++) {
              const int fast = 8 * g4 + 4 * (lane >> 5), slow = lane & 31;
              const int row = OUT_NC ? m * B + slow : wn * 32 + slow, col = OUT_NC ? wn * 32 + fast : m * B + fast;
              union { u32x2 raw; T e[4]; } u;
#pragma unroll
              for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(acc[m][4 * g4 + e]);
              *reinterpret_cast<u32x2 *>(buf + row * LDR + col) = u.raw;
            }
        }
        BSP_WAIT_VM(63);
        asm volatile("" ::: "memory");
        __builtin_amdgcn_s_barrier();
        asm volatile("" ::: "memory");
        const int m0 = (line_here + hh * HALF) * B, rows = g.lines * B - m0;      // first row of the half; how many there are
#pragma unroll
        for (int i = 0; i < HALF; i++) {
          const int c = tid + i * 512, row = c / (CW / 8), col = (c % (CW / 8)) * 8;
          const u32x4 v = *reinterpret_cast<const u32x4 *>(buf + row * LDR + col);
          T *dst = OUT_NC ? oz + (int64_t)(m0 + row) * ldo + n0 + col : oz + (int64_t)(n0 + row) * ldo + m0 + col;
          if (decltype(whole)::value || (OUT_NC ? row < rows && n0 + col < NF : col < rows && n0 + row < NF)) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(dst));
        }
      }
#pragma unroll
      for (int m = 0; m < HALF; m++)
#pragma unroll
        for (int v = 0; v < M::NACC; v++) acc[m][v] = 0.f;
    };
    // the next tile's first chunk was asked for before the stores of this one, which need not be waited for where their number is known
    if (line_here + kChunkLines <= g.lines && n0 + kChunkN <= NF) {
      store(Const<1>{});
      if (!more) break;
      BSP_WAIT_VM(2 * HALF);
    } else {
      store(Const<0>{});
      if (!more) break;
      BSP_WAIT_VM(0);
    }
    w += tiles.stride;
    here = then;
  }
}

template <typename T> int launch_xsd_list_dl(const XsdArgs &g, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st) {
  const int64_t n_wg = (int64_t)g.n_pgroups * ((g.NF + kChunkN - 1) / kChunkN) * g.Z;
  if (n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  constexpr int SMEM = 2 * (kChunkCols * kChunkN + kChunkBlocks * 32) * kTK * 2;
  dim3 grid((unsigned)(n_wg < 256 ? n_wg : 256)), wg(512);
#define BSP_XSD_LIST_LAUNCH(ST, DK, ON)                                                                                 \
  do {                                                                                                                  \
    static std::atomic<uint64_t> done{0};                                                                               \
    if (!raise_lds_limit((const void *)k_xsd_list_dl<T, ST, DK, ON>, SMEM, done)) return BSP_ERR_HIP;                   \
    hipLaunchKernelGGL((k_xsd_list_dl<T, ST, DK, ON>), grid, wg, SMEM, st, g);                                          \
  } while (0)
  const int key = (sp_trans ? 4 : 0) | (dn_kc ? 2 : 0) | (out_nc ? 1 : 0);
  switch (key) {
    case 0: BSP_XSD_LIST_LAUNCH(false, false, false); break;
    case 1: BSP_XSD_LIST_LAUNCH(false, false, true); break;
    case 2: BSP_XSD_LIST_LAUNCH(false, true, false); break;
    case 3: BSP_XSD_LIST_LAUNCH(false, true, true); break;
    case 4: BSP_XSD_LIST_LAUNCH(true, false, false); break;
    case 5: BSP_XSD_LIST_LAUNCH(true, false, true); break;
    case 6: BSP_XSD_LIST_LAUNCH(true, true, false); break;
    default: BSP_XSD_LIST_LAUNCH(true, true, true); break;
  }
#undef BSP_XSD_LIST_LAUNCH
  return BSP_OK;
}

// ---------------------------------------------------------------------------------------------------------
// sdd with a long reduction (hundreds of elements or more), blocks of 32, fp16 / bf16.  One output block is a 32 x 32
// product: a workgroup per block (or per 2 x 2 pack of the reference's table) fetches 2 + 2 KiB per 65 kflop and is bound
// by the feed from L2 at a thirteenth of the matrix peak.  Here a workgroup takes a group of four consecutive block-rows
// (128 rows of A, the group plan of bsp_group_plan_build) and eight of the block-columns in which any of them has a
// block (256 rows of B, gathered), and runs the dense 128 x 256 product over the whole reduction with the pipeline
// of k_xsd_dl; only the blocks that exist are written.  Computing the absent ones as well costs matrix time that the
// launch has to spare (it waits for operands either way) and removes all bookkeeping from the reduction loop: no
// table is read in it.  Operand bytes per useful flop drop by 2 at a quarter of the blocks kept.
// ---------------------------------------------------------------------------------------------------------
constexpr int kSddColsElems = 256;   // columns of the gathered B tile: 8 block-columns of 32, 16 of 16

// BLOCK = 32: the group plan of the layout itself, entries (position, id of each member's block or -1).
// BLOCK = 16: the same 128 x 256 product from blocks of 16.  The plan is over PAIRS of block-rows (a member = two
// consecutive block-rows = 32 rows of A, present at a block-column if either has a block there), so that a group is
// still 128 consecutive rows of A; a workgroup gathers sixteen block-columns of 16; an entry is (position, 4 member
// flags, then the ids of the two blocks of each member, -1 where absent): 13 ints.
template <typename T, bool A_KC, bool B_KC, int BLOCK>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2))) k_sdd_rg_dl(SddArgs g, int chunks) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  constexpr int B = 32, G = BSP_GROUP, CB = BLOCK, J = kSddColsElems / CB, TM = G * B, TN = J * CB;
  constexpr int SUB = B / CB;                         // block-rows per member: 1 or 2
  constexpr int ENT = SUB == 1 ? G + 1 : G + 1 + G * SUB;
  static_assert(BLOCK == 16 || BLOCK == 32, "blocks of 16 or 32");
  static_assert(TN == kTN, "the gathered B tile is the dense tile of the other kernels");
  typedef DlTile<T, TM, A_KC> XT;
  typedef DlTile<T, TN, B_KC> YT;
  constexpr int STAGE = XT::BYTES + YT::BYTES;
  constexpr int XL = XT::LOADS / 4, YL = YT::LOADS / 4, L = XL + YL;
  constexpr int RM = 2, RN = 4;                       // 2 x 2 wavefronts of 64 x 128
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t per_z = (int64_t)g.n_pgroups * chunks;
  const int64_t w = xcd_remap(blockIdx.x, per_z * g.Z);
  const int z = (int)(w / per_z);
  const int chunk = (int)((w % per_z) % chunks);      // chunk fastest: the chunks of a group share its rows of A in L2
  const table_ptr hd = as_table(g.gplan) + 4 * ((w % per_z) / chunks);
  const int e0 = hd[0], ne = hd[1], h = hd[2], code = hd[3];
  if (chunk * J >= ne) return;                        // (the grid is sized for the longest possible group)
  static_assert(J == kSddColsElems / BLOCK, "launch_sdd_rg_dl sizes the grid with the same J");
  const int left = ne - chunk * J;                    // entries of this chunk: min(left, J)
  const int line0 = (code & 0xffffff) * G;
  const int rows_a = g.lines * B;                     // rows of op(A) per head
  const int64_t lda = g.lda, ldb = g.ldb;
  const T *pa = reinterpret_cast<const T *>(g.a) + z * g.a_sz + h * g.a_sh + (int64_t)line0 * B * (A_KC ? lda : 1);
  const T *pb = reinterpret_cast<const T *>(g.b) + z * g.b_sz + h * g.b_sh;

  // Loop-invariant part of every load address.  A: rows line0 * 32 .. + 127 (rows past the end of the matrix read its
  // last rows; their blocks do not exist).  B: row n of the tile is row n % 32 of block-column pos[n / 32].
  uint32_t xoff[XL], yoff[YL];
#pragma unroll
  for (int i = 0; i < XL; i++) {
    const int ld = wave * XL + i;
    if constexpr (A_KC) {
      const int row = ld * 16 + (lane >> 2), chunk16 = (lane & 3) ^ kc_swz(row);
      const int r = line0 * B + row < rows_a ? row : rows_a - 1 - line0 * B;
      xoff[i] = (uint32_t)(r * lda + chunk16 * 8) * 2u;
    } else {
      constexpr int CPR = TM / 8;
      const int j = ld * 64 + lane, k = j / CPR, slot = j % CPR;
      const int c = (((slot >> 1) ^ ks_swz<TM>(k)) << 1) | (slot & 1);
      const int r = line0 * B + c * 8 < rows_a ? c * 8 : rows_a - 8 - line0 * B;
      xoff[i] = (uint32_t)(k * lda + r) * 2u;
    }
  }
#pragma unroll
  for (int i = 0; i < YL; i++) {
    const int ld = wave * YL + i;
    if constexpr (B_KC) {
      const int row = ld * 16 + (lane >> 2), chunk16 = (lane & 3) ^ kc_swz(row);
      const int jj = row / CB;
      const int pos = as_table(g.gplan)[4 * (int64_t)g.n_pgroups + (int64_t)ENT * (e0 + chunk * J + (jj < left ? jj : left - 1))];
      yoff[i] = (uint32_t)(((int64_t)pos * CB + (row % CB)) * ldb + chunk16 * 8) * 2u;
    } else {
      constexpr int CPR = TN / 8;
      const int j = ld * 64 + lane, k = j / CPR, slot = j % CPR;
      const int c = (((slot >> 1) ^ ks_swz<TN>(k)) << 1) | (slot & 1);
      const int jj = c / (CB / 8);                    // CB / 8 chunks of 8 columns per block-column
      const int pos = as_table(g.gplan)[4 * (int64_t)g.n_pgroups + (int64_t)ENT * (e0 + chunk * J + (jj < left ? jj : left - 1))];
      yoff[i] = (uint32_t)(k * ldb + (int64_t)pos * CB + (c % (CB / 8)) * 8) * 2u;
    }
  }
  typename M::acc_t acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; i++)
#pragma unroll
    for (int j = 0; j < RN; j++)
#pragma unroll
      for (int v = 0; v < M::NACC; v++) acc[i][j][v] = 0.f;
  // which of this wavefront's 2 x 4 blocks exist: the others are neither multiplied nor (if a whole row or column of
  // them is absent) read from LDS.  The loads into LDS stay dense: their count per stage is fixed.
  unsigned present = 0;
  {
    const table_ptr ids = as_table(g.gplan) + 4 * (int64_t)g.n_pgroups + (int64_t)ENT * (e0 + chunk * J);
#pragma unroll
    for (int i = 0; i < RM; i++)
#pragma unroll
      for (int j = 0; j < RN; j++) {
        // a 32 x 32 tile of the product covers one member and 32 / CB entries; the member's flag of an entry says
        // whether any of its blocks exists there
        const int m = wm * RM + i;
        bool any = false;
#pragma unroll
        for (int t = 0; t < B / CB; t++) {
          const int jj = (wn * RN + j) * (B / CB) + t;
          any = any || (jj < left && ids[ENT * (jj < left ? jj : left - 1) + 1 + m] >= 0);
        }
        present |= any ? 1u << (i * RN + j) : 0u;
      }
  }
  const int ksteps = g.K / kTK;
  auto issue = [&](int s, unsigned char *st) {
    const int64_t k0 = (int64_t)s * kTK;
    const T *xb = pa + (A_KC ? k0 : k0 * lda);
    const T *yb = pb + (B_KC ? k0 : k0 * ldb);
#pragma unroll
    for (int i = 0; i < XL; i++)
      load_lds16(xb, xoff[i], st + (wave * XL + i) * 1024);
#pragma unroll
    for (int i = 0; i < YL; i++)
      load_lds16(yb, yoff[i], st + XT::BYTES + (wave * YL + i) * 1024);
  };
  static_assert(kStages == 3, "two steps ahead");
  issue(0, smem);
  if (ksteps > 1) issue(1, smem + STAGE);
  auto step = [&](auto stage, int s) {
    constexpr int S = decltype(stage)::value;
    if (s + 1 < ksteps) BSP_WAIT_VM(L * (kStages - 2));
    else BSP_WAIT_VM(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + 2 < ksteps) issue(s + 2, smem + (S + 2) % kStages * STAGE);
    const unsigned char *st = smem + S * STAGE;
#pragma unroll
    for (int kk = 0; kk < kTK / 16; kk++) {
      frag_t xf[RM] = {}, yf[RN] = {};
#pragma unroll
      for (int i = 0; i < RM; i++)
        if ((present >> (i * RN)) & ((1u << RN) - 1)) xf[i] = XT::frag(st, (wm * RM + i) * 32, kk, lane);
#pragma unroll
      for (int j = 0; j < RN; j++)
        if ((present >> j) & 0x11u) yf[j] = YT::frag(st + XT::BYTES, (wn * RN + j) * 32, kk, lane);
      static_assert(RM == 2 && RN == 4, "the column test above reads bits j and j + RN");
#pragma unroll
      for (int i = 0; i < RM; i++)
#pragma unroll
        for (int j = 0; j < RN; j++)
          if ((present >> (i * RN + j)) & 1u) acc[i][j] = M::run(yf[j], xf[i], acc[i][j]);   // 4 consecutive values run along the block's columns
    }
  };
  for (int s = 0; s < ksteps; s += kStages) ring_round(s, ksteps, step);
  BSP_WAIT_VM(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // epilogue: the 128 x 256 tile through LDS, then the blocks that exist, each 2 KiB of consecutive addresses
  constexpr int LDR = TN + 8;
  static_assert(TM * LDR * 2 <= kStages * STAGE, "the staged tile fits into the ring");
  T *stage = reinterpret_cast<T *>(smem);
#pragma unroll
  for (int i = 0; i < RM; i++)
#pragma unroll
    for (int j = 0; j < RN; j++)
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++) {
        const int row = (wm * RM + i) * 32 + (lane & 31), col = (wn * RN + j) * 32 + 8 * g4 + 4 * (lane >> 5);
        union { u32x2 raw; T e[4]; } u;
#pragma unroll
        for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(acc[i][j][4 * g4 + e]);
        *reinterpret_cast<u32x2 *>(stage + row * LDR + col) = u.raw;
      }
  __syncthreads();
  T *pc = reinterpret_cast<T *>(g.c) + z * g.c_sz;
  const int32_t *ids = g.gplan + 4 * (int64_t)g.n_pgroups + (int64_t)ENT * (e0 + chunk * J);   // vector loads: the id differs from lane to lane
  constexpr int CPB = CB * CB / 8;                    // 16-byte chunks per block
  constexpr int MR = G * SUB;                         // block-rows of the tile
#pragma unroll 4
  for (int c = tid; c < MR * J * CPB; c += 256) {
    const int blk = c / CPB, within = c % CPB;
    const int mr = blk / J, jj = blk % J;             // block-row of the tile (member mr / SUB, its block-row mr % SUB), entry
    const int id = jj < left ? ids[ENT * jj + (SUB == 1 ? 1 + mr : 1 + G + mr)] : -1;
    if (id >= 0) {
      const int r = within / (CB / 8), cc = (within % (CB / 8)) * 8;
      *reinterpret_cast<u32x4 *>(pc + (int64_t)id * (CB * CB) + within * 8) = *reinterpret_cast<const u32x4 *>(stage + (mr * CB + r) * LDR + jj * CB + cc);
    }
  }
}

template <typename T, int BLOCK> int launch_sdd_rg_dl(const SddArgs &g, bool a_kc, bool b_kc, hipStream_t st) {
  constexpr int J = kSddColsElems / BLOCK;
  const int chunks = (g.cols + J - 1) / J;
  const int64_t n_wg = (int64_t)g.n_pgroups * chunks * g.Z;
  if (n_wg <= 0) return BSP_OK;
  if (n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  constexpr int SMEM = kStages * (BSP_GROUP * 32 + kTN) * kTK * 2;
  dim3 grid((unsigned)n_wg), wg(256);
#define BSP_SDD_RG_LAUNCH(AK, BK)                                                                                       \
  do {                                                                                                                  \
    static std::atomic<uint64_t> done{0};                                                                               \
    if (!raise_lds_limit((const void *)k_sdd_rg_dl<T, AK, BK, BLOCK>, SMEM, done)) return BSP_ERR_HIP;                  \
    hipLaunchKernelGGL((k_sdd_rg_dl<T, AK, BK, BLOCK>), grid, wg, SMEM, st, g, chunks);                                \
  } while (0)
  if (a_kc && b_kc) BSP_SDD_RG_LAUNCH(true, true);
  else if (a_kc) BSP_SDD_RG_LAUNCH(true, false);
  else if (b_kc) BSP_SDD_RG_LAUNCH(false, true);
  else BSP_SDD_RG_LAUNCH(false, false);
#undef BSP_SDD_RG_LAUNCH
  return BSP_OK;
}

// ---------------------------------------------------------------------------------------------------------
// sdd with a long reduction, blocks of 32, fp16 / bf16, layouts that hold a fair share of their blocks: a workgroup of eight
// wavefronts takes sixteen consecutive block-rows (512 rows of A) and up to sixteen block-columns gathered so that at most 64 blocks
// lie in them (512 rows of B), and computes those blocks and no others: each wavefront eight of them, from a list, in registers over
// the whole reduction.  What bounds k_sdd_rg_dl at these layouts is work and feed for absent blocks: it multiplies its whole 128 x 256
// tile, of which a quarter to a third of the blocks exist.  Here a step's 64 KiB at most serve up to 64 blocks, all of them wanted, and
// a wavefront reads both fragments of every block (2 KiB a matrix instruction), so that nothing in a step depends on the list but the
// addresses, which are computed once.  128 KiB of LDS: one workgroup a compute unit.  What bounds it is the feed and the step's barrier:
// 10 TB/s from L2, matrix units busy 32 % of the cycles, LDS 33 %.
// 16 heads of 64 x 64 blocks, a quarter of them there, batch 8, reduction 2048, fp16: 1594 -> 1071 us (513 TFLOP/s), 1668 -> 965 with
// A transposed.
// Tiles (bsp_sdd_tiles_build), kTileInts ints each: head, first block-row, block-columns n, blocks m, the 16 block-columns (the last
// repeated), per block its id, per block its row in the tile + 256 * its column in the tile (the first repeated past m).
// ---------------------------------------------------------------------------------------------------------
constexpr int kTileRows = 16, kTileCols = 16, kTileBlocks = 64, kTileInts = 4 + kTileCols + 2 * kTileBlocks;

template <typename T, bool A_KC, bool B_KC>
__global__ void __launch_bounds__(512) __attribute__((amdgpu_waves_per_eu(2, 2))) k_sdd_list_dl(SddArgs g) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  constexpr int TM = kTileRows * 32, TN = kTileCols * 32, PER = kTileBlocks / 8;
  typedef DlTile<T, TM, A_KC> XT;
  typedef DlTile<T, TN, B_KC> YT;
  constexpr int STAGE = XT::BYTES + YT::BYTES;
  constexpr int XL = XT::LOADS / 8, YL = YT::LOADS / 8;
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int64_t w = xcd_remap(blockIdx.x, (int64_t)g.n_pgroups * g.Z);
  const int z = (int)(w / g.n_pgroups);
  const table_ptr tile = as_table(g.gplan) + (int64_t)kTileInts * (w % g.n_pgroups);
  const int h = tile[0], row0 = tile[1] * 32, n_cols = tile[2], m = tile[3];
  const table_ptr cols = tile + 4, where = tile + 4 + kTileCols + kTileBlocks;
  const int rows_a = g.lines * 32;                    // rows of op(A) per head
  const int64_t lda = g.lda, ldb = g.ldb;
  const T *pa = reinterpret_cast<const T *>(g.a) + z * g.a_sz + h * g.a_sh + (int64_t)row0 * (A_KC ? lda : 1);
  const T *pb = reinterpret_cast<const T *>(g.b) + z * g.b_sz + h * g.b_sh;
  // Loop-invariant part of every load address, as in k_sdd_rg_dl: rows past the end of A read its last rows
  uint32_t xoff[XL], yoff[YL];
#pragma unroll
  for (int i = 0; i < XL; i++) {
    const int ld = wave * XL + i;
    if constexpr (A_KC) {
      const int row = ld * 16 + (lane >> 2), chunk16 = (lane & 3) ^ kc_swz(row);
      const int r = row0 + row < rows_a ? row : rows_a - 1 - row0;
      xoff[i] = (uint32_t)(r * lda + chunk16 * 8) * 2u;
    } else {
      constexpr int CPR = TM / 8;
      const int j = ld * 64 + lane, k = j / CPR, slot = j % CPR;
      const int c = (((slot >> 1) ^ ks_swz<TM>(k)) << 1) | (slot & 1);
      const int r = row0 + c * 8 < rows_a ? c * 8 : rows_a - 8 - row0;
      xoff[i] = (uint32_t)(k * lda + r) * 2u;
    }
  }
#pragma unroll
  for (int i = 0; i < YL; i++) {
    const int ld = wave * YL + i;
    if constexpr (B_KC) {
      const int row = ld * 16 + (lane >> 2), chunk16 = (lane & 3) ^ kc_swz(row);
      yoff[i] = (uint32_t)(((int64_t)cols[ld / 2] * 32 + (row & 31)) * ldb + chunk16 * 8) * 2u;
    } else {
      constexpr int CPR = TN / 8;
      const int j = ld * 64 + lane, k = j / CPR, slot = j % CPR;
      const int c = (((slot >> 1) ^ ks_swz<TN>(k)) << 1) | (slot & 1);
      const int32_t *vcols = g.gplan + (int64_t)kTileInts * (w % g.n_pgroups) + 4;     // (the column differs from lane to lane)
      yoff[i] = (uint32_t)(k * ldb + (int64_t)vcols[c >> 2] * 32 + (c & 3) * 8) * 2u;
    }
  }
  // The wavefront's blocks: an equal share of the list, in its order (by rows).  LDS byte addresses of their fragments of the first
  // stage; a row or column of blocks further is 2 KiB where the reduction is contiguous, 64 bytes (under the swizzle, so an
  // exclusive-or) where it is strided.
  const int first = wave * m / 8, count = (wave + 1) * m / 8 - first;
  const uint32_t base = (uint32_t)(uintptr_t)((const void __attribute__((address_space(3))) *)smem);
  const uint32_t xlane = A_KC ? (uint32_t)kc_offset(lane & 31, lane >> 5) : (uint32_t)ks_offset<TM>(8 * (lane >> 5) + ((lane & 15) >> 2), 16 * ((lane >> 4) & 1) + 4 * (lane & 3));
  const uint32_t ylane = B_KC ? (uint32_t)kc_offset(lane & 31, lane >> 5) : (uint32_t)ks_offset<TN>(8 * (lane >> 5) + ((lane & 15) >> 2), 16 * ((lane >> 4) & 1) + 4 * (lane & 3));
  uint32_t xa[PER], ya[PER];
#pragma unroll
  for (int i = 0; i < PER; i++) {
    const int rc = where[i < count ? first + i : first < m ? first : 0];
    xa[i] = base + (A_KC ? xlane + (uint32_t)(rc & 255) * 2048u : xlane ^ ((uint32_t)(rc & 255) * 64u));
    ya[i] = base + XT::BYTES + (B_KC ? ylane + (uint32_t)(rc >> 8) * 2048u : ylane ^ ((uint32_t)(rc >> 8) * 64u));
  }
  typename M::acc_t acc[PER];
#pragma unroll
  for (int i = 0; i < PER; i++)
#pragma unroll
    for (int v = 0; v < M::NACC; v++) acc[i][v] = 0.f;
  const int ksteps = g.K / kTK;
  auto issue = [&](int s, const unsigned char *st) {
    const int64_t k0 = (int64_t)s * kTK;
    const T *xb = pa + (A_KC ? k0 : k0 * lda);
    const T *yb = pb + (B_KC ? k0 : k0 * ldb);
#pragma unroll
    for (int i = 0; i < XL; i++) load_lds16(xb, xoff[i], st + (wave * XL + i) * 1024);
#pragma unroll
    for (int i = 0; i < YL; i++)
      if (!B_KC || (wave * YL + i) / 2 < n_cols) load_lds16(yb, yoff[i], st + XT::BYTES + (wave * YL + i) * 1024);
  };
  // the fragment of reduction indices 16 kk .. at the address of indices 0 ..
  auto fragment = [&](auto kcontig, auto rows, uint32_t at, int kk) {
    typedef typename Mma<T, 32>::frag_t __attribute__((address_space(3))) * frag_ptr;
    typedef s16x4 __attribute__((address_space(3))) * tr_ptr;
    if constexpr (decltype(kcontig)::value) {
      return *(frag_ptr)(uintptr_t)(at ^ (uint32_t)(kk << 5));
    } else {
      constexpr int ROW = decltype(rows)::value * 2;
      const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)(at + kk * 16 * ROW)), hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tr_ptr)(uintptr_t)(at + (kk * 16 + 4) * ROW));
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      return __builtin_bit_cast(frag_t, (s16x8)__builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
    }
  };
  issue(0, smem);
  for (int s = 0; s < ksteps; s++) {
    BSP_WAIT_VM(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    if (s + 1 < ksteps) issue(s + 1, smem + ((s + 1) & 1) * STAGE);
    const uint32_t at = (uint32_t)(s & 1) * STAGE;
#pragma unroll
    for (int kk = 0; kk < kTK / 16; kk++)
#pragma unroll
      for (int i0 = 0; i0 < PER; i0 += 4) {
        frag_t xf[4], yf[4];
#pragma unroll
        for (int i = 0; i < 4; i++) {
          xf[i] = fragment(Const<A_KC>{}, Const<TM>{}, xa[i0 + i] + at, kk);
          yf[i] = fragment(Const<B_KC>{}, Const<TN>{}, ya[i0 + i] + at, kk);
        }
#pragma unroll
        for (int i = 0; i < 4; i++) acc[i0 + i] = M::run(yf[i], xf[i], acc[i0 + i]);     // 4 consecutive values run along the block's columns
      }
  }
  BSP_WAIT_VM(0);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // each block through the wavefront's piece of LDS to 2 KiB of consecutive addresses
  constexpr int LDR = 40;
  T *stage = reinterpret_cast<T *>(smem) + wave * 32 * LDR;
  T *pc = reinterpret_cast<T *>(g.c) + z * g.c_sz;
#pragma unroll
  for (int i = 0; i < PER; i++)
    if (i < count) {
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++) {
        union { u32x2 raw; T e[4]; } u;
#pragma unroll
        for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(acc[i][4 * g4 + e]);
        *reinterpret_cast<u32x2 *>(stage + (lane & 31) * LDR + 8 * g4 + 4 * (lane >> 5)) = u.raw;
      }
      __builtin_amdgcn_wave_barrier();                 // (the LDS operations of one wavefront complete in order)
      T *dst = pc + (int64_t)tile[4 + kTileCols + first + i] * 1024;
#pragma unroll
      for (int c = lane; c < 128; c += 64) *reinterpret_cast<u32x4 *>(dst + c * 8) = *reinterpret_cast<const u32x4 *>(stage + (c >> 2) * LDR + (c & 3) * 8);
      __builtin_amdgcn_wave_barrier();
    }
}

template <typename T> int launch_sdd_list_dl(const SddArgs &g, bool a_kc, bool b_kc, hipStream_t st) {
  constexpr int SMEM = 2 * (kTileRows + kTileCols) * 32 * kTK * 2;
  const int64_t n_wg = (int64_t)g.n_pgroups * g.Z;
  if (n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  dim3 grid((unsigned)n_wg), wg(512);
#define BSP_SDD_LIST_LAUNCH(AK, BK)                                                                                     \
  do {                                                                                                                  \
    static std::atomic<uint64_t> done{0};                                                                               \
    if (!raise_lds_limit((const void *)k_sdd_list_dl<T, AK, BK>, SMEM, done)) return BSP_ERR_HIP;                       \
    hipLaunchKernelGGL((k_sdd_list_dl<T, AK, BK>), grid, wg, SMEM, st, g);                                              \
  } while (0)
  if (a_kc && b_kc) BSP_SDD_LIST_LAUNCH(true, true);
  else if (a_kc) BSP_SDD_LIST_LAUNCH(true, false);
  else if (b_kc) BSP_SDD_LIST_LAUNCH(false, true);
  else BSP_SDD_LIST_LAUNCH(false, false);
#undef BSP_SDD_LIST_LAUNCH
  return BSP_OK;
}

// ---------------------------------------------------------------------------------------------------------
// sdd over a long reduction into few blocks of 128 (the weight gradient of a block-sparse linear layer: 102 blocks,
// reduction over 8192 tokens).  One workgroup per block leaves most of the chip idle, four 64 x 64 workgroups per block
// fetch every operand row twice.  Here a workgroup computes a whole 128 x 128 block over a PART of the reduction with
// the pipeline of k_xsd_dl (128 x 128 x 32 steps, three LDS stages of 16 KiB, three workgroups per CU) and leaves an
// fp32 partial block in the caller's workspace; k_sdd_splitk_sum adds the parts of a block in part order and writes
// it.  Deterministic, no locks, no atomics: this is what the reference's split-K lock path (matmul.py:186-203, dead
// there) was meant for.  With a single part the block is written directly.
// Work item w: block fastest, then part, then batch: the workgroups that start together on an XCD (a contiguous range
// of w) then work on the same part of the reduction, and blocks of one block-row (neighbours in the table) find the
// rows of A they share in L2, as blocks of one block-column do with B.
// ---------------------------------------------------------------------------------------------------------
struct SplitK { int parts; int steps_per_part; float *ws; };

template <typename T, bool A_KC, bool B_KC>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 3))) k_sdd128_splitk(SddArgs g, SplitK sk) {
  typedef Mma<T, 32> M;
  typedef typename M::frag_t frag_t;
  constexpr int BL = 128;
  typedef DlTile<T, BL, A_KC> XT;
  typedef DlTile<T, BL, B_KC> YT;
  constexpr int STAGE = XT::BYTES + YT::BYTES;
  constexpr int XL = XT::LOADS / 4, YL = YT::LOADS / 4, L = XL + YL;
  constexpr int RM = 2, RN = 2;                       // 2 x 2 wavefronts of 64 x 64
  extern __shared__ __attribute__((aligned(1024))) unsigned char smem[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int64_t per_z = g.n_groups * sk.parts;
  const int64_t w = xcd_remap(blockIdx.x, per_z * g.Z);
  const int z = (int)(w / per_z);
  const int64_t grp = (w % per_z) % g.n_groups;
  const int part = (int)((w % per_z) / g.n_groups);
  if (g.valid && !g.valid[grp]) return;
  const table_ptr e = as_table(g.lut) + grp * 4;
  const int h = e[0], bi = e[1], bj = e[2], id = e[3];
  const int64_t lda = g.lda, ldb = g.ldb;
  const int ksteps_all = g.K / kTK;
  const int s0 = part * sk.steps_per_part;
  const int ksteps = min(sk.steps_per_part, ksteps_all - s0);
  // (a part past the end of the reduction has nothing to add: it leaves a zero block, so that the sum reads no garbage)
  const T *pa = reinterpret_cast<const T *>(g.a) + z * g.a_sz + h * g.a_sh + (A_KC ? (int64_t)bi * BL * lda : (int64_t)bi * BL);
  const T *pb = reinterpret_cast<const T *>(g.b) + z * g.b_sz + h * g.b_sh + (B_KC ? (int64_t)bj * BL * ldb : (int64_t)bj * BL);
  uint32_t xoff[XL], yoff[YL];
#pragma unroll
  for (int i = 0; i < XL; i++) xoff[i] = A_KC ? XT::lane_offset(wave * XL + i, lane, lda, 1) : XT::lane_offset(wave * XL + i, lane, 1, lda);
#pragma unroll
  for (int i = 0; i < YL; i++) yoff[i] = B_KC ? YT::lane_offset(wave * YL + i, lane, ldb, 1) : YT::lane_offset(wave * YL + i, lane, 1, ldb);
  typename M::acc_t acc[RM][RN];
#pragma unroll
  for (int i = 0; i < RM; i++)
#pragma unroll
    for (int j = 0; j < RN; j++)
#pragma unroll
      for (int v = 0; v < M::NACC; v++) acc[i][j][v] = 0.f;
  auto issue = [&](int s, unsigned char *st) {
    const int64_t k0 = (int64_t)(s0 + s) * kTK;
    const T *xb = pa + (A_KC ? k0 : k0 * lda);
    const T *yb = pb + (B_KC ? k0 : k0 * ldb);
#pragma unroll
    for (int i = 0; i < XL; i++)
      load_lds16(xb, xoff[i], st + (wave * XL + i) * 1024);
#pragma unroll
    for (int i = 0; i < YL; i++)
      load_lds16(yb, yoff[i], st + XT::BYTES + (wave * YL + i) * 1024);
  };
  if (ksteps > 0) {
    issue(0, smem);
    if (ksteps > 1) issue(1, smem + STAGE);
    auto step = [&](auto stage, int s) {
      constexpr int S = decltype(stage)::value;
      if (s + 1 < ksteps) BSP_WAIT_VM(L * (kStages - 2));
      else BSP_WAIT_VM(0);
      asm volatile("" ::: "memory");
      __builtin_amdgcn_s_barrier();
      asm volatile("" ::: "memory");
      if (s + 2 < ksteps) issue(s + 2, smem + (S + 2) % kStages * STAGE);
      const unsigned char *st = smem + S * STAGE;
      frag_t xf[kTK / 16][RM], yf[kTK / 16][RN];
#pragma unroll
      for (int kk = 0; kk < kTK / 16; kk++) {
#pragma unroll
        for (int i = 0; i < RM; i++) xf[kk][i] = XT::frag(st, (wm * RM + i) * 32, kk, lane);
#pragma unroll
        for (int j = 0; j < RN; j++) yf[kk][j] = YT::frag(st + XT::BYTES, (wn * RN + j) * 32, kk, lane);
      }
#pragma unroll
      for (int kk = 0; kk < kTK / 16; kk++)
#pragma unroll
        for (int i = 0; i < RM; i++)
#pragma unroll
          for (int j = 0; j < RN; j++) acc[i][j] = M::run(yf[kk][j], xf[kk][i], acc[i][j]);   // 4 consecutive values run along the block's columns
    };
    for (int s = 0; s < ksteps; s += kStages) ring_round(s, ksteps, step);
    BSP_WAIT_VM(0);
  }
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  // acc[i][j][4 * g4 + e] = C[row (wm * RM + i) * 32 + lane % 32][col (wn * RN + j) * 32 + 8 * g4 + 4 * (lane / 32) + e]
  if (sk.parts > 1) {
    // fp32 partial block, 16 bytes per lane (the parts of a block are summed by k_sdd_splitk_sum)
    float *ws = sk.ws + (((int64_t)z * g.n_groups + grp) * sk.parts + part) * (BL * BL);
#pragma unroll
    for (int i = 0; i < RM; i++)
#pragma unroll
      for (int j = 0; j < RN; j++)
#pragma unroll
        for (int g4 = 0; g4 < 4; g4++) {
          const int row = (wm * RM + i) * 32 + (lane & 31), col = (wn * RN + j) * 32 + 8 * g4 + 4 * (lane >> 5);
          const f32x4 v = {acc[i][j][4 * g4 + 0], acc[i][j][4 * g4 + 1], acc[i][j][4 * g4 + 2], acc[i][j][4 * g4 + 3]};
          *reinterpret_cast<f32x4 *>(ws + row * BL + col) = v;
        }
    return;
  }
  constexpr int LDR = BL + 8;
  static_assert(BL * LDR * 2 <= kStages * STAGE, "the staged block fits into the ring");
  T *stage = reinterpret_cast<T *>(smem);
#pragma unroll
  for (int i = 0; i < RM; i++)
#pragma unroll
    for (int j = 0; j < RN; j++)
#pragma unroll
      for (int g4 = 0; g4 < 4; g4++) {
        const int row = (wm * RM + i) * 32 + (lane & 31), col = (wn * RN + j) * 32 + 8 * g4 + 4 * (lane >> 5);
        union { u32x2 raw; T e[4]; } u;
#pragma unroll
        for (int e2 = 0; e2 < 4; e2++) u.e[e2] = from_float<T>(acc[i][j][4 * g4 + e2]);
        *reinterpret_cast<u32x2 *>(stage + row * LDR + col) = u.raw;
      }
  __syncthreads();
  T *pc = reinterpret_cast<T *>(g.c) + z * g.c_sz + (int64_t)id * (BL * BL);
#pragma unroll 4
  for (int c = tid; c < BL * BL / 8; c += 256) {
    const int row = c >> 4, cc = (c & 15) * 8;
    *reinterpret_cast<u32x4 *>(pc + row * BL + cc) = *reinterpret_cast<const u32x4 *>(stage + row * LDR + cc);
  }
}

// c[z, id] = sum over the parts, in part order, of the fp32 partial blocks; one thread per 8 elements
template <typename T>
__global__ void __launch_bounds__(256) k_sdd_splitk_sum(SddArgs g, SplitK sk) {
  constexpr int BB = 128 * 128;
  const int64_t chunk = (int64_t)blockIdx.x * 256 + threadIdx.x;      // 8 consecutive elements of one block
  const int64_t blk = chunk / (BB / 8);                               // z * n_groups + grp
  if (blk >= g.n_groups * g.Z) return;
  const int64_t grp = blk % g.n_groups, z = blk / g.n_groups;
  if (g.valid && !g.valid[grp]) return;
  const int within = (int)(chunk % (BB / 8)) * 8;
  const float *ws = sk.ws + blk * sk.parts * BB + within;
  f32x4 lo = {0.f, 0.f, 0.f, 0.f}, hi = {0.f, 0.f, 0.f, 0.f};
  for (int p = 0; p < sk.parts; p++) {
    lo += __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(ws + (int64_t)p * BB));
    hi += __builtin_nontemporal_load(reinterpret_cast<const f32x4 *>(ws + (int64_t)p * BB + 4));
  }
  union { u32x4 raw; T e[8]; } u;
#pragma unroll
  for (int k = 0; k < 4; k++) { u.e[k] = from_float<T>(lo[k]); u.e[4 + k] = from_float<T>(hi[k]); }
  const int id = as_table(g.lut)[grp * 4 + 3];
  *reinterpret_cast<u32x4 *>(reinterpret_cast<T *>(g.c) + z * g.c_sz + (int64_t)id * BB + within) = u.raw;
}

template <typename T> int launch_sdd128_splitk(const SddArgs &g, const SplitK &sk, bool a_kc, bool b_kc, hipStream_t st) {
  const int64_t n_wg = g.n_groups * g.Z * sk.parts;
  if (n_wg <= 0) return BSP_OK;
  if (n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  constexpr int SMEM = kStages * 2 * 128 * kTK * 2;
  dim3 grid((unsigned)n_wg), wg(256);
#define BSP_SPLITK_LAUNCH(AK, BK)                                                                                       \
  do {                                                                                                                  \
    static std::atomic<uint64_t> done{0};                                                                               \
    if (!raise_lds_limit((const void *)k_sdd128_splitk<T, AK, BK>, SMEM, done)) return BSP_ERR_HIP;                     \
    hipLaunchKernelGGL((k_sdd128_splitk<T, AK, BK>), grid, wg, SMEM, st, g, sk);                                       \
  } while (0)
  if (a_kc && b_kc) BSP_SPLITK_LAUNCH(true, true);
  else if (a_kc) BSP_SPLITK_LAUNCH(true, false);
  else if (b_kc) BSP_SPLITK_LAUNCH(false, true);
  else BSP_SPLITK_LAUNCH(false, false);
#undef BSP_SPLITK_LAUNCH
  if (sk.parts > 1) {
    const int64_t chunks = g.n_groups * g.Z * (128 * 128 / 8);
    hipLaunchKernelGGL((k_sdd_splitk_sum<T>), dim3((unsigned)((chunks + 255) / 256)), dim3(256), 0, st, g, sk);
  }
  return BSP_OK;
}

template <typename T, int BLOCK> int launch_dl(const XsdArgs &g0, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st) {
  const int64_t n_wg = (int64_t)g0.width * ((g0.NF + kTN - 1) / kTN) * g0.Z;
  if (n_wg <= 0) return BSP_OK;
  if (n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  XsdArgs g = g0;
  if (n_wg > 16 * 256) g.order = nullptr;            // longest segments first only in short launches (see launch_xsd_bw)
  constexpr int SMEM = kStages * (BLOCK + kTN) * kTK * 2;
  dim3 grid((unsigned)n_wg), wg(256);
#define BSP_DL_LAUNCH(ST, DK, ON)                                                                                       \
  do {                                                                                                                  \
    static std::atomic<uint64_t> done{0};                                                                               \
    if (!raise_lds_limit((const void *)k_xsd_dl<T, BLOCK, ST, DK, ON>, SMEM, done)) return BSP_ERR_HIP;                 \
    hipLaunchKernelGGL((k_xsd_dl<T, BLOCK, ST, DK, ON>), grid, wg, SMEM, st, g);                                       \
  } while (0)
  const int key = (sp_trans ? 4 : 0) | (dn_kc ? 2 : 0) | (out_nc ? 1 : 0);
  switch (key) {
    case 0: BSP_DL_LAUNCH(false, false, false); break;
    case 1: BSP_DL_LAUNCH(false, false, true); break;
    case 2: BSP_DL_LAUNCH(false, true, false); break;
    case 3: BSP_DL_LAUNCH(false, true, true); break;
    case 4: BSP_DL_LAUNCH(true, false, false); break;
    case 5: BSP_DL_LAUNCH(true, false, true); break;
    case 6: BSP_DL_LAUNCH(true, true, false); break;
    default: BSP_DL_LAUNCH(true, true, true); break;
  }
#undef BSP_DL_LAUNCH
  return BSP_OK;
}

}  // namespace

// The kernels of this file keep the per-lane part of a load's address in 32 bits of bytes from the operand's tile (or, for the
// gathered operand of sdd_dl, from its first row).
static bool near_rows(int64_t rows, int64_t ld) { return ld >= 0 && ld < ((int64_t)1 << 31) / rows; }

// 1 = launched, 0 = not applicable (the caller takes another kernel), 2 = the general kernel's, < 0 = error
int xsd_dl(int dtype, const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st) {
  if (dtype == BSP_F32 || g.NF < 256 || !near_rows(kTN, g.ldd)) return 0;
  if (block == 32) {   // needs the group plan (whole blocks, no split chains)
    // Groups of four lines times tiles of 256 columns leave most of the chip idle in a small launch, where the general
    // kernel's smaller workgroups win.  Single dsd products at a quarter of the blocks, this kernel / the general one, dense
    // reduction strided (contiguous): 1024^3, 32 workgroups here, 20.8 / 14.9 us (19.8 / 16.0); 4096 x 2048 x 4096, 256 of
    // them, 70.5 / 60.8 (68.1 / 67.0); 8 products of 2048^3, 1024 of them, 87 / 111 (91 against 108 of this kernel with its
    // table read and its addresses computed in every step).  (The host chooses the plan by the same rule: _plan_for in matmul.py.)
    if ((g.width + 3) / 4 * (int64_t)((g.NF + kTN - 1) / kTN) * g.Z < 384) return 0;
    if (!g.gplan || g.n_pgroups <= 0 || g.lines <= 0 || g.n_split != 0) return 0;
    const int rc = dtype == BSP_F16 ? launch_rg_dl<f16>(g, sp_trans, dn_kc, out_nc, st) : launch_rg_dl<bf16>(g, sp_trans, dn_kc, out_nc, st);
    return rc == BSP_OK ? 1 : rc;
  }
  if (block != 64 && block != 128) return 0;
  // ... the same at blocks of 64 with the dense reduction contiguous, whose tiles the general kernel reads well: 1024^3 (64
  // workgroups here) 13.7 / 12.2 us, 4096 x 2048 x 4096 (512) 56.7 / 55.5, 8 products of 2048^3 (2048) 89 / 104; with it
  // strided 13.9 / 15.0, 52.4 / 75.1 and 76 / 110
  const int64_t n_wg = (int64_t)g.width * ((g.NF + kTN - 1) / kTN) * g.Z;
  if (block == 64 && dn_kc && n_wg <= 512) return 0;
  // Tiles of 256 on less than half of the compute units: the general kernel's narrower ones.  fp16, this kernel / the general one, us:
  // blocks of 128, a tenth to half of the blocks there, 512^3 (8 workgroups here) 8-12 / 6-8, 1024 x 512 x 2048 in 2 heads (32) 16-29 / 10-21,
  // 1024^3 in 3 (96) 13-19 / 10-15; on 128 13-31 / 8-27, but 16 x 512^3 up to 12.8 / 13.9; on 160 17.8 / 20.1.  Blocks of 64, 16 workgroups 6-8 / 5-6,
  // 64 8-18 / 7-14; 192 8-14 / 7-15.
  if (n_wg < 128) return 2;
  int rc;
  if (dtype == BSP_F16) rc = block == 128 ? launch_dl<f16, 128>(g, sp_trans, dn_kc, out_nc, st) : launch_dl<f16, 64>(g, sp_trans, dn_kc, out_nc, st);
  else rc = block == 128 ? launch_dl<bf16, 128>(g, sp_trans, dn_kc, out_nc, st) : launch_dl<bf16, 64>(g, sp_trans, dn_kc, out_nc, st);
  return rc == BSP_OK ? 1 : rc;
}

// The same from the chunks of bsp_xsd_chunks_build (g.gplan, g.n_pgroups groups of them)
int xsd_list(int dtype, const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st) {
  if (dtype == BSP_F32 || block != 32 || !g.gplan || g.n_pgroups <= 0 || g.lines <= 0 || g.NF < kChunkN || !near_rows(kTN, g.ldd)) return 0;
  if (g.n_pgroups % ((g.lines + kChunkLines - 1) / kChunkLines)) return BSP_ERR_ARG;
  const int rc = dtype == BSP_F16 ? launch_xsd_list_dl<f16>(g, sp_trans, dn_kc, out_nc, st) : launch_xsd_list_dl<bf16>(g, sp_trans, dn_kc, out_nc, st);
  return rc == BSP_OK ? 1 : rc;
}

// sdd at blocks of 128 over a reduction cut into `parts` parts (pack-1 table rows; ws: parts fp32 blocks per table row and
// batch, may be null when parts == 1): BSP_OK = launched, BSP_ERR_UNSUPPORTED = not this kernel's case
int sdd128_splitk(int dtype, const SddArgs &g, int parts, float *ws, bool a_kc, bool b_kc, hipStream_t st) {
  if (dtype == BSP_F32 || parts < 1 || g.K % kTK || (parts > 1 && !ws) || !near_rows(128, g.lda) || !near_rows(128, g.ldb)) return BSP_ERR_UNSUPPORTED;
  const int steps = g.K / kTK;
  SplitK sk;
  sk.parts = parts; sk.steps_per_part = (steps + parts - 1) / parts; sk.ws = ws;
  return dtype == BSP_F16 ? launch_sdd128_splitk<f16>(g, sk, a_kc, b_kc, st) : launch_sdd128_splitk<bf16>(g, sk, a_kc, b_kc, st);
}

// The same from the tiles of bsp_sdd_tiles_build (g.gplan, g.n_pgroups of them; g.lines: block-rows, g.cols: block-columns of a head):
// 2 = launched, every block of the layout written; 0 = not applicable, < 0 = error
int sdd_list(int dtype, const SddArgs &g, int block, bool a_kc, bool b_kc, hipStream_t st) {
  if (dtype == BSP_F32 || block != 32 || !g.gplan || g.n_pgroups <= 0 || g.lines <= 0 || g.cols <= 0) return 0;
  if (g.K < 256 || g.K % kTK || !near_rows(kTileRows * 32, g.lda) || !near_rows(b_kc ? (int64_t)g.cols * 32 : kTK, g.ldb)) return 0;
  const int rc = dtype == BSP_F16 ? launch_sdd_list_dl<f16>(g, a_kc, b_kc, st) : launch_sdd_list_dl<bf16>(g, a_kc, b_kc, st);
  return rc == BSP_OK ? 2 : rc;
}

// sdd with a long reduction at blocks of 32 from the group plan alone: 2 = launched (every block of the layout is
// written), 0 = not applicable, < 0 = error
int sdd_dl(int dtype, const SddArgs &g, int block, bool rowpair_plan, bool a_kc, bool b_kc, hipStream_t st) {
  if (dtype == BSP_F32 || (block != 32 && block != 16) || !g.gplan || g.n_pgroups <= 0 || g.lines <= 0 || g.cols <= 0) return 0;
  if ((block == 16) != rowpair_plan) return 0;        // blocks of 16 come with the plan over pairs of block-rows, and only they
  if (g.K < 256 || g.K % kTK || !near_rows(BSP_GROUP * 32, g.lda) || !near_rows(b_kc ? (int64_t)g.cols * block : kTK, g.ldb)) return 0;
  int rc;
  if (block == 32) rc = dtype == BSP_F16 ? launch_sdd_rg_dl<f16, 32>(g, a_kc, b_kc, st) : launch_sdd_rg_dl<bf16, 32>(g, a_kc, b_kc, st);
  else rc = dtype == BSP_F16 ? launch_sdd_rg_dl<f16, 16>(g, a_kc, b_kc, st) : launch_sdd_rg_dl<bf16, 16>(g, a_kc, b_kc, st);
  return rc == BSP_OK ? 2 : rc;
}

}  // namespace bsp

static int sdd_tiles_build(const uint8_t *layout, int H, int R, int C, int32_t *out, int64_t cap, int64_t *n_tiles) {
  using namespace bsp;
  if (!layout || !n_tiles || H <= 0 || R <= 0 || C <= 0 || cap < 0 || (cap > 0 && !out)) return BSP_ERR_ARG;
  int64_t n = 0, blocks_before = 0;
  std::vector<int64_t> row_first((size_t)R + 1);             // id of the first block of a block-row
  for (int h = 0; h < H; h++) {
    const uint8_t *lay = layout + (int64_t)h * R * C;
    row_first[0] = blocks_before;
    for (int r = 0; r < R; r++) row_first[r + 1] = row_first[r] + std::count_if(lay + (int64_t)r * C, lay + (int64_t)(r + 1) * C, [](uint8_t v) { return v != 0; });
    blocks_before = row_first[R];
    for (int r0 = 0; r0 < R; r0 += kTileRows) {
      const int rows = R - r0 < kTileRows ? R - r0 : kTileRows;
      // a tile's blocks: those of whole columns, except that its first column may lack its first rows and its last one its last rows,
      // which the tile before and the next one have (64 x 64 blocks a head, 90 % of them there: tiles of whole columns 3147 us, these 2555)
      int cols[kTileCols], n_cols = 0, m = 0, from = 0, upto = rows;
      int64_t next[kTileRows];                         // id of the row's next block
      for (int r = 0; r < rows; r++) next[r] = row_first[r0 + r];
      auto flush = [&]() {
        if (m && (n + 1) * kTileInts <= cap) {
          int32_t *t = out + n * kTileInts, at = 0;
          t[0] = h; t[1] = r0; t[2] = n_cols; t[3] = m;
          for (int c = 0; c < kTileCols; c++) t[4 + c] = cols[c < n_cols ? c : n_cols - 1];
          for (int r = 0; r < rows; r++)
            for (int c = 0; c < n_cols; c++)
              if (lay[(int64_t)(r0 + r) * C + cols[c]] && (c > 0 || r >= from) && (c < n_cols - 1 || r < upto)) {
                t[4 + kTileCols + at] = (int32_t)next[r]++;
                t[4 + kTileCols + kTileBlocks + at++] = r | c << 8;
              }
          for (; at < kTileBlocks; at++) t[4 + kTileCols + at] = -1, t[4 + kTileCols + kTileBlocks + at] = t[4 + kTileCols + kTileBlocks];
        }
        if (m) n++;
        n_cols = m = 0;
        from = 0;
        upto = rows;
      };
      for (int c = 0; c < C; c++) {
        int here = 0;
        for (int r = 0; r < rows; r++) here += lay[(int64_t)(r0 + r) * C + c] != 0;
        if (!here) continue;
        if (n_cols == kTileCols || m == kTileBlocks) flush();
        cols[n_cols++] = c;
        if (m + here <= kTileBlocks) {
          m += here;
          continue;
        }
        int r = 0, left = kTileBlocks - m;             // the rows before r fill the tile
        for (; left > 0; r++) left -= lay[(int64_t)(r0 + r) * C + c] != 0;
        here -= kTileBlocks - m;
        m = kTileBlocks;
        upto = r;
        flush();
        cols[n_cols++] = c;
        m = here;
        from = r;
      }
      flush();
    }
  }
  *n_tiles = n;
  return n * kTileInts > cap ? BSP_ERR_CAPACITY : BSP_OK;
}
extern "C" int bsp_sdd_tiles_build(const uint8_t *layout, int H, int R, int C, int32_t *out, int64_t cap, int64_t *n_tiles) {
  return bsp::no_throw([&] { return sdd_tiles_build(layout, H, R, C, out, cap, n_tiles); });
}

static int xsd_chunks_build(const uint8_t *layout, int H, int R, int C, int rows, int32_t *out, int64_t cap, int *n_groups, int64_t *n_ints) {
  using namespace bsp;
  if (!layout || !n_groups || !n_ints || H <= 0 || R <= 0 || C <= 0 || cap < 0 || (cap > 0 && !out)) return BSP_ERR_ARG;
  const int L = rows ? R : C, K = rows ? C : R, per_head = (L + kChunkLines - 1) / kChunkLines;
  const int64_t first = 4 * (int64_t)H * per_head;     // the records start behind the groups
  int64_t n = 0, blocks_before = 0, group = 0;
  std::vector<int32_t> id((int64_t)R * C);             // of the head's blocks, -1: none
  for (int h = 0; h < H; h++) {
    for (int64_t i = 0; i < (int64_t)R * C; i++) id[i] = layout[h * (int64_t)R * C + i] ? (int32_t)blocks_before++ : -1;
    for (int l0 = 0; l0 < L; l0 += kChunkLines, group++) {
      const int lines = L - l0 < kChunkLines ? L - l0 : kChunkLines;
      const int64_t before = n;
      int cols[kChunkCols], n_cols = 0, m = 0;
      auto block_at = [&](int l, int k) { return rows ? id[(int64_t)(l0 + l) * C + k] : id[(int64_t)k * C + l0 + l]; };
      auto flush = [&]() {
        if (m && first + (n + 1) * kChunkInts <= cap) {
          int32_t *r = out + first + n * kChunkInts;
          std::fill(r, r + kChunkInts, 0);
          r[0] = n_cols; r[1] = m;
          int at = 0;
          for (int c = 0; c < n_cols; c++) r[4 + c] = cols[c];
          for (int l = 0; l < lines; l++)
            for (int c = 0; c < n_cols; c++)
              if (const int32_t b = block_at(l, cols[c]); b >= 0) {
                const int bit = l * kChunkCols + c;
                r[2 + bit / 32] = (int32_t)((uint32_t)r[2 + bit / 32] | 1u << bit % 32);
                r[8 + at++] = b;
              }
        }
        if (m) n++;
        n_cols = m = 0;
      };
      for (int k = 0; k < K; k++) {
        int here = 0;
        for (int l = 0; l < lines; l++) here += block_at(l, k) >= 0;
        if (!here) continue;
        if (n_cols == kChunkCols || m + here > kChunkBlocks) flush();
        cols[n_cols++] = k;
        m += here;
      }
      flush();
      if (n == before) {                               // no block: one record without any
        if (first + (n + 1) * kChunkInts <= cap) std::fill(out + first + n * kChunkInts, out + first + (n + 1) * kChunkInts, 0);
        n++;
      }
      if (4 * (group + 1) <= cap) {
        int32_t *g = out + 4 * group;
        g[0] = h; g[1] = l0; g[2] = (int32_t)before; g[3] = (int32_t)(n - before);
      }
    }
  }
  *n_groups = H * per_head;
  *n_ints = first + n * kChunkInts;
  return *n_ints > cap ? BSP_ERR_CAPACITY : BSP_OK;
}
extern "C" int bsp_xsd_chunks_build(const uint8_t *layout, int H, int R, int C, int rows, int32_t *out, int64_t cap, int *n_groups, int64_t *n_ints) {
  return bsp::no_throw([&] { return xsd_chunks_build(layout, H, R, C, rows, out, cap, n_groups, n_ints); });
}
