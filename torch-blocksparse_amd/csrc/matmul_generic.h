// General block-sparse matmul kernels for gfx950: every block size (16/32/64/128), fp16 / bf16 / fp32,
// every trans_a / trans_b / trans_c combination.
//
// Replaces the reference's single Triton-C kernel with its SDD / DSD / DDS branches (matmul.py:6-205).
// Structure: a workgroup of four wavefronts owns one output tile; both operand tiles are staged through LDS
// An operand whose reduction dimension is contiguous in memory sits in LDS as rows of TK elements plus padding
// and every MFMA operand is one 16-byte LDS read; an operand stored with the reduction dimension strided sits in
// LDS as it lies in memory and is read with the transposing LDS load (16-bit types; 32-bit ones are transposed
// while they are written).  Global loads for step s+1 are issued before
// the MFMAs of step s (two LDS buffers, one barrier per step).  fp32 accumulation in 16x16 MFMA tiles.
//
// "xsd" is the kernel behind both dsd and dds: dds is dsd with the roles of rows and columns exchanged
// (C^T = B_sparse^T . A^T), which only changes the three orientation flags.
#pragma once
#include "bsp_common.h"

namespace bsp {

// ---------------------------------------------------------------------------------------------------------
// MFMA per element type and tile size MS (16 or 32).  Lane l supplies row (l % MS) of its operand, reduction
// indices (l / MS) * KV .. + KV - 1.  Result: MS = 16 -> element e is (row 4*(l/16) + e, column l % 16);
// MS = 32 -> element 4*g + e is (row 8*g + 4*(l/32) + e, column l % 32).
// ---------------------------------------------------------------------------------------------------------
template <typename T> struct Mma16;
template <> struct Mma16<f16> {
  static constexpr int KSTEP = 32, KV = 8;
  typedef f16x8 frag_t;
  static __device__ __forceinline__ f32x4 run(frag_t a, frag_t b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_f16(a, b, c, 0, 0, 0); }
};
template <> struct Mma16<bf16> {
  static constexpr int KSTEP = 32, KV = 8;
  typedef bf16x8 frag_t;
  static __device__ __forceinline__ f32x4 run(frag_t a, frag_t b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0); }
};
template <> struct Mma16<float> {
  static constexpr int KSTEP = 4, KV = 1;
  typedef float frag_t;
  static __device__ __forceinline__ f32x4 run(frag_t a, frag_t b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }
};

template <typename T, int MS> struct Mma;
template <typename T> struct Mma<T, 16> : Mma16<T> {
  static constexpr int NACC = 4;
  typedef f32x4 acc_t;
};
template <> struct Mma<f16, 32> {
  static constexpr int KSTEP = 16, KV = 8, NACC = 16;
  typedef f16x8 frag_t;
  typedef f32x16 acc_t;
  static __device__ __forceinline__ acc_t run(frag_t a, frag_t b, acc_t c) { return __builtin_amdgcn_mfma_f32_32x32x16_f16(a, b, c, 0, 0, 0); }
};
template <> struct Mma<bf16, 32> {
  static constexpr int KSTEP = 16, KV = 8, NACC = 16;
  typedef bf16x8 frag_t;
  typedef f32x16 acc_t;
  static __device__ __forceinline__ acc_t run(frag_t a, frag_t b, acc_t c) { return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0); }
};
template <> struct Mma<float, 32> {
  static constexpr int KSTEP = 2, KV = 1, NACC = 16;
  typedef float frag_t;
  typedef f32x16 acc_t;
  static __device__ __forceinline__ acc_t run(frag_t a, frag_t b, acc_t c) { return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0); }
};

// Reduction step: 64 bytes; rows of the tiles 16 bytes more.  Steps of 128 bytes in fp32 win up to 15 % in sdd at blocks of 32 with a long
// reduction and lose 60 % with one of 32; blocks of 16, 64 and 128 lose up to 12 %, dsd and dds up to 20 % in large launches.
template <typename T> struct TileK { static constexpr int TK = 64 / sizeof(T), PAD = 16 / sizeof(T); };

// ---------------------------------------------------------------------------------------------------------
// One operand tile: ROWS x TK, fetched by NT threads in 16-byte chunks, kept in registers until the LDS
// buffer is free.  The address of a chunk is split into the part that never changes for a thread (computed once, before
// the reduction loop) and the part that is the same for all threads of a step (scalar arithmetic on the step's table
// values): a load costs one 64-bit add, not the multiplications and selects of a full index computation.
//   View::part_k(row, k) / part_r(row, k) -> Part{off, ok, sel, k}: element offset of chunk (row, k..k+VE-1) resp.
//     (row..row+VE-1, k) inside the step, whether the rows exist, which of the step's blocks it belongs to
//   View::step(k0) -> Step{..., live[NB], klim}: raw table values of the reduction step starting at k0
//   View::scalar_k(step, i) / scalar_r(step, i) -> element offset of block i of the step
// ---------------------------------------------------------------------------------------------------------
struct Part { int64_t off; bool ok; int sel; int k; };

// MS: rows of the MFMA tiles that read it
template <typename T, int ROWS, int NT, bool KCONTIG, int MS> struct TileLoader {
  static constexpr int TK = TileK<T>::TK, LDK = TK + TileK<T>::PAD;
  static constexpr int VE = 16 / sizeof(T);
  static constexpr int NCH = ROWS * TK / VE, THREADS = NT;
  static constexpr int ITER = (NCH + NT - 1) / NT;
  static constexpr int CPR = TK / VE;    // chunks per row when the reduction is contiguous
  static constexpr int RCH = ROWS / VE;  // chunks per reduction index otherwise
  // An operand stored with the reduction dimension strided is kept in LDS as it lies in memory, [TK][ROWS + 8].  A
  // 16-bit one is handed to the MFMA through the transposing LDS read; a 32-bit one needs no transposition at all:
  // its MFMA operand is a single element per lane, read where it lies.
  static constexpr bool ASIS = !KCONTIG;
  static constexpr bool TR = ASIS && sizeof(T) == 2;
  // Padding of a row of the as-is layout.  16-bit: the transposing read of a 16-lane group takes 32 contiguous bytes from
  // each of four consecutive reduction rows, and two groups half a row block apart are served together; with rows of
  // 64 bytes more than a multiple of 256 these eight pieces fall into different banks (the LDS serves 256 bytes per
  // clock: measured, bank-conflict cycles 46-50 % -> 10-20 % of the LDS-active cycles against a padding of 16 bytes).
  // 32-bit: a read takes MS elements of each of 64 / MS rows that are four apart (frag4): with 8 elements more than a multiple of
  // 16 (MS 16: 4 more) four rows are half (a quarter) of the 64 banks.
  static constexpr int LDR = ROWS + (sizeof(T) == 2 ? 32 : MS == 16 ? 4 : 8);
  static constexpr int ELEMS = ASIS ? TK * LDR : ROWS * LDK;
  u32x4 reg[ITER];
  bool ok[ITER];

  __device__ __forceinline__ void store(T *S, int tid) const {
#pragma unroll
    for (int it = 0; it < ITER; it++) {
      const int c = tid + it * NT;
      if (NCH % NT == 0 || c < NCH) {
        const u32x4 z = {0u, 0u, 0u, 0u};
        const u32x4 val = ok[it] ? reg[it] : z;
        if constexpr (KCONTIG) {
          *reinterpret_cast<u32x4 *>(S + (c / CPR) * LDK + (c % CPR) * VE) = val;
        } else {
          *reinterpret_cast<u32x4 *>(S + (c / RCH) * LDR + (c % RCH) * VE) = val;
        }
      }
    }
  }
  // fp32: the operands of four MFMAs that start at reduction index k0 of the tile.  NEXT: a lane group takes four neighbouring
  // indices, one an MFMA (which is told two, or four, that are four apart: both operands alike, so that the products are the
  // same, in another order): where the reduction is contiguous one 128-bit read, in place of four of 32 bits whose rows met in the
  // same banks.
  template <class M, bool NEXT> __device__ __forceinline__ static f32x4 frag4(const T *S, int row0, int k0, int lane) {
    const int k = k0 + (NEXT ? 4 : 1) * (lane / MS), row = row0 + lane % MS;
    if constexpr (KCONTIG) {
      static_assert(NEXT, "read as one");
      return *reinterpret_cast<const f32x4 *>(S + row * LDK + k);
    } else {
      constexpr int D = (NEXT ? 1 : M::KSTEP) * LDR;
      const T *p = S + k * LDR + row;
      return f32x4{p[0], p[D], p[2 * D], p[3 * D]};
    }
  }
  // operand fragment of an MS-row MFMA tile starting at tile row `row0`, reduction step kk (KSTEP wide); 16-bit types
  template <class M> __device__ __forceinline__ static typename M::frag_t frag(const T *S, int row0, int kk, int lane) {
    if constexpr (TR) {
      typedef s16x4 __attribute__((address_space(3))) * lds_ptr;
      const int t = lane & 15, gi = lane >> 4;
      // MS 16: the four 16-lane groups are the four reduction groups; MS 32: two row halves x two reduction groups
      const int kq = (MS == 16) ? gi : (gi >> 1), rh = (MS == 16) ? 0 : 16 * (gi & 1);
      const T *p = S + (kk * M::KSTEP + 8 * kq + (t >> 2)) * LDR + row0 + rh + 4 * (t & 3);
      s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)p);
      s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(p + 4 * LDR));
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      s16x8 v = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
      return __builtin_bit_cast(typename M::frag_t, v);
    } else {
      return *reinterpret_cast<const typename M::frag_t *>(S + (row0 + lane % MS) * LDK + (lane / MS) * M::KV + kk * M::KSTEP);
    }
  }
};

// The thread-invariant half of a loader's addressing (one per operand, shared by all ring stages).
template <class Loader, bool KCONTIG> struct TileAddr {
  typedef Loader L;
  Part part[L::ITER];
  template <class View> __device__ __forceinline__ void init(const View &v, int tid) {
#pragma unroll
    for (int it = 0; it < L::ITER; it++) {
      int c = tid + it * L::THREADS;
      if (L::NCH % L::THREADS != 0 && c >= L::NCH) c = L::NCH - 1;
      if constexpr (KCONTIG) part[it] = v.part_k(c / L::CPR, (c % L::CPR) * L::VE);
      else part[it] = v.part_r((c % L::RCH) * L::VE, c / L::RCH);
    }
  }
  // Every thread issues exactly ITER loads whatever the tile holds (chunks outside the operand read a dummy line
  // and are zeroed afterwards): with a fixed count the wait before a stage is consumed is exact.
  template <class View> __device__ __forceinline__ void load(L &dst, const View &v, const typename View::Step &st) const {
    constexpr int NB = View::NB;
    int64_t so[NB];
#pragma unroll
    for (int i = 0; i < NB; i++) so[i] = KCONTIG ? v.scalar_k(st, i) : v.scalar_r(st, i);
#pragma unroll
    for (int it = 0; it < L::ITER; it++) {
      int64_t o = so[0];
      bool live = st.live[0];
#pragma unroll
      for (int i = 1; i < NB; i++) {
        o = part[it].sel == i ? so[i] : o;
        live = part[it].sel == i ? st.live[i] : live;
      }
      const bool good = part[it].ok && live && part[it].k < st.klim;
      dst.ok[it] = good;                // zero-filling happens when the stage is consumed, not here: a use of the loaded
      dst.reg[it] = *reinterpret_cast<const u32x4 *>(good ? v.base + part[it].off + o : v.base);   // value right away would make the wait for it immediate
    }
  }
};

// ---------------------------------------------------------------------------------------------------------
// The tile product.  X supplies TM rows ("m"), Y supplies TN rows ("n"); out(m, n) = sum_k X(m,k) * Y(n,k).
// WGM x WGN wavefronts, each RM x RN MFMA tiles.  OUT_NCONTIG chooses which index the four values of a lane
// run along, so that the epilogue writes 4 consecutive elements whatever the output orientation.
// ---------------------------------------------------------------------------------------------------------
constexpr int stage_tiles(int nc, int ms, int ve, int bytes_per_elem_all_waves, int limit) {
  int cg = nc;
  while (cg > 1 && ms * (cg * ms + ve) * bytes_per_elem_all_waves > limit) cg /= 2;
  return cg;
}

template <typename T, int TM, int TN, int WGM, int WGN, bool X_KCONTIG, bool Y_KCONTIG, bool OUT_NCONTIG> struct TileGemm {
  static constexpr int NT = 64 * WGM * WGN;
  static constexpr int TK = TileK<T>::TK;
  // 32x32 MFMA tiles when a wavefront's region allows it (half the LDS operand traffic per flop), 16x16 otherwise
  static constexpr int MS = (TM / WGM >= 32 && TN / WGN >= 32) ? 32 : 16;
  static constexpr int RM = TM / (MS * WGM), RN = TN / (MS * WGN);
  typedef Mma<T, MS> M;
  typedef TileLoader<T, TM, NT, X_KCONTIG, MS> XL;
  typedef TileLoader<T, TN, NT, Y_KCONTIG, MS> YL;
  static constexpr int X_ELEMS = (XL::ELEMS + 7) & ~7, Y_ELEMS = (YL::ELEMS + 7) & ~7;
  static constexpr int SMEM_BYTES = 2 * (X_ELEMS + Y_ELEMS) * (int)sizeof(T);

  // ksteps = number of TK-wide reduction steps.  Store(m, n, vals): vals[4] run along n (OUT_NCONTIG) or m.
  // SUB > 0: the output consists of SUB x SUB blocks that are each contiguous in memory (the sparse result of sdd);
  // the epilogue then writes block by block.  SUB == 0: the output is a matrix with long rows.
  // PARTIAL: the result is a part of a sum; store takes the fp32 values (f32x4) as they are.
  template <int SUB = 0, bool PARTIAL = false, class XView, class YView, class Store>
  static __device__ __forceinline__ void run(const XView &xv, const YView &yv, int ksteps, T *smem, const Store &store) {
    const int tid = threadIdx.x % NT, lane = tid & 63, wave = tid >> 6;   // (a workgroup may hold several products of one wavefront)
    const int wm = wave / WGN, wn = wave % WGN;
    T *Xs[2] = {smem, smem + X_ELEMS + Y_ELEMS};
    T *Ys[2] = {smem + X_ELEMS, smem + 2 * X_ELEMS + Y_ELEMS};
    typename M::acc_t acc[RM][RN];
#pragma unroll
    for (int i = 0; i < RM; i++)
#pragma unroll
      for (int j = 0; j < RN; j++)
#pragma unroll
        for (int v = 0; v < M::NACC; v++) acc[i][j][v] = 0.f;
    // Register ring of NS stages (two: deeper rings were measured slower or equal, on large tiles and on the small ones of short
    // launches, the loop is not waiting for its loads): global loads run NS - 1 reduction steps ahead of their use; two LDS buffers, one
    // barrier per step.  Step s first writes stage s + 1 to the other LDS buffer, then reads stage s and issues its
    // MFMAs, then refills the ring slot it has just emptied, and only then meets the barrier: the LDS write and the
    // barrier wait pass while the matrix pipe works instead of in front of it.  The loop runs whole rounds of NS
    // steps; steps past the end hold zeros.
    constexpr int NS = 2;
    static_assert(NS % 2 == 0, "the LDS buffer of a step is chosen by the ring slot's parity");
    XL xl[NS];
    YL yl[NS];
    TileAddr<XL, X_KCONTIG> xa;
    TileAddr<YL, Y_KCONTIG> ya;
    xa.init(xv, tid);
    ya.init(yv, tid);
#pragma unroll
    for (int u = 0; u < NS; u++) {
      xa.load(xl[u], xv, xv.step(u * TK));
      ya.load(yl[u], yv, yv.step(u * TK));
    }
    xl[0].store(Xs[0], tid);
    yl[0].store(Ys[0], tid);
    xa.load(xl[0], xv, xv.step(NS * TK));
    ya.load(yl[0], yv, yv.step(NS * TK));
    // The table look-ups run one step ahead of the refill that uses them: started a whole step before they are needed,
    // their (scalar) latency is not in front of the loads.
    auto xst = xv.step((NS + 1) * TK);
    auto yst = yv.step((NS + 1) * TK);
    __syncthreads();
    for (int s0 = 0; s0 < ksteps; s0 += NS) {
#pragma unroll
      for (int u = 0; u < NS; u++) {
        const int s = s0 + u;
        const int cur = u & 1, nxt = cur ^ 1, u1 = (u + 1) % NS;
        xl[u1].store(Xs[nxt], tid);   // stage s + 1; this buffer was last read in step s - 1, before the previous barrier
        yl[u1].store(Ys[nxt], tid);
        // (steps past the end multiply zeros: cheaper than a branch, which would copy the accumulators around)
        auto product = [&](auto &xf, auto &yf, auto &&of) {
#pragma unroll
          for (int i = 0; i < RM; i++)
#pragma unroll
            for (int j = 0; j < RN; j++) {
              if constexpr (OUT_NCONTIG) acc[i][j] = M::run(of(yf[j]), of(xf[i]), acc[i][j]);   // result rows = n, column = m
              else acc[i][j] = M::run(of(xf[i]), of(yf[j]), acc[i][j]);                          // result rows = m, column = n
            }
        };
        if constexpr (sizeof(T) == 4) {
          // with the reduction strided in both operands rows of 32 lose 2-7 % to NEXT, rows of 16 win 2-8 %
          constexpr bool NEXT = X_KCONTIG || Y_KCONTIG || MS == 16;
#pragma unroll
          for (int k0 = 0; k0 < TK; k0 += 4 * M::KSTEP) {
            f32x4 xf[RM], yf[RN];
#pragma unroll
            for (int i = 0; i < RM; i++) xf[i] = XL::template frag4<M, NEXT>(Xs[cur], (wm * RM + i) * MS, k0, lane);
#pragma unroll
            for (int j = 0; j < RN; j++) yf[j] = YL::template frag4<M, NEXT>(Ys[cur], (wn * RN + j) * MS, k0, lane);
#pragma unroll
            for (int e = 0; e < 4; e++) product(xf, yf, [&](const f32x4 &v) { return v[e]; });
          }
        } else {
#pragma unroll
          for (int kk = 0; kk < TK / M::KSTEP; kk++) {
            typename M::frag_t xf[RM], yf[RN];
#pragma unroll
            for (int i = 0; i < RM; i++) xf[i] = XL::template frag<M>(Xs[cur], (wm * RM + i) * MS, kk, lane);
#pragma unroll
            for (int j = 0; j < RN; j++) yf[j] = YL::template frag<M>(Ys[cur], (wn * RN + j) * MS, kk, lane);
            product(xf, yf, [](const typename M::frag_t &v) { return v; });
          }
        }
        const auto xnext = xv.step((s + NS + 2) * TK);
        const auto ynext = yv.step((s + NS + 2) * TK);
        xa.load(xl[u1], xv, xst);   // stage s + 1 + NS into the slot emptied above
        ya.load(yl[u1], yv, yst);
        xst = xnext;
        yst = ynext;
        __syncthreads();
      }
    }
    // Epilogue.  A lane's values come in groups of 4 consecutive positions along the output's contiguous index
    // (4*(lane/16) for MS 16, 8*g + 4*(lane/32) for MS 32) at row lane % MS of a tile, so a direct store would write
    // 8- or 16-byte pieces of 32 different rows per instruction.  Each wavefront instead passes one row of tiles at a
    // time through its own piece of LDS (free after the last barrier) and writes whole 16-byte chunks, consecutive
    // lanes along a row.  store(r, c, chunk): r = row (m if OUT_NCONTIG, else n), c = first of VE consecutive columns.
    constexpr int VE = 16 / (int)sizeof(T);
    if constexpr (PARTIAL) {
      // (straight from the accumulators, 16 bytes a lane: parts are few, and what reads them next finds them in L2)
#pragma unroll
      for (int i = 0; i < RM; i++)
#pragma unroll
        for (int j = 0; j < RN; j++)
#pragma unroll
          for (int g4 = 0; g4 < M::NACC / 4; g4++) {
            const int m0 = (wm * RM + i) * MS, nn0 = (wn * RN + j) * MS, along = MS == 16 ? 4 * (lane >> 4) : 8 * g4 + 4 * (lane >> 5);
            store(lane % MS + (OUT_NCONTIG ? m0 : nn0), along + (OUT_NCONTIG ? nn0 : m0),
                  f32x4{acc[i][j][4 * g4], acc[i][j][4 * g4 + 1], acc[i][j][4 * g4 + 2], acc[i][j][4 * g4 + 3]});
          }
    } else {
    if constexpr (SUB > 0 && OUT_NCONTIG && TM * (TN + VE) * (int)sizeof(T) <= SMEM_BYTES) {
      // Blocked output: the whole TM x TN tile is staged (all wavefronts, two barriers) and then written block by
      // block, consecutive lanes on consecutive 16-byte chunks of one block: 512 contiguous bytes per 32 lanes at
      // block 16, where row-wise stores would write 32-byte pieces.
      constexpr int LDS_ROW = TN + VE, CPB = SUB * SUB / VE, BPR = TN / SUB, CHUNKS = TM * TN / VE;
      const int cc = lane % MS;
#pragma unroll
      for (int i = 0; i < RM; i++)
#pragma unroll
        for (int j = 0; j < RN; j++)
#pragma unroll
          for (int g4 = 0; g4 < M::NACC / 4; g4++) {
            const int rr = (MS == 16) ? 4 * (lane >> 4) : 8 * g4 + 4 * (lane >> 5);
            T *dst = smem + ((wm * RM + i) * MS + cc) * LDS_ROW + (wn * RN + j) * MS + rr;
            if constexpr (sizeof(T) == 4) {
              *reinterpret_cast<f32x4 *>(dst) = f32x4{acc[i][j][4 * g4 + 0], acc[i][j][4 * g4 + 1], acc[i][j][4 * g4 + 2], acc[i][j][4 * g4 + 3]};
            } else {
              union { u32x2 raw; T e[4]; } u;
#pragma unroll
              for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(acc[i][j][4 * g4 + e]);
              *reinterpret_cast<u32x2 *>(dst) = u.raw;
            }
          }
      __syncthreads();
#pragma unroll
      for (int it = 0; it < (CHUNKS + NT - 1) / NT; it++) {
        const int idx = it * NT + tid;
        if (CHUNKS % NT == 0 || idx < CHUNKS) {
          const int blk = idx / CPB, within = idx % CPB;
          const int m = (blk / BPR) * SUB + within / (SUB / VE), n = (blk % BPR) * SUB + (within % (SUB / VE)) * VE;
          store(m, n, *reinterpret_cast<const u32x4 *>(smem + m * LDS_ROW + n));
        }
      }
      return;
    }
    constexpr int NR = OUT_NCONTIG ? RM : RN, NC = OUT_NCONTIG ? RN : RM;   // tiles along the row / contiguous index
    // tiles staged per pass: all NC of them if that fits the tile buffers, else half, a quarter ...
    constexpr int CG = stage_tiles(NC, MS, VE, (int)sizeof(T) * WGM * WGN, SMEM_BYTES);
    constexpr int CW = CG * MS, LDS_ROW = CW + VE;                            // staged row, padded by one chunk
    static_assert(MS * LDS_ROW * (int)sizeof(T) * WGM * WGN <= SMEM_BYTES, "epilogue staging must fit the tile buffers");
    T *stage = smem + wave * (MS * LDS_ROW);
    const int cc = lane % MS;
    const int r_wave = OUT_NCONTIG ? wm * RM * MS : wn * RN * MS, c_wave = OUT_NCONTIG ? wn * RN * MS : wm * RM * MS;
#pragma unroll
    for (int pass = 0; pass < NR * (NC / CG); pass++) {
      const int rt = pass / (NC / CG), c0 = (pass % (NC / CG)) * CG;
#pragma unroll
      for (int ct = 0; ct < CG; ct++)
#pragma unroll
        for (int g4 = 0; g4 < M::NACC / 4; g4++) {
          const typename M::acc_t &t = OUT_NCONTIG ? acc[rt][c0 + ct] : acc[c0 + ct][rt];
          const int rr = (MS == 16) ? 4 * (lane >> 4) : 8 * g4 + 4 * (lane >> 5);
          T *dst = stage + cc * LDS_ROW + ct * MS + rr;
          if constexpr (sizeof(T) == 4) {
            *reinterpret_cast<f32x4 *>(dst) = f32x4{t[4 * g4 + 0], t[4 * g4 + 1], t[4 * g4 + 2], t[4 * g4 + 3]};
          } else {
            union { u32x2 raw; T e[4]; } u;
#pragma unroll
            for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(t[4 * g4 + e]);
            *reinterpret_cast<u32x2 *>(dst) = u.raw;
          }
        }
      __builtin_amdgcn_wave_barrier();   // the LDS operations of one wavefront complete in order
      constexpr int CHUNKS = MS * CW / VE;
#pragma unroll
      for (int it = 0; it < (CHUNKS + 63) / 64; it++) {
        const int idx = it * 64 + lane;
        if (CHUNKS % 64 == 0 || idx < CHUNKS) {
          const int row = idx / (CW / VE), ch = idx % (CW / VE);
          store(r_wave + rt * MS + row, c_wave + c0 * MS + ch * VE, *reinterpret_cast<const u32x4 *>(stage + row * LDS_ROW + ch * VE));
        }
      }
      __builtin_amdgcn_wave_barrier();
    }
    }
  }
};

// ---------------------------------------------------------------------------------------------------------
// sdd: C[z, blockid] = op(A)[z,h, i-th block-row, :K] . op(B)[z,h, :K, j-th block-col]
// One workgroup per super-block of PACK x PACK blocks of the sdd table (reference kernel matmul.py:30-54,
// 163-176: rows come from the table entries (bm, 0), columns from (0, bn), the head from entry (0, 0), the
// output block from entry (bm, bn)).
// ---------------------------------------------------------------------------------------------------------
struct SddArgs {
  const void *a, *b; void *c;
  int Z, K;
  int64_t a_sz, a_sh, lda, b_sz, b_sh, ldb, c_sz;
  const int32_t *lut; const uint8_t *valid;
  int64_t n_groups;
  const int32_t *gplan; int n_pgroups; int lines;   // optional group plan (by rows), its groups, block-rows per head
  int cols = 0;                                       // block-columns per head when known (a call with the plan alone), else 0
  // the reduction cut into parts of part_k elements, whose fp32 sums go to ws [part][Z][n_blocks][block][block]
  int parts = 1, part_k = 0;
  int64_t n_blocks = 0;
  float *ws = nullptr;
};

struct SddLevel { int pack; const int32_t *lut; const uint8_t *valid; int64_t n; };   // one pack level of the sdd table, n super-blocks

template <typename T, int BLOCK, int PACK, bool KCONTIG> struct SddView {
  // idx is a vector, not an array: an array member makes the compiler keep the view in scratch memory and turn the
  // selection in blk() into an indexed scratch load, a full memory round trip before a workgroup's first load
  typedef int idx_t __attribute__((ext_vector_type(PACK == 1 ? 2 : PACK)));
  const T *base; int64_t ld; int K; idx_t idx;   // base doubles as the dummy address of out-of-range chunks
  int off = 0;                                        // first row of the tile inside its block (tiles smaller than a block)
  int first = 0;                                      // where the reduction starts (K: where it ends)
  static constexpr int NB = 1;
  struct Step { int k0; bool live[1]; int klim; };
  __device__ __forceinline__ Step step(int k0) const { return Step{first + k0, {true}, K - first - k0}; }
  __device__ __forceinline__ int blk(int row) const {
    int r = idx[0];
#pragma unroll
    for (int p = 1; p < PACK; p++) r = (row / BLOCK == p) ? idx[p] : r;
    return r * BLOCK + off + row % BLOCK;
  }
  __device__ __forceinline__ Part part_k(int row, int k) const { return Part{(int64_t)blk(row) * ld + k, true, 0, k}; }
  __device__ __forceinline__ Part part_r(int row, int k) const { return Part{(int64_t)k * ld + blk(row), true, 0, k}; }
  __device__ __forceinline__ int64_t scalar_k(const Step &st, int) const { return st.k0; }
  __device__ __forceinline__ int64_t scalar_r(const Step &st, int) const { return (int64_t)st.k0 * ld; }
};

template <int T_> struct SddShape { static constexpr int WG = T_ >= 32 ? 2 : 1; };

// One super-block, by the SddShape<BLOCK * PACK>::WG squared wavefronts that call it together
template <typename T, int BLOCK, int PACK, bool A_KCONTIG, bool B_KCONTIG, bool PARTS>
__device__ __forceinline__ void sdd_super_block(const SddArgs &g, const int32_t *lut, const uint8_t *all_valid, int part, int z, int64_t grp, bool keep, unsigned char *smem) {
  constexpr int TT = BLOCK * PACK, WG = SddShape<TT>::WG;
  typedef TileGemm<T, TT, TT, WG, WG, A_KCONTIG, B_KCONTIG, true> G;
  const table_ptr e = as_table(lut) + grp * (PACK * PACK * 4);
  const int h = e[0];
  SddView<T, BLOCK, PACK, A_KCONTIG> av;
  SddView<T, BLOCK, PACK, B_KCONTIG> bv;
  av.base = reinterpret_cast<const T *>(g.a) + z * g.a_sz + h * g.a_sh; av.ld = g.lda; av.K = g.K;
  bv.base = reinterpret_cast<const T *>(g.b) + z * g.b_sz + h * g.b_sh; bv.ld = g.ldb; bv.K = g.K;
#pragma unroll
  for (int p = 0; p < PACK; p++) {
    av.idx[p] = e[(p * PACK) * 4 + 1];   // block-row of entries (p, 0)
    bv.idx[p] = e[p * 4 + 2];            // block-col of entries (0, p)
  }
  if constexpr (PARTS) {
    av.first = bv.first = part * g.part_k;
    if (av.first + g.part_k < g.K) av.K = bv.K = av.first + g.part_k;
  }
  T *cz = reinterpret_cast<T *>(g.c) + z * g.c_sz;
  const uint8_t *valid = all_valid ? all_valid + grp * (PACK * PACK) : nullptr;
  // The entry differs from lane to lane here, so the output block is looked up through an ordinary pointer (a vector
  // load): through the constant address space the compiler fetches all PACK * PACK entries with scalar loads and
  // indexes them per lane in scratch memory.
  const int32_t *eg = lut + grp * (PACK * PACK * 4);
  auto store = [&](int m, int n, u32x4 v) {
    const int ent = (m / BLOCK) * PACK + n / BLOCK;
    if (!keep || (valid && !valid[ent])) return;
    const int64_t bk = eg[ent * 4 + 3];
    *reinterpret_cast<u32x4 *>(cz + bk * (BLOCK * BLOCK) + (m % BLOCK) * BLOCK + n % BLOCK) = v;
  };
  if constexpr (PARTS) {
    float *ws = g.ws + ((int64_t)part * g.Z + z) * g.n_blocks * (BLOCK * BLOCK);
    auto store_part = [&](int m, int n, f32x4 v) {
      const int ent = (m / BLOCK) * PACK + n / BLOCK;
      if (!keep || (valid && !valid[ent])) return;
      *reinterpret_cast<f32x4 *>(ws + (int64_t)eg[ent * 4 + 3] * (BLOCK * BLOCK) + (m % BLOCK) * BLOCK + n % BLOCK) = v;
    };
    // (every part of every wavefront runs the same number of steps: those past the end of the reduction multiply zeros)
    G::template run<BLOCK, true>(av, bv, (g.part_k + G::TK - 1) / G::TK, reinterpret_cast<T *>(smem), store_part);
  } else {
    G::template run<BLOCK>(av, bv, (g.K + G::TK - 1) / G::TK, reinterpret_cast<T *>(smem), store);
  }
}

template <typename T, int BLOCK, bool A_KCONTIG, bool B_KCONTIG, bool PARTS>
__global__ void __launch_bounds__(64 * SddShape<BLOCK>::WG * SddShape<BLOCK>::WG) k_sdd(SddArgs g) {
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int64_t n_wg = g.n_groups * g.Z;
  const uint32_t w = (uint32_t)xcd_remap(blockIdx.x, PARTS ? n_wg * g.parts : n_wg), part = PARTS ? w / (uint32_t)n_wg : 0;
  const Quotient z((PARTS ? w - part * (uint32_t)n_wg : w), (uint32_t)g.n_groups);
  sdd_super_block<T, BLOCK, 1, A_KCONTIG, B_KCONTIG, PARTS>(g, g.lut, g.valid, (int)part, (int)z.q, z.r, true, smem_raw);
}

// The second pass of an sdd in parts: the parts of every block in order, rounded once
template <typename T> __global__ void __launch_bounds__(256) k_sdd_parts_sum(SddArgs g, int64_t per_z) {   // per_z: groups of four values of a batch's blocks
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x, all = per_z * g.Z;
  if (i >= all) return;
  const f32x4 *ws = reinterpret_cast<const f32x4 *>(g.ws) + i;
  f32x4 sum = ws[0];
  for (int p = 1; p < g.parts; p++) {
    const f32x4 v = ws[p * all];
#pragma unroll
    for (int e = 0; e < 4; e++) sum[e] += v[e];
  }
  T *c = reinterpret_cast<T *>(g.c) + (i / per_z) * g.c_sz + (i % per_z) * 4;
  if constexpr (sizeof(T) == 4) {
    *reinterpret_cast<f32x4 *>(c) = sum;
  } else {
    union { u32x2 raw; T e[4]; } u;
#pragma unroll
    for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(sum[e]);
    *reinterpret_cast<u32x2 *>(c) = u.raw;
  }
}

// Blocks of 16 and 32: every pack level of the table in one launch, the largest super-blocks first.  A launch per level
// leaves the chip idle between them and at the end of each: fp32, block 16, 256 x 512 x 384 in 8 heads and batches, half of
// the blocks, takes 11.3 + 9.5 us in two launches and 14.7 in one.  The host makes one launch less, too.
// The last level of block 16 has super-blocks of one wavefront, four of which share a workgroup: they run the same number of steps and
// so of barriers, and the ones past the end of the level repeat its last super-block and keep nothing.
template <int BLOCK> struct SddLevels {
  static constexpr int N = BLOCK == 16 ? 3 : 2;
  const int32_t *lut[N];                 // by pack: 64 / BLOCK, half of that, ..., 1
  const uint8_t *valid[N];
  int64_t n[N];                          // super-blocks
};
constexpr int max_of(int a, int b) { return a > b ? a : b; }
template <typename T, int BLOCK, bool AK, bool BK> struct SddLevelsShape {
  static constexpr int PACK0 = 64 / BLOCK, LAST_PER_WG = BLOCK == 16 ? 4 : 1;
  template <int P> using G = TileGemm<T, BLOCK * P, BLOCK * P, SddShape<BLOCK * P>::WG, SddShape<BLOCK * P>::WG, AK, BK, true>;
  static constexpr int SMEM = max_of(max_of(G<PACK0>::SMEM_BYTES, G<PACK0 / 2>::SMEM_BYTES), LAST_PER_WG * G<1>::SMEM_BYTES);
};

template <typename T, int BLOCK, bool A_KCONTIG, bool B_KCONTIG, bool PARTS>
__global__ void __launch_bounds__(256) k_sdd_levels(SddArgs g, SddLevels<BLOCK> lv, int64_t per_part) {
  typedef SddLevelsShape<T, BLOCK, A_KCONTIG, B_KCONTIG> S;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int part = PARTS ? (int)(blockIdx.x / (uint32_t)per_part) : 0;
  int64_t w = PARTS ? blockIdx.x % (uint32_t)per_part : blockIdx.x, n = lv.n[0] * g.Z;
  if (w < n) {
    const Quotient z((uint32_t)xcd_remap(w, n), (uint32_t)lv.n[0]);
    sdd_super_block<T, BLOCK, S::PACK0, A_KCONTIG, B_KCONTIG, PARTS>(g, lv.lut[0], lv.valid[0], part, (int)z.q, z.r, true, smem_raw);
    return;
  }
  w -= n;
  if constexpr (BLOCK == 16) {
    n = lv.n[1] * g.Z;
    if (w < n) {
      const Quotient z((uint32_t)xcd_remap(w, n), (uint32_t)lv.n[1]);
      sdd_super_block<T, 16, 2, A_KCONTIG, B_KCONTIG, PARTS>(g, lv.lut[1], lv.valid[1], part, (int)z.q, z.r, true, smem_raw);
      return;
    }
    w -= n;
  }
  constexpr int LAST = SddLevels<BLOCK>::N - 1, PER = S::LAST_PER_WG;
  const int64_t last = lv.n[LAST] * g.Z;
  w = xcd_remap(w, (last + PER - 1) / PER);
  const int own = PER == 1 ? 0 : __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int64_t i = w * PER + own, j = i < last ? i : last - 1;
  const Quotient z((uint32_t)j, (uint32_t)lv.n[LAST]);
  sdd_super_block<T, BLOCK, 1, A_KCONTIG, B_KCONTIG, PARTS>(g, lv.lut[LAST], lv.valid[LAST], part, (int)z.q, z.r, i < last,
                                                            smem_raw + own * S::template G<1>::SMEM_BYTES);
}

// sdd with SPLIT x SPLIT workgroups per block (pack 1): for layouts with so few blocks that one workgroup per block
// would leave most of the chip idle (a 10 % dense 32 x 32 layout of 128-blocks has 100 blocks for 256 CUs).  The
// sub-tiles of a block are neighbours in the grid, so that they meet their shared operand rows in L2.
template <typename T, int BLOCK, int SPLIT, bool A_KCONTIG, bool B_KCONTIG, bool PARTS>
__global__ void __launch_bounds__(64 * SddShape<BLOCK / SPLIT>::WG * SddShape<BLOCK / SPLIT>::WG) k_sdd_split(SddArgs g) {
  constexpr int TT = BLOCK / SPLIT, WG = SddShape<TT>::WG;
  typedef TileGemm<T, TT, TT, WG, WG, A_KCONTIG, B_KCONTIG, true> G;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int64_t n_wg = g.n_groups * g.Z * (SPLIT * SPLIT);
  const uint32_t w = (uint32_t)xcd_remap(blockIdx.x, PARTS ? n_wg * g.parts : n_wg);
  const int sub = (int)(w % (SPLIT * SPLIT)), part = PARTS ? (int)(w / (uint32_t)n_wg) : 0;
  const Quotient batch((PARTS ? w - part * (uint32_t)n_wg : w) / (SPLIT * SPLIT), (uint32_t)g.n_groups);
  const int z = (int)batch.q;
  const int64_t grp = batch.r;
  const table_ptr e = as_table(g.lut) + grp * 4;
  if (g.valid && !g.valid[grp]) return;
  SddView<T, BLOCK, 1, A_KCONTIG> av;
  SddView<T, BLOCK, 1, B_KCONTIG> bv;
  av.base = reinterpret_cast<const T *>(g.a) + z * g.a_sz + e[0] * g.a_sh; av.ld = g.lda; av.K = g.K;
  bv.base = reinterpret_cast<const T *>(g.b) + z * g.b_sz + e[0] * g.b_sh; bv.ld = g.ldb; bv.K = g.K;
  av.idx[0] = e[1]; av.off = (sub / SPLIT) * TT;
  bv.idx[0] = e[2]; bv.off = (sub % SPLIT) * TT;
  if constexpr (PARTS) {
    av.first = bv.first = part * g.part_k;
    if (av.first + g.part_k < g.K) av.K = bv.K = av.first + g.part_k;
    float *ws = g.ws + (((int64_t)part * g.Z + z) * g.n_blocks + e[3]) * (BLOCK * BLOCK) + av.off * BLOCK + bv.off;
    G::template run<0, true>(av, bv, (g.part_k + G::TK - 1) / G::TK, reinterpret_cast<T *>(smem_raw), [&](int m, int n, f32x4 v) { *reinterpret_cast<f32x4 *>(ws + m * BLOCK + n) = v; });
    return;
  }
  T *cb = reinterpret_cast<T *>(g.c) + z * g.c_sz + (int64_t)e[3] * (BLOCK * BLOCK) + av.off * BLOCK + bv.off;
  auto store = [&](int m, int n, u32x4 v) { *reinterpret_cast<u32x4 *>(cb + m * BLOCK + n) = v; };
  G::run(av, bv, (g.K + G::TK - 1) / G::TK, reinterpret_cast<T *>(smem_raw), store);
}

// ---------------------------------------------------------------------------------------------------------
// xsd: out[col*BLOCK + m, n] = sum over the blocks t of one table segment  S_t(m, :) . D(n, pos_t + :)
// (dsd: S = op(A) blocks, D = op(B)^T rows; dds: S = op(B)^T blocks, D = op(A) rows).
// One workgroup per (segment, tile of the dense free dimension, batch).  Reads the segment header
// of the reference table (offset, length, column, depth; matmul.py:57-63) and the per-block positions.
// ---------------------------------------------------------------------------------------------------------
struct XsdArgs {
  const void *sp, *dn; void *out;
  int Z, NF;                            // batch, size of the dense free dimension
  int64_t sp_sz, dn_sz, dn_sh, ldd, out_sz, out_sh, ldo;
  const int32_t *lut; const int32_t *plan; int width; int div2;   // div2 = 2 * block / step of the table
  const int32_t *order;                 // order[p] = segment dispatched p-th (head by head, longest first inside a head), or null
  int n_tiles;                          // 64-wide tiles of the free dimension (specialised kernels)
  const int32_t *gplan; int n_pgroups; int lines;   // optional group plan, its groups, lines (block-rows or -columns) per head
  int n_split = 0;                      // split chains of the plan; their fp32 partial tiles (caller's workspace)
  float *partials = nullptr;
  // general kernels: segments of more than part_blocks blocks run in parts of that many (at most `parts` of them), whose fp32 tiles
  // go to partials [part][Z][width][tiles]
  int parts = 1, part_blocks = 0;
};

// A reduction step of TK elements lies inside one block (BLOCK >= TK) or covers TK / BLOCK whole blocks.
template <typename T, int BLOCK> struct StepBlocks { static constexpr int TK = TileK<T>::TK, NB = TK > BLOCK ? TK / BLOCK : 1; };

// The Step of a view holds the raw table values only; all arithmetic on them happens when the addresses are formed,
// so that a look-up started one step ahead is not waited for before it is needed.
template <typename T, int BLOCK, bool TRANS> struct SparseView {   // element (m, k) of the segment's blocks
  const T *base; table_ptr plan; int nblk;
  static constexpr int NB = StepBlocks<T, BLOCK>::NB;
  struct Step { int32_t bid[NB]; bool live[NB]; int kin; int klim; };   // storage index of each block, whether it exists, offset inside
  __device__ __forceinline__ Step step(int k0) const {
    Step st;
    st.kin = k0 % BLOCK;
    st.klim = 1 << 30;
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int ord = k0 / BLOCK + i;
      // unconditional read of a clamped index (nblk >= 1): a load under a branch could not be started early
      st.bid[i] = plan[2 * (ord < nblk ? ord : nblk - 1) + 1];
      st.live[i] = ord < nblk;
    }
    return st;
  }
  // stored [m][k] (part_k) or [k][m] (part_r); k / BLOCK picks the block when a step spans several
  __device__ __forceinline__ Part part_k(int row, int k) const { return Part{(int64_t)row * BLOCK + k % BLOCK, true, k / BLOCK, k}; }
  __device__ __forceinline__ Part part_r(int row, int k) const { return Part{(int64_t)(k % BLOCK) * BLOCK + row, true, k / BLOCK, k}; }
  __device__ __forceinline__ int64_t scalar_k(const Step &st, int i) const { return (int64_t)st.bid[i] * (BLOCK * BLOCK) + st.kin; }
  __device__ __forceinline__ int64_t scalar_r(const Step &st, int i) const { return (int64_t)st.bid[i] * (BLOCK * BLOCK) + st.kin * BLOCK; }
};

template <typename T, int BLOCK> struct DenseView {                   // element (n, k): dense row/col n, reduction position k
  const T *base; table_ptr plan; int nblk; int64_t ld; int n0, NF;
  static constexpr int NB = StepBlocks<T, BLOCK>::NB;
  struct Step { int32_t pos[NB]; bool live[NB]; int kin; int klim; };  // position of each block in the dense operand, whether it exists
  __device__ __forceinline__ Step step(int k0) const {
    Step st;
    st.kin = k0 % BLOCK;
    st.klim = 1 << 30;
#pragma unroll
    for (int i = 0; i < NB; i++) {
      const int ord = k0 / BLOCK + i;
      st.pos[i] = plan[2 * (ord < nblk ? ord : nblk - 1)];
      st.live[i] = ord < nblk;
    }
    return st;
  }
  // stored [n][k] (part_k) or [k][n] (part_r); rows past the free dimension are zero-filled
  __device__ __forceinline__ Part part_k(int row, int k) const { return Part{(int64_t)(n0 + row) * ld + k % BLOCK, n0 + row < NF, k / BLOCK, k}; }
  __device__ __forceinline__ Part part_r(int row, int k) const { return Part{(int64_t)(k % BLOCK) * ld + n0 + row, n0 + row < NF, k / BLOCK, k}; }
  __device__ __forceinline__ int64_t scalar_k(const Step &st, int i) const { return (int64_t)st.pos[i] + st.kin; }
  __device__ __forceinline__ int64_t scalar_r(const Step &st, int i) const { return ((int64_t)st.pos[i] + st.kin) * ld; }
};

// Tile of the dense free dimension, TN: 64, 128 or 256 wide.  Wide tiles for blocks of 32 and 128: a wavefront then reuses each fragment
// of the sparse block for two or four MFMAs (LDS reads per MFMA are what bounds these kernels); measured +13 % at block 32.  A free
// dimension up to 64 or 128 (the head dimension of an attention product) takes a tile that it fills: fp32, block 32, 18 blocks a row, 128
// wide, 52 us on tiles of 256, half of them padding.
constexpr int xsd_tile(int block, int free_dim) { return free_dim <= 64 || block == 16 ? 64 : block == 64 || free_dim <= 128 ? 128 : 256; }
template <int BLOCK, int TN_> struct XsdShape {
  static constexpr int TN = TN_;
  // wider than 64: 32 -> 1x4 wavefronts of 32x32 / 32x64; 64 -> 2x2 of 32x64; 128 -> 2x2 of 64x64 / 64x128.  64: 16 -> 1x4 of 16x16;
  // 32 -> 2x2 of 16x32; 64 -> 2x2 of 32x32; 128 -> 2x2 of 64x32
  static constexpr int WGM = (TN > 64 ? BLOCK >= 64 : BLOCK >= 32) ? 2 : 1;
  static constexpr int WGN = 4 / WGM;
};

// Which (batch, tile of the free dimension, position in the dispatch order) a workgroup of the dsd / dds kernels takes.
// Segment index fastest: consecutive workgroups (same XCD after the re-numbering) walk the segments of a head against one
// slab of columns of the dense operand, which then stays in L2 between its uses.  With a dispatch order (g.order:
// longest segments first, short launches only) "first" has to mean first on every XCD: an XCD works on a contiguous
// eighth of the launch, so inside its eighth the position in the order is the slow index and the tile the fast one.
// One batch with a number of tiles that divides by 8: every XCD gets all segments for its own tiles; a batch that
// divides by 8: every XCD gets whole batches.
__device__ __forceinline__ void xsd_work_item(const XsdArgs &g, int n_tiles, uint32_t wg, int &z, int &nt, int &seg0) {
  const uint32_t per_z = (uint32_t)g.width * n_tiles, total = per_z * (uint32_t)g.Z;   // (a launch has fewer than 2^31 workgroups)
  const uint32_t w = (uint32_t)xcd_remap(wg, total);
  if (g.order && total % 8 == 0 && ((g.Z == 1 && n_tiles % 8 == 0) || g.Z % 8 == 0)) {
    const Quotient x(w, total / 8);
    if (g.Z % 8) {
      const Quotient s(x.r, (uint32_t)n_tiles / 8);
      z = 0;
      seg0 = (int)s.q;
      nt = (int)(x.q * (n_tiles / 8) + s.r);
    } else {
      const Quotient b(x.r, per_z), s(b.r, (uint32_t)n_tiles);
      z = (int)(x.q * (g.Z / 8) + b.q);
      seg0 = (int)s.q;
      nt = (int)s.r;
    }
    return;
  }
  const Quotient b(w, per_z), t(b.r, (uint32_t)g.width);
  z = (int)b.q;
  nt = (int)t.q;
  seg0 = (int)t.r;
}

// (at least two wavefronts per SIMD: the 128 x 256 tile of block 128 would otherwise take 266 registers and run alone)
template <typename T, int BLOCK, int TN_, bool SP_TRANS, bool DN_KCONTIG, bool OUT_NCONTIG, bool PARTS>
__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2))) k_xsd(XsdArgs g) {
  typedef XsdShape<BLOCK, TN_> S;
  typedef TileGemm<T, BLOCK, S::TN, S::WGM, S::WGN, !SP_TRANS, DN_KCONTIG, OUT_NCONTIG> G;
  extern __shared__ __attribute__((aligned(16))) unsigned char smem_raw[];
  const int n_tiles = (g.NF + S::TN - 1) / S::TN;
  const int64_t n_wg = (int64_t)g.width * n_tiles * g.Z;
  const int part = PARTS ? (int)(blockIdx.x / (uint32_t)n_wg) : 0;
  int z, nt, seg0;
  xsd_work_item(g, n_tiles, PARTS ? blockIdx.x % (uint32_t)n_wg : blockIdx.x, z, nt, seg0);
  const int seg = g.order ? as_table(g.order)[seg0] : seg0;   // longest first only where the launch is short (see the dispatcher)
  const table_ptr hd = as_table(g.lut) + 6 * (int64_t)seg;
  const int offset = hd[0], seglen = hd[1], column = hd[2], depth = hd[3];
  const int whole = seglen / BLOCK;
  int nblk = whole;
  if constexpr (PARTS) {
    nblk = whole - part * g.part_blocks;
    if (part > 0 && nblk <= 0) return;
    if (nblk > g.part_blocks) nblk = g.part_blocks;
  }
  if (nblk == 0) {
    // The table carries zero-length segments.  One that stands alone is an empty row/column of the layout and
    // must zero-fill its output tile; one that follows a real segment of the same row/column must not touch it.
    if (seg > 0 && hd[-6 + 2] == column && hd[-6 + 3] == depth) return;
  }
  const int t0 = (offset - 6 * g.width) / g.div2 + part * g.part_blocks;   // first block of the segment (the part) in table order
  SparseView<T, BLOCK, SP_TRANS> sv;
  sv.base = reinterpret_cast<const T *>(g.sp) + z * g.sp_sz; sv.plan = as_table(g.plan) + 2 * (int64_t)t0; sv.nblk = nblk;
  DenseView<T, BLOCK> dv;
  dv.base = reinterpret_cast<const T *>(g.dn) + z * g.dn_sz + depth * g.dn_sh; dv.plan = sv.plan; dv.nblk = nblk; dv.ld = g.ldd;
  dv.n0 = nt * S::TN; dv.NF = g.NF;
  T *oz = reinterpret_cast<T *>(g.out) + z * g.out_sz + depth * g.out_sh;
  const int NF = g.NF, n0 = nt * S::TN;
  const int64_t ldo = g.ldo;
  // r, c = (m, n) when the output has n contiguous, (n, m) otherwise; c is the first of a 16-byte chunk
  // streaming stores: the dense result is not read again by the sparse chain and should not displace what is
  auto store = [&](int r, int c, u32x4 v) {
    if constexpr (OUT_NCONTIG) {
      if (n0 + c < NF) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(oz + ((int64_t)column * BLOCK + r) * ldo + n0 + c));
    } else {
      if (n0 + r < NF) __builtin_nontemporal_store(v, reinterpret_cast<u32x4 *>(oz + (int64_t)(n0 + r) * ldo + column * BLOCK + c));
    }
  };
  if (nblk == 0) {   // nothing to read (the views below assume at least one block): write the zeros and leave
    const u32x4 zero = {0u, 0u, 0u, 0u};
    constexpr int VE = 16 / (int)sizeof(T), CW = OUT_NCONTIG ? S::TN : BLOCK;   // chunks run along the contiguous index
    for (int i = threadIdx.x; i < BLOCK * S::TN / VE; i += 256) store(i / (CW / VE), (i % (CW / VE)) * VE, zero);
    return;
  }
  if constexpr (PARTS) {
    if (whole > g.part_blocks) {
      constexpr int CW = OUT_NCONTIG ? S::TN : BLOCK;
      float *ws = g.partials + ((((int64_t)part * g.Z + z) * g.width + seg) * n_tiles + nt) * (BLOCK * S::TN);
      G::template run<0, true>(sv, dv, (nblk * BLOCK + G::TK - 1) / G::TK, reinterpret_cast<T *>(smem_raw), [&](int r, int c, f32x4 v) { *reinterpret_cast<f32x4 *>(ws + r * CW + c) = v; });
      return;
    }
  }
  G::run(sv, dv, (nblk * BLOCK + G::TK - 1) / G::TK, reinterpret_cast<T *>(smem_raw), store);
}

// The second pass of segments in parts: a workgroup per segment, tile and batch adds the parts in order
template <typename T, int BLOCK, int TN, bool OUT_NCONTIG> __global__ void __launch_bounds__(256) k_xsd_parts_sum(XsdArgs g) {
  constexpr int CW = OUT_NCONTIG ? TN : BLOCK;
  const int n_tiles = (g.NF + TN - 1) / TN;
  const int seg = blockIdx.x % g.width, nt = (blockIdx.x / g.width) % n_tiles, z = blockIdx.x / g.width / n_tiles;
  const table_ptr hd = as_table(g.lut) + 6 * (int64_t)seg;
  const int nblk = hd[1] / BLOCK, column = hd[2], depth = hd[3];
  if (nblk <= g.part_blocks) return;
  const int parts = (nblk + g.part_blocks - 1) / g.part_blocks;
  const int64_t stride = (int64_t)g.Z * g.width * n_tiles * (BLOCK * TN);
  const float *ws = g.partials + (((int64_t)z * g.width + seg) * n_tiles + nt) * (BLOCK * TN);
  T *oz = reinterpret_cast<T *>(g.out) + z * g.out_sz + depth * g.out_sh;
  for (int i = threadIdx.x * 4; i < BLOCK * TN; i += 1024) {
    const int r = i / CW, c = i % CW;
    if (nt * TN + (OUT_NCONTIG ? c : r) >= g.NF) continue;
    f32x4 sum = *reinterpret_cast<const f32x4 *>(ws + i);
    for (int p = 1; p < parts; p++) {
      const f32x4 v = *reinterpret_cast<const f32x4 *>(ws + p * stride + i);
#pragma unroll
      for (int e = 0; e < 4; e++) sum[e] += v[e];
    }
    T *dst = OUT_NCONTIG ? oz + ((int64_t)column * BLOCK + r) * g.ldo + nt * TN + c : oz + (int64_t)(nt * TN + r) * g.ldo + column * BLOCK + c;
    if constexpr (sizeof(T) == 4) *reinterpret_cast<f32x4 *>(dst) = sum;
    else {
      union { u32x2 raw; T e[4]; } u;
#pragma unroll
      for (int e = 0; e < 4; e++) u.e[e] = from_float<T>(sum[e]);
      *reinterpret_cast<u32x2 *>(dst) = u.raw;
    }
  }
}

// ---------------------------------------------------------------------------------------------------------
// host-side launch helpers shared by the per-type translation units
// ---------------------------------------------------------------------------------------------------------
template <typename T, int BLOCK> int launch_sdd_b(const SddArgs &g, bool a_kc, bool b_kc, hipStream_t st) {
  constexpr int WG = SddShape<BLOCK>::WG;
  const int64_t n_wg = g.n_groups * g.Z * g.parts;
  if (n_wg <= 0) return BSP_OK;
  if (n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  dim3 grid((unsigned)n_wg), blockdim(64 * WG * WG);
#define BSP_SDD_LAUNCH(AK, BK)                                                                                   \
  do {                                                                                                           \
    constexpr int SMEM = TileGemm<T, BLOCK, BLOCK, WG, WG, AK, BK, true>::SMEM_BYTES;                            \
    if (g.parts > 1) hipLaunchKernelGGL((k_sdd<T, BLOCK, AK, BK, true>), grid, blockdim, SMEM, st, g);           \
    else hipLaunchKernelGGL((k_sdd<T, BLOCK, AK, BK, false>), grid, blockdim, SMEM, st, g);                      \
  } while (0)
  if (a_kc && b_kc) BSP_SDD_LAUNCH(true, true);
  else if (a_kc && !b_kc) BSP_SDD_LAUNCH(true, false);
  else if (!a_kc && b_kc) BSP_SDD_LAUNCH(false, true);
  else BSP_SDD_LAUNCH(false, false);
#undef BSP_SDD_LAUNCH
  return BSP_OK;
}

template <typename T, int BLOCK> int launch_sdd_levels(const SddArgs &g, const SddLevel *levels, int n_levels, bool a_kc, bool b_kc, hipStream_t st) {
  SddLevels<BLOCK> lv{};
  int64_t n_wg = 0;
  for (int i = 0; i < n_levels; i++) {
    int at = 0;
    while (at < SddLevels<BLOCK>::N && (64 / BLOCK) >> at != levels[i].pack) at++;
    if (at == SddLevels<BLOCK>::N || lv.n[at]) return BSP_ERR_UNSUPPORTED;
    lv.lut[at] = levels[i].lut; lv.valid[at] = levels[i].valid; lv.n[at] = levels[i].n;
    const int per = BLOCK == 16 && levels[i].pack == 1 ? 4 : 1;
    n_wg += (levels[i].n * g.Z + per - 1) / per;
  }
  if (n_wg <= 0) return BSP_OK;
  if (n_wg * g.parts >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  dim3 grid((unsigned)(n_wg * g.parts)), blockdim(256);
#define BSP_SDD_LAUNCH(AK, BK)                                                                                   \
  do {                                                                                                           \
    constexpr int SMEM = SddLevelsShape<T, BLOCK, AK, BK>::SMEM;                                                 \
    if (g.parts > 1) hipLaunchKernelGGL((k_sdd_levels<T, BLOCK, AK, BK, true>), grid, blockdim, SMEM, st, g, lv, n_wg); \
    else hipLaunchKernelGGL((k_sdd_levels<T, BLOCK, AK, BK, false>), grid, blockdim, SMEM, st, g, lv, n_wg);     \
  } while (0)
  if (a_kc && b_kc) BSP_SDD_LAUNCH(true, true);
  else if (a_kc && !b_kc) BSP_SDD_LAUNCH(true, false);
  else if (!a_kc && b_kc) BSP_SDD_LAUNCH(false, true);
  else BSP_SDD_LAUNCH(false, false);
#undef BSP_SDD_LAUNCH
  return BSP_OK;
}

template <typename T, int BLOCK, int SPLIT> int launch_sdd_split(const SddArgs &g, bool a_kc, bool b_kc, hipStream_t st) {
  constexpr int TT = BLOCK / SPLIT, WG = SddShape<TT>::WG;
  const int64_t n_wg = g.n_groups * g.Z * (SPLIT * SPLIT) * g.parts;
  if (n_wg <= 0) return BSP_OK;
  if (n_wg >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  dim3 grid((unsigned)n_wg), blockdim(64 * WG * WG);
#define BSP_SDD_LAUNCH(AK, BK)                                                                                   \
  do {                                                                                                           \
    constexpr int SMEM = TileGemm<T, TT, TT, WG, WG, AK, BK, true>::SMEM_BYTES;                                  \
    if (g.parts > 1) hipLaunchKernelGGL((k_sdd_split<T, BLOCK, SPLIT, AK, BK, true>), grid, blockdim, SMEM, st, g); \
    else hipLaunchKernelGGL((k_sdd_split<T, BLOCK, SPLIT, AK, BK, false>), grid, blockdim, SMEM, st, g);         \
  } while (0)
  if (a_kc && b_kc) BSP_SDD_LAUNCH(true, true);
  else if (a_kc && !b_kc) BSP_SDD_LAUNCH(true, false);
  else if (!a_kc && b_kc) BSP_SDD_LAUNCH(false, true);
  else BSP_SDD_LAUNCH(false, false);
#undef BSP_SDD_LAUNCH
  return BSP_OK;
}

template <typename T> int launch_sdd_whole(const SddArgs &g0, int block, const SddLevel *levels, int n_levels, bool a_kc, bool b_kc, hipStream_t st) {
  if (block == 16) return launch_sdd_levels<T, 16>(g0, levels, n_levels, a_kc, b_kc, st);
  if (block == 32) return launch_sdd_levels<T, 32>(g0, levels, n_levels, a_kc, b_kc, st);
  if (n_levels != 1 || levels[0].pack != 1) return BSP_ERR_UNSUPPORTED;
  SddArgs g = g0;
  g.lut = levels[0].lut; g.valid = levels[0].valid; g.n_groups = levels[0].n;
  // fewer than two workgroups per CU: four 64 x 64 workgroups per 128-block instead of one
  if (block == 128 && g.n_groups * g.Z < 512) return launch_sdd_split<T, 128, 2>(g, a_kc, b_kc, st);
  if (block == 64) return launch_sdd_b<T, 64>(g, a_kc, b_kc, st);
  if (block == 128) return launch_sdd_b<T, 128>(g, a_kc, b_kc, st);
  return BSP_ERR_UNSUPPORTED;
}

template <typename T> int launch_sdd(const SddArgs &g, int block, const SddLevel *levels, int n_levels, bool a_kc, bool b_kc, hipStream_t st) {
  const int rc = launch_sdd_whole<T>(g, block, levels, n_levels, a_kc, b_kc, st);
  if (rc != BSP_OK || g.parts <= 1) return rc;
  const int64_t per_z = g.n_blocks * (block * block / 4);
  hipLaunchKernelGGL((k_sdd_parts_sum<T>), dim3((unsigned)((per_z * g.Z + 255) / 256)), dim3(256), 0, st, g, per_z);
  return BSP_OK;
}

template <typename T, int BLOCK, int TN_> int launch_xsd_bw(const XsdArgs &g0, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st) {
  typedef XsdShape<BLOCK, TN_> S;
  const int64_t n_wg = (int64_t)g0.width * ((g0.NF + S::TN - 1) / S::TN) * g0.Z;
  if (n_wg <= 0) return BSP_OK;
  if (n_wg * g0.parts >= ((int64_t)1 << 31)) return BSP_ERR_UNSUPPORTED;
  // Longest segments first only in short launches (a few workgroups per CU), where the last workgroups to start
  // decide when the launch ends: 7 % on an 8192 x 4096 x 4096 linear layer at block 128 and 10 % density (1024
  // workgroups).  A long launch balances by itself and reads the sparse blocks in storage order without it (1 %
  // faster at 65536 workgroups).
  XsdArgs g = g0;
  if (n_wg > 16 * 256) g.order = nullptr;
  dim3 grid((unsigned)(n_wg * g.parts)), blockdim(256);
#define BSP_XSD_LAUNCH(ST, DK, ON)                                                                               \
  do {                                                                                                           \
    constexpr int SMEM = TileGemm<T, BLOCK, S::TN, S::WGM, S::WGN, !ST, DK, ON>::SMEM_BYTES;                     \
    if constexpr (sizeof(T) == 4)                                                                                \
      if (g.parts > 1) {                                                                                         \
        hipLaunchKernelGGL((k_xsd<T, BLOCK, TN_, ST, DK, ON, true>), grid, blockdim, SMEM, st, g);              \
        hipLaunchKernelGGL((k_xsd_parts_sum<T, BLOCK, TN_, ON>), dim3((unsigned)n_wg), blockdim, 0, st, g);     \
        break;                                                                                                   \
      }                                                                                                          \
    hipLaunchKernelGGL((k_xsd<T, BLOCK, TN_, ST, DK, ON, false>), grid, blockdim, SMEM, st, g);                 \
  } while (0)
  const int key = (sp_trans ? 4 : 0) | (dn_kc ? 2 : 0) | (out_nc ? 1 : 0);
  switch (key) {
    case 0: BSP_XSD_LAUNCH(false, false, false); break;
    case 1: BSP_XSD_LAUNCH(false, false, true); break;
    case 2: BSP_XSD_LAUNCH(false, true, false); break;
    case 3: BSP_XSD_LAUNCH(false, true, true); break;
    case 4: BSP_XSD_LAUNCH(true, false, false); break;
    case 5: BSP_XSD_LAUNCH(true, false, true); break;
    case 6: BSP_XSD_LAUNCH(true, true, false); break;
    default: BSP_XSD_LAUNCH(true, true, true); break;
  }
#undef BSP_XSD_LAUNCH
  return BSP_OK;
}

template <typename T, int BLOCK> int launch_xsd_b(const XsdArgs &g, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st) {
  int tile = xsd_tile(BLOCK, g.NF);
  // 16-bit, blocks of 32: a launch on tiles of 256 has two workgroups a compute unit from 512 on; fewer leave the chip waiting for the few
  // steps in flight, and tiles of 128 are twice as many.  Tiles of 256 / 128, us, of the launches on 256: 128 of them 20.7 / 16.3 (31 blocks
  // a line) and 7.9 / 6.3 (8), 256 20.1 / 17.2, 384 25.7 / 23.4; 512 10.6 / 10.9, 14.3 / 14.3, 17.6 / 20.3; 768 18.2 / 19.1, 25.2 / 27.6.
  if (sizeof(T) == 2 && BLOCK == 32 && tile == 256 && (int64_t)g.width * ((g.NF + 255) / 256) * g.Z < 512) tile = 128;
  // fp32, whose matrix pipe makes long steps: tiles as narrow as it takes to have two workgroups a compute unit.  1024^3 in 8 heads and batches, a
  // quarter of the blocks, blocks of 128: tiles of 256 94-103 us, of 128 79-86; 512^3 in 2 heads, of 128 55-61 -> 20-21 on tiles of 64, of 64
  // 18-20 -> 11-12, of 32 17-22 -> 8-10.  (Parts have their own rule, on the width that xsd_tile gives.)
  // 16-bit, blocks of 64 and 128: one a compute unit (1024 x 200 x 1024 in 4 heads, of 128, 14-23 -> 8-13 us, of 64 7-13 -> 6-10; 256
  // workgroups on tiles of 128 lose 4-10 % on twice as many of 64: 1024 x 128 x 1024 in 16 heads, of 64, half of the blocks, 11.9 -> 13.2).
  if (sizeof(T) == 4 ? g.parts <= 1 : BLOCK >= 64)
    while (tile > 64 && (int64_t)g.width * ((g.NF + tile - 1) / tile) * g.Z < (sizeof(T) == 4 ? 512 : 256)) tile /= 2;
  if constexpr (BLOCK == 32 || BLOCK == 128)
    if (tile == 256) return launch_xsd_bw<T, BLOCK, 256>(g, sp_trans, dn_kc, out_nc, st);
  if constexpr (BLOCK != 16)
    if (tile == 128) return launch_xsd_bw<T, BLOCK, 128>(g, sp_trans, dn_kc, out_nc, st);
  return launch_xsd_bw<T, BLOCK, 64>(g, sp_trans, dn_kc, out_nc, st);
}

template <typename T> int launch_xsd(const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st) {
  switch (block) {
    case 16: return launch_xsd_b<T, 16>(g, sp_trans, dn_kc, out_nc, st);
    case 32: return launch_xsd_b<T, 32>(g, sp_trans, dn_kc, out_nc, st);
    case 64: return launch_xsd_b<T, 64>(g, sp_trans, dn_kc, out_nc, st);
    case 128: return launch_xsd_b<T, 128>(g, sp_trans, dn_kc, out_nc, st);
    default: return BSP_ERR_UNSUPPORTED;
  }
}

// implemented once per element type (matmul_f16.hip, matmul_bf16.hip, matmul_f32.hip)
int sdd_generic_f16(const SddArgs &g, int block, const SddLevel *levels, int n_levels, bool a_kc, bool b_kc, hipStream_t st);
int sdd_generic_bf16(const SddArgs &g, int block, const SddLevel *levels, int n_levels, bool a_kc, bool b_kc, hipStream_t st);
int sdd_generic_f32(const SddArgs &g, int block, const SddLevel *levels, int n_levels, bool a_kc, bool b_kc, hipStream_t st);
int xsd_generic_f16(const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st);
int xsd_generic_bf16(const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st);
int xsd_generic_f32(const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st);


// specialised block-64 16-bit kernels (matmul_fast64.hip): 1 = launched, 0 = not applicable, < 0 = error
int sdd_fast64(int dtype, const SddArgs &g, int block, int pack, bool a_kc, bool b_kc, hipStream_t st);
int xsd_fast64(int dtype, const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st);
// dsd / dds for a wide free dimension at blocks 64 / 128, 16-bit (matmul_dl.hip): same return convention
int xsd_dl(int dtype, const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st);
int xsd_list(int dtype, const XsdArgs &g, int block, bool sp_trans, bool dn_kc, bool out_nc, hipStream_t st);
// sdd with a long reduction at blocks of 32, from the group plan alone (matmul_dl.hip): 2 = launched and every block written
int sdd_dl(int dtype, const SddArgs &g, int block, bool rowpair_plan, bool a_kc, bool b_kc, hipStream_t st);
int sdd_list(int dtype, const SddArgs &g, int block, bool a_kc, bool b_kc, hipStream_t st);   // ... from the tiles of bsp_sdd_tiles_build
int sdd128_splitk(int dtype, const SddArgs &g, int parts, float *ws, bool a_kc, bool b_kc, hipStream_t st);

}  // namespace bsp
