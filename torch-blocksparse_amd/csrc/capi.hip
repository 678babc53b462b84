// C-ABI entry points of the matmul launchers: argument validation and dispatch.  (The table builders and
// the softmax entry points live next to their kernels in lut.hip / softmax.hip.)
#include "matmul_generic.h"
#include <mutex>

using namespace bsp;

namespace {
bool no_groups(int flags) { return (flags & BSP_FLAG_NO_GROUPS) != 0; }
bool general_only(int flags) { return (flags & BSP_FLAG_GENERAL_ONLY) != 0; }
bool no_wide(int flags) { return (flags & (BSP_FLAG_NO_WIDE | BSP_FLAG_GENERAL_ONLY)) != 0; }
// the reduction of an sdd product: a multiple of 16 (reference matmul.py:318-319), or any number of rows where both operands hold
// it as rows and the caller says so (the general kernels then read row by row up to the last)
bool sdd_k_ok(int K, int trans_a, int trans_b, int flags) { return K % 16 == 0 || ((flags & BSP_FLAG_ANY_K) && trans_a && !trans_b); }
bool rowpair(int flags) { return (flags & BSP_FLAG_PLAN_ROWPAIR) != 0; }
bool aligned16(const void *p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }
bool block_ok(int block) { return block == 16 || block == 32 || block == 64 || block == 128; }
int elems16(int dtype) { return dtype == BSP_F32 ? 4 : 8; }   // elements per 16 bytes
}  // namespace

extern "C" int bsp_version(void) { return 1; }

extern "C" const char *bsp_strerror(int status) {
  switch (status) {
    case BSP_OK: return "ok";
    case BSP_OK_WHOLE_LAYOUT: return "ok, every block of the layout written (skip the remaining pack levels)";
    case BSP_NEEDS_TABLE: return "nothing launched: this product needs the sdd table (call again with it)";
    case BSP_ERR_ARG: return "invalid argument (null pointer, bad size or operand not 16-byte aligned)";
    case BSP_ERR_UNSUPPORTED: return "unsupported block size, dtype or problem size";
    case BSP_ERR_CAPACITY: return "caller-provided table or workspace too small";
    case BSP_ERR_EMPTY_HEAD: return "a head of the layout has no nonzero block";
    case BSP_ERR_HIP: return "HIP runtime error";
    case BSP_ERR_ROW_TOO_LONG: return "Reductions larger than 32768 elements are not yet implemented";
    case BSP_ERR_K_MULTIPLE: return "Reduction size for SDD must be a multiple of 16";
    case BSP_ERR_SCRATCH_LIMIT: return "the launch needs more (split chain, tile, batch) slots than the library's static scratch buffer holds; use bsp_dsd_matmul with a workspace";
    default: return "unknown status";
  }
}

// Into how many parts the reduction of an sdd product on the general kernels is cut: launches that do not fill the chip (three
// workgroups a compute unit) and whose workgroups run many steps one after the other.  Whole / in parts, us, blocks as workgroups
// (a block of 128 counts as four): fp32, 92 of them, 340 steps 136 / 54 (8 parts), 53 steps 24 / 20 (3); 197, 125 steps 53 / 48
// (4); 407, 512 steps 345 / 269 (4); 24, 120 steps 53 / 15 (7); 28 + 2 of four blocks of 32, 60 steps 26 / 13 (3); 174, 44 steps 22 / 22;
// 254, 32 steps 15.5 / 17.4; 24 steps and fewer: the second launch costs more than the parts gain.  16-bit types take twice the
// elements a step and less time for it: 92, 170 steps 40 / 19 (8); 24, 32 steps 9.2 / 11.8; 407, 256 steps 73 / 77.
extern "C" int bsp_sdd_parts(int dtype, int block, int n_levels, const int *packs, const int64_t *n_groups, int Z, int K, int flags) {
  if (!block_ok(block) || n_levels < 1 || !packs || !n_groups || Z <= 0 || K <= 0 || (flags & BSP_FLAG_WHOLE_K)) return 1;
  int64_t wgs = 0;
  for (int i = 0; i < n_levels; i++) {
    const int tile = block * packs[i];
    wgs += tile >= 128 ? n_groups[i] * (n_groups[i] * Z < 512 ? 4 : 1) : tile < 32 ? (n_groups[i] + 3) / 4 : n_groups[i];
  }
  wgs *= Z;
  const bool f32 = dtype == BSP_F32;
  const int unit = f32 ? 16 : 32, steps = (K + unit - 1) / unit;
  if (wgs <= 0 || wgs > (f32 ? 512 : 256) || steps < (f32 ? 48 : 96)) return 1;
  int64_t parts = 800 / wgs;
  if (f32 && parts < steps / 128) parts = steps / 128;
  if (parts > steps / 16) parts = steps / 16;
  if (parts > 16) parts = 16;
  if (parts <= 1) return 1;
  const int per = (int)((steps + parts - 1) / parts);
  return (steps + per - 1) / per;                      // (no part is empty)
}

// Blocks of 16 and 32, 16-bit, a reduction that is no multiple of 32: as it is on the general kernel, or as copies with whole steps on
// k_sdd_rg_dl.  The copies take 10 to 100 us, and that kernel is the faster one only with a large result (with a small one it has too few
// workgroups for its long chains of steps), so they need many elements, many of them per row copied, and much work.  As it is / with
// copies, us, fp16, the density and in brackets the rows of the reduction.
// Block 32, 4096 x 4096: .1 257 / 281 (8170); .25 47 / 59 (1000), 103 / 89 (2041), 548 / 295 (8170); .5 41 / 46 (531), 80 / 60 (1000),
// 963 / 309 (8170).  2048 x 2048: .5 91 / 127 (4090), 206 / 233 (8170).  1024 x 1024: .5 74 / 210 (8170).
// Block 16, 4096 x 4096: .1 52 / 59 (1000), 133 / 89 (2041), 746 / 319 (8170); .25 29 / 33 (271), 56 / 46 (531); .5 54 / 35 (271).
// 2048 x 2048: .25 66 / 74 (2041), 147 / 125 (4090), 352 / 231 (8170).  1024 x 1024: .5 126 / 206 (8170).
// Block 128, whose kernel for whole steps is k_sdd128_splitk: as it is everywhere, 4096 x 4096, .1 8 / 34 (531), 75 / 158 (8170), .5
// 23 / 39 (531), 224 / 294 (8170).
extern "C" int bsp_sdd_whole_steps(int dtype, int block, int64_t n_blocks, int64_t rows, int64_t cols, int K) {
  if (dtype == BSP_F32 || (block != 16 && block != 32) || K < 256 || K % 32 == 0 || n_blocks <= 0) return 0;
  const int64_t elems = n_blocks * block * block, few = block == 16 ? 1000000 : 3000000, work = block == 16 ? 2200000000 : 6000000000;
  return elems >= few && elems >= 8 * block * (rows + cols) && elems * K >= work;
}

extern "C" int64_t bsp_sdd_parts_workspace_bytes(int block, int64_t n_blocks, int Z, int parts) {
  return parts > 1 && n_blocks > 0 && Z > 0 ? (int64_t)parts * Z * n_blocks * block * block * (int64_t)sizeof(float) : 0;
}

extern "C" int bsp_sdd_matmul_levels(int dtype, const void *a, const void *b, void *c, int trans_a, int trans_b, int Z, int K,
                                     int64_t a_stride_z, int64_t a_stride_h, int64_t lda, int64_t b_stride_z, int64_t b_stride_h,
                                     int64_t ldb, int64_t c_stride_z, int block, int n_levels, const int *packs, const int32_t *const *d_luts,
                                     const uint8_t *const *d_valids, const int64_t *n_groups, const int32_t *d_gplan, int n_plan_groups,
                                     int plan_lines, int parts, int64_t n_blocks, void *d_ws, int64_t ws_bytes, int flags, void *stream) {
  if (!a || !b || !c || Z <= 0 || K <= 0 || n_levels < 1 || n_levels > 3 || !packs || !d_luts || !d_valids || !n_groups) return BSP_ERR_ARG;
  SddLevel levels[3];
  for (int i = 0; i < n_levels; i++) {
    if (!d_luts[i] || n_groups[i] < 0) return BSP_ERR_ARG;
    levels[i] = SddLevel{packs[i], d_luts[i], d_valids[i], n_groups[i]};
  }
  if (!block_ok(block)) return BSP_ERR_UNSUPPORTED;
  if (!sdd_k_ok(K, trans_a, trans_b, flags)) return BSP_ERR_K_MULTIPLE;
  const int u = elems16(dtype);
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return BSP_ERR_ARG;
  if (a_stride_z % u || a_stride_h % u || lda % u || b_stride_z % u || b_stride_h % u || ldb % u || c_stride_z % u) return BSP_ERR_ARG;
  SddArgs g;
  g.a = a; g.b = b; g.c = c; g.Z = Z; g.K = K;
  g.a_sz = a_stride_z; g.a_sh = a_stride_h; g.lda = lda;
  g.b_sz = b_stride_z; g.b_sh = b_stride_h; g.ldb = ldb; g.c_sz = c_stride_z;
  g.lut = levels[0].lut; g.valid = levels[0].valid; g.n_groups = levels[0].n;
  g.gplan = no_groups(flags) ? nullptr : d_gplan; g.n_pgroups = n_plan_groups; g.lines = plan_lines;
  if (g.gplan && (n_plan_groups <= 0 || plan_lines == 0)) return BSP_ERR_ARG;
  if (rowpair(flags)) g.gplan = nullptr;   // a plan over pairs of block-rows serves the long-reduction kernel only
  // op(A)[m][k]: reduction contiguous unless A is read transposed; op(B)[k][n]: contiguous when B is read transposed
  const bool a_kc = !trans_a, b_kc = trans_b != 0;
  hipStream_t st = as_stream(stream);
  if (parts > 1) {
    if (n_blocks <= 0 || !d_ws || !aligned16(d_ws) || c_stride_z < n_blocks * block * block) return BSP_ERR_ARG;
    if (ws_bytes < bsp_sdd_parts_workspace_bytes(block, n_blocks, Z, parts)) return BSP_ERR_CAPACITY;
    const int unit = dtype == BSP_F32 ? 16 : 32;       // whole reduction steps
    g.parts = parts; g.n_blocks = n_blocks; g.ws = reinterpret_cast<float *>(d_ws);
    g.part_k = ((K + unit - 1) / unit + parts - 1) / parts * unit;
    if ((int64_t)g.part_k * (parts - 1) >= K) return BSP_ERR_ARG;   // (a part would be empty)
  }
  int rc = general_only(flags) || K % 16 || parts > 1 ? 0 : sdd_fast64(dtype, g, block, packs[0], a_kc, b_kc, st);
  if (rc < 0) return rc;
  // (a kernel that works from the plan writes the whole layout; the one for a single level serves blocks of 64, which have no other)
  if (rc >= 1) { BSP_LAUNCH_CHECK(); return rc == 2 ? BSP_OK_WHOLE_LAYOUT : BSP_OK; }
  switch (dtype) {
    case BSP_F16: rc = sdd_generic_f16(g, block, levels, n_levels, a_kc, b_kc, st); break;
    case BSP_BF16: rc = sdd_generic_bf16(g, block, levels, n_levels, a_kc, b_kc, st); break;
    case BSP_F32: rc = sdd_generic_f32(g, block, levels, n_levels, a_kc, b_kc, st); break;
    default: return BSP_ERR_UNSUPPORTED;
  }
  if (rc != BSP_OK) return rc;
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}

extern "C" int bsp_sdd_matmul(int dtype, const void *a, const void *b, void *c, int trans_a, int trans_b, int Z, int K,
                              int64_t a_stride_z, int64_t a_stride_h, int64_t lda, int64_t b_stride_z, int64_t b_stride_h,
                              int64_t ldb, int64_t c_stride_z, int block, int pack, const int32_t *d_lut,
                              const uint8_t *d_valid, int64_t n_groups, const int32_t *d_gplan, int n_plan_groups,
                              int plan_lines, int flags, void *stream) {
  if (d_lut)
    return bsp_sdd_matmul_levels(dtype, a, b, c, trans_a, trans_b, Z, K, a_stride_z, a_stride_h, lda, b_stride_z, b_stride_h, ldb, c_stride_z, block,
                                 1, &pack, &d_lut, &d_valid, &n_groups, d_gplan, n_plan_groups, plan_lines, 1, 0, nullptr, 0, flags, stream);
  if (!a || !b || !c || Z <= 0 || K <= 0 || n_groups < 0) return BSP_ERR_ARG;
  if (!d_gplan || no_groups(flags) || general_only(flags)) return d_gplan ? BSP_NEEDS_TABLE : BSP_ERR_ARG;
  if (!block_ok(block)) return BSP_ERR_UNSUPPORTED;
  if (K % 16) return BSP_ERR_K_MULTIPLE;   // reference matmul.py:318-319
  const int u = elems16(dtype);
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return BSP_ERR_ARG;
  if (a_stride_z % u || a_stride_h % u || lda % u || b_stride_z % u || b_stride_h % u || ldb % u || c_stride_z % u) return BSP_ERR_ARG;
  if (n_plan_groups <= 0 || plan_lines == 0) return BSP_ERR_ARG;
  // the plan alone: n_groups then carries an upper bound on the entries of a group (at most the block-columns of the layout)
  SddArgs g;
  g.a = a; g.b = b; g.c = c; g.Z = Z; g.K = K;
  g.a_sz = a_stride_z; g.a_sh = a_stride_h; g.lda = lda;
  g.b_sz = b_stride_z; g.b_sh = b_stride_h; g.ldb = ldb; g.c_sz = c_stride_z;
  g.lut = nullptr; g.valid = d_valid; g.n_groups = 0; g.cols = (int)n_groups;
  g.gplan = d_gplan; g.n_pgroups = n_plan_groups; g.lines = plan_lines;
  const bool a_kc = !trans_a, b_kc = trans_b != 0;
  hipStream_t st = as_stream(stream);
  const bool tiles = (flags & BSP_FLAG_PLAN_TILES) != 0;
  int rc = no_wide(flags) ? 0 : tiles ? sdd_list(dtype, g, block, a_kc, b_kc, st) : sdd_dl(dtype, g, block, rowpair(flags), a_kc, b_kc, st);
  if (rc < 0) return rc;
  if (rc == 2) { BSP_LAUNCH_CHECK(); return BSP_OK_WHOLE_LAYOUT; }
  if (rowpair(flags) || tiles) return BSP_NEEDS_TABLE;      // a plan over pairs of block-rows serves the long-reduction kernel only
  rc = sdd_fast64(dtype, g, block, pack, a_kc, b_kc, st);
  if (rc < 0) return rc;
  if (rc >= 1) { BSP_LAUNCH_CHECK(); return rc == 2 ? BSP_OK_WHOLE_LAYOUT : BSP_OK; }
  return BSP_NEEDS_TABLE;                          // no kernel that works from the plan applies
}

extern "C" int64_t bsp_sdd_splitk_workspace_bytes(int Z, int64_t n_groups, int parts) {
  if (Z <= 0 || n_groups <= 0 || parts <= 1) return 0;
  return (int64_t)Z * n_groups * parts * (int64_t)(128 * 128 * sizeof(float));
}

extern "C" int bsp_sdd_matmul_splitk(int dtype, const void *a, const void *b, void *c, int trans_a, int trans_b, int Z, int K,
                                     int64_t a_stride_z, int64_t a_stride_h, int64_t lda, int64_t b_stride_z, int64_t b_stride_h,
                                     int64_t ldb, int64_t c_stride_z, int block, const int32_t *d_lut, const uint8_t *d_valid,
                                     int64_t n_groups, int parts, void *d_ws, int64_t ws_bytes, int flags, void *stream) {
  if (!a || !b || !c || !d_lut || Z <= 0 || K <= 0 || n_groups < 0 || parts < 1 || parts > 64) return BSP_ERR_ARG;
  if (block != 128 || (dtype != BSP_F16 && dtype != BSP_BF16) || general_only(flags) || no_wide(flags)) return BSP_ERR_UNSUPPORTED;
  if (K % 16) return BSP_ERR_K_MULTIPLE;
  if (K % 32) return BSP_ERR_UNSUPPORTED;
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return BSP_ERR_ARG;
  if (a_stride_z % 8 || a_stride_h % 8 || lda % 8 || b_stride_z % 8 || b_stride_h % 8 || ldb % 8 || c_stride_z % 8) return BSP_ERR_ARG;
  if (parts > 1) {
    if (!d_ws || !aligned16(d_ws)) return BSP_ERR_ARG;
    if (ws_bytes < bsp_sdd_splitk_workspace_bytes(Z, n_groups, parts)) return BSP_ERR_CAPACITY;
  }
  SddArgs g;
  g.a = a; g.b = b; g.c = c; g.Z = Z; g.K = K;
  g.a_sz = a_stride_z; g.a_sh = a_stride_h; g.lda = lda;
  g.b_sz = b_stride_z; g.b_sh = b_stride_h; g.ldb = ldb; g.c_sz = c_stride_z;
  g.lut = d_lut; g.valid = d_valid; g.n_groups = n_groups;
  g.gplan = nullptr; g.n_pgroups = 0; g.lines = 0;
  const int rc = sdd128_splitk(dtype, g, parts, reinterpret_cast<float *>(d_ws), !trans_a, trans_b != 0, as_stream(stream));
  if (rc != BSP_OK) return rc;
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}

// Workspace of a plan with split chains: BSP_CHAIN_PARTS fp32 tiles of 64 x 64 per (split chain, free tile, batch).
static int64_t xsd_ws_slots(int n_split, int free_dim, int Z) { return (int64_t)n_split * ((free_dim + 63) / 64) * Z; }

extern "C" int64_t bsp_xsd_workspace_bytes(int n_split, int free_dim, int Z) {
  if (n_split <= 0 || free_dim <= 0 || Z <= 0) return 0;
  return xsd_ws_slots(n_split, free_dim, Z) * BSP_CHAIN_PARTS * (int64_t)(64 * 64 * sizeof(float));
}

// Fills in the workspace fields of the arguments.
static int xsd_workspace(XsdArgs &g, int n_split, int free_dim, void *d_ws, int64_t ws_bytes) {
  g.n_split = 0; g.partials = nullptr;
  if (n_split < 0) return BSP_ERR_ARG;
  if (!g.gplan || n_split == 0) return BSP_OK;
  if (!d_ws || (reinterpret_cast<uintptr_t>(d_ws) & 255)) return BSP_ERR_ARG;
  if (ws_bytes < bsp_xsd_workspace_bytes(n_split, free_dim, g.Z)) return BSP_ERR_CAPACITY;
  g.n_split = n_split;
  g.partials = reinterpret_cast<float *>(d_ws);
  return BSP_OK;
}

static int xsd_dispatch(int dtype, XsdArgs g, int block, bool sp_trans, bool dn_kc, bool out_nc, int flags, void *stream) {
  hipStream_t st = as_stream(stream);
  // a wide free dimension at blocks 64 / 128: the kernels bound by the matrix cores and the feed from L2
  const bool chunks = (flags & BSP_FLAG_PLAN_TILES) != 0;
  int rc = no_wide(flags) ? 0 : chunks ? xsd_list(dtype, g, block, sp_trans, dn_kc, out_nc, st) : xsd_dl(dtype, g, block, sp_trans, dn_kc, out_nc, st);
  if (rc < 0) return rc;
  if (rc == 1) { BSP_LAUNCH_CHECK(); return BSP_OK; }
  if (chunks) g.gplan = nullptr;                       // (the chunks serve no other kernel)
  rc = general_only(flags) || rc == 2 ? 0 : xsd_fast64(dtype, g, block, sp_trans, dn_kc, out_nc, st);
  if (rc < 0) return rc;
  if (rc == 1) { BSP_LAUNCH_CHECK(); return BSP_OK; }
  switch (dtype) {
    case BSP_F16: rc = xsd_generic_f16(g, block, sp_trans, dn_kc, out_nc, st); break;
    case BSP_BF16: rc = xsd_generic_bf16(g, block, sp_trans, dn_kc, out_nc, st); break;
    case BSP_F32: rc = xsd_generic_f32(g, block, sp_trans, dn_kc, out_nc, st); break;
    default: return BSP_ERR_UNSUPPORTED;
  }
  if (rc != BSP_OK) return rc;
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}

extern "C" int bsp_dsd_matmul(int dtype, const void *a, const void *b, void *c, int trans_a, int trans_b, int trans_c, int Z,
                              int N, int64_t a_stride_z, int64_t b_stride_z, int64_t b_stride_h, int64_t ldb,
                              int64_t c_stride_z, int64_t c_stride_h, int64_t ldc, int block, const int32_t *d_lut,
                              const int32_t *d_plan, int width, const int32_t *d_gplan, int n_plan_groups, int plan_lines,
                              int n_split, void *d_ws, int64_t ws_bytes, int flags, void *stream) {
  if (!a || !b || !c || !d_lut || !d_plan || Z <= 0 || N <= 0 || width < 0) return BSP_ERR_ARG;
  if (d_gplan && (n_plan_groups <= 0 || plan_lines == 0)) return BSP_ERR_ARG;
  if (!block_ok(block)) return BSP_ERR_UNSUPPORTED;
  const int u = elems16(dtype);
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return BSP_ERR_ARG;
  // (a free dimension whose elements are whole rows on both sides may have any size, one that lies along the rows is read and
  // written in chunks of 16 bytes)
  if ((N % u && !(trans_b && trans_c)) || a_stride_z % u || b_stride_z % u || b_stride_h % u || ldb % u || c_stride_z % u || c_stride_h % u || ldc % u) return BSP_ERR_ARG;
  XsdArgs g;
  g.sp = a; g.dn = b; g.out = c; g.Z = Z; g.NF = N;
  g.sp_sz = a_stride_z; g.dn_sz = b_stride_z; g.dn_sh = b_stride_h; g.ldd = ldb;
  g.out_sz = c_stride_z; g.out_sh = c_stride_h; g.ldo = ldc;
  g.lut = d_lut; g.order = d_plan; g.plan = d_plan + bsp_dxx_plan_pairs_offset(width); g.width = width;
  g.div2 = 2 * (block / (dtype == BSP_F32 ? 8 : 16));   // step of the table: 8 for fp32, 16 otherwise (matmul.py:617)
  g.n_tiles = (N + 63) / 64;
  g.gplan = (no_groups(flags) || general_only(flags)) ? nullptr : d_gplan; g.n_pgroups = n_plan_groups; g.lines = plan_lines;
  if (int rc = xsd_workspace(g, n_split, N, d_ws, ws_bytes)) return rc;
  // rows of the kernel = rows of op(A); op(A)(m,k) is stored [k][m] when trans_a.  Dense (n,k) = op(B)[k][n]:
  // reduction contiguous when B is read transposed.  C[m][n] has n contiguous unless written transposed.
  return xsd_dispatch(dtype, g, block, trans_a != 0, trans_b != 0, !trans_c, flags, stream);
}

// Segments of how many blocks a dsd / dds product of the general kernels takes whole; returns how many parts the longest one makes (1:
// all are taken whole).  fp32 only: the 16-bit kernels have plans of their own for long lines.  A launch ends with its longest
// segments, which run alone: a global column of an attention layout is 64 blocks where the others are 4.  Whole / in parts, us, the
// transposed product of 'fixed' layouts with a head dimension of 64 (longest segment, average): block 32, 64 of 19 blocks 62 / 53,
// 61 of 10 59 / 39, 121 of 12 85 / 45; block 64, 16 of 7 30 / 21; block 16, 125 of 18 48 / 39, but 128 of 35 51 / 55 (its parts are read
// and written as often as the blocks, so the line lies higher).  Launches that do not fill the chip: 27 segments of up to 54 blocks of
// 64 107 / 27, 64 of up to 64 blocks of 32 115 / 38.  With equal segments, or more workgroups than the chip holds, parts only cost (19 of
// 19 36 / 42; 14 of 5, 1161 workgroups 79 / 83).
extern "C" int bsp_xsd_parts(int dtype, int block, int width, int longest, int64_t nnz, int free_dim, int Z, int flags, int *part_blocks) {
  *part_blocks = 0;
  if (dtype != BSP_F32 || !block_ok(block) || width <= 0 || free_dim <= 0 || Z <= 0 || longest <= 0 || (flags & BSP_FLAG_WHOLE_K)) return 1;
  const int tile = xsd_tile(block, free_dim);
  const int64_t wgs = (int64_t)width * ((free_dim + tile - 1) / tile) * Z;
  const int steps = longest * (block / 16);
  if (wgs > 1024 || steps < 48) return 1;
  int64_t parts = 1;
  if ((int64_t)longest * width >= (block == 16 ? 4 : 2) * nnz) parts = steps / (block == 16 ? 32 : 16);
  if (wgs <= 384 && parts < 800 / wgs) parts = 800 / wgs < steps / 16 ? 800 / wgs : steps / 16;
  if (parts > 8) parts = 8;
  if (parts <= 1) return 1;
  const int per = (longest + (int)parts - 1) / (int)parts;
  if (bsp_xsd_parts_workspace_bytes(block, width, free_dim, Z, (longest + per - 1) / per) > ((int64_t)256 << 20)) return 1;
  *part_blocks = per;
  return (longest + per - 1) / per;
}

extern "C" int64_t bsp_xsd_parts_workspace_bytes(int block, int width, int free_dim, int Z, int parts) {
  if (parts <= 1) return 0;
  const int tile = xsd_tile(block, free_dim);
  return (int64_t)parts * Z * width * ((free_dim + tile - 1) / tile) * block * tile * (int64_t)sizeof(float);
}

extern "C" int bsp_xsd_matmul_parts(int is_dds, int dtype, const void *sp, const void *dn, void *c, int trans_a, int trans_b, int trans_c, int Z, int free_dim,
                                    int64_t sp_stride_z, int64_t dn_stride_z, int64_t dn_stride_h, int64_t ldd, int64_t c_stride_z, int64_t c_stride_h,
                                    int64_t ldc, int block, const int32_t *d_lut, const int32_t *d_plan, int width, int parts, int part_blocks, void *d_ws,
                                    int64_t ws_bytes, void *stream) {
  if (!sp || !dn || !c || !d_lut || !d_plan || Z <= 0 || free_dim <= 0 || width < 0 || parts < 2 || part_blocks < 1 || !d_ws) return BSP_ERR_ARG;
  if (!block_ok(block) || dtype != BSP_F32) return BSP_ERR_UNSUPPORTED;
  if (!aligned16(sp) || !aligned16(dn) || !aligned16(c) || !aligned16(d_ws)) return BSP_ERR_ARG;
  if (sp_stride_z % 4 || dn_stride_z % 4 || dn_stride_h % 4 || ldd % 4 || c_stride_z % 4 || c_stride_h % 4 || ldc % 4) return BSP_ERR_ARG;
  const bool whole_rows = is_dds ? !trans_a && !trans_c : trans_b && trans_c;
  if (free_dim % 4 && !whole_rows) return BSP_ERR_ARG;
  if (ws_bytes < bsp_xsd_parts_workspace_bytes(block, width, free_dim, Z, parts)) return BSP_ERR_CAPACITY;
  XsdArgs g;
  g.sp = sp; g.dn = dn; g.out = c; g.Z = Z; g.NF = free_dim;
  g.sp_sz = sp_stride_z; g.dn_sz = dn_stride_z; g.dn_sh = dn_stride_h; g.ldd = ldd;
  g.out_sz = c_stride_z; g.out_sh = c_stride_h; g.ldo = ldc;
  g.lut = d_lut; g.order = d_plan; g.plan = d_plan + bsp_dxx_plan_pairs_offset(width); g.width = width;
  g.div2 = 2 * (block / 8);
  g.n_tiles = (free_dim + 63) / 64;
  g.gplan = nullptr; g.n_pgroups = 0; g.lines = 0;
  g.parts = parts; g.part_blocks = part_blocks; g.partials = reinterpret_cast<float *>(d_ws);
  // (orientations as in bsp_dsd_matmul and bsp_dds_matmul)
  const int rc = is_dds ? xsd_generic_f32(g, block, trans_b == 0, trans_a == 0, trans_c != 0, as_stream(stream))
                        : xsd_generic_f32(g, block, trans_a != 0, trans_b != 0, trans_c == 0, as_stream(stream));
  if (rc != BSP_OK) return rc;
  BSP_LAUNCH_CHECK();
  return BSP_OK;
}

// Whether a dsd launch with these properties is taken by a kernel that runs split chains and so uses the workspace:
// the row-group kernels on 64 x 64 tiles (block 64, or block 16 with a plan over tiles: negative line count), 16-bit
// types, dense operand not reduction-contiguous, output rows contiguous, whole 64-wide tiles of the free dimension,
// and at block 64 a free dimension the wide kernel (xsd_dl, which comes first in xsd_dispatch) leaves alone.
static bool split_chains_run(int dtype, int block, int N, bool dn_kc, bool out_nc, int plan_lines, int flags) {
  if (dtype == BSP_F32 || dn_kc || !out_nc || N % 64) return false;
  if (no_groups(flags) || general_only(flags)) return false;
  if (block == 16) return plan_lines < 0;
  if (block == 64) return plan_lines > 0 && (N < 256 || no_wide(flags));
  return false;
}

// ---------------------------------------------------------------------------------------------------------
// The allocation-free variant of bsp_dsd_matmul: the workspace of the split chains is a static device array.
// In host code the array's name only stands for the symbol; its device address differs from GPU to GPU and is looked
// up once per device with hipGetSymbolAddress, with that device current, and kept.  Everything below uses that
// address, never the name.
// ---------------------------------------------------------------------------------------------------------
static __device__ __align__(256) unsigned char scratch[BSP_NOALLOC_SCRATCH_BYTES];

namespace {
constexpr int kMaxDevices = 64;
std::mutex g_scratch_mutex;
void *g_scratch_ptr[kMaxDevices] = {};   // per device: the address of its copy of `scratch`

// the device address of `scratch` on the current device (nullptr on failure)
void *scratch_address() {
  int dev = -1;
  if (hipGetDevice(&dev) != hipSuccess || dev < 0 || dev >= kMaxDevices) return nullptr;
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (!g_scratch_ptr[dev]) {
    void *p = nullptr;
    if (hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)) != hipSuccess || !p) return nullptr;
    g_scratch_ptr[dev] = p;
  }
  return g_scratch_ptr[dev];
}

}  // namespace

extern "C" int bsp_dsd_matmul_noalloc(int dtype, const void *a, const void *b, void *c, int trans_a, int trans_b, int trans_c, int Z,
                                      int N, int64_t a_stride_z, int64_t b_stride_z, int64_t b_stride_h, int64_t ldb,
                                      int64_t c_stride_z, int64_t c_stride_h, int64_t ldc, int block, const int32_t *d_lut,
                                      const int32_t *d_plan, int width, const int32_t *d_gplan, int n_plan_groups,
                                      int plan_lines, int n_split, int flags, void *stream) {
  if (n_split < 0 || Z <= 0 || N <= 0) return BSP_ERR_ARG;
  void *ws = nullptr;
  int64_t ws_bytes = 0;
  if (d_gplan && n_split > 0 && !split_chains_run(dtype, block, N, trans_b != 0, !trans_c, plan_lines, flags)) {
    // A kernel that does not know split chains takes this launch (the wide kernel, the general one, fp32, ...): it
    // needs no scratch memory whatever the sizes, and must not see a plan whose chains are cut into parts.
    d_gplan = nullptr; n_plan_groups = 0; plan_lines = 0; n_split = 0;
  }
  if (d_gplan && n_split > 0) {
    if (xsd_ws_slots(n_split, N, Z) > BSP_NOALLOC_MAX_SLOTS) return BSP_ERR_SCRATCH_LIMIT;
    ws = scratch_address();
    if (!ws) return BSP_ERR_HIP;
    ws_bytes = BSP_NOALLOC_SCRATCH_BYTES;
    // (the buffer keeps what the last call left, which is harmless: every tile that is read was written by this call)
  }
  return bsp_dsd_matmul(dtype, a, b, c, trans_a, trans_b, trans_c, Z, N, a_stride_z, b_stride_z, b_stride_h, ldb, c_stride_z,
                        c_stride_h, ldc, block, d_lut, d_plan, width, d_gplan, n_plan_groups, plan_lines, n_split, ws, ws_bytes,
                        flags, stream);
}

extern "C" int bsp_dds_matmul(int dtype, const void *a, const void *b, void *c, int trans_a, int trans_b, int trans_c, int Z,
                              int M, int64_t a_stride_z, int64_t a_stride_h, int64_t lda, int64_t b_stride_z,
                              int64_t c_stride_z, int64_t c_stride_h, int64_t ldc, int block, const int32_t *d_lut,
                              const int32_t *d_plan, int width, const int32_t *d_gplan, int n_plan_groups, int plan_lines,
                              int n_split, void *d_ws, int64_t ws_bytes, int flags, void *stream) {
  if (!a || !b || !c || !d_lut || !d_plan || Z <= 0 || M <= 0 || width < 0) return BSP_ERR_ARG;
  if (d_gplan && (n_plan_groups <= 0 || plan_lines == 0)) return BSP_ERR_ARG;
  if (!block_ok(block)) return BSP_ERR_UNSUPPORTED;
  const int u = elems16(dtype);
  if (!aligned16(a) || !aligned16(b) || !aligned16(c)) return BSP_ERR_ARG;
  if ((M % u && (trans_a || trans_c)) || a_stride_z % u || a_stride_h % u || lda % u || b_stride_z % u || c_stride_z % u || c_stride_h % u || ldc % u) return BSP_ERR_ARG;
  XsdArgs g;
  g.sp = b; g.dn = a; g.out = c; g.Z = Z; g.NF = M;
  g.sp_sz = b_stride_z; g.dn_sz = a_stride_z; g.dn_sh = a_stride_h; g.ldd = lda;
  g.out_sz = c_stride_z; g.out_sh = c_stride_h; g.ldo = ldc;
  g.lut = d_lut; g.order = d_plan; g.plan = d_plan + bsp_dxx_plan_pairs_offset(width); g.width = width;
  g.div2 = 2 * (block / (dtype == BSP_F32 ? 8 : 16));
  g.n_tiles = (M + 63) / 64;
  g.gplan = (no_groups(flags) || general_only(flags)) ? nullptr : d_gplan; g.n_pgroups = n_plan_groups; g.lines = plan_lines;
  if (int rc = xsd_workspace(g, n_split, M, d_ws, ws_bytes)) return rc;
  // dds is dsd on the transposed problem: kernel rows = columns of op(B) (stored [k][col] unless trans_b), dense
  // rows = rows of op(A) (reduction contiguous unless trans_a), and C[row][col] has the kernel's m index contiguous
  // unless written transposed.
  return xsd_dispatch(dtype, g, block, !trans_b, !trans_a, trans_c != 0, flags, stream);
}
