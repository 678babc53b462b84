// The host side of a launch in native code: operand checks, the output, strides and pointers, and the call of the C entry point
// (include/bsp.h).  A CPython extension, torch_blocksparse._launch: the functions take tensors as Python objects and know
// nothing of them but the methods a Python caller has, so that allocation (torch.empty), streams and autograd stay where they are.
//
// Every function returns None where a call is not the ordinary one (an operand to be copied or padded, a table that has yet to be
// built, a shape that does not fit): nothing has been launched then, and the caller goes the general way in Python, which does
// what is needed or raises the error.  An entry point that fails raises what _lib.check raises for it.
//
// Why: such a call passes 25 to 40 numbers; collecting them in Python and converting them one by one takes longer than the kernels of
// small problems (a 4 us product: 24 us of host time for the call, 11 of them here).
#define PY_SSIZE_T_CLEAN
#include <Python.h>
#include <cstdint>
#include <initializer_list>
#include <new>
#include "../../include/bsp.h"

namespace {

PyObject *g_torch, *g_check, *g_raw_stream, *g_tensor, *g_parameter, *g_dtypes[3], *g_matmul_class;   // (borrowed for the life of the process)
PyObject *s_shape, *s_stride, *s_data_ptr, *s_dtype, *s_device, *s_get_device, *s_empty, *s_uint8, *s_float32, *s_target;
PyObject *k_dtype_device;                               // ('dtype', 'device')

struct Ref {                                            // an owned reference
  PyObject *o;
  explicit Ref(PyObject *p = nullptr) : o(p) {}
  ~Ref() { Py_XDECREF(o); }
  Ref(const Ref &) = delete;
  Ref &operator=(const Ref &) = delete;
  PyObject *release() { PyObject *p = o; o = nullptr; return p; }
};

// A tensor as the launchers see it.  read() is false for what is not a plain tensor on a GPU in one of the three types.
struct Operand {
  PyObject *obj = nullptr;
  int dim = 0, dtype = -1, dev = -1;
  int64_t size[4], stride[4];
  uintptr_t ptr = 0;

  bool read(PyObject *o, int max_dim = 4) {
    obj = o;
    if ((PyObject *)Py_TYPE(o) != g_tensor && (PyObject *)Py_TYPE(o) != g_parameter && PyObject_IsInstance(o, g_tensor) != 1) return no();
    Ref dev_o(PyObject_CallMethodNoArgs(o, s_get_device));
    if (!dev_o.o) return no();
    dev = (int)PyLong_AsLong(dev_o.o);
    if (dev < 0) return no();
    Ref dt(PyObject_GetAttr(o, s_dtype)), sh(PyObject_GetAttr(o, s_shape));
    if (!dt.o || !sh.o) return no();
    for (int i = 0; i < 3; i++) if (dt.o == g_dtypes[i]) dtype = i;
    if (dtype < 0 || !PyTuple_Check(sh.o) || PyTuple_GET_SIZE(sh.o) > max_dim || PyTuple_GET_SIZE(sh.o) < 1) return false;
    Ref st(PyObject_CallMethodNoArgs(o, s_stride)), p(PyObject_CallMethodNoArgs(o, s_data_ptr));
    if (!st.o || !p.o || !PyTuple_Check(st.o) || PyTuple_GET_SIZE(st.o) != PyTuple_GET_SIZE(sh.o)) return no();
    dim = (int)PyTuple_GET_SIZE(sh.o);
    for (int i = 0; i < dim; i++) {
      size[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(sh.o, i));
      stride[i] = PyLong_AsLongLong(PyTuple_GET_ITEM(st.o, i));
    }
    ptr = (uintptr_t)PyLong_AsUnsignedLongLong(p.o);
    return !PyErr_Occurred() || no();
  }
  static bool no() { PyErr_Clear(); return false; }
  void *data() const { return reinterpret_cast<void *>(ptr); }
  int vec() const { return dtype == BSP_F32 ? 4 : 8; }
  // 16-byte accesses along a unit inner stride
  bool vectors() const {
    if (stride[dim - 1] != 1 || ptr & 15) return false;
    for (int i = 0; i + 1 < dim; i++) if (stride[i] % vec()) return false;
    return true;
  }
  bool contiguous() const {
    int64_t want = 1;
    for (int i = dim - 1; i >= 0; i--) {
      if (size[i] != 1 && stride[i] != want) return false;
      want *= size[i];
    }
    return true;
  }
  int64_t numel() const { int64_t n = 1; for (int i = 0; i < dim; i++) n *= size[i]; return n; }
};

// torch.empty(size, dtype = dtype, device = that of `like`): looked up at every call, as any caller does
PyObject *empty(const int64_t *size, int n, PyObject *dtype, PyObject *like) {
  Ref fn(PyObject_GetAttr(g_torch, s_empty)), dev(PyObject_GetAttr(like, s_device)), shape(PyTuple_New(n));
  if (!fn.o || !dev.o || !shape.o) return nullptr;
  for (int i = 0; i < n; i++) {
    PyObject *v = PyLong_FromLongLong(size[i]);
    if (!v) return nullptr;
    PyTuple_SET_ITEM(shape.o, i, v);
  }
  PyObject *args[] = {shape.o, dtype, dev.o};
  return PyObject_Vectorcall(fn.o, args, 1, k_dtype_device);
}
PyObject *empty_like_type(const int64_t *size, int n, const Operand &like) { return empty(size, n, g_dtypes[like.dtype], like.obj); }
PyObject *empty_bytes(int64_t n, PyObject *like) {
  Ref dt(PyObject_GetAttr(g_torch, s_uint8));
  return dt.o ? empty(&n, 1, dt.o, like) : nullptr;
}
PyObject *empty_floats(const int64_t *size, int n, PyObject *like) {
  Ref dt(PyObject_GetAttr(g_torch, s_float32));
  return dt.o ? empty(size, n, dt.o, like) : nullptr;
}
bool pointer(PyObject *t, void **out) {
  Ref p(PyObject_CallMethodNoArgs(t, s_data_ptr));
  if (!p.o) return false;
  *out = PyLong_AsVoidPtr(p.o);
  return !PyErr_Occurred();
}
// memory for the fp32 parts of one call, which has it to itself until its launches are made (_scratch in matmul.py)
bool scratch(int64_t n, PyObject *like, Ref &held, void **out) {
  Py_XSETREF(held.o, empty_bytes(n, like));
  return held.o && pointer(held.o, out);
}
bool stream_of(int dev, void **out) {
  Ref d(PyLong_FromLong(dev));
  Ref s(d.o ? PyObject_CallOneArg(g_raw_stream, d.o) : nullptr);
  if (!s.o) return false;
  *out = PyLong_AsVoidPtr(s.o);
  return !PyErr_Occurred();
}
bool truth(PyObject *o) { return o == Py_True || (o != Py_False && PyObject_IsTrue(o) == 1); }
bool checked(int rc, const char *what) {                // true, or false with the error set
  if (rc == BSP_OK) return true;
  Ref r(PyObject_CallFunction(g_check, "is", rc, what));
  if (r.o) PyErr_Format(PyExc_RuntimeError, "%s failed (status %d)", what, rc);
  return false;
}

// An entry point without the interpreter's lock: a launch waits where the queue is full.  (f touches no Python object.)
template <class F> int unlocked(F &&f) {
  PyThreadState *t = PyEval_SaveThread();
  const int rc = f();
  PyEval_RestoreThread(t);
  return rc;
}

// ---- tables: numbers and pointers that stay the same for an operator, with the tensors behind the pointers ----
struct Plan { const int32_t *table; int n_groups, lines, n_split; };
struct Xsd {
  PyObject *keep;                                       // a tuple, the ordinary plan its second, the wide one its third member
  const int32_t *lut, *plan;
  int width, block, dtype, dev, longest;
  int64_t nnz, H, R, C;
  Plan ordinary, wide;
  int wide_flags;                                       // that go with the wide plan
  int wide_state;                                       // 0: there is none, 1: not built yet, 2: built
};
struct Sdd {
  PyObject *keep;                                       // a tuple, the SddTables first
  int block, dtype, dev;
  int64_t nnz, H, R, C;
  Plan ordinary, longk, tiles;
  int tiles_state, tiles_launch, tile_blocks;           // as wide_state; SddTables.TILES_LAUNCH, TILE_BLOCKS
  int long_state, long_rowpair, long_entries;           // as wide_state
  int n_levels, any_k;                                  // n_levels -1: the tables are not built yet
  int packs[3];
  const int32_t *luts[3];
  const uint8_t *valids[3];
  int64_t widths[3];
};
struct Rows {                                           // softmax
  PyObject *keep;
  const int32_t *lut;
  int maxlut, dev;
  int64_t nnz, H, R, C, block;
};
struct Attn {
  PyObject *keep;
  const int32_t *rows, *items, *split;
  int lines, columns, n_items, n_slots, n_split, dev, longest;
  int64_t H, R, C, block;
};
template <class S> void drop(PyObject *cap) {
  S *s = static_cast<S *>(PyCapsule_GetPointer(cap, PyCapsule_GetName(cap)));
  if (s) { Py_XDECREF(s->keep); delete s; }
}
template <class S> PyObject *capsule(const S &tables, const char *name) {
  S *s = new (std::nothrow) S(tables);
  if (!s) return PyErr_NoMemory();
  Py_INCREF(s->keep);
  PyObject *c = PyCapsule_New(s, name, drop<S>);
  if (!c) { Py_XDECREF(s->keep); delete s; }
  return c;
}
const char *kXsd = "torch_blocksparse.xsd", *kSdd = "torch_blocksparse.sdd", *kRows = "torch_blocksparse.rows", *kAttn = "torch_blocksparse.attn";

PyObject *make_xsd(PyObject *, PyObject *args) {
  Xsd s{};
  unsigned long long lut, planbuf, gp, wp;
  if (!PyArg_ParseTuple(args, "OKKiiiiiLLLL(Kiii)(Kiii)ii", &s.keep, &lut, &planbuf, &s.width, &s.block, &s.dtype, &s.dev, &s.longest, &s.nnz, &s.H, &s.R, &s.C, &gp,
                        &s.ordinary.n_groups, &s.ordinary.lines, &s.ordinary.n_split, &wp, &s.wide.n_groups, &s.wide.lines, &s.wide.n_split, &s.wide_flags, &s.wide_state))
    return nullptr;
  s.lut = reinterpret_cast<const int32_t *>(lut); s.plan = reinterpret_cast<const int32_t *>(planbuf);
  s.ordinary.table = reinterpret_cast<const int32_t *>(gp); s.wide.table = reinterpret_cast<const int32_t *>(wp);
  return capsule(s, kXsd);
}

PyObject *make_sdd(PyObject *, PyObject *args) {
  Sdd s{};
  unsigned long long gp, lp, tp;
  PyObject *levels;
  if (!PyArg_ParseTuple(args, "OiiiLLLL(Kiii)(Kiii)iiii(Kiii)iiiO", &s.keep, &s.block, &s.dtype, &s.dev, &s.nnz, &s.H, &s.R, &s.C, &gp, &s.ordinary.n_groups,
                        &s.ordinary.lines, &s.ordinary.n_split, &lp, &s.longk.n_groups, &s.longk.lines, &s.longk.n_split, &s.long_state, &s.long_rowpair,
                        &s.long_entries, &s.any_k, &tp, &s.tiles.n_groups, &s.tiles.lines, &s.tiles.n_split, &s.tiles_state, &s.tiles_launch, &s.tile_blocks, &levels))
    return nullptr;
  s.tiles.table = reinterpret_cast<const int32_t *>(tp);
  s.ordinary.table = reinterpret_cast<const int32_t *>(gp); s.longk.table = reinterpret_cast<const int32_t *>(lp);
  s.n_levels = -1;
  if (levels != Py_None) {
    if (!PyTuple_Check(levels) || PyTuple_GET_SIZE(levels) > 3) { PyErr_SetString(PyExc_ValueError, "at most three pack levels"); return nullptr; }
    s.n_levels = (int)PyTuple_GET_SIZE(levels);
    for (int i = 0; i < s.n_levels; i++) {
      unsigned long long l, v;
      long long w;
      if (!PyArg_ParseTuple(PyTuple_GET_ITEM(levels, i), "iKKL", &s.packs[i], &l, &v, &w)) return nullptr;
      s.luts[i] = reinterpret_cast<const int32_t *>(l); s.valids[i] = reinterpret_cast<const uint8_t *>(v); s.widths[i] = w;
    }
  }
  return capsule(s, kSdd);
}

PyObject *make_rows(PyObject *, PyObject *args) {
  Rows s{};
  unsigned long long lut;
  if (!PyArg_ParseTuple(args, "OKiiLLLLL", &s.keep, &lut, &s.maxlut, &s.dev, &s.nnz, &s.H, &s.R, &s.C, &s.block)) return nullptr;
  s.lut = reinterpret_cast<const int32_t *>(lut);
  return capsule(s, kRows);
}

PyObject *make_attn(PyObject *, PyObject *args) {
  Attn s{};
  unsigned long long r, i, p;
  if (!PyArg_ParseTuple(args, "OKKKiiiiiiiLLLL", &s.keep, &r, &i, &p, &s.lines, &s.columns, &s.n_items, &s.n_slots, &s.n_split, &s.dev, &s.longest, &s.H, &s.R, &s.C,
                        &s.block))
    return nullptr;
  s.rows = reinterpret_cast<const int32_t *>(r); s.items = reinterpret_cast<const int32_t *>(i); s.split = reinterpret_cast<const int32_t *>(p);
  return capsule(s, kAttn);
}

// ---- products ----
// xsd(tables, is_dds, a, b, trans_a, trans_b, trans_c, flags): bsp_dsd_matmul / bsp_dds_matmul
PyObject *xsd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 8) { PyErr_SetString(PyExc_TypeError, "xsd takes 8 arguments"); return nullptr; }
  const Xsd *s = static_cast<const Xsd *>(PyCapsule_GetPointer(args[0], kXsd));
  if (!s) return nullptr;
  const bool dds = truth(args[1]), ta = truth(args[4]), tb = truth(args[5]), tc = truth(args[6]);
  int flags = (int)PyLong_AsLong(args[7]);
  Operand sp, dn;
  if (!sp.read(args[dds ? 3 : 2]) || !dn.read(args[dds ? 2 : 3])) Py_RETURN_NONE;
  if (dn.dtype != s->dtype || sp.dtype != s->dtype || dn.dev != s->dev || sp.dev != s->dev || dn.dim != 4 || sp.dim < 3) Py_RETURN_NONE;
  const int64_t Z = dn.size[0], block = s->block;
  // dense: op(dn) has its reduction over the layout's rows or columns, its free dimension of any size
  const int64_t red = block * (dds ? (tb ? s->C : s->R) : (ta ? s->R : s->C)), out_sp = block * (dds ? (tb ? s->R : s->C) : (ta ? s->C : s->R));
  const int red_at = dds ? (ta ? 2 : 3) : (tb ? 3 : 2);
  const int64_t free_dim = dn.size[5 - red_at];
  if (Z <= 0 || free_dim <= 0 || dn.size[1] != s->H || dn.size[red_at] != red || !dn.vectors()) Py_RETURN_NONE;
  if (sp.size[sp.dim - 1] != block || sp.size[sp.dim - 2] != block || sp.size[sp.dim - 3] != s->nnz || !sp.contiguous() || sp.ptr & 15) Py_RETURN_NONE;
  if (sp.dim == 4 && sp.size[0] != 1 && sp.size[0] != Z) Py_RETURN_NONE;
  const bool whole_rows = dds ? !ta && !tc : tb && tc;  // the free dimension lies along whole rows on both sides
  if ((free_dim % dn.vec() && !whole_rows) || free_dim > INT32_MAX) Py_RETURN_NONE;
  Plan plan = s->ordinary;
  // (_plan_for in matmul.py)
  if (block == 32 && free_dim >= 256 && s->dtype != BSP_F32 && s->wide_state && (int64_t)(s->width + 3) / 4 * ((free_dim + 255) / 256) * Z >= 384) {
    if (s->wide_state != 2) Py_RETURN_NONE;
    plan = s->wide;
    flags |= s->wide_flags;
  }
  const bool out_free_last = dds ? tc : !tc;            // the result's free dimension is its last one
  const int64_t shape[4] = {Z, s->H, out_free_last ? out_sp : free_dim, out_free_last ? free_dim : out_sp};
  Ref c(empty_like_type(shape, 4, dn));
  void *cp, *wsp = nullptr, *st;
  if (!c.o || !pointer(c.o, &cp) || !stream_of(dn.dev, &st)) return nullptr;
  long long ws_bytes = 0;
  if (plan.table && plan.n_split) {                     // the plan keeps its workspace (GroupPlan.workspace_address)
    unsigned long long at;
    Ref ws(PyObject_CallMethod(PyTuple_GET_ITEM(s->keep, plan.table == s->wide.table ? 2 : 1), "workspace_address", "LL", (long long)free_dim, (long long)Z));
    if (!ws.o || !PyArg_ParseTuple(ws.o, "KL", &at, &ws_bytes)) return nullptr;
    wsp = reinterpret_cast<void *>(at);
  }
  const int64_t sp_sz = sp.dim == 4 && sp.size[0] > 1 ? sp.stride[0] : 0, ldc = shape[3], c_sh = shape[2] * shape[3], c_sz = s->H * c_sh;
  int part_blocks = 0;
  const int parts = bsp_xsd_parts(s->dtype, s->block, s->width, s->longest, s->nnz, (int)free_dim, (int)Z, flags, &part_blocks);
  if (parts > 1) {
    const int64_t need = bsp_xsd_parts_workspace_bytes(s->block, s->width, (int)free_dim, (int)Z, parts);
    Ref ws;
    if (!scratch(need, dn.obj, ws, &wsp)) return nullptr;
    const int rc = unlocked([&] {
      return bsp_xsd_matmul_parts(dds, s->dtype, sp.data(), dn.data(), cp, ta, tb, tc, (int)Z, (int)free_dim, sp_sz, dn.stride[0], dn.stride[1], dn.stride[2], c_sz, c_sh, ldc,
                                  s->block, s->lut, s->plan, s->width, parts, part_blocks, wsp, need, st);
    });
    return checked(rc, "bsp_xsd_matmul_parts") ? c.release() : nullptr;
  }
  const int rc = unlocked([&] {
    return dds ? bsp_dds_matmul(s->dtype, dn.data(), sp.data(), cp, ta, tb, tc, (int)Z, (int)free_dim, dn.stride[0], dn.stride[1], dn.stride[2], sp_sz,
                                c_sz, c_sh, ldc, s->block, s->lut, s->plan, s->width, plan.table, plan.n_groups, plan.lines, plan.n_split, wsp, ws_bytes,
                                flags, st)
               : bsp_dsd_matmul(s->dtype, sp.data(), dn.data(), cp, ta, tb, tc, (int)Z, (int)free_dim, sp_sz, dn.stride[0], dn.stride[1], dn.stride[2],
                                c_sz, c_sh, ldc, s->block, s->lut, s->plan, s->width, plan.table, plan.n_groups, plan.lines, plan.n_split, wsp, ws_bytes,
                                flags, st);
  });
  return checked(rc, dds ? "bsp_dds_matmul" : "bsp_dsd_matmul") ? c.release() : nullptr;
}

// sdd(tables, a, b, trans_a, trans_b, trans_c, flags): bsp_sdd_matmul with the plan alone where a kernel takes it, else all pack levels
PyObject *sdd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 7) { PyErr_SetString(PyExc_TypeError, "sdd takes 7 arguments"); return nullptr; }
  const Sdd *s = static_cast<const Sdd *>(PyCapsule_GetPointer(args[0], kSdd));
  if (!s) return nullptr;
  const bool swap = truth(args[5]);                 // C^T = op(B)^T . op(A)^T (matmul.py:303-305)
  bool ta = truth(args[3]), tb = truth(args[4]);
  if (swap) { const bool t = !tb; tb = !ta; ta = t; }
  int flags = (int)PyLong_AsLong(args[6]);
  Operand a, b;
  if (!a.read(args[swap ? 2 : 1]) || !b.read(args[swap ? 1 : 2])) Py_RETURN_NONE;
  if (a.dtype != s->dtype || b.dtype != s->dtype || a.dev != s->dev || b.dev != s->dev || a.dim != 4 || b.dim != 4 || !a.vectors() || !b.vectors()) Py_RETURN_NONE;
  const int64_t Z = a.size[0], K = a.size[ta ? 2 : 3];
  const bool f32 = s->dtype == BSP_F32;
  if (Z <= 0 || K <= 0 || K > INT32_MAX || b.size[0] != Z || a.size[1] != s->H || b.size[1] != s->H || b.size[tb ? 3 : 2] != K) Py_RETURN_NONE;
  if (a.size[ta ? 3 : 2] != s->block * s->R || b.size[tb ? 2 : 3] != s->block * s->C) Py_RETURN_NONE;
  const bool by_rows = s->any_k && ta && !tb;
  if (by_rows && s->long_state && bsp_sdd_whole_steps(s->dtype, s->block, s->nnz, s->block * s->R, s->block * s->C, (int)K)) Py_RETURN_NONE;   // (copied)
  const bool any_k = K % 16 != 0;
  if (any_k && !by_rows) Py_RETURN_NONE;
  if (any_k) flags |= BSP_FLAG_ANY_K;
  const bool long_k = (s->block == 16 || s->block == 32) && K >= 256 && K % 32 == 0 && !f32 && s->long_state;
  if ((long_k && s->long_state != 2) || (s->n_levels < 0 && (any_k || (!long_k && !s->ordinary.table)))) Py_RETURN_NONE;
  bool tiles = long_k && s->tiles_state && s->nnz * Z >= (int64_t)s->tiles_launch * s->tile_blocks;       // SddTables.tiles_for
  if (tiles && s->tiles_state != 2) Py_RETURN_NONE;
  tiles = tiles && (int64_t)s->tiles.n_groups * Z >= s->tiles_launch && s->nnz >= (int64_t)s->tile_blocks * s->tiles.n_groups;
  int parts = 0;
  if (s->n_levels == 1 && s->block == 128 && !f32 && K % 32 == 0 && K >= 512 && s->packs[0] == 1 && !(flags & (BSP_FLAG_GENERAL_ONLY | BSP_FLAG_NO_WIDE))) {
    Ref t(PyObject_GetAttr(g_matmul_class, s_target));  // _sdd_splitk in matmul.py
    if (!t.o) return nullptr;
    const int64_t target = PyLong_AsLongLong(t.o), blocks = s->widths[0] * Z;
    if (blocks > 0 && blocks < target) {
      int64_t p = target / blocks;
      if (p > K / 256) p = K / 256;
      if (p > 16) p = 16;
      parts = p < 1 ? 1 : (int)p;
    }
  }
  const int64_t shape[4] = {Z, s->nnz, s->block, s->block}, c_sz = s->nnz * s->block * s->block;
  Ref c(empty_like_type(shape, 4, a)), ws;
  void *cp, *wsp = nullptr, *st;
  if (!c.o || !pointer(c.o, &cp) || !stream_of(a.dev, &st)) return nullptr;
#define BSP_OPERANDS s->dtype, a.data(), b.data(), cp, ta, tb, (int)Z, (int)K, a.stride[0], a.stride[1], a.stride[2], b.stride[0], b.stride[1], b.stride[2], c_sz, s->block
  int rc = BSP_NEEDS_TABLE;
  if (tiles)
    rc = unlocked([&] {
      return bsp_sdd_matmul(BSP_OPERANDS, 0, nullptr, nullptr, s->C, s->tiles.table, s->tiles.n_groups, s->tiles.lines, flags | BSP_FLAG_PLAN_TILES, st);
    });
  if (rc != BSP_NEEDS_TABLE) {
  } else if (long_k)
    rc = unlocked([&] { return bsp_sdd_matmul(BSP_OPERANDS, 0, nullptr, nullptr, s->long_entries < s->C ? s->long_entries : s->C, s->longk.table, s->longk.n_groups, s->longk.lines,
                        flags | (s->long_rowpair ? BSP_FLAG_PLAN_ROWPAIR : 0), st); });
  else if (s->n_levels < 0)
    rc = unlocked([&] { return bsp_sdd_matmul(BSP_OPERANDS, 0, nullptr, nullptr, s->C, s->ordinary.table, s->ordinary.n_groups, s->ordinary.lines, flags, st); });
  if (rc == BSP_OK_WHOLE_LAYOUT) return c.release();
  if (rc != BSP_NEEDS_TABLE) return checked(rc, "bsp_sdd_matmul") ? c.release() : nullptr;
  if (s->n_levels < 0) Py_RETURN_NONE;                  // (nothing was launched)
  if (parts) {
    const int64_t need = bsp_sdd_splitk_workspace_bytes((int)Z, s->widths[0], parts);
    if (need && !scratch(need, a.obj, ws, &wsp)) return nullptr;
    rc = unlocked([&] { return bsp_sdd_matmul_splitk(BSP_OPERANDS, s->luts[0], s->valids[0], s->widths[0], parts, wsp, need, flags, st); });
    if (rc != BSP_ERR_UNSUPPORTED) return checked(rc, "bsp_sdd_matmul_splitk") ? c.release() : nullptr;
  }
  if (s->n_levels == 0) return c.release();
  parts = bsp_sdd_parts(s->dtype, s->block, s->n_levels, s->packs, s->widths, (int)Z, (int)K, flags);
  const int64_t need = bsp_sdd_parts_workspace_bytes(s->block, s->nnz, (int)Z, parts);
  if (need && !scratch(need, a.obj, ws, &wsp)) return nullptr;
  rc = unlocked([&] {
    return bsp_sdd_matmul_levels(BSP_OPERANDS, s->n_levels, s->packs, s->luts, s->valids, s->widths, s->ordinary.table, s->ordinary.n_groups, s->ordinary.lines, parts, s->nnz,
                                 wsp, need, flags, st);
  });
#undef BSP_OPERANDS
  return rc == BSP_OK_WHOLE_LAYOUT || checked(rc, "bsp_sdd_matmul_levels") ? c.release() : nullptr;
}

// ---- softmax ----
struct Mask { Operand t; bool given = false; };
// a mask of the softmax: unit inner stride, 16-byte aligned rows, the type of x
bool mask_ok(PyObject *o, const Operand &x, Mask &m) {
  if (o == Py_None) return true;
  m.given = true;
  return m.t.read(o) && m.t.dtype == x.dtype && m.t.dev == x.dev && m.t.vectors();
}

// softmax_fwd(tables, x, scale, rpe, key_padding_mask, attn_mask, kp_mul, attn_mul) -> True: bsp_softmax_fwd in place on x
PyObject *softmax_fwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 8) { PyErr_SetString(PyExc_TypeError, "softmax_fwd takes 8 arguments"); return nullptr; }
  const Rows *s = static_cast<const Rows *>(PyCapsule_GetPointer(args[0], kRows));
  if (!s) return nullptr;
  Operand x;
  if (!x.read(args[1]) || x.dim != 4 || x.dev != s->dev || x.size[0] <= 0 || x.size[1] != s->nnz || x.size[2] != s->block || x.size[3] != s->block ||
      !x.contiguous() || x.ptr & 15 || (int64_t)s->maxlut * s->block >= 32768)
    Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(args[2]);
  if (PyErr_Occurred()) return nullptr;
  const int64_t Z = x.size[0], rows = s->R * s->block, cols = s->C * s->block;
  Mask rpe, kpm, att;
  if (!mask_ok(args[3], x, rpe) || !mask_ok(args[4], x, kpm) || !mask_ok(args[5], x, att)) Py_RETURN_NONE;
  if (kpm.given && (kpm.t.dim != 2 || (kpm.t.size[0] != 1 && kpm.t.size[0] != Z) || kpm.t.size[1] < cols)) Py_RETURN_NONE;
  if (att.given && (att.t.dim != 2 || att.t.size[0] < rows || att.t.size[1] < cols)) Py_RETURN_NONE;
  int64_t r[4] = {0, 0, 0, 0};                          // the embedding's strides over (z, h, row), broadcast dimensions 0
  if (rpe.given) {
    const int d = rpe.t.dim;
    if (d < 2 || rpe.t.size[d - 2] < rows || rpe.t.size[d - 1] < cols) Py_RETURN_NONE;
    r[2] = rpe.t.stride[d - 2];
    if (d > 2) {
      if (rpe.t.size[d - 3] != 1 && rpe.t.size[d - 3] != s->H) Py_RETURN_NONE;
      r[1] = rpe.t.size[d - 3] == 1 ? 0 : rpe.t.stride[d - 3];
    }
    if (d > 3) {
      if (rpe.t.size[0] != 1 && rpe.t.size[0] != Z) Py_RETURN_NONE;
      r[0] = rpe.t.size[0] == 1 ? 0 : rpe.t.stride[0];
    }
  }
  const int kpm_mul = truth(args[6]), att_mul = truth(args[7]);
  const int64_t kpm_sz = kpm.given && kpm.t.size[0] > 1 ? kpm.t.stride[0] : 0, att_ld = att.given ? att.t.stride[0] : 0;
  void *st;
  if (PyErr_Occurred() || !stream_of(x.dev, &st)) return nullptr;
  const int rc = unlocked([&] {
    return bsp_softmax_fwd(x.dtype, x.data(), (float)scale, s->lut, s->maxlut, rpe.given ? rpe.t.data() : nullptr, r[0], r[1], r[2],
                           kpm.given ? kpm.t.data() : nullptr, kpm_sz, kpm_mul, att.given ? att.t.data() : nullptr, att_ld, att_mul,
                           (int)Z, (int)s->H, (int)s->R, (int)s->block, s->nnz * s->block * s->block, st);
  });
  if (!checked(rc, "bsp_softmax_fwd")) return nullptr;
  Py_RETURN_TRUE;
}

// softmax_bwd(tables, y, dy, scale) -> True: bsp_softmax_bwd in place on dy
PyObject *softmax_bwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 4) { PyErr_SetString(PyExc_TypeError, "softmax_bwd takes 4 arguments"); return nullptr; }
  const Rows *s = static_cast<const Rows *>(PyCapsule_GetPointer(args[0], kRows));
  if (!s) return nullptr;
  Operand y, dy;
  if (!y.read(args[1]) || !dy.read(args[2]) || y.dim != 4 || dy.dim != 4 || y.dev != s->dev || dy.dev != s->dev || y.dtype != dy.dtype || y.size[0] <= 0 ||
      y.size[0] != dy.size[0] || y.size[1] != s->nnz || dy.size[1] != s->nnz || y.size[2] != s->block || y.size[3] != s->block || dy.size[2] != s->block ||
      dy.size[3] != s->block || !y.contiguous() || !dy.contiguous() || (y.ptr | dy.ptr) & 15)
    Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(args[3]);
  void *st;
  if (PyErr_Occurred() || !stream_of(y.dev, &st)) return nullptr;
  const int64_t sz = s->nnz * s->block * s->block;
  const int rc = unlocked([&] { return bsp_softmax_bwd(y.dtype, y.data(), dy.data(), (float)scale, s->lut, s->maxlut, (int)y.size[0], (int)s->H, (int)s->R, (int)s->block, sz, sz, st); });
  if (!checked(rc, "bsp_softmax_bwd")) return nullptr;
  Py_RETURN_TRUE;
}

// ---- attention without per-element masks ----
// what the kernels address (_near in attention_core.py): 16-byte rows that do not overlap, within 4 GiB of a head's first
bool near_rows(const Operand &t) {
  return t.dim == 4 && t.stride[3] == 1 && !((t.stride[0] | t.stride[1] | t.stride[2]) % 8) && t.stride[2] >= t.size[3] && !(t.ptr & 15) &&
         t.stride[2] * t.size[2] * 2 < (int64_t)1 << 32;
}
bool attn_shape(const Attn *s, const Operand &q, const Operand &k, const Operand &v, bool f32 = false) {
  if ((q.dtype == BSP_F32) != f32 || k.dtype != q.dtype || v.dtype != q.dtype || q.dev != s->dev || k.dev != q.dev || v.dev != q.dev) return false;
  if (q.dim != 4 || k.dim != 4 || v.dim != 4 || (q.size[3] != 64 && q.size[3] != 128) || q.size[0] <= 0) return false;
  for (const Operand *t : {&q, &k, &v})
    if (t->size[0] != q.size[0] || t->size[1] != s->H || t->size[3] != q.size[3] || t->size[2] != (t == &q ? s->R : s->C) * s->block) return false;
  return true;
}

// attn_usable(tables, q, k, v): do the kernels take these operands (copied, where they have to be)?  (fp32: those of attention_f32.hip,
// which keep three parts of two bytes an element within 4 GiB of a head's first)
PyObject *attn_usable(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 4) { PyErr_SetString(PyExc_TypeError, "attn_usable takes 4 arguments"); return nullptr; }
  const Attn *s = static_cast<const Attn *>(PyCapsule_GetPointer(args[0], kAttn));
  if (!s) return nullptr;
  Operand q, k, v;
  if (!q.read(args[1]) || !k.read(args[2]) || !v.read(args[3])) Py_RETURN_NONE;
  const bool f32 = q.dtype == BSP_F32;
  return PyBool_FromLong(attn_shape(s, q, k, v, f32) && s->longest > 0 && s->longest * 64 < 32768 &&
                         (!f32 || (s->R > s->C ? s->R : s->C) * s->block * q.size[3] * 6 < (int64_t)1 << 32));
}

// attn_fwd(tables, q, k, v, scale, kpm, kpm_stride, kpm_mul, keep) -> (o, lse or None): bsp_attention_rows_fwd
PyObject *attn_fwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 9) { PyErr_SetString(PyExc_TypeError, "attn_fwd takes 9 arguments"); return nullptr; }
  const Attn *s = static_cast<const Attn *>(PyCapsule_GetPointer(args[0], kAttn));
  if (!s) return nullptr;
  Operand q, k, v;
  if (!q.read(args[1]) || !k.read(args[2]) || !v.read(args[3]) || !attn_shape(s, q, k, v) || !near_rows(q) || !near_rows(k) || !near_rows(v)) Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(args[4]);
  const int64_t kpm_sz = PyLong_AsLongLong(args[6]);
  const int mul = (int)PyLong_AsLong(args[7]);
  void *kpm = nullptr, *op, *lp = nullptr, *st;
  if (PyErr_Occurred() || (args[5] != Py_None && !pointer(args[5], &kpm)) || !stream_of(q.dev, &st)) return nullptr;
  const int64_t Z = q.size[0], rows = s->R * s->block, D = q.size[3], shape[4] = {Z, s->H, rows, D}, lshape[4] = {Z, s->H, 2, (int64_t)s->lines * 64};
  Ref o(empty_like_type(shape, 4, q)), lse;
  if (!o.o || !pointer(o.o, &op)) return nullptr;
  if (truth(args[8])) {
    lse.o = empty_floats(lshape, 4, q.obj);
    if (!lse.o || !pointer(lse.o, &lp)) return nullptr;
  }
  const int rc = unlocked([&] { return bsp_attention_rows_fwd(q.dtype | BSP_ROWS_WITH_REST, q.data(), k.data(), v.data(), op, static_cast<float *>(lp), (int)Z, (int)s->H, s->lines, k.size[2],
                                        (int)D, q.stride[0], q.stride[1], q.stride[2], k.stride[0], k.stride[1], k.stride[2], v.stride[0], v.stride[1], v.stride[2],
                                        s->H * rows * D, rows * D, D, (int64_t)s->lines * 128, (float)scale, s->rows, kpm, kpm_sz, mul, st); });
  if (!checked(rc, "bsp_attention_rows_fwd")) return nullptr;
  return PyTuple_Pack(2, o.o, lse.o ? lse.o : Py_None);
}

// attn_bwd(tables, do, q, k, v, o, lse, scale, kpm, kpm_stride, kpm_mul, need_q, need_k, need_v) -> (dq, dk, dv): the row kernel
// (bsp_attention_rows_bwd) where dq or dk is asked for, the column kernel (bsp_attention_cols_bwd) where dk is.  (dv without dk: Python)
PyObject *attn_bwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 14) { PyErr_SetString(PyExc_TypeError, "attn_bwd takes 14 arguments"); return nullptr; }
  const Attn *s = static_cast<const Attn *>(PyCapsule_GetPointer(args[0], kAttn));
  if (!s) return nullptr;
  const bool need_q = truth(args[11]), need_k = truth(args[12]), need_v = truth(args[13]);
  Operand g, q, k, v, o;
  if ((need_v && !need_k) || !(need_q || need_k) || !g.read(args[1]) || !q.read(args[2]) || !k.read(args[3]) || !v.read(args[4]) || !o.read(args[5]) ||
      !attn_shape(s, q, k, v))
    Py_RETURN_NONE;
  if (g.dim != 4 || g.dtype != q.dtype || o.dtype != q.dtype || g.dev != q.dev) Py_RETURN_NONE;
  for (int i = 0; i < 4; i++) if (g.size[i] != q.size[i] || o.size[i] != q.size[i]) Py_RETURN_NONE;
  if (!near_rows(g) || !near_rows(q) || !near_rows(k) || !near_rows(v) || !near_rows(o)) Py_RETURN_NONE;
  const double scale = PyFloat_AsDouble(args[7]);
  const int64_t kpm_sz = PyLong_AsLongLong(args[9]);
  const int mul = (int)PyLong_AsLong(args[10]);
  void *lse, *kpm = nullptr, *st, *delta = nullptr, *dq_p, *dk_p, *dv_p, *part = nullptr;
  if (PyErr_Occurred() || !pointer(args[6], &lse) || (args[8] != Py_None && !pointer(args[8], &kpm)) || !stream_of(q.dev, &st)) return nullptr;
  const int64_t Z = q.size[0], H = s->H, D = q.size[3], R = q.size[2], C = k.size[2], row_sh = (int64_t)s->lines * 128;
  const int64_t qs[4] = {Z, H, R, D}, ks[4] = {Z, H, C, D}, ds[4] = {Z, H, 2, (int64_t)s->lines * 64}, ps[5] = {Z, s->n_slots, 2, 64, D};
  // Each kernel's results are allocated in front of its launch, in the order of the general host side, so that they lie where they lie
  // there: with all of them allocated first the module's default at 8 x 16 x 4096 took up to 2 % longer in some processes
  Ref delta_o, dq, dk, dv, part_o;
  if (need_k) {                                         // (the rows of a head as far apart as those of lse; the second half is not used)
    delta_o.o = empty_floats(ds, 4, q.obj);
    if (!delta_o.o || !pointer(delta_o.o, &delta)) return nullptr;
  }
  dq.o = empty_like_type(qs, 4, q);
  if (!dq.o || !pointer(dq.o, &dq_p)) return nullptr;
  const int type = q.dtype | BSP_ROWS_WITH_REST;
  int rc = unlocked([&] { return bsp_attention_rows_bwd(type, g.data(), q.data(), k.data(), v.data(), o.data(), static_cast<const float *>(lse), dq_p, static_cast<float *>(delta), (int)Z, (int)H,
                                  s->lines, C, (int)D, g.stride[0], g.stride[1], g.stride[2], q.stride[0], q.stride[1], q.stride[2], k.stride[0], k.stride[1], k.stride[2],
                                  v.stride[0], v.stride[1], v.stride[2], o.stride[0], o.stride[1], o.stride[2], H * R * D, R * D, D, row_sh, (float)scale, s->rows, kpm, kpm_sz,
                                  mul, st); });
  if (!checked(rc, "bsp_attention_rows_bwd")) return nullptr;
  if (need_k) {
    dk.o = empty_like_type(ks, 4, k);
    dv.o = empty_like_type(ks, 4, v);
    if (!dk.o || !dv.o || !pointer(dk.o, &dk_p) || !pointer(dv.o, &dv_p)) return nullptr;
    if (s->n_slots) {
      part_o.o = empty_floats(ps, 5, q.obj);
      if (!part_o.o || !pointer(part_o.o, &part)) return nullptr;
    }
    rc = unlocked([&] { return bsp_attention_cols_bwd(type, g.data(), q.data(), k.data(), v.data(), static_cast<const float *>(lse), static_cast<const float *>(delta), dk_p, dv_p, (int)Z, (int)H,
                                s->columns, R, (int)D, g.stride[0], g.stride[1], g.stride[2], q.stride[0], q.stride[1], q.stride[2], k.stride[0], k.stride[1], k.stride[2],
                                v.stride[0], v.stride[1], v.stride[2], H * C * D, C * D, D, H * C * D, C * D, D, row_sh, (float)scale, s->items, s->n_items,
                                static_cast<float *>(part), s->n_slots, s->split, s->n_split, kpm, kpm_sz, mul, st); });
    if (!checked(rc, "bsp_attention_cols_bwd")) return nullptr;
  }
  return PyTuple_Pack(3, need_q ? dq.o : Py_None, need_k ? dk.o : Py_None, need_v ? dv.o : Py_None);
}

// ... in fp32
bool f32_rows(const Operand &t) {                       // _vec32 in attention_core.py
  return t.dim == 4 && t.stride[3] == 1 && !((t.stride[0] | t.stride[1] | t.stride[2]) % 4) && t.stride[2] >= t.size[3] && !(t.ptr & 15);
}
void put_strides(int64_t *to, const int64_t *size) {    // of a contiguous tensor
  to[0] = size[1] * size[2] * size[3]; to[1] = size[2] * size[3]; to[2] = size[3];
}
// the call's sizes and masks; masks: scale, kpm, kpm_stride, kpm_mul
bool f32_call(const Attn *s, int64_t Z, int64_t D, PyObject *const *masks, bsp_attention_f32_call *c) {
  *c = bsp_attention_f32_call{};
  c->Z = (int)Z; c->H = (int)s->H; c->R = s->lines; c->D = (int)D;
  c->keys = s->C * s->block;
  c->d_rows = s->rows;
  c->scale = (float)PyFloat_AsDouble(masks[0]);
  c->kpm_stride_z = PyLong_AsLongLong(masks[2]);
  c->kpm_mul = (int)PyLong_AsLong(masks[3]);
  void *kpm = nullptr;
  if (PyErr_Occurred() || (masks[1] != Py_None && !pointer(masks[1], &kpm))) return false;
  c->kpm = static_cast<const float *>(kpm);
  return true;
}

// attn32_fwd(tables, q, k, v, scale, kpm, kpm_stride, kpm_mul, keep) -> (o, planes, stats or None, copy of o or None): bsp_attention_f32_fwd
PyObject *attn32_fwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 9) { PyErr_SetString(PyExc_TypeError, "attn32_fwd takes 9 arguments"); return nullptr; }
  const Attn *s = static_cast<const Attn *>(PyCapsule_GetPointer(args[0], kAttn));
  if (!s) return nullptr;
  Operand q, k, v;
  if (!q.read(args[1]) || !k.read(args[2]) || !v.read(args[3]) || !attn_shape(s, q, k, v, true) || !f32_rows(q) || !f32_rows(k) || !f32_rows(v)) Py_RETURN_NONE;
  const int64_t Z = q.size[0], rows = q.size[2], D = q.size[3], shape[4] = {Z, s->H, rows, D}, sshape[4] = {Z, s->H, 2, rows};
  const bool keep = truth(args[8]);
  bsp_attention_f32_call c;
  void *op, *sp = nullptr, *cp = nullptr, *st;
  if (!f32_call(s, Z, D, args + 4, &c) || !stream_of(q.dev, &st)) return nullptr;
  Ref planes(empty_bytes(bsp_attention_f32_bytes((int)Z, (int)s->H, keep ? rows : 0, c.keys, (int)D), q.obj)), o(planes.o ? empty_like_type(shape, 4, q) : nullptr), stats, copy;
  if (!o.o || !pointer(planes.o, &c.planes) || !pointer(o.o, &op)) return nullptr;
  if (keep) {
    stats.o = empty_floats(sshape, 4, q.obj);
    copy.o = stats.o ? empty_like_type(shape, 4, q) : nullptr;
    if (!copy.o || !pointer(stats.o, &sp) || !pointer(copy.o, &cp)) return nullptr;
  }
  c.stats = static_cast<float *>(sp);
  c.o_copy = static_cast<float *>(cp);
  for (int i = 0; i < 3; i++) c.strides[i] = q.stride[i], c.strides[3 + i] = k.stride[i], c.strides[6 + i] = v.stride[i];
  put_strides(c.strides + 9, shape);
  const int rc = unlocked([&] { return bsp_attention_f32_fwd(&c, static_cast<const float *>(q.data()), static_cast<const float *>(k.data()), static_cast<const float *>(v.data()),
                                                             static_cast<float *>(op), st); });
  if (!checked(rc, "bsp_attention_f32_fwd")) return nullptr;
  return PyTuple_Pack(4, o.o, planes.o, stats.o ? stats.o : Py_None, copy.o ? copy.o : Py_None);
}

// attn32_bwd(tables, do, o, planes, stats, scale, kpm, kpm_stride, kpm_mul, need_q, need_k, need_v) -> (dq, dk, dv): bsp_attention_f32_bwd
PyObject *attn32_bwd(PyObject *, PyObject *const *args, Py_ssize_t n) {
  if (n != 12) { PyErr_SetString(PyExc_TypeError, "attn32_bwd takes 12 arguments"); return nullptr; }
  const Attn *s = static_cast<const Attn *>(PyCapsule_GetPointer(args[0], kAttn));
  if (!s) return nullptr;
  const bool need_q = truth(args[9]), need_k = truth(args[10]), need_v = truth(args[11]), columns = need_k || need_v;
  Operand g, o;
  if (!g.read(args[1]) || !o.read(args[2]) || g.dim != 4 || o.dim != 4 || g.dtype != BSP_F32 || o.dtype != BSP_F32 || g.dev != o.dev || o.dev != s->dev) Py_RETURN_NONE;
  for (int i = 0; i < 4; i++) if (g.size[i] != o.size[i]) Py_RETURN_NONE;
  if (o.size[1] != s->H || o.size[2] != (int64_t)s->lines * 64 || !f32_rows(g) || !f32_rows(o)) Py_RETURN_NONE;
  const int64_t Z = o.size[0], rows = o.size[2], D = o.size[3];
  bsp_attention_f32_call c;
  void *sp, *st, *dq_p, *dk_p = nullptr, *dv_p = nullptr, *parts_p = nullptr, *delta_p = nullptr, *slots_p = nullptr;
  if (!f32_call(s, Z, D, args + 5, &c) || !pointer(args[3], &c.planes) || !pointer(args[4], &sp) || !stream_of(o.dev, &st)) return nullptr;
  c.stats = static_cast<float *>(sp);
  const int64_t qs[4] = {Z, s->H, rows, D}, ks[4] = {Z, s->H, c.keys, D}, ds[3] = {Z, s->H, rows}, ps[4] = {bsp_attention_f32_slots((int)Z, s->n_slots), 2, 64, D};
  Ref dq(empty_like_type(qs, 4, o)), dk, dv, parts, delta, slots;
  if (!dq.o || !pointer(dq.o, &dq_p)) return nullptr;
  if (columns) {
    dk.o = empty_like_type(ks, 4, o);
    dv.o = dk.o ? empty_like_type(ks, 4, o) : nullptr;
    delta.o = dv.o ? empty_floats(ds, 3, o.obj) : nullptr;
    parts.o = delta.o ? empty_bytes(bsp_attention_f32_bytes((int)Z, (int)s->H, rows, 0, (int)D), o.obj) : nullptr;
    if (!parts.o || !pointer(dk.o, &dk_p) || !pointer(dv.o, &dv_p) || !pointer(delta.o, &delta_p) || !pointer(parts.o, &parts_p)) return nullptr;
    if (s->n_slots) {
      slots.o = empty_floats(ps, 4, o.obj);
      if (!slots.o || !pointer(slots.o, &slots_p)) return nullptr;
    }
  }
  for (int i = 0; i < 3; i++) c.strides[i] = g.stride[i], c.strides[3 + i] = o.stride[i];
  put_strides(c.strides + 6, qs);
  put_strides(c.strides + 9, ks);
  put_strides(c.strides + 12, ks);
  const int rc = unlocked([&] { return bsp_attention_f32_bwd(&c, static_cast<const float *>(g.data()), static_cast<const float *>(o.data()), static_cast<float *>(dq_p), static_cast<float *>(dk_p),
                                                             static_cast<float *>(dv_p), parts_p, static_cast<float *>(delta_p), s->items, s->n_items, static_cast<float *>(slots_p), s->n_slots,
                                                             s->split, s->n_split, st); });
  if (!checked(rc, "bsp_attention_f32_bwd")) return nullptr;
  return PyTuple_Pack(3, need_q ? dq.o : Py_None, need_k ? dk.o : Py_None, need_v ? dv.o : Py_None);
}

// setup(torch, _lib.check, raw stream of a device, Parameter, the class with SPLITK_TARGET_WORKGROUPS)
PyObject *setup(PyObject *, PyObject *args) {
  PyObject *torch, *check, *stream, *parameter, *cls;
  if (!PyArg_ParseTuple(args, "OOOOO", &torch, &check, &stream, &parameter, &cls)) return nullptr;
  const char *types[] = {"float16", "bfloat16", "float32"};     // in the order of BSP_F16, BSP_BF16, BSP_F32
  PyObject *tensor = PyObject_GetAttrString(torch, "Tensor"), *d[3];
  for (int i = 0; i < 3; i++) if (!(d[i] = PyObject_GetAttrString(torch, types[i]))) return nullptr;
  if (!tensor) return nullptr;
  for (PyObject *o : {torch, check, stream, parameter, cls}) Py_INCREF(o);
  g_torch = torch; g_check = check; g_raw_stream = stream; g_parameter = parameter; g_matmul_class = cls; g_tensor = tensor;
  for (int i = 0; i < 3; i++) g_dtypes[i] = d[i];
  Py_RETURN_NONE;
}

#define BSP_FAST(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {{"setup", setup, METH_VARARGS, nullptr}, {"make_xsd", make_xsd, METH_VARARGS, nullptr}, {"make_sdd", make_sdd, METH_VARARGS, nullptr},
                         {"make_rows", make_rows, METH_VARARGS, nullptr}, {"make_attn", make_attn, METH_VARARGS, nullptr}, BSP_FAST(xsd), BSP_FAST(sdd), BSP_FAST(softmax_fwd),
                         BSP_FAST(softmax_bwd), BSP_FAST(attn_usable), BSP_FAST(attn_fwd), BSP_FAST(attn_bwd), BSP_FAST(attn32_fwd), BSP_FAST(attn32_bwd), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_launch", "host side of the launches", -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

static_assert(BSP_F16 == 0 && BSP_BF16 == 1 && BSP_F32 == 2, "the order of the types in setup()");

PyMODINIT_FUNC PyInit__launch(void) {
  struct { PyObject **at; const char *name; } names[] = {{&s_shape, "shape"}, {&s_stride, "stride"}, {&s_data_ptr, "data_ptr"}, {&s_dtype, "dtype"}, {&s_device, "device"},
                                                         {&s_get_device, "get_device"}, {&s_empty, "empty"}, {&s_uint8, "uint8"}, {&s_float32, "float32"},
                                                         {&s_target, "SPLITK_TARGET_WORKGROUPS"}};
  for (auto &e : names) if (!(*e.at = PyUnicode_InternFromString(e.name))) return nullptr;
  if (!(k_dtype_device = PyTuple_Pack(2, s_dtype, s_device))) return nullptr;
  return PyModule_Create(&module);
}
