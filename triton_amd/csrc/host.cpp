// Host side of the hot entry points as a CPython extension: argument checks, output allocation and the call into the C
// ABI, without going through Python objects, ctypes structures and the dispatcher for every field.
//
// What bounds it: at decode sizes a layer's kernels take 35 us and the Python host code of its five calls took 120
// (matmul 19 us, routing 14, reduce 10, ...): the GPU waited for the host.  Here a call costs the
// reading of its arguments (about 50 ns per attribute), one caching-allocator request and the launch.
//
// Every function covers the calls that need no conversion and no error message -- GPU tensors of the types, layouts
// and shapes that the kernels take as they are -- and answers None for anything else; the Python code then runs the
// general path, which is also where every misuse is reported.  A call that is covered does exactly what the general
// path does.  There is no state besides interned names and the addresses handed over by init().
#define PY_SSIZE_T_CLEAN
#include <Python.h>

#include <ATen/ATen.h>
#include <c10/core/InferenceMode.h>
#include <c10/hip/HIPStream.h>
#include <torch/csrc/DynamicTypes.h>
#include <torch/csrc/Dtype.h>
#include <torch/csrc/autograd/python_variable.h>

#include <cmath>
#include <cstring>

#include "../../include/triton_amd.h"
#include "tile_rules.h"

namespace {

// ------------------------------------------------------------------ addresses and Python objects handed over by init()
struct Abi {
  int (*matmul)(const tamd_matmul_args *, size_t, void *);
  int (*routing)(const void *, int, int64_t, int, int, int, void *, int16_t *, uint32_t *, int64_t, int64_t, int32_t *,
                 int32_t *, int32_t *, int32_t *, void *, int32_t *, int64_t, int32_t *, int64_t, int, int32_t *, void *);
  int (*reduce)(const void *, int, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, const void *, int64_t, int64_t,
                int64_t, const void *, int64_t, int64_t, int64_t, void *, int, int64_t, int64_t, void *);
  int (*downcast)(const void *, int, int64_t, int64_t, int64_t, int64_t, int64_t, int64_t, void *, int, int64_t, int64_t,
                  void *, int64_t, int64_t, int, void *);
  int (*upcast)(const void *, int, int64_t, int64_t, const void *, int64_t, int64_t, void *, int, int64_t, int64_t, int64_t,
                int64_t, int64_t, int64_t, void *);
} abi;
PyObject *cls_tensor, *cls_value_layout, *cls_scale_layout, *obj_fp4, *ctx_constraints, *ctx_flags;

struct Names {
  PyObject *storage, *data, *layout, *dtype, *shape, *c_mx_scale, *c_microblock_size, *c_value_pack_factor, *a_mx_tensor_scale,
      *b_mx_tensor_scale, *acc_scale, *a_mx_scale, *a_microblock_size, *b_mx_scale, *b_microblock_size, *flex_ctx, *lhs_data,
      *rhs_data, *out_data, *acc_data, *scale, *expected_scale, *actual_scale, *checksum_scale, *out_dtype,
      *flexpoint_saturate_inf, *specs, *name, *fn_arg_names, *fn_args, *reduction_n, *slice_sizes, *slice_offs,
      *block_offs_data, *block_schedule_data, *expected_slice_size, *native;
} nm;

// ------------------------------------------------------------------ small helpers
struct Ref {  // owned reference
  PyObject *p;
  explicit Ref(PyObject *q) : p(q) {}
  Ref(const Ref &) = delete;
  ~Ref() { Py_XDECREF(p); }
  bool none() const { return p == Py_None; }
};
struct Miss {};  // "not covered here": the general path takes the call

PyObject *attr(PyObject *o, PyObject *name) {
  PyObject *v = PyObject_GetAttr(o, name);
  if (!v) {
    PyErr_Clear();
    throw Miss{};
  }
  return v;
}
inline void need(bool ok) {
  if (!ok) throw Miss{};
}
inline const at::Tensor &tensor(PyObject *o) {
  need(THPVariable_Check(o));
  return THPVariable_Unpack(o);
}
// a GPU tensor on device `dev` (any device when dev < 0, which is then set)
inline const at::Tensor &gpu_tensor(PyObject *o, int &dev) {
  const at::Tensor &t = tensor(o);
  need(t.is_cuda());
  const int d = t.get_device();
  if (dev < 0) dev = d;
  need(d == dev);
  return t;
}
inline int64_t as_int(PyObject *o) {
  need(PyLong_Check(o));
  const long long v = PyLong_AsLongLong(o);
  if (v == -1 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Miss{};
  }
  return v;
}
inline double as_double(PyObject *o) {
  need(PyFloat_Check(o) || PyLong_Check(o));
  const double v = PyFloat_AsDouble(o);
  if (v == -1.0 && PyErr_Occurred()) {
    PyErr_Clear();
    throw Miss{};
  }
  return v;
}
inline int type_code(at::ScalarType t) {
  switch (t) {
    case at::kFloat: return TAMD_F32;
    case at::kHalf: return TAMD_F16;
    case at::kBFloat16: return TAMD_BF16;
    case at::ScalarType::Float8_e4m3fn: return TAMD_FP8_E4M3;
    case at::ScalarType::Float8_e5m2: return TAMD_FP8_E5M2;
    default: throw Miss{};
  }
}
inline bool is_fp8_code(int c) { return c == TAMD_FP8_E4M3 || c == TAMD_FP8_E5M2; }
inline void *stream_of(int dev) { return (void *)c10::hip::getCurrentHIPStream((c10::DeviceIndex)dev).stream(); }
inline at::Tensor new_empty(at::IntArrayRef sizes, at::ScalarType t, int dev) {
  return at::empty(sizes, at::TensorOptions().dtype(t).device(at::Device(at::kCUDA, (c10::DeviceIndex)dev)));
}
// a float32 scalar on the device, or null
inline const float *scalar_ptr(PyObject *o, int &dev) {
  if (o == Py_None) return nullptr;
  const at::Tensor &t = gpu_tensor(o, dev);
  need(t.numel() == 1 && t.scalar_type() == at::kFloat);
  return (const float *)t.data_ptr();
}
template <typename F>
int without_gil(F f) {
  int rc;
  Py_BEGIN_ALLOW_THREADS rc = f();
  Py_END_ALLOW_THREADS return rc;
}
// runs `f` (a new reference, or a throw of Miss); any other C++ exception becomes a Python one
template <typename F>
PyObject *covered(F f) {
  try {
    return f();
  } catch (const Miss &) {
    Py_RETURN_NONE;
  } catch (const c10::OutOfMemoryError &e) {
    // torch's own class for it, as torch.empty raises
    PyObject *torch = PyImport_ImportModule("torch");
    PyObject *cls = torch ? PyObject_GetAttrString(torch, "OutOfMemoryError") : nullptr;
    PyErr_SetString(cls ? cls : PyExc_RuntimeError, e.what_without_backtrace());
    Py_XDECREF(cls);
    Py_XDECREF(torch);
    return nullptr;
  } catch (const std::exception &e) {
    PyErr_SetString(PyExc_RuntimeError, e.what());
    return nullptr;
  }
}
// a tensor over part of another one's storage; element offset, sizes and strides in elements of `t`
at::Tensor alias(const at::Tensor &base, at::ScalarType t, int64_t offset, at::IntArrayRef sizes, at::IntArrayRef strides) {
  at::Tensor v = at::detail::make_tensor<c10::TensorImpl>(c10::Storage(base.storage()), base.key_set(),
                                                          caffe2::TypeMeta::fromScalarType(t));
  v.unsafeGetTensorImpl()->set_storage_offset(offset);
  v.unsafeGetTensorImpl()->set_sizes_and_strides(sizes, strides);
  return v;
}
// the type a plain torch.dtype object stands for
inline at::ScalarType dtype_of(PyObject *o) {
  need(THPDtype_Check(o));
  return ((THPDtype *)o)->scalar_type;
}

// ------------------------------------------------------------------ tile choice
// Row block of a ragged or dense problem: the rule of make_opt_flags (matmul_details/opt_flags.py) without constraints;
// a test compares the two.
int choose_block_m(int64_t m, int64_t n_slices, bool ragged, int64_t expected, bool fp8_rows) {
  int64_t rows = m;
  if (ragged) {
    const int64_t mean = m / (n_slices > 1 ? n_slices : 1);
    rows = expected >= 0 ? expected : (mean > 1 ? mean : 1);
  }
  const double cover = ragged ? (double)rows + 2.0 * std::pow((double)rows, 0.5) : (double)rows;
  int bm = cover <= 16 ? 16 : cover <= 32 ? 32 : cover <= 64 ? 64 : 128;
  if (ragged && fp8_rows && bm == 16) bm = 32;
  return bm;
}
// tiles_block_m of the same file; the same test compares the two.
int tiles_block_m(int bm, int64_t m, int64_t n, int64_t k, int64_t n_slices, int64_t expected, bool mxfp4_weights, bool fp8_rows,
                  bool not_streamed) {
  constexpr int64_t cus = 256;
  const int64_t mean = m / (n_slices > 1 ? n_slices : 1), rows = expected >= 0 ? expected : (mean > 1 ? mean : 1);
  const int64_t slices = n_slices < m ? n_slices : m, cols = (n + 255) / 256;
  auto tiles = [&](int64_t b) { return slices * ((rows + b - 1) / b) * cols; };
  const double cover = (double)rows + 2.0 * std::pow((double)rows, 0.5);
  if (bm == 16 && mxfp4_weights && (not_streamed || (tiles(32) > cus * 3 / 4 && k <= 1152))) return 32;
  if (bm == 128 && tiles(128) <= (mxfp4_weights ? cus : cus / 2)) bm = 64;
  if (bm == 64 && tiles(64) <= (mxfp4_weights ? cus * 3 / 4 : cus * 3 / 8)) bm = 32;
  if (bm == 32 && mxfp4_weights && !not_streamed &&
      (fp8_rows ? cover <= 16 && tiles(32) <= cus * 5 / 16 && k >= 640 : cover <= 32 && tiles(32) <= cus / 4))
    bm = 16;
  return bm;
}
int64_t n_blocks(int64_t n_slices, int64_t rows, int64_t block) {  // RaggedTensorMetadata.n_blocks
  if (rows <= n_slices) return rows;
  return n_slices - 1 + (rows - n_slices + 1 + block - 1) / block;
}

// ------------------------------------------------------------------ matmul
// (a, b, bias, a_ragged_metadata, gather_indx, scatter_indx, precision_config, betas, gammas, out_alpha, c,
//  fused_activation, epilogue); the remaining arguments of `matmul` are at their defaults.  A tensor: done; an int: the
//  library's error code; None: not covered.
PyObject *py_matmul(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 13);
    PyObject *a_o = v[0], *b_o = v[1], *bias_o = v[2], *md = v[3], *gather_o = v[4], *scatter_o = v[5], *pc = v[6],
             *betas_o = v[7], *gammas_o = v[8], *alpha_o = v[9], *c_o = v[10], *fa = v[11], *ep = v[12];
    {  // forced flags or constraints of the calling context
      PyObject *q = nullptr;
      need(PyContextVar_Get(ctx_constraints, Py_None, &q) == 0);
      Ref rq(q);
      need(q == Py_None || (PyDict_Check(q) && PyDict_GET_SIZE(q) == 0));
      PyObject *f = nullptr;
      need(PyContextVar_Get(ctx_flags, Py_None, &f) == 0);
      Ref rf(f);
      need(f == Py_None);
    }
    int dev = -1;
    const at::Tensor &a = gpu_tensor(a_o, dev);
    need(a.dim() == 2);
    const at::ScalarType a_type = a.scalar_type();
    const bool a4 = a_type == at::kByte;  // packed e2m1 rows (with block scales)
    const int64_t K = a.size(1) * (a4 ? 2 : 1), a_rows = a.size(0);
    need(a.stride(1) == 1 && a.size(1) > 1);
    tamd_matmul_args g;
    std::memset(&g, 0, sizeof g);
    g.x_dtype = a4 ? TAMD_MXFP4 : type_code(a_type);
    need(g.x_dtype != TAMD_F32);
    const bool a8 = is_fp8_code(g.x_dtype);
    if (a4)  // what the kernel for them reads as it is (_packed_rows_direct; rows of less than a stage, and what is widened, are
             // the general path's)
      need(K >= 256 && a.stride(0) % 16 == 0 && (uintptr_t)a.data_ptr() % 16 == 0);

    // ---- precision options
    bool mx_out = false, a_mx = false;
    at::ScalarType out_type = a_type;
    bool out_type_set = false;
    int rhs_type = -1;
    Ref b_scale_o(pc == Py_None ? (Py_INCREF(Py_None), Py_None) : attr(pc, nm.b_mx_scale));
    if (pc != Py_None) {
      Ref r1(attr(pc, nm.a_mx_tensor_scale)), r2(attr(pc, nm.b_mx_tensor_scale)), r3(attr(pc, nm.acc_scale));
      need(r1.none() && r2.none() && as_double(r3.p) == 1.0);
      Ref od(attr(pc, nm.out_dtype));
      if (!od.none()) out_type = dtype_of(od.p), out_type_set = true;
      Ref ams(attr(pc, nm.a_mx_scale));
      if (!ams.none()) {
        a_mx = true;
        need(g.x_dtype == TAMD_FP8_E4M3 || a4);
        const at::Tensor &s = gpu_tensor(ams.p, dev);
        need(s.scalar_type() == at::kByte && s.dim() == 2 && s.size(0) == a_rows && s.size(1) == K / 32 &&
             (s.stride(1) == 1 || s.size(1) == 1));
        Ref mb(attr(pc, nm.a_microblock_size));
        need(mb.none() || as_int(mb.p) == 32);
        g.x_mx_scale = (const uint8_t *)s.data_ptr();
        g.x_mx_stride_m = s.stride(0);
        if (!out_type_set) out_type = at::kBFloat16;
      }
      Ref cms(attr(pc, nm.c_mx_scale));
      mx_out = !cms.none();
      if (mx_out) {
        Ref pf(attr(pc, nm.c_value_pack_factor)), mb(attr(pc, nm.c_microblock_size));
        need(as_int(pf.p) == 1);
        if (mb.none()) {  // left out: filled in for the caller, as the general path does
          Ref size(PyLong_FromLong(32));
          if (!size.p || PyObject_SetAttr(pc, nm.c_microblock_size, size.p) != 0) {
            PyErr_Clear();
            throw Miss{};
          }
        } else {
          need(as_int(mb.p) == 32);
        }
      }
      Ref fc(attr(pc, nm.flex_ctx));
      Ref lhs(attr(fc.p, nm.lhs_data)), rhs(attr(fc.p, nm.rhs_data)), outd(attr(fc.p, nm.out_data)), accd(attr(fc.p, nm.acc_data));
      Ref ls(attr(lhs.p, nm.scale)), rs(attr(rhs.p, nm.scale)), as(attr(accd.p, nm.scale));
      need(as.none());
      Ref ld(attr(lhs.p, nm.dtype));
      need(ld.none() || (!a8 && !a4) || (a8 && dtype_of(ld.p) == a_type));  // (another 8-bit type: reinterpreted by the general path)
      g.x_scale = scalar_ptr(ls.p, dev);
      g.w_scale = scalar_ptr(rs.p, dev);
      Ref rd(attr(rhs.p, nm.dtype));  // (weights of another 8-bit type: reinterpreted by the general path)
      if (!rd.none()) rhs_type = (int)dtype_of(rd.p);
      Ref es(attr(outd.p, nm.expected_scale)), acs(attr(outd.p, nm.actual_scale)), cks(attr(outd.p, nm.checksum_scale));
      need(cks.none());
      g.y_expected_scale = scalar_ptr(es.p, dev);
      g.y_actual_scale = (float *)scalar_ptr(acs.p, dev);
      Ref si(attr(pc, nm.flexpoint_saturate_inf));
      need(PyBool_Check(si.p));
      g.y_saturate_inf = si.p == Py_True;
    }
    need(!a4 || a_mx);
    // ---- epilogue and activation
    if (ep != Py_None) {
      Ref sp(attr(ep, nm.specs));
      Ref en(attr(sp.p, nm.name));
      need(PyUnicode_Check(en.p));
      const char *s = PyUnicode_AsUTF8(en.p);
      need(s != nullptr);
      if (std::strcmp(s, "dflt") == 0) need(!mx_out);
      else need(mx_out && (std::strcmp(s, "QUANTIZE_MXFP8") == 0 || std::strcmp(s, "quantize_mxfp8") == 0));
    } else {
      need(!mx_out);
    }
    int64_t red_n = 1;
    if (fa != Py_None) {
      Ref sp(attr(fa, nm.specs));
      Ref n(attr(sp.p, nm.name)), rn(attr(sp.p, nm.reduction_n));
      need(PyUnicode_Check(n.p));
      red_n = as_int(rn.p);
      const char *s = PyUnicode_AsUTF8(n.p);
      need(s != nullptr);
      if (std::strcmp(s, "swiglu") == 0) {
        Ref names(attr(sp.p, nm.fn_arg_names)), args(attr(fa, nm.fn_args));
        need(red_n == 2 && PyTuple_Check(names.p) && PyTuple_Check(args.p) && PyTuple_GET_SIZE(names.p) == 2 &&
             PyTuple_GET_SIZE(args.p) == 2);
        need(PyUnicode_Check(PyTuple_GET_ITEM(names.p, 0)) && PyUnicode_Check(PyTuple_GET_ITEM(names.p, 1)) &&
             PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(names.p, 0), "alpha") == 0 &&
             PyUnicode_CompareWithASCIIString(PyTuple_GET_ITEM(names.p, 1), "limit") == 0);
        g.activation = TAMD_ACT_SWIGLU;
        g.act_alpha = (float)as_double(PyTuple_GET_ITEM(args.p, 0));
        PyObject *lim = PyTuple_GET_ITEM(args.p, 1);
        g.act_has_limit = lim != Py_None;
        g.act_limit = lim != Py_None ? (float)as_double(lim) : 0.f;
      } else {
        need(std::strcmp(s, "dflt") == 0 && red_n == 1);
      }
    }
    // ---- weights
    int64_t n_mat, K_W, N;
    bool w_fp4 = false, w_blocks = false;
    if (Py_TYPE(b_o) == (PyTypeObject *)cls_tensor) {
      Ref dt(attr(b_o, nm.dtype)), st(attr(b_o, nm.storage)), sh(attr(b_o, nm.shape));
      need(dt.p == obj_fp4 && PyList_Check(sh.p) && PyList_GET_SIZE(sh.p) == 3);
      Ref lay(attr(st.p, nm.layout)), data(attr(st.p, nm.data));
      need(Py_TYPE(lay.p) == (PyTypeObject *)cls_value_layout && rhs_type < 0);
      n_mat = as_int(PyList_GET_ITEM(sh.p, 0)), K_W = as_int(PyList_GET_ITEM(sh.p, 1)), N = as_int(PyList_GET_ITEM(sh.p, 2));
      const at::Tensor &w = gpu_tensor(data.p, dev);
      need(w.dim() == 3 && w.is_contiguous() && w.scalar_type() == at::kByte && w.size(0) == n_mat &&
           w.size(1) == (N + 63) / 64 && w.size(2) == (K_W + 127) / 128 * 4096);
      g.w = w.data_ptr();
      g.w_layout = TAMD_W_CDNA4_BLOCKS;
      g.w_stride_e = w.stride(0), g.w_stride_k = 1, g.w_stride_n = 0;
      w_fp4 = w_blocks = true;
    } else {
      const at::Tensor &w = gpu_tensor(b_o, dev);
      need((w.dim() == 3 || w.dim() == 2) && w.stride(-2) == 1 && w.size(-2) > 1);
      w_fp4 = w.scalar_type() == at::kByte;
      need(w_fp4 || (w.scalar_type() == a_type && !a4));
      if (a8 && !w_fp4)  // fp8 x fp8: whole, aligned 16-byte chunks along K (otherwise widened by the general path)
        need(!a_mx && K % 16 == 0 && w.stride(-1) % 16 == 0 && (w.dim() == 2 || w.stride(0) % 16 == 0) && a.stride(0) % 16 == 0 &&
             ((uintptr_t)w.data_ptr() | (uintptr_t)a.data_ptr()) % 16 == 0);
      need(rhs_type < 0 || (at::ScalarType)rhs_type == w.scalar_type());
      need(w.stride(-1) != 1);
      n_mat = w.dim() == 3 ? w.size(0) : 1;
      K_W = w.size(-2) * (w_fp4 ? 2 : 1), N = w.size(-1);
      g.w = w.data_ptr();
      g.w_stride_e = w.dim() == 3 ? w.stride(0) : w.size(-2) * w.stride(-2);
      g.w_stride_k = 1, g.w_stride_n = w.stride(-1);
      if (w.dim() == 3 && w.size(0) > 1) need(w.stride(0) != 1);
    }
    need(K == K_W && N > 0 && n_mat > 0);
    g.w_dtype = w_fp4 ? TAMD_MXFP4 : g.x_dtype;
    if (w_fp4) {
      need(!b_scale_o.none());
      Ref mb(attr(pc, nm.b_microblock_size));
      need(!mb.none() && as_int(mb.p) == 32 && K % 32 == 0);
      const int64_t G = K / 32;
      PyObject *s_o = b_scale_o.p;
      Ref data(nullptr);
      bool shuffled = false;
      if (Py_TYPE(s_o) == (PyTypeObject *)cls_tensor) {
        Ref st(attr(s_o, nm.storage)), sh(attr(s_o, nm.shape));
        Ref lay(attr(st.p, nm.layout));
        data.p = attr(st.p, nm.data);
        shuffled = Py_TYPE(lay.p) == (PyTypeObject *)cls_scale_layout;
        if (shuffled) {
          need(PyList_Check(sh.p));
          const Py_ssize_t nd = PyList_GET_SIZE(sh.p);
          need(nd == 2 || nd == 3);
          need((nd == 2 ? 1 : as_int(PyList_GET_ITEM(sh.p, 0))) == n_mat && as_int(PyList_GET_ITEM(sh.p, nd - 2)) == G &&
               as_int(PyList_GET_ITEM(sh.p, nd - 1)) == N);
        }
        s_o = data.p;
      }
      const at::Tensor &s = gpu_tensor(s_o, dev);
      need(s.scalar_type() == at::kByte && s.numel() > 0);
      g.w_mx_scale = (const uint8_t *)s.data_ptr();
      if (shuffled) {
        need(s.dim() == 3 && s.size(0) == n_mat && s.size(1) == (G + 7) / 8 * 8 * 32 && s.size(2) == (N + 31) / 32 &&
             s.stride(1) == 1 && s.stride(2) == s.size(1));
        g.w_mx_layout = TAMD_SCALE_CDNA4;
        g.w_mx_stride_e = s.stride(0);
      } else {
        need((s.dim() == 3 || s.dim() == 2) && s.size(-2) == G && s.size(-1) == N && (s.dim() == 2 ? 1 : s.size(0)) == n_mat);
        g.w_mx_stride_e = s.dim() == 3 ? s.stride(0) : s.size(0) * s.stride(0);
        g.w_mx_stride_k = s.stride(-2), g.w_mx_stride_n = s.stride(-1);
      }
    } else {
      need(b_scale_o.none());
    }
    // ---- rows
    const bool ragged = md != Py_None;
    int64_t M = a_rows;
    auto index = [&](PyObject *o) -> const at::Tensor * {
      if (o == Py_None) return nullptr;
      const at::Tensor &t = gpu_tensor(o, dev);
      need(t.scalar_type() == at::kInt && t.dim() == 1 && t.is_contiguous());
      return &t;
    };
    auto factors = [&](PyObject *o) -> const float * {
      if (o == Py_None) return nullptr;
      const at::Tensor &t = gpu_tensor(o, dev);
      need(t.scalar_type() == at::kFloat && t.is_contiguous());
      return (const float *)t.data_ptr();
    };
    const at::Tensor *gather = index(gather_o), *scatter = index(scatter_o);
    if (gather) M = gather->size(0);
    const int64_t rows_out = scatter ? scatter->size(0) : M;
    need(M > 0 && N % red_n == 0);
    if (bias_o != Py_None) {
      const at::Tensor &bt = gpu_tensor(bias_o, dev);
      need((bt.dim() == 1 || bt.dim() == 2) && bt.stride(-1) == 1 && bt.size(-1) == N);
      g.bias = bt.data_ptr();
      g.bias_dtype = type_code(bt.scalar_type());
      need(!is_fp8_code(g.bias_dtype));
      g.bias_stride_e = bt.dim() == 2 ? bt.stride(0) : N;
    }
    g.betas = factors(betas_o), g.gammas = factors(gammas_o);
    g.out_alpha = alpha_o == Py_None ? 1.0f : (float)as_double(alpha_o);
    int64_t n_slices = 1;
    if (ragged) {
      Ref ss(attr(md, nm.slice_sizes)), so(attr(md, nm.slice_offs)), bo(attr(md, nm.block_offs_data)),
          bs(attr(md, nm.block_schedule_data)), ex(attr(md, nm.expected_slice_size));
      const at::Tensor &tss = gpu_tensor(ss.p, dev), &tso = gpu_tensor(so.p, dev), &tbo = gpu_tensor(bo.p, dev),
                       &tbs = gpu_tensor(bs.p, dev);
      need(tss.dim() == 1 && tss.scalar_type() == at::kInt && tso.scalar_type() == at::kInt && tbo.scalar_type() == at::kInt &&
           tbs.scalar_type() == at::kInt && tbo.dim() == 2 && tbs.dim() == 2 && tbo.size(0) == 5 && tbs.size(0) == 5 &&
           (tbo.stride(1) == 1 || tbo.size(1) == 1) && (tbs.stride(1) == 1 || tbs.size(1) == 1));
      n_slices = tss.size(0);
      need(n_slices > 0 && n_slices <= n_mat && N <= 0x7FFFFFFF && K <= 0x7FFFFFFF && (!g.bias || tensor(bias_o).dim() == 2));
      const int64_t expected = ex.none() ? -1 : as_int(ex.p);
      g.N = (int)N, g.K = (int)K, g.n_experts = (int)n_slices;
      g.block_offs = (const int32_t *)tbo.data_ptr(), g.block_schedule = (const int32_t *)tbs.data_ptr();
      const int bm = tiles_block_m(choose_block_m(M, n_slices, true, expected, (a8 || a4) && w_fp4), M, N, K, n_slices, expected,
                                   w_fp4, a8, mx_out || !tamd::blocks_of_16_stream(g));
      const int row = bm == 16 ? 0 : bm == 32 ? 1 : bm == 64 ? 2 : 3;
      g.slice_sizes = (const int32_t *)tss.data_ptr(), g.slice_offs = (const int32_t *)tso.data_ptr();
      g.block_offs = (const int32_t *)tbo.data_ptr() + row * tbo.stride(0);
      g.block_schedule = (const int32_t *)tbs.data_ptr() + row * tbs.stride(0);
      g.block_m = bm;
      const int64_t gm = n_blocks(n_slices, M, bm);
      need(gm <= tbs.size(1));
      g.grid_m = (int)gm;
    } else {
      need(n_mat == 1);
      // (a long K over few rows is split by the general path)
      need(!a4 || M > 256 || K < 8192);
      need(!(M <= 256 && K >= 8192 && !scatter && !w_blocks && g.w_mx_layout != TAMD_SCALE_CDNA4));
    }
    // ---- output
    const int64_t n_out = N / red_n;
    at::Tensor out;
    PyObject *ret = nullptr;
    if (mx_out) {
      Ref cms(attr(pc, nm.c_mx_scale));
      need(!g.y_expected_scale && !g.y_actual_scale && c_o == Py_None);
      if (!out_type_set) out_type = at::ScalarType::Float8_e4m3fn;
      need(out_type == at::ScalarType::Float8_e4m3fn);
      const at::Tensor &cs = gpu_tensor(cms.p, dev);
      const int64_t groups = (n_out + 31) / 32;
      need(cs.scalar_type() == at::kByte && cs.dim() == 2 && cs.size(0) == rows_out && cs.size(1) == groups &&
           (cs.stride(1) == 1 || groups == 1));
      g.y_mx_scale = (uint8_t *)cs.data_ptr(), g.y_mx_stride_m = cs.stride(0), g.y_mx_stride_z = rows_out * cs.stride(0);
    }
    if (c_o == Py_None) {
      g.y_dtype = type_code(out_type);
      out = new_empty({rows_out, n_out}, out_type, dev);
      g.y_stride_m = n_out, g.y_stride_z = rows_out * n_out;
    } else {
      out = gpu_tensor(c_o, dev);
      need(out.dim() == 2 && out.size(0) == rows_out && out.size(1) == n_out && out.stride(1) == 1);
      g.y_dtype = type_code(out.scalar_type());
      g.y_stride_m = out.stride(0), g.y_stride_z = rows_out * out.stride(0);
    }
    need(M <= 0x7FFFFFFF && N <= 0x7FFFFFFF && K <= 0x7FFFFFFF && n_slices <= 0x7FFFFFFF);
    g.x = a.data_ptr();
    g.x_stride_m = a.stride(0);
    g.x_rows = a_rows;
    g.y = out.data_ptr();
    g.y_rows = rows_out;
    g.M = (int)M, g.N = (int)N, g.K = (int)K, g.n_experts = (int)n_slices;
    g.gather_indx = gather ? (const int32_t *)gather->data_ptr() : nullptr;
    g.scatter_indx = scatter ? (const int32_t *)scatter->data_ptr() : nullptr;
    void *st = stream_of(dev);
    const int rc = without_gil([&] { return abi.matmul(&g, sizeof g, st); });
    if (rc != 0) return PyLong_FromLong(rc);
    if (c_o != Py_None) {
      Py_INCREF(c_o);
      return c_o;
    }
    ret = THPVariable_Wrap(out);
    return ret;
  });
}

// ------------------------------------------------------------------ routing
// (logits, k, layouts): `layouts` is routing._layouts, (rows, experts, k, type code) -> layout of one call's arena; its part
// "native" holds the numbers that follow as 64-bit integers (arena's length, sizes of the tables, byte offset of every part).
// (arena, layout), an error code, or None.  (Checks and the look-up in Python took 0.9 us of the 5 of a call of one launch.)
PyObject *py_routing(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 3 && PyDict_Check(v[2]));
    int dev = -1;
    const at::Tensor &x = gpu_tensor(v[0], dev);
    need(x.dim() == 2 && x.stride(1) == 1);
    const int code = type_code(x.scalar_type());
    const int64_t T = x.size(0), E = x.size(1), k = as_int(v[1]);
    Ref key(Py_BuildValue("LLLi", (long long)T, (long long)E, (long long)k, code));
    if (!key.p) return nullptr;
    PyObject *lay = PyDict_GetItem(v[2], key.p);
    need(lay != nullptr && PyDict_Check(lay));
    const Ref held(Py_NewRef(lay));   // (the launch lets other threads run)
    PyObject *numbers = PyDict_GetItem(lay, nm.native);
    int64_t o[16];
    need(numbers && PyBytes_Check(numbers) && PyBytes_GET_SIZE(numbers) == sizeof o);
    std::memcpy(o, PyBytes_AS_STRING(numbers), sizeof o);
    at::Tensor arena = new_empty({o[0]}, at::kInt, dev);
    uint8_t *b = (uint8_t *)arena.data_ptr();
    void *st = stream_of(dev);
    auto p = [&](int i) { return (int32_t *)(b + o[i]); };
    const int rc = without_gil([&] {
      return abi.routing(x.data_ptr(), code, x.stride(0), (int)T, (int)E, (int)k, p(5), (int16_t *)p(6), (uint32_t *)p(7), 1,
                         o[4], p(8), p(9), p(10), p(11), p(12), p(13), o[2], p(14), o[3], (int)o[1], p(15), st);
    });
    if (rc != 0) return PyLong_FromLong(rc);
    Ref t(THPVariable_Wrap(arena));
    return t.p ? PyTuple_Pack(2, t.p, lay) : nullptr;
  });
}

// (base, numbers): int32 tensors over parts of `base`'s storage, a tuple; five 64-bit integers each: element offset, size0,
// stride0, size1 (-1: one dimension), stride1.
PyObject *py_int_views(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 2 && PyBytes_Check(v[1]));
    const at::Tensor &t = tensor(v[0]);
    constexpr size_t kEach = 5 * sizeof(int64_t);
    const Py_ssize_t n = PyBytes_GET_SIZE(v[1]) / (Py_ssize_t)kEach;
    // (ordinary tensors also under inference mode: who asks for one of them there may write to another, or save it for a backward pass, later)
    const c10::InferenceMode ordinary(false);
    Ref all(PyTuple_New(n));
    if (!all.p) return nullptr;
    for (Py_ssize_t i = 0; i < n; ++i) {
      int64_t o[5];
      std::memcpy(o, PyBytes_AS_STRING(v[1]) + i * kEach, kEach);
      const int64_t sizes[2] = {o[1], o[3]}, strides[2] = {o[2], o[4]};
      const size_t nd = o[3] < 0 ? 1 : 2;
      PyObject *w = THPVariable_Wrap(alias(t, at::kInt, o[0], at::IntArrayRef(sizes, nd), at::IntArrayRef(strides, nd)));
      if (!w) return nullptr;
      PyTuple_SET_ITEM(all.p, i, w);
    }
    return Py_NewRef(all.p);
  });
}

// (base, dtype, element offset, size0, stride0, size1, stride1): a tensor over part of `base`'s storage; size1 < 0: one
// dimension.
PyObject *py_view(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 7);
    const at::Tensor &t = tensor(v[0]);
    const int64_t n1 = as_int(v[5]);
    const int64_t sizes[2] = {as_int(v[3]), n1}, strides[2] = {as_int(v[4]), as_int(v[6])};
    const size_t nd = n1 < 0 ? 1 : 2;
    return THPVariable_Wrap(alias(t, dtype_of(v[1]), as_int(v[2]), at::IntArrayRef(sizes, nd), at::IntArrayRef(strides, nd)));
  });
}

// ------------------------------------------------------------------ reduce
// (x, dim): the plain sum of a 3-D tensor over one axis, in its own type.
PyObject *py_reduce(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 2);
    int dev = -1;
    const at::Tensor &x = gpu_tensor(v[0], dev);
    int64_t dim = as_int(v[1]);
    need(x.dim() == 3 && dim >= -3 && dim < 3);
    if (dim < 0) dim += 3;
    const int code = type_code(x.scalar_type());
    need(!is_fp8_code(code));
    const int d0 = dim == 0 ? 1 : 0, d1 = dim == 2 ? 1 : 2;
    const int64_t S0 = x.size(d0), R = x.size(dim), S1 = x.size(d1);
    need(R < 512 && S0 > 0 && S1 > 0);  // (a longer axis may be cut into chunks by the general path)
    at::Tensor y = new_empty({S0, S1}, x.scalar_type(), dev);
    void *st = stream_of(dev);
    const int rc = without_gil([&] {
      return abi.reduce(x.data_ptr(), code, S0, R, S1, x.stride(d0), x.stride(dim), x.stride(d1), nullptr, 0, 0, 0, nullptr, 0,
                        0, 0, y.data_ptr(), code, S1, 1, st);
    });
    if (rc != 0) return PyLong_FromLong(rc);
    return THPVariable_Wrap(y);
  });
}

// ------------------------------------------------------------------ microscaled conversion
PyObject *pair(const at::Tensor &a, const at::Tensor &b) {
  Ref x(THPVariable_Wrap(a)), y(THPVariable_Wrap(b));
  if (!x.p || !y.p) return nullptr;
  return PyTuple_Pack(2, x.p, y.p);
}

// (x, value dtype: uint8 = packed e2m1, or an fp8 type, axis, rounding mode): contiguous 2-D or 3-D rows quantised along
// the last axis, or (e2m1) along the one before it.  (values, scales), an error code, or None.
PyObject *py_downcast(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 4);
    int dev = -1;
    const at::Tensor &x = gpu_tensor(v[0], dev);
    const at::ScalarType vt = dtype_of(v[1]);
    const bool fp4 = vt == at::kByte;
    const int nd = (int)x.dim();
    int64_t axis = as_int(v[2]);
    need((nd == 2 || nd == 3) && x.is_contiguous() && x.numel() > 0 && axis >= -nd && axis < nd);
    if (axis < 0) axis += nd;
    const int code = type_code(x.scalar_type());
    need(!is_fp8_code(code));
    const int vcode = fp4 ? TAMD_MXFP4 : type_code(vt);
    need(fp4 || is_fp8_code(vcode));
    const int mode = (int)as_int(v[3]);
    const int64_t L = x.size(axis);
    need(L % 32 == 0);
    const int64_t Lv = fp4 ? L / 2 : L, G = L / 32;
    void *st = stream_of(dev);
    int rc;
    at::Tensor val, sc;
    if (axis == nd - 1) {
      const int64_t rows = x.numel() / L;
      if (nd == 2) val = new_empty({rows, Lv}, vt, dev), sc = new_empty({rows, G}, at::kByte, dev);
      else val = new_empty({x.size(0), x.size(1), Lv}, vt, dev), sc = new_empty({x.size(0), x.size(1), G}, at::kByte, dev);
      rc = without_gil([&] {
        return abi.downcast(x.data_ptr(), code, rows, L, 1, L, 1, 0, val.data_ptr(), vcode, Lv, 0, sc.data_ptr(), G, 0, mode, st);
      });
    } else {
      need(fp4 && axis == nd - 2 && x.size(-1) > 1);
      const int64_t nb = nd == 3 ? x.size(0) : 1, nr = x.size(-1);
      // storage with unit stride along the quantised axis
      at::Tensor vs = new_empty({nb, nr, Lv}, vt, dev), ss = new_empty({nb, nr, G}, at::kByte, dev);
      rc = without_gil([&] {
        return abi.downcast(x.data_ptr(), code, nb, L, nr, L * nr, nr, 1, vs.data_ptr(), vcode, Lv * nr, Lv, ss.data_ptr(), G * nr, G,
                            mode, st);
      });
      const int64_t vsz[3] = {nb, Lv, nr}, vst[3] = {Lv * nr, 1, Lv}, ssz[3] = {nb, G, nr}, sst[3] = {G * nr, 1, G};
      const int skip = nd == 3 ? 0 : 1;
      val = alias(vs, vt, 0, at::IntArrayRef(vsz + skip, nd), at::IntArrayRef(vst + skip, nd));
      sc = alias(ss, at::kByte, 0, at::IntArrayRef(ssz + skip, nd), at::IntArrayRef(sst + skip, nd));
    }
    if (rc != 0) return PyLong_FromLong(rc);
    return pair(val, sc);
  });
}

// (values, scales, target dtype, axis): the inverse, for values and scales with unit stride along the axis and dense rows.
PyObject *py_upcast(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 4);
    int dev = -1;
    const at::Tensor &q = gpu_tensor(v[0], dev), &s = gpu_tensor(v[1], dev);
    const at::ScalarType ot = dtype_of(v[2]);
    const int ocode = type_code(ot);
    need(!is_fp8_code(ocode) && s.scalar_type() == at::kByte);
    const bool fp4 = q.scalar_type() == at::kByte;
    const int vcode = fp4 ? TAMD_MXFP4 : type_code(q.scalar_type());
    need(fp4 || is_fp8_code(vcode));
    const int nd = (int)q.dim();
    int64_t axis = as_int(v[3]);
    need((nd == 2 || nd == 3) && s.dim() == nd && q.numel() > 0 && axis >= -nd && axis < nd);
    if (axis < 0) axis += nd;
    const int64_t Lv = q.size(axis), L = fp4 ? 2 * Lv : Lv, G = L / 32;
    need(L % 32 == 0);
    for (int d = 0; d < nd; ++d) need(s.size(d) == (d == axis ? G : q.size(d)));
    void *st = stream_of(dev);
    if (axis == nd - 1) {
      need(q.is_contiguous() && s.is_contiguous());
      const int64_t rows = q.numel() / Lv;
      at::Tensor out = nd == 2 ? new_empty({rows, L}, ot, dev) : new_empty({q.size(0), q.size(1), L}, ot, dev);
      const int rc = without_gil([&] {
        return abi.upcast(q.data_ptr(), vcode, Lv, 0, s.data_ptr(), G, 0, out.data_ptr(), ocode, rows, L, 1, L, 1, 0, st);
      });
      if (rc != 0) return PyLong_FromLong(rc);
      return THPVariable_Wrap(out);
    }
    need(fp4 && axis == nd - 2 && q.size(-1) > 1);
    const int64_t nb = nd == 3 ? q.size(0) : 1, nr = q.size(-1);
    need(q.stride(-2) == 1 && q.stride(-1) == Lv && s.stride(-2) == 1 && s.stride(-1) == G);
    need(nb == 1 || (q.stride(0) == Lv * nr && s.stride(0) == G * nr));
    at::Tensor out = nd == 2 ? new_empty({L, nr}, ot, dev) : new_empty({nb, L, nr}, ot, dev);
    const int rc = without_gil([&] {
      return abi.upcast(q.data_ptr(), vcode, Lv * nr, Lv, s.data_ptr(), G * nr, G, out.data_ptr(), ocode, nb, L, nr, L * nr, nr, 1, st);
    });
    if (rc != 0) return PyLong_FromLong(rc);
    return THPVariable_Wrap(out);
  });
}

// ------------------------------------------------------------------ module
PyObject *py_choose_block_m(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 5 || nargs == 9);
    const int bm = choose_block_m(as_int(v[0]), as_int(v[1]), v[2] == Py_True, as_int(v[3]), v[4] == Py_True);
    if (nargs == 5) return PyLong_FromLong(bm);
    return PyLong_FromLong(tiles_block_m(bm, as_int(v[0]), as_int(v[5]), as_int(v[6]), as_int(v[1]), as_int(v[3]), v[7] == Py_True,
                                             v[4] == Py_True, v[8] == Py_True));
  });
}

// (address of a tamd_matmul_args): whether its row blocks of 16 would take the streaming kernel.
PyObject *py_blocks_of_16_stream(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 1);
    tamd_matmul_args a;
    std::memcpy(&a, (const void *)(intptr_t)as_int(v[0]), sizeof a);
    return PyBool_FromLong(tamd::blocks_of_16_stream(a));
  });
}

// (address of a tamd_matmul_args, compute units): the row block of a dense product.
PyObject *py_dense_block_m(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 2);
    tamd_matmul_args a;
    std::memcpy(&a, (const void *)(intptr_t)as_int(v[0]), sizeof a);
    return PyLong_FromLong(tamd::dense_block_m(a, (int)as_int(v[1])));
  });
}

// (address of a tamd_matmul_args, compute units): the row block of the persistent kernel for few rows per slice, or 0.
PyObject *py_ring_rows(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 2);
    tamd_matmul_args a;
    std::memcpy(&a, (const void *)(intptr_t)as_int(v[0]), sizeof a);
    return PyLong_FromLong(a.w_dtype == TAMD_MXFP4 ? tamd::ring_rows(a, (int)as_int(v[1])) : tamd::kk_ring_rows(a, (int)as_int(v[1])));
  });
}

// (rows, experts, picks per row): rows to a workgroup of the routing's two launches, 0 where others take them.
PyObject *py_routing_block_rows(PyObject *, PyObject *const *v, Py_ssize_t nargs) {
  return covered([&]() -> PyObject * {
    need(nargs == 3);
    const int64_t T = as_int(v[0]), E = as_int(v[1]), k = as_int(v[2]);
    need(E >= 1 && k >= 1 && k <= 64 && k <= E && E <= 1 << 20);
    tamd::RowPlan p;
    return PyLong_FromLong(tamd::make_row_plan(T, (int)E, (int)k, tamd::lanes_per_row((int)E, (int)k), INT64_MAX, p) ? p.RB : 0);
  });
}

// (addresses of the C ABI functions by name, Tensor, CDNA4MXValueLayout, CDNA4MXScaleLayout, FP4, constraints ContextVar,
//  flags ContextVar)
PyObject *py_init(PyObject *, PyObject *args) {
  PyObject *addr;
  if (!PyArg_ParseTuple(args, "O!OOOOOO", &PyDict_Type, &addr, &cls_tensor, &cls_value_layout, &cls_scale_layout, &obj_fp4,
                        &ctx_constraints, &ctx_flags))
    return nullptr;
  for (PyObject *o : {cls_tensor, cls_value_layout, cls_scale_layout, obj_fp4, ctx_constraints, ctx_flags}) Py_INCREF(o);
  auto take = [&](const char *name, void *slot) {
    PyObject *o = PyDict_GetItemString(addr, name);
    void *p = o ? PyLong_AsVoidPtr(o) : nullptr;
    std::memcpy(slot, &p, sizeof p);
    return p != nullptr;
  };
  if (!take("tamd_matmul_sized", &abi.matmul) || !take("tamd_routing_gates", &abi.routing) || !take("tamd_reduce", &abi.reduce) ||
      !take("tamd_downcast_mxfp", &abi.downcast) || !take("tamd_upcast_mxfp", &abi.upcast)) {
    PyErr_SetString(PyExc_RuntimeError, "an entry point of the library is missing");
    return nullptr;
  }
#define TAMD_NAME(n) nm.n = PyUnicode_InternFromString(#n)
  TAMD_NAME(storage), TAMD_NAME(data), TAMD_NAME(layout), TAMD_NAME(dtype), TAMD_NAME(shape), TAMD_NAME(c_mx_scale),
      TAMD_NAME(c_microblock_size), TAMD_NAME(c_value_pack_factor), TAMD_NAME(a_mx_tensor_scale), TAMD_NAME(b_mx_tensor_scale),
      TAMD_NAME(acc_scale), TAMD_NAME(a_mx_scale), TAMD_NAME(a_microblock_size), TAMD_NAME(b_mx_scale),
      TAMD_NAME(b_microblock_size), TAMD_NAME(flex_ctx), TAMD_NAME(lhs_data), TAMD_NAME(rhs_data), TAMD_NAME(out_data),
      TAMD_NAME(acc_data), TAMD_NAME(scale), TAMD_NAME(expected_scale), TAMD_NAME(actual_scale), TAMD_NAME(checksum_scale),
      TAMD_NAME(out_dtype), TAMD_NAME(flexpoint_saturate_inf), TAMD_NAME(specs), TAMD_NAME(name), TAMD_NAME(fn_arg_names),
      TAMD_NAME(fn_args), TAMD_NAME(reduction_n), TAMD_NAME(slice_sizes), TAMD_NAME(slice_offs), TAMD_NAME(block_offs_data),
      TAMD_NAME(block_schedule_data), TAMD_NAME(expected_slice_size), TAMD_NAME(native);
#undef TAMD_NAME
  Py_RETURN_NONE;
}

#define TAMD_FAST(f) (PyCFunction)(void (*)(void)) f, METH_FASTCALL, nullptr
PyMethodDef methods[] = {{"init", py_init, METH_VARARGS, nullptr},
                         {"matmul", TAMD_FAST(py_matmul)},
                         {"routing", TAMD_FAST(py_routing)},
                         {"view", TAMD_FAST(py_view)},
                         {"int_views", TAMD_FAST(py_int_views)},
                         {"routing_block_rows", TAMD_FAST(py_routing_block_rows)},
                         {"reduce", TAMD_FAST(py_reduce)},
                         {"downcast", TAMD_FAST(py_downcast)},
                         {"upcast", TAMD_FAST(py_upcast)},
                         {"choose_block_m", TAMD_FAST(py_choose_block_m)},
                         {"blocks_of_16_stream", TAMD_FAST(py_blocks_of_16_stream)},
                         {"dense_block_m", TAMD_FAST(py_dense_block_m)},
                         {"ring_rows", TAMD_FAST(py_ring_rows)},
                         {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

// `built_for`: the torch whose headers and libraries this file was compiled against; the loader compares it before anything
// here touches a tensor
PyMODINIT_FUNC PyInit__host() {
  PyObject *m = PyModule_Create(&module);
  if (m && PyModule_AddStringConstant(m, "built_for", TAMD_TORCH_VERSION) != 0) Py_CLEAR(m);
  return m;
}
