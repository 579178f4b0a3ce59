// host_layer.cpp — a whole decoder layer as a CPython extension (triton_int_amd._layer_host).
//
// The seven to eight launches of W8A8OPTDecoderLayer.forward cost 60 us of Python (module calls, attribute
// look-ups, views, one allocation per step) where their kernels on a 1024-wide layer take 30.  This is the same
// sequence of C ABI calls on the modules' buffers as they are now: nothing is kept from one call for the next.
// Intermediates share one allocation.  Anything that Python would notice (hooks, another module type, a method replaced on
// an instance or on a class, a launcher replaced in the module that calls it) or that the plain sequence does not cover is
// declined, as is a status from the library: the steps before it have written nothing that the Python path, which then
// runs them all, does not write again.
#include "host_common.h"

namespace {

PyObject* key(const char* name) { return PyUnicode_InternFromString(name); }
struct Names {
  PyObject *modules = key("_modules"), *buffers = key("_buffers"), *weight = key("weight"), *bias = key("bias"), *a = key("a"), *b = key("b"),
           *eps = key("eps"), *input_scale = key("input_scale"), *qkv = key("_qkv"), *hidden = key("hidden"), *heads = key("heads"),
           *causal = key("causal"), *qk_alpha = key("qk_alpha"), *score_scale = key("score_scale"), *pv_alpha = key("pv_alpha"),
           *fused_attention = key("fused_attention"), *min_queries = key("fused_attention_min_queries"), *fused_residual = key("fused_residual");
  PyObject* replaced[5] = {key("forward"), key("_launch"), key("forward_add"), key("_call_impl"), key("_compiled_call_impl")};
  PyObject* hooks[4] = {key("_forward_hooks"), key("_forward_pre_hooks"), key("_backward_hooks"), key("_backward_pre_hooks")};
  PyObject* layer_methods[7] = {key("forward"), key("_forward_steps"), key("_qkv_pack"), key("_heads"), key("_append"), key("_at_once"), key("_kernel_takes")};
  PyObject* steps[8] = {key("ln1"), key("q_proj"), key("k_proj"), key("v_proj"), key("out_proj"), key("ln2"), key("fc1"), key("fc2")};
};
const Names& names() {
  static const Names n;  // created under the interpreter's lock
  return n;
}

// the instance dictionary (borrowed: the object keeps it)
PyObject* dict_of(PyObject* o) {
  PyObject** d = _PyObject_GetDictPtr(o);
  need(d && *d);
  return *d;
}

PyObject* item(PyObject* dict, PyObject* name) {
  PyObject* v = PyDict_GetItem(dict, name);
  need(v != nullptr);
  return v;
}

bool none_of(PyObject* dict, PyObject* const* names_, int n) {
  for (int i = 0; i < n; ++i)
    if (PyDict_GetItem(dict, names_[i])) return false;
  return true;
}

// A submodule of exactly the given type that nobody has hooked into: its instance dictionary
PyObject* step(PyObject* modules, int i, PyObject* type) {
  PyObject* m = item(modules, names().steps[i]);
  need((PyObject*)Py_TYPE(m) == type);
  PyObject* d = dict_of(m);
  need(none_of(d, names().replaced, 5));
  for (PyObject* h : names().hooks) {
    PyObject* hooks = item(d, h);
    need(PyDict_Check(hooks) && PyDict_Size(hooks) == 0);
  }
  return d;
}

// The tensors that a call reads, held until it returns: another thread may replace a module's buffer, or what a tensor object
// holds, while this one launches without the interpreter's lock.  The references stay valid: nothing moves within the
// inline storage.
struct Held {
  c10::SmallVector<Tensor, 40> all;
  const Tensor& tensor(PyObject* o, int dev, ScalarType type) {
    need(all.size() < 40);
    all.push_back(::tensor(o, dev, type));
    return all.back();
  }
  const void* vector(PyObject* o, int dev, ScalarType type, int64_t n) {
    const void* at = ::vector(o, dev, type, n);
    if (at) tensor(o, dev, type);
    return at;
  }
};

// the buffers of an int8 linear [N, K]
struct Linear {
  const int8_t* w;
  const void* bias;
  const float *a = nullptr, *b = nullptr;
  int64_t N, ldw;
  Linear(Held& held, PyObject* dict, int dev, int64_t K, ScalarType bias_type, bool scales) {
    PyObject* buffers = item(dict, names().buffers);
    need(PyDict_Check(buffers));
    const Tensor& wt = held.tensor(item(buffers, names().weight), dev, ScalarType::Char);
    need(wt.dim() == 2 && wt.size(1) == K && wt.stride(1) == 1);
    N = wt.size(0), ldw = wt.stride(0), w = (const int8_t*)ptr(wt);
    bias = held.vector(item(buffers, names().bias), dev, bias_type, N);
    need(bias);
    if (!scales) return;
    for (int i = 0; i < 2; ++i) {
      const Tensor& t = held.tensor(item(buffers, i ? names().b : names().a), dev, ScalarType::Float);
      need(t.numel() == 1);
      (i ? b : a) = (const float*)ptr(t);
    }
  }
};

struct Norm {
  const float *g, *b;
  float eps;
  Norm(Held& held, PyObject* dict, int dev, int64_t H) {
    PyObject* buffers = item(dict, names().buffers);
    need(PyDict_Check(buffers));
    g = (const float*)held.vector(item(buffers, names().weight), dev, ScalarType::Float, H);
    b = (const float*)held.vector(item(buffers, names().bias), dev, ScalarType::Float, H);
    need(g != nullptr);
    eps = (float)number(item(dict, names().eps));
  }
};

// What the Python steps look up in classes and modules while they run, as (class or module dictionary, name, what was found
// there when the package was loaded): nobody has replaced any of it.  The 41 look-ups cost 0.3 us of
// the call's 21.
void unchanged(PyObject* found) {
  need(PyTuple_Check(found));
  for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(found); ++i) {
    PyObject* e = PyTuple_GET_ITEM(found, i);
    need(PyTuple_Check(e) && PyTuple_GET_SIZE(e) == 3);
    PyObject *where = PyTuple_GET_ITEM(e, 0), *name = PyTuple_GET_ITEM(e, 1);
    need(PyDict_Check(where) || PyType_Check(where));
    need((PyDict_Check(where) ? PyDict_GetItem(where, name) : _PyType_Lookup((PyTypeObject*)where, name)) == PyTuple_GET_ITEM(e, 2));
  }
}

// decoder_layer(layer, hidden, kv_cache, types, global_hooks): W8A8OPTDecoderLayer.forward without trace and marks.  types: of the layer
// and of its eight steps, then what unchanged() takes; global_hooks: torch's dictionaries of hooks on every module.
PyObject* decoder_layer(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 5, [&]() -> PyObject* {
    const Names& nm = names();
    need(PyTuple_Check(v[3]) && PyTuple_GET_SIZE(v[3]) == 10 && PyTuple_Check(v[4]));
    need((PyObject*)Py_TYPE(v[0]) == PyTuple_GET_ITEM(v[3], 0));
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(v[4]); ++i) need(PyDict_Check(PyTuple_GET_ITEM(v[4], i)) && PyDict_Size(PyTuple_GET_ITEM(v[4], i)) == 0);
    PyObject* self = dict_of(v[0]);
    need(none_of(self, nm.layer_methods, 7));
    unchanged(PyTuple_GET_ITEM(v[3], 9));
    need(flag(item(self, nm.fused_attention)) && flag(item(self, nm.fused_residual)));
    PyObject* modules = item(self, nm.modules);
    need(PyDict_Check(modules));
    PyObject* d[8];
    for (int i = 0; i < 8; ++i) d[i] = step(modules, i, PyTuple_GET_ITEM(v[3], i + 1));

    Held held;
    const Tensor& x = held.tensor(v[1], -1, ScalarType::Float);
    const Call c(x);
    need(x.dim() == 3 && x.numel() > 0);
    const int64_t B = x.size(0), S = x.size(1), H = x.size(2), M = B * S, x_rs = row_pitch(x);
    const int64_t heads = integer(item(self, nm.heads)), D = 128;
    need(integer(item(self, nm.hidden)) == H && heads > 0 && heads * D == H && B * heads <= 32767);
    const int M32 = int32_size(M), S32 = int32_size(S), B32 = (int)B, H32 = int32_size(H);
    int32_size(3 * H);

    const Norm ln1(held, d[0], c.dev, H), ln2(held, d[5], c.dev, H);
    // the projections' buffers have to be slices of the pack, whose rows are contiguous
    PyObject* pack = item(self, nm.qkv);
    need(PyTuple_Check(pack) && PyTuple_GET_SIZE(pack) == 4);
    const Tensor& w3 = held.tensor(PyTuple_GET_ITEM(pack, 0), c.dev, ScalarType::Char);
    need(w3.dim() == 2 && w3.size(0) == 3 * H && w3.size(1) == H && w3.is_contiguous());
    const int8_t* b3 = (const int8_t*)held.vector(PyTuple_GET_ITEM(pack, 1), c.dev, ScalarType::Char, 3 * H);
    const float *a3 = (const float*)held.vector(PyTuple_GET_ITEM(pack, 2), c.dev, ScalarType::Float, 3),
                *s3 = (const float*)held.vector(PyTuple_GET_ITEM(pack, 3), c.dev, ScalarType::Float, 3);
    need(b3 && a3 && s3);
    for (int i = 0; i < 3; ++i) {
      const Linear p(held, d[1 + i], c.dev, H, ScalarType::Char, true);
      need(p.N == H && p.ldw == H && p.w == (const int8_t*)ptr(w3) + i * H * H && p.bias == b3 + i * H && p.a == a3 + i && p.b == s3 + i);
    }
    const Linear out_proj(held, d[4], c.dev, H, ScalarType::Int, false), fc1(held, d[6], c.dev, H, ScalarType::Float, true),
        fc2(held, d[7], c.dev, fc1.N, ScalarType::Float, true);
    need(out_proj.N == H && fc2.N == H);
    const int F32 = int32_size(fc1.N);

    const float in_scale = (float)number(item(d[5], nm.input_scale)), qk_alpha = (float)number(item(self, nm.qk_alpha)),
                score_scale = (float)number(item(self, nm.score_scale)), pv_alpha = (float)number(item(self, nm.pv_alpha));
    const int causal = flag(item(self, nm.causal)) ? S32 : 0;
    const int64_t min_queries = integer(item(self, nm.min_queries));
    need(score_scale > 0.0f);

    // keys and values: a cache, or this call's own
    const bool cached = v[2] != Py_None;
    int64_t T = S;
    const int8_t *k = nullptr, *vt = nullptr;
    int64_t k_ss = S * 3 * H, k_hs = D, k_rs = 3 * H, vt_rs = (S + 15) / 16 * 16, vt_hs = D * vt_rs;
    int8_t *k_dst = nullptr, *vt_dst = nullptr;
    int64_t dst_hs = 0, dst_rs = 0;
    if (cached) {
      need(PyTuple_Check(v[2]) && PyTuple_GET_SIZE(v[2]) == 2);
      const Caches kv(PyTuple_GET_ITEM(v[2], 0), PyTuple_GET_ITEM(v[2], 1), c.dev, S);
      need(kv.k && kv.BH == B * heads && kv.D == D);
      T = kv.T;
      k_dst = kv.k, vt_dst = kv.vt, dst_hs = kv.k_hs, dst_rs = kv.k_rs, vt_rs = kv.vt_rs;
      k = kv.k - (T - S) * kv.k_rs, vt = kv.vt - (T - S);
      k_hs = kv.k_hs, k_rs = kv.k_rs, k_ss = heads * k_hs;
      held.tensor(PyTuple_GET_ITEM(v[2], 0), c.dev, ScalarType::Char);
      vt_hs = held.tensor(PyTuple_GET_ITEM(v[2], 1), c.dev, ScalarType::Char).stride(0);
      need(k_rs >= D && (((int64_t)k | k_hs | k_rs) & 15) == 0 && vt_rs >= T);
    }
    need(S >= min_queries || T <= 4096);
    const int T32 = int32_size(T);

    const bool few = M <= 4 && H >= 1024 && (x_rs & 3) == 0 && (((uintptr_t)ptr(x) | (uintptr_t)ln1.g | (uintptr_t)ln1.b | (uintptr_t)ln2.g |
                                                                              (uintptr_t)ln2.b) & 15) == 0;  // the norms go into the launches after them
    int rc = TI_OK;
    Tensor out;
    {
      const NoGil unlocked;
      const auto up = [](int64_t bytes) { return (bytes + 511) & ~(int64_t)511; };
      const int64_t sizes[8] = {up(M * H), up(3 * M * H), up(M * H), up(4 * M * H), up(4 * M * H), up(M * H), up(M * fc1.N), cached ? 0 : up(B * heads * vt_hs)};
      int64_t total = 0, at[8];
      for (int i = 0; i < 8; ++i) at[i] = total, total += sizes[i];
      const Tensor scratch = c.empty({total}, ScalarType::Byte);
      out = c.empty(x.sizes(), ScalarType::Float);
      char* base = (char*)mptr(scratch);
      int8_t *h8 = (int8_t*)base + at[0], *qkv = (int8_t*)base + at[1], *ctx = (int8_t*)base + at[2], *h8b = (int8_t*)base + at[5], *f8 = (int8_t*)base + at[6];
      int32_t* acc = (int32_t*)(base + at[3]);
      float* resid = (float*)(base + at[4]);
      const float* xp = (const float*)ptr(x);
      const int next_reads = 0xff | TI_CONFIG_NEXT_READS;
      const auto run = [&]() {
        bool appended = false;
        if (few && cached) {
          rc = ti_layernorm_qkv_decode_i8_seqs(xp, x_rs, ln1.g, ln1.b, ln1.eps, (const int8_t*)ptr(w3), H, b3, a3, s3, qkv, 3 * H, B32, M32, H32, H32, k_dst, dst_hs,
                                               dst_rs, vt_dst, vt_rs, (int)D, c.stream);
          if (rc && rc != TI_E_COMBO) return;
          appended = rc == TI_OK;
        }
        if (!appended && (rc = ti_layernorm_q(xp, x_rs, ln1.g, ln1.b, ln1.eps, h8, H, M32, H32, 0, TI_ROUND_RNE_CLAMP, nullptr, nullptr, c.stream))) return;
        int8_t* const vd = cached ? vt_dst : (int8_t*)base + at[7];
        if (!appended && M <= 64 && H >= 1024 && ((((int64_t)k_dst | dst_hs | dst_rs) & 3) == 0)) {
          rc = ti_qkv_append_i8_seqs(h8, H, (const int8_t*)ptr(w3), H, b3, a3, s3, qkv, 3 * H, B32, M32, H32, H32, k_dst, dst_hs, dst_rs, vd, vt_rs, (int)D, c.stream);
          if (rc && rc != TI_E_COMBO) return;
          appended = rc == TI_OK;
        }
        if (!appended) {
          if ((rc = ti_bmm_i8_grouped(h8, 0, H, 1, (const int8_t*)ptr(w3), H * H, H, 1, qkv, H, 3 * H, 1, 3, M32, H32, H32, b3, TI_BIAS_I8, H, a3, s3, 1,
                                      TI_EPI_SCALE_I8, TI_I8, TI_ROUND_RNE_CLAMP, next_reads, c.stream))) return;
          if ((rc = ti_kv_append_i8_seqs(cached ? qkv + H : nullptr, cached ? 3 * H : 0, qkv + 2 * H, 3 * H, k_dst, dst_hs, dst_rs, vd, vt_rs, B32, S32,
                                         (int)heads, (int)D, c.stream))) return;
        }
        if ((rc = ti_attention_i8_heads(qkv, S * 3 * H, D, 3 * H, cached ? k : qkv + H, k_ss, k_hs, k_rs, cached ? vt : (int8_t*)base + at[7], heads * vt_hs, vt_hs,
                                        vt_rs, ctx, S * H, D, H, B32, (int)heads, S32, T32, (int)D, qk_alpha, score_scale, pv_alpha, causal, c.stream))) return;
        if ((rc = ti_bmm_i8_config(ctx, 0, H, 1, out_proj.w, 0, out_proj.ldw, 1, acc, 0, H, 1, 1, M32, H32, H32, out_proj.bias, TI_BIAS_I32, nullptr, nullptr,
                                   TI_EPI_I32, TI_I32, TI_ROUND_RNE_CLAMP, -1, c.stream))) return;
        rc = few ? ti_dq_add_layernorm_linear_gelu_i8(acc, H, in_scale, xp, x_rs, ln2.g, ln2.b, ln2.eps, resid, H, fc1.w, fc1.ldw, (const float*)fc1.bias, fc1.a, fc1.b,
                                                      f8, fc1.N, M32, F32, H32, c.stream)
                 : TI_E_COMBO;
        if (rc && rc != TI_E_COMBO) return;
        if (rc) {
          if ((rc = ti_dq_add_layernorm_q(acc, H, in_scale, nullptr, xp, x_rs, ln2.g, ln2.b, ln2.eps, resid, H, h8b, H, nullptr, H, M32, H32, TI_ROUND_RNE_CLAMP,
                                          nullptr, nullptr, c.stream))) return;
          if ((rc = ti_bmm_i8_config(h8b, 0, H, 1, fc1.w, 0, fc1.ldw, 1, f8, 0, fc1.N, 1, 1, M32, F32, H32, fc1.bias, TI_BIAS_F32, fc1.a, fc1.b, TI_EPI_GELU_I8, TI_I8,
                                     TI_ROUND_RNE_CLAMP, next_reads, c.stream))) return;
        }
        rc = ti_linear_i8_residual_f32(f8, fc1.N, fc2.w, fc2.ldw, (const float*)fc2.bias, fc2.a, fc2.b, resid, H, (float*)mptr(out), H, M32, H32, F32, c.stream);
      };
      run();
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

PyMethodDef methods[] = {{"decoder_layer", (PyCFunction)(void (*)(void))decoder_layer, METH_FASTCALL, nullptr}, {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_layer_host", "A decoder layer's host path (see csrc/host_layer.cpp).", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__layer_host() { return PyModule_Create(&module); }
