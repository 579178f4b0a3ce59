// host.cpp — the launchers' host path as a CPython extension (triton_int_amd._host).
//
// A launch of libtriton_int_hip.so through ctypes costs about as much again as the launch itself, and the
// argument checks, views and allocations around it in Python three times as much: 15.9 us for a 512 x 768 x 768
// linear module whose kernel runs 5 us.  These functions take the tensors as they are, check what the Python
// launchers check, allocate the output and call the C ABI.
//
// Every function returns None, having done nothing, when an argument is anything but the ordinary case (a
// tensor subclass, another device than the current one, a layout that needs a copy, a python-float scale, a
// wrong dtype or size, a status from the library, an exception from torch, e.g. out of memory).  The Python
// launcher then takes its own path, which converts or raises: there is one definition of every conversion and
// every error, its type included.
//
// The allocations and the C ABI call run without the interpreter's lock (NoGil), as a ctypes call does: a launch can
// wait (a full hardware queue, a kernel's first launch, a workspace that grows), and other Python threads, host
// callbacks of the stream among them, go on meanwhile.  So every argument is read before.
#include "host_common.h"

namespace {

// linear(a, w, bias, alpha, beta, out, epilogue, out_dtype, round_mode, config, groups): kernels/_gemm.py linear and,
// with groups > 0, linear_group
PyObject* linear(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 11, [&]() -> PyObject* {
    const Tensor& a = tensor(v[0], -1, ScalarType::Char);
    const Call c(a);
    const Tensor& w = tensor(v[1], c.dev, ScalarType::Char);
    need(w.dim() == 2);
    const int64_t groups = integer(v[10]), N = w.size(0), per = groups ? N / groups : N;
    need(!groups || N % groups == 0);
    const int N32 = int32_size(N), per32 = int32_size(per);
    const Rows r(a, w.size(1));
    int bk = TI_BIAS_NONE;
    const void* bias = nullptr;
    if (v[2] != Py_None) {
      const Tensor& b = tensor(v[2], c.dev);
      bk = bias_kind(b.scalar_type());
      need(b.numel() == N && b.is_contiguous());
      bias = ptr(b);
    }
    const float *alpha = scale(v[3], c.dev), *beta = scale(v[4], c.dev);
    const int epilogue = (int)integer(v[6]), dt = (int)integer(v[7]), round_mode = (int)integer(v[8]), config = (int)integer(v[9]);
    const ScalarType type = out_type(dt);
    const auto sizes = with_last(a, N);
    Tensor out;
    if (v[5] != Py_None) {
      const Tensor& o = tensor(v[5], c.dev, type);
      need(o.numel() == (int64_t)r.M * N && o.is_contiguous());
      out = o.view(sizes);
    }
    if (groups) {
      for (int i = 3; i < 5; ++i)
        if (v[i] != Py_None) need(THPVariable_Unpack(v[i]).numel() == groups && THPVariable_Unpack(v[i]).is_contiguous());
    }
    int rc;
    {
      const NoGil unlocked;
      if (!out.defined()) out = c.empty(sizes, type);
      if (groups) {
        rc = ti_bmm_i8_grouped((const int8_t*)ptr(a), 0, r.pitch, 1, (const int8_t*)ptr(w), per * w.stride(0), w.stride(0), w.stride(1),
                               mptr(out), per, N, 1, (int)groups, r.M, per32, r.K, bias, bk, per, alpha, beta, 1, epilogue, dt, round_mode,
                               config, c.stream);
      } else {
        rc = ti_bmm_i8_config((const int8_t*)ptr(a), 0, r.pitch, 1, (const int8_t*)ptr(w), 0, w.stride(0), w.stride(1), mptr(out), 0, N, 1, 1,
                              r.M, N32, r.K, bias, bk, alpha, beta, epilogue, dt, round_mode, config, c.stream);
      }
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

// bmm(a, b, b_is_kn, alpha, out, epilogue, out_dtype, round_mode, config): kernels/_gemm.py bmm
PyObject* bmm(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 9, [&]() -> PyObject* {
    const Tensor& a = tensor(v[0], -1, ScalarType::Char);
    const Call c(a);
    const Tensor& b = tensor(v[1], c.dev, ScalarType::Char);
    need(a.dim() == 3 && b.dim() == 3 && a.size(0) == b.size(0));
    const bool kn = flag(v[2]);  // b is [B, K, N]
    need(a.size(2) == b.size(kn ? 1 : 2));
    const int64_t B = a.size(0), M = a.size(1), K = a.size(2), N = b.size(kn ? 2 : 1);
    const int B32 = int32_size(B), M32 = int32_size(M), N32 = int32_size(N), K32 = int32_size(K);
    const int epilogue = (int)integer(v[5]), dt = (int)integer(v[6]), round_mode = (int)integer(v[7]), config = (int)integer(v[8]);
    const float* alpha = scale(v[3], c.dev);
    const ScalarType type = out_type(dt);
    Tensor out;
    if (v[4] != Py_None) {
      out = tensor(v[4], c.dev, type);
      need(out.dim() == 3 && out.size(0) == B && out.size(1) == M && out.size(2) == N);
    }
    int rc;
    {
      const NoGil unlocked;
      if (!out.defined()) out = c.empty({B, M, N}, type);
      rc = ti_bmm_i8_config((const int8_t*)ptr(a), a.stride(0), a.stride(1), a.stride(2), (const int8_t*)ptr(b), b.stride(0),
                            b.stride(kn ? 2 : 1), b.stride(kn ? 1 : 2), mptr(out), out.stride(0), out.stride(1), out.stride(2), B32, M32, N32, K32,
                            nullptr, TI_BIAS_NONE, alpha, nullptr, epilogue, dt, round_mode, config, c.stream);
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

// linear_residual(a, w, bias, alpha, beta, residual): linear_a8_w8_bfp32_ofp32_residual without `out`
PyObject* linear_residual(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 6, [&]() -> PyObject* {
    const Tensor& a = tensor(v[0], -1, ScalarType::Char);
    const Call c(a);
    const Tensor& w = tensor(v[1], c.dev, ScalarType::Char);
    need(w.dim() == 2 && w.stride(1) == 1);
    const int64_t N = w.size(0);
    const Rows r(a, w.size(1));
    const float *bias = (const float*)vector(v[2], c.dev, ScalarType::Float, N), *alpha = scale(v[3], c.dev), *beta = scale(v[4], c.dev);
    need(alpha && beta);
    const Tensor& res = tensor(v[5], c.dev, ScalarType::Float);
    need(res.numel() == (int64_t)r.M * N && (res.is_contiguous() || res.size(-1) == N));
    const int64_t res_pitch = res.is_contiguous() ? N : row_pitch(res);
    const int N32 = int32_size(N);
    Tensor out;
    int rc;
    {
      const NoGil unlocked;
      out = c.empty(with_last(a, N), ScalarType::Float);
      rc = ti_linear_i8_residual_f32((const int8_t*)ptr(a), r.pitch, (const int8_t*)ptr(w), w.stride(0), bias, alpha, beta, (const float*)ptr(res), res_pitch,
                                     (float*)mptr(out), N, r.M, N32, r.K, c.stream);
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

// layernorm_q(x, weight, bias, eps, rms, round_mode)
PyObject* layernorm_q(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 6, [&]() -> PyObject* {
    const Tensor& x = tensor(v[0], -1, ScalarType::Float);
    const Call c(x);
    need(x.dim() >= 1 && x.size(-1) > 0);
    const int64_t N = x.size(-1), pitch = row_pitch(x);
    const float *g = (const float*)vector(v[1], c.dev, ScalarType::Float, N), *b = (const float*)vector(v[2], c.dev, ScalarType::Float, N);
    need(g);
    const int rows = int32_size(x.numel() / N), cols = int32_size(N), round_mode = (int)integer(v[5]);
    const float eps = (float)number(v[3]);
    const bool rms = flag(v[4]);
    Tensor out;
    int rc;
    {
      const NoGil unlocked;
      out = c.empty(x.sizes(), ScalarType::Char);
      rc = ti_layernorm_q((const float*)ptr(x), pitch, g, b, eps, (int8_t*)mptr(out), N, rows, cols, rms, round_mode, nullptr, nullptr, c.stream);
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

// dq_add_layernorm_q(acc, scale, residual, gamma, beta, eps, round_mode) -> (residual_out, int8)
PyObject* dq_add_layernorm_q(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 7, [&]() -> PyObject* {
    const Tensor& acc = tensor(v[0], -1, ScalarType::Int);
    const Call c(acc);
    const Tensor& res = tensor(v[2], c.dev, ScalarType::Float);
    need(acc.dim() >= 1 && acc.sizes() == res.sizes() && acc.size(-1) > 0);
    const int64_t H = acc.size(-1), pitch = row_pitch(acc), res_pitch = row_pitch(res);
    const float *g = (const float*)vector(v[3], c.dev, ScalarType::Float, H), *b = (const float*)vector(v[4], c.dev, ScalarType::Float, H);
    need(g);
    const int rows = int32_size(acc.numel() / H), cols = int32_size(H), round_mode = (int)integer(v[6]);
    const float s = (float)number(v[1]), eps = (float)number(v[5]);
    Tensor rout, y;
    int rc;
    {
      const NoGil unlocked;
      rout = c.empty(acc.sizes(), ScalarType::Float);
      y = c.empty(acc.sizes(), ScalarType::Char);
      rc = ti_dq_add_layernorm_q((const int32_t*)ptr(acc), pitch, s, nullptr, (const float*)ptr(res), res_pitch, g, b, eps, (float*)mptr(rout), H,
                                 (int8_t*)mptr(y), H, nullptr, H, rows, cols, round_mode, nullptr, nullptr, c.stream);
    }
    need(rc == TI_OK);
    PyObject* pair = PyTuple_New(2);
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(rout));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(y));
    return pair;
  });
}

// layernorm_fp(x, skip, weight, bias, eps, rms, want_out, want_skip_out) -> (out or None, skip_out or None)
PyObject* layernorm_fp(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 8, [&]() -> PyObject* {
    const Tensor& x = tensor(v[0]);
    const Call c(x);
    const ScalarType type = x.scalar_type();
    const int dt = dtype_code(type);
    need(x.dim() >= 1 && x.size(-1) > 0);
    const int64_t N = x.size(-1), pitch = row_pitch(x);
    int64_t skip_pitch = 0;
    const void *g = vector(v[2], c.dev, type, N), *b = vector(v[3], c.dev, type, N), *skip = nullptr;
    need(g);
    if (v[1] != Py_None) {
      const Tensor& s = tensor(v[1], c.dev, type);
      need(s.numel() == x.numel() && s.size(-1) == N);
      skip_pitch = row_pitch(s);
      skip = ptr(s);
    }
    const int rows = int32_size(x.numel() / N), cols = int32_size(N);
    const float eps = (float)number(v[4]);
    const bool rms = flag(v[5]), want_out = flag(v[6]), want_skip_out = flag(v[7]);
    Tensor out, sout;
    int rc;
    {
      const NoGil unlocked;
      if (want_out) out = c.empty(x.sizes(), type);
      if (want_skip_out) sout = c.empty(x.sizes(), type);
      rc = ti_layernorm_fp(ptr(x), pitch, skip, skip_pitch, dt, g, b, eps, rms, want_out ? mptr(out) : nullptr, N,
                           want_skip_out ? mptr(sout) : nullptr, N, rows, cols, c.stream);
    }
    need(rc == TI_OK);
    PyObject* pair = PyTuple_New(2);
    const Tensor* both[2] = {&out, &sout};
    for (int i = 0; i < 2; ++i) {
      PyObject* o = both[i]->defined() ? THPVariable_Wrap(*both[i]) : (Py_INCREF(Py_None), Py_None);
      PyTuple_SET_ITEM(pair, i, o);
    }
    return pair;
  });
}

// gelu_q(x, scale, round_mode)
PyObject* gelu_q(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 3, [&]() -> PyObject* {
    const Tensor& x = tensor(v[0], -1, ScalarType::Float);
    const Call c(x);
    need(x.is_contiguous());
    const float* s = scale(v[1], c.dev);
    need(s);
    const int round_mode = (int)integer(v[2]);
    Tensor out;
    int rc;
    {
      const NoGil unlocked;
      out = c.empty(x.sizes(), ScalarType::Char);
      rc = ti_gelu_q((const float*)ptr(x), s, (int8_t*)mptr(out), x.numel(), round_mode, c.stream);
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

// softmax_q(x, scale, causal_q_len)
PyObject* softmax_q(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 3, [&]() -> PyObject* {
    const Tensor& x = tensor(v[0], -1, ScalarType::Char);
    const Call c(x);
    need(x.dim() >= 1 && x.size(-1) > 0);
    const int64_t cols = x.size(-1), pitch = row_pitch(x);
    const int rows = int32_size(x.numel() / cols), cols32 = int32_size(cols), causal = (int)integer(v[2]);
    const float s = (float)number(v[1]);
    Tensor out;
    int rc;
    {
      const NoGil unlocked;
      out = c.empty(x.sizes(), ScalarType::Char);
      rc = ti_softmax_q((const int8_t*)ptr(x), pitch, s, (int8_t*)mptr(out), cols, rows, cols32, causal, c.stream);
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

// quantize_per_token(x) -> (int8, scale)
PyObject* quantize_per_token(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 1, [&]() -> PyObject* {
    const Tensor& x = tensor(v[0]);
    const Call c(x);
    need(x.scalar_type() == ScalarType::Float || x.scalar_type() == ScalarType::Half);
    need(x.dim() >= 1 && x.size(-1) > 0);
    const int64_t cols = x.size(-1), pitch = row_pitch(x);
    const int rows = int32_size(x.numel() / cols), cols32 = int32_size(cols);
    Tensor q, s;
    int rc;
    {
      const NoGil unlocked;
      q = c.empty(x.sizes(), ScalarType::Char);
      s = c.empty(with_last(x, 1), x.scalar_type());
      rc = ti_quantize_per_token_absmax(ptr(x), dtype_code(x.scalar_type()), pitch, (int8_t*)mptr(q), cols, mptr(s), rows, cols32, c.stream);
    }
    need(rc == TI_OK);
    PyObject* pair = PyTuple_New(2);
    PyTuple_SET_ITEM(pair, 0, THPVariable_Wrap(q));
    PyTuple_SET_ITEM(pair, 1, THPVariable_Wrap(s));
    return pair;
  });
}

// quantize_per_tensor(x, weight_scale) -> (int8, scale, alpha)
PyObject* quantize_per_tensor(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 2, [&]() -> PyObject* {
    const Tensor& x = tensor(v[0]);
    const Call c(x);
    need(x.scalar_type() == ScalarType::Float || x.scalar_type() == ScalarType::Half);
    need(x.is_contiguous() && x.numel() > 0);
    const float* ws = scale(v[1], c.dev);
    Tensor q, s, al, work;
    int rc;
    {
      const NoGil unlocked;
      q = c.empty(x.sizes(), ScalarType::Char);
      s = c.empty({}, x.scalar_type());
      al = c.empty({}, ScalarType::Float);
      work = c.empty({TI_QUANT_TENSOR_WORKSPACE}, ScalarType::Byte);
      rc = ti_quantize_per_tensor_absmax(ptr(x), dtype_code(x.scalar_type()), x.numel(), (int8_t*)mptr(q), mptr(s), ws, (float*)mptr(al),
                                         mptr(work), c.stream);
    }
    need(rc == TI_OK);
    PyObject* triple = PyTuple_New(3);
    PyTuple_SET_ITEM(triple, 0, THPVariable_Wrap(q));
    PyTuple_SET_ITEM(triple, 1, THPVariable_Wrap(s));
    PyTuple_SET_ITEM(triple, 2, THPVariable_Wrap(al));
    return triple;
  });
}

// strides of [seqs, heads, rows, D] or [heads, rows, D] with unit last stride
struct Heads {
  int64_t ss, hs, rs;
  int seqs, heads;
  explicit Heads(const Tensor& t) {
    const int64_t d = t.dim();
    need(d == 3 || d == 4);
    need(t.stride(d - 1) == 1 || t.size(d - 1) == 1);
    ss = d == 4 ? t.stride(0) : 0;
    hs = t.stride(d - 3);
    rs = t.stride(d - 2);
    seqs = d == 4 ? int32_size(t.size(0)) : 1;
    heads = int32_size(t.size(d - 3));
  }
};

// attention(q, k, vt, qk_alpha, score_scale, pv_alpha, causal_q_len, out)
PyObject* attention(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 8, [&]() -> PyObject* {
    const Tensor& q = tensor(v[0], -1, ScalarType::Char);
    const Call c(q);
    const Tensor &k = tensor(v[1], c.dev, ScalarType::Char), &vt = tensor(v[2], c.dev, ScalarType::Char);
    const Heads hq(q), hk(k), hv(vt);
    const int64_t S = q.size(-2), D = q.size(-1), T = k.size(-2);
    need(k.dim() == q.dim() && vt.dim() == q.dim() && hk.seqs == hq.seqs && hv.seqs == hq.seqs && hk.heads == hq.heads && hv.heads == hq.heads);
    need(k.size(-1) == D && vt.size(-2) == D && vt.size(-1) == T);
    const int S32 = int32_size(S), T32 = int32_size(T), D32 = int32_size(D), causal = (int)integer(v[6]);
    const float qk_alpha = (float)number(v[3]), score_scale = (float)number(v[4]), pv_alpha = (float)number(v[5]);
    Tensor out;
    if (v[7] != Py_None) {
      out = tensor(v[7], c.dev, ScalarType::Char);
      need(out.sizes() == q.sizes());
    }
    int rc;
    {
      const NoGil unlocked;
      if (!out.defined()) out = c.empty(q.sizes(), ScalarType::Char);
      const Heads ho(out);
      rc = ti_attention_i8_heads((const int8_t*)ptr(q), hq.ss, hq.hs, hq.rs, (const int8_t*)ptr(k), hk.ss, hk.hs, hk.rs, (const int8_t*)ptr(vt),
                                 hv.ss, hv.hs, hv.rs, (int8_t*)mptr(out), ho.ss, ho.hs, ho.rs, hq.seqs, hq.heads, S32, T32, D32, qk_alpha,
                                 score_scale, pv_alpha, causal, c.stream);
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

// qkv_decode(a, w3, bias3, alpha3, beta3, k_cache, vt_cache, seqs)
PyObject* qkv_decode(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 8, [&]() -> PyObject* {
    const Tensor& a = tensor(v[0], -1, ScalarType::Char);
    const Call c(a);
    const Tensor& w = tensor(v[1], c.dev, ScalarType::Char);
    const int64_t seqs = integer(v[7]);
    need(a.dim() == 2 && w.dim() == 2 && w.is_contiguous() && w.size(0) % 3 == 0 && seqs > 0 && a.size(0) % seqs == 0 && a.size(0) <= 16);
    const Rows r(a, w.size(1));
    const int64_t N = w.size(0) / 3;
    const Caches kv(v[5], v[6], c.dev, r.M / seqs);
    need(kv.k && kv.BH * kv.D == seqs * N && r.K >= 1024);
    const int8_t* bias = (const int8_t*)vector(v[2], c.dev, ScalarType::Char, 3 * N);
    const float *al = (const float*)vector(v[3], c.dev, ScalarType::Float, 3), *be = (const float*)vector(v[4], c.dev, ScalarType::Float, 3);
    need(bias && al && be);
    const int N32 = int32_size(N);
    Tensor out;
    int rc;
    {
      const NoGil unlocked;
      out = c.empty({r.M, 3 * N}, ScalarType::Char);
      rc = ti_qkv_decode_i8_seqs((const int8_t*)ptr(a), r.pitch, (const int8_t*)ptr(w), r.K, bias, al, be, (int8_t*)mptr(out), 3 * N, (int)seqs,
                                 r.M, N32, r.K, kv.k, kv.k_hs, kv.k_rs, kv.vt, kv.vt_rs, (int)kv.D, c.stream);
    }
    need(rc == TI_OK);
    return THPVariable_Wrap(out);
  });
}

// kv_append(k_new, v_new, k_cache, vt_cache, seqs) -> True
PyObject* kv_append(PyObject*, PyObject* const* v, Py_ssize_t n) {
  return guarded(n, 5, [&]() -> PyObject* {
    const Tensor& vn = tensor(v[1], -1, ScalarType::Char);
    const Call c(vn);
    const int64_t seqs = integer(v[4]);
    need(vn.dim() == 2 && vn.stride(1) == 1 && seqs > 0 && vn.size(0) % seqs == 0);
    const int64_t S = vn.size(0) / seqs;
    const Caches kv(v[2], v[3], c.dev, S);
    need(kv.BH % seqs == 0 && kv.BH / seqs * kv.D == vn.size(1));
    const int8_t* ksrc = nullptr;
    int64_t k_rs = 0;
    if (kv.k) {
      const Tensor& kn = tensor(v[0], c.dev, ScalarType::Char);
      need(kn.sizes() == vn.sizes() && kn.stride(1) == 1);
      ksrc = (const int8_t*)ptr(kn);
      k_rs = kn.stride(0);
    }
    const int S32 = int32_size(S);
    int rc;
    {
      const NoGil unlocked;
      rc = ti_kv_append_i8_seqs(ksrc, k_rs, (const int8_t*)ptr(vn), vn.stride(0), kv.k, kv.k_hs, kv.k_rs, kv.vt, kv.vt_rs, (int)seqs, S32,
                                (int)(kv.BH / seqs), (int)kv.D, c.stream);
    }
    need(rc == TI_OK);
    Py_RETURN_TRUE;
  });
}

#define TI_METHOD(name) {#name, (PyCFunction)(void (*)(void))name, METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    TI_METHOD(linear), TI_METHOD(bmm), TI_METHOD(linear_residual), TI_METHOD(layernorm_q), TI_METHOD(dq_add_layernorm_q),
    TI_METHOD(layernorm_fp), TI_METHOD(gelu_q), TI_METHOD(softmax_q), TI_METHOD(quantize_per_token), TI_METHOD(quantize_per_tensor), TI_METHOD(attention),
    TI_METHOD(qkv_decode), TI_METHOD(kv_append), {nullptr, nullptr, 0, nullptr}};
PyModuleDef module = {PyModuleDef_HEAD_INIT, "_host", "Host path of the launchers (see csrc/host.cpp).", -1, methods};

}  // namespace

PyMODINIT_FUNC PyInit__host() { return PyModule_Create(&module); }
