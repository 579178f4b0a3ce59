// The LayerNorm-in-front entry points on addresses that share memory or do not.  Prints "case status launches" a line.
#include "fake_hip.h"

typedef char* P;
static P at(size_t n) { return (P)fake_address(n); }

static void said(const char* name, int rc) {
  printf("%s %d %d\n", name, rc, launches);
  launches = 0;
}

struct Fc1 {
  int M = 2, N = 8192, K = 2048;
  int64_t acc_rs = K, x_rs = K, ro_rs = K;
  P acc = at(1), x = at(2), gamma = at(3), beta = at(4), ro = at(5), W = at(6), bias = at(7), a = at(8), b = at(9), C = at(10);
  int call() const {
    return ti_dq_add_layernorm_linear_gelu_i8((const int32_t*)acc, acc_rs, 1e-5f, (const float*)x, x_rs, (const float*)gamma, (const float*)beta, 1e-5f, (float*)ro, ro_rs,
                                              (const int8_t*)W, K, (const float*)bias, (const float*)a, (const float*)b, (int8_t*)C, N, M, N, K, (void*)16);
  }
};

struct Qkv {
  int M = 2, seqs = 2, heads = 8, K = 2048, T = 64, D = 128, N = heads * D;
  int64_t x_rs = K;
  P x = at(1), gamma = at(2), beta = at(3), W = at(4), bias = at(5), a = at(6), b = at(7), C = at(8), k = at(9), v = at(10);
  int call() const {
    return ti_layernorm_qkv_decode_i8_seqs((const float*)x, x_rs, (const float*)gamma, (const float*)beta, 1e-5f, (const int8_t*)W, K, (const int8_t*)bias, (const float*)a,
                                           (const float*)b, (int8_t*)C, 3 * N, seqs, M, N, K, (int8_t*)k, (int64_t)T * D, D, (int8_t*)v, T, D, (void*)16);
  }
};

template <class T, class F>
static void with(const char* name, F change) {
  T t;
  change(t);
  said(name, t.call());
}

int main() {
  room = 0;
  const int row = 2048 * 4;
  with<Fc1>("fc1", [](Fc1&) {});
  with<Fc1>("fc1_no_bias", [](Fc1& t) { t.beta = t.bias = nullptr; });
  with<Fc1>("fc1_out_after_acc", [=](Fc1& t) { t.C = t.acc + 2 * row; });
  with<Fc1>("fc1_out_before_x", [=](Fc1& t) { t.C = t.x - 2 * 8192; });
  with<Fc1>("fc1_out_is_acc", [](Fc1& t) { t.C = t.acc; });
  with<Fc1>("fc1_out_in_x", [=](Fc1& t) { t.C = t.x + 2 * row - 16; });
  with<Fc1>("fc1_out_in_gamma", [](Fc1& t) { t.C = t.gamma + 16; });
  with<Fc1>("fc1_out_in_beta", [](Fc1& t) { t.C = t.beta - 16; });
  with<Fc1>("fc1_out_in_resid_out", [](Fc1& t) { t.C = t.ro + 16; });
  with<Fc1>("fc1_resid_out_is_x", [](Fc1& t) { t.ro = t.x; });
  with<Fc1>("fc1_resid_out_in_acc", [=](Fc1& t) { t.ro = t.acc + row; });
  with<Fc1>("fc1_resid_out_in_gamma", [](Fc1& t) { t.ro = t.gamma + 16; });
  with<Fc1>("fc1_resid_out_in_weights", [](Fc1& t) { t.ro = t.W + 2048 * 16; });
  with<Fc1>("fc1_resid_out_in_bias", [](Fc1& t) { t.ro = t.bias + 16; });
  with<Qkv>("qkv", [](Qkv&) {});
  with<Qkv>("qkv_out_after_x", [=](Qkv& t) { t.C = t.x + 2 * row; });
  with<Qkv>("qkv_out_is_x", [](Qkv& t) { t.C = t.x; });
  with<Qkv>("qkv_out_in_gamma", [](Qkv& t) { t.C = t.gamma + 16; });
  with<Qkv>("qkv_k_in_x", [=](Qkv& t) { t.k = t.x + row; });
  with<Qkv>("qkv_k_ends_in_x", [](Qkv& t) { t.k = t.x - (2 * 8 - 1) * 64 * 128 - 112; });
  with<Qkv>("qkv_k_ends_before_x", [](Qkv& t) { t.k = t.x - (2 * 8 - 1) * 64 * 128 - 128; });
  with<Qkv>("qkv_v_in_beta", [](Qkv& t) { t.v = t.beta + 16; });
  for (int m = 1; m <= 2; ++m) {
    const char* const names[2][5] = {{"fc1_one_row", "fc1_one_row_odd_x", "fc1_one_row_odd_acc", "fc1_one_row_odd_resid_out", "qkv_one_row_odd_x"},
                                     {"fc1_two_rows", "fc1_two_rows_odd_x", "fc1_two_rows_odd_acc", "fc1_two_rows_odd_resid_out", "qkv_two_rows_odd_x"}};
    with<Fc1>(names[m - 1][0], [=](Fc1& t) { t.M = m, t.x_rs += 4, t.acc_rs += 8, t.ro_rs += 12; });
    with<Fc1>(names[m - 1][1], [=](Fc1& t) { t.M = m, t.x_rs += 2; });
    with<Fc1>(names[m - 1][2], [=](Fc1& t) { t.M = m, t.acc_rs += 1; });
    with<Fc1>(names[m - 1][3], [=](Fc1& t) { t.M = m, t.ro_rs += 3; });
    with<Qkv>(names[m - 1][4], [=](Qkv& t) { t.M = t.seqs = m, t.x_rs += 2; });
  }
  with<Fc1>("fc1_no_columns", [](Fc1& t) { t.N = 0; });
  with<Fc1>("fc1_empty", [](Fc1& t) { t.M = 0; });
  with<Fc1>("fc1_empty_no_columns", [](Fc1& t) { t.M = t.N = 0; });
  return 0;
}
