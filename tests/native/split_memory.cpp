// GEMM launches with little memory or under capture.  Arguments: `capturing` or `none`, bytes that hipMalloc gives in all, then
// launches of "M,N,K" (fp32 out), each on the same stream.  Prints a line per launch: status, configuration, K splits, launches, bytes held.
#include "fake_hip.h"

int main(int argc, char** argv) {
  capturing = !strcmp(argv[1], "capturing");
  room = strtoull(argv[2], nullptr, 0);
  for (int i = 3; i < argc; ++i) {
    int M, N, K;
    if (sscanf(argv[i], "%d,%d,%d", &M, &N, &K) != 3) return 2;
    const auto at = fake_address;
    launches = 0;
    const int rc = ti_bmm_i8((const int8_t*)at(1), 0, K, 1, (const int8_t*)at(2), 0, K, 1, at(3), 0, N, 1, 1, M, N, K, nullptr, TI_BIAS_NONE, (const float*)at(4),
                             nullptr, TI_EPI_SCALE_F, TI_F32, TI_ROUND_RNE_CLAMP, (void*)16);
    printf("%d %s %d %d %zu\n", rc, ti_gemm_config_name(ti_gemm_last_config()), ti_gemm_last_splits(), launches, held);
  }
  return 0;
}
