// attention_i8.hip — int8 attention for one block of query rows without the score round trip.
//
// The reference's callers chain three launches per attention block (nn/bmm.py:10-29 for Q.K^T,
// a softmax in the caller, nn/bmm.py:10-29 / :54-74 for P.V):
//     scores = q8(qk_alpha * (q . k))                      int8 [BH, S, T]   (kernels/bmm.py:576-612)
//     probs  = rne(127 * softmax(scores * score_scale))    int8 [BH, S, T]   values 0..127
//     ctx    = q8(pv_alpha * (probs . v))                  int8 [BH, S, D]   (kernels/bmm.py:576-612)
// At 2048 x 2048 scores per head the two intermediates are 4 x 168 MB of HBM traffic for 40 heads.
// This kernel computes the same three steps per 32 x 32 block of scores in registers: the int8
// score quantisation, the probability quantisation and the context quantisation are the same
// fp32 operations as in the three kernels, and a row's exponentials are summed as integers (see
// the softmax-quantise arithmetic in ti_common.h), so the result is the three-kernel chain's bit
// for bit although the keys are visited in another order.
//
// Three passes over the keys of a query block.  Pass 0 finds each row's largest score (the
// exponent's reference point): the quantisation is monotone in the int32 accumulator, so it is a
// maximum over accumulators, one instruction per two scores.  Pass 1 recomputes the scores
// (K = 128 deep: cheap) and sums the exponentials.  Pass 2 recomputes them once more, forms the
// int8 probabilities in the MFMA operand layout straight from the accumulator registers (two
// half-wave swaps put a row's keys in order) and feeds them to the P.V MFMAs, so P never goes
// through memory.
//
// (Launches of few query rows take attention_decode_i8_kernel, and of one row attention_row_i8_kernel, further down instead.)
//
// Workgroup = 4 waves = 128 query rows of one head; a wave owns 32 rows.  K and V^T are staged
// through LDS in tiles of 64 keys, double-buffered, one barrier per tile.  Causal masking skips
// whole key tiles beyond a wave's last visible key and masks inside the tiles on the diagonal.
#include <type_traits>

#include "ti_common.h"

namespace ti {

constexpr int AT_D = 128;                // head dimension this kernel is written for
constexpr int AT_ROWS = 128;             // query rows per workgroup
constexpr int AT_KT = 64;                // keys per LDS tile
constexpr int AT_KP = AT_D + 16;         // K tile row pitch (bytes): 16-byte reads of 16 rows hit 64 different banks
constexpr int AT_VP = AT_KT + 16;        // V^T tile row pitch
constexpr int AT_KBYTES = AT_KT * AT_KP;
constexpr int AT_VBYTES = AT_D * AT_VP;

struct AttnParams {
  const int8_t* q; const int8_t* k; const int8_t* vt; int8_t* out;
  // strides of a sequence, of a head inside it, of a row inside that
  int64_t sQb, sQh, sQm, sKb, sKh, sKn, sVb, sVh, sVd, sOb, sOh, sOm;
  int S, T, causal_q_len, nblk;
  int batch, heads;  // batch = sequences * heads
  float qk_alpha, s2, pv_alpha;  // s2 = score_scale * log2(e)
};

__device__ __forceinline__ int attn_limit(const AttnParams& p, int row) {
  return p.causal_q_len > 0 ? min(p.T, (row % p.causal_q_len) + (p.T - p.causal_q_len) + 1) : p.T;
}

// Any number of keys, all sequences of a batch in one launch: what a length that is no multiple of 16 used to
// cost was the three-launch chain with P.V through byte gathers, once per sequence.  Whole layer, before ->
// after: two prompts of 333 tokens (4096 wide) 377 -> 239 us, sixteen sequences decoding at position 1007
// 1105 -> 284 us.
//
// VANY: rows of V^T start anywhere (a row pitch that is no multiple of 16: a cache allocated at exactly its
// length; load16_tail).  Otherwise they are 16-byte aligned, and a chunk that
// crosses T is loaded whole: an aligned 16-byte chunk that holds at least one key of the row lies inside the
// row's pitch, and the keys past T are multiplied by probabilities that are exactly 0.
template <bool VANY>
__global__ __launch_bounds__(256, 2) void attention_i8_kernel(AttnParams p) {
  __shared__ __attribute__((aligned(16))) char lds[2 * (AT_KBYTES + AT_VBYTES)];
  __shared__ int wg_lim[4];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lrow = lane & 31, lhi = lane >> 5;
  // Work item = (head, block of 128 query rows).  Under a causal mask a later row block sees more
  // keys, and every workgroup of a launch of this size is resident at once, workgroup i on the same
  // CU as i + 256 and i + 512 (measured placement).  The items are therefore taken in order of
  // decreasing work and dealt to the workgroup indices in a snake: 0..255 forward, 256..511
  // backward, ..., which gives every CU about the same total.
  const int n_items = p.nblk * p.batch;
  const int pass = (int)blockIdx.x >> 8, c = (int)blockIdx.x & 255;
  const int cnt = min(256, n_items - pass * 256);
  const int pos = pass * 256 + ((pass & 1) ? cnt - 1 - c : c);
  const int bh = pos % p.batch;
  const int m0 = (p.nblk - 1 - pos / p.batch) * AT_ROWS + wave * 32;
  const int seq = bh / p.heads, head = bh - seq * p.heads;
  const int8_t* qb = p.q + (int64_t)seq * p.sQb + (int64_t)head * p.sQh;
  const int8_t* kb_ = p.k + (int64_t)seq * p.sKb + (int64_t)head * p.sKh;
  const int8_t* vb = p.vt + (int64_t)seq * p.sVb + (int64_t)head * p.sVh;

  // ---- per-lane row, visible-key limit; wave and workgroup bounds
  const int row = m0 + lrow;
  const int rowc = min(row, p.S - 1);                       // rows past S repeat the last row, never stored
  const int lim_lane = attn_limit(p, min(max(rowc, 0), p.S - 1));
  int lim_hi = lim_lane, lim_lo = lim_lane;
#pragma unroll
  for (int off = 16; off > 0; off >>= 1) {
    lim_hi = max(lim_hi, __shfl_xor(lim_hi, off, 64));
    lim_lo = min(lim_lo, __shfl_xor(lim_lo, off, 64));
  }
  lim_hi = __builtin_amdgcn_readfirstlane(lim_hi);
  lim_lo = __builtin_amdgcn_readfirstlane(lim_lo);
  const bool wave_live = m0 < p.S;                          // a wave wholly past S computes nothing
  if (lane == 0) wg_lim[wave] = wave_live ? lim_hi : 0;
  __syncthreads();
  const int wg_hi = max(max(wg_lim[0], wg_lim[1]), max(wg_lim[2], wg_lim[3]));
  const int ntiles = __builtin_amdgcn_readfirstlane((wg_hi + AT_KT - 1) / AT_KT);

  // ---- this wave's Q fragments (32 rows x 128 d): lane (row, half) holds 16 bytes per 32-deep step
  v4i qf[4];
#pragma unroll
  for (int ds = 0; ds < 4; ++ds)
    qf[ds] = *(const v4i*)(qb + (int64_t)rowc * p.sQm + ds * 32 + lhi * 16);

  // ---- tile staging: thread t copies two 16-byte chunks of the K tile and two of the V^T tile
  v4i kreg[2], vreg[2];
  auto fetch = [&](int t, bool with_v) {
    const int key0 = t * AT_KT;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int q_ = c * 256 + tid;          // chunk index: 64 keys x 8 chunks
      const int kr = q_ >> 3, kc = q_ & 7;
      const bool in = key0 + kr < p.T;
      kreg[c] = in ? *(const v4i*)(kb_ + (int64_t)(key0 + kr) * p.sKn + kc * 16) : (v4i){0, 0, 0, 0};
    }
    if (with_v) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int q_ = c * 256 + tid;        // chunk index: 128 d x 4 chunks of 16 keys
        const int vr = q_ >> 2, vc = q_ & 3;
        const int8_t* row = vb + (int64_t)vr * p.sVd;
        if constexpr (VANY) {
          vreg[c] = load16_tail(row, key0 + vc * 16, p.T);
        } else {
          const bool in = key0 + vc * 16 < p.T;
          vreg[c] = in ? *(const v4i*)(row + key0 + vc * 16) : (v4i){0, 0, 0, 0};
        }
      }
    }
  };
  auto stash = [&](int buf, bool with_v) {
    char* kt = lds + buf * (AT_KBYTES + AT_VBYTES);
    char* vt = kt + AT_KBYTES;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const int q_ = c * 256 + tid;
      *(v4i*)(kt + (q_ >> 3) * AT_KP + (q_ & 7) * 16) = kreg[c];
    }
    if (with_v) {
#pragma unroll
      for (int c = 0; c < 2; ++c) {
        const int q_ = c * 256 + tid;
        *(v4i*)(vt + (q_ >> 2) * AT_VP + (q_ & 3) * 16) = vreg[c];
      }
    }
  };

  const float MAGIC = 12582912.0f;  // 1.5 * 2^23: adding it rounds to the nearest even integer

  // ================= pass 0: each row's largest score =================
  // q8(alpha * f(acc)) does not decrease with acc when alpha >= 0 (and does not increase when
  // alpha < 0), so the largest score is the quantised largest (smallest) accumulator.
  const bool want_max = p.qk_alpha >= 0.0f;
  int ext = want_max ? (int)0x80000000 : 0x7fffffff;
  auto score_ext_t = [&](const char* kt, int key0, auto mask_tag, auto max_tag) {
    constexpr bool MASK = decltype(mask_tag)::value;
    constexpr bool MAX = decltype(max_tag)::value;
    v4i kf[2][4];
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
#pragma unroll
      for (int b = 0; b < 2; ++b) kf[b][ds] = *(const v4i*)(kt + (b * 32 + lrow) * AT_KP + ds * 32 + lhi * 16);
    v16i s[2];
    const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        s[b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[b][ds], qf[ds], ds == 0 ? zero : s[b], 0, 0, 0);
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        int v = s[b][r];
        if constexpr (MASK) {
          const int key = key0 + 32 * b + 8 * (r >> 2) + 4 * lhi + (r & 3);
          v = key < lim_lane ? v : (MAX ? (int)0x80000000 : 0x7fffffff);
        }
        ext = MAX ? max(ext, v) : min(ext, v);
      }
  };
  auto score_ext = [&](const char* kt, int key0) {
    const bool mask = key0 + AT_KT > lim_lo;
    if (want_max) {
      if (mask) score_ext_t(kt, key0, std::true_type{}, std::true_type{});
      else score_ext_t(kt, key0, std::false_type{}, std::true_type{});
    } else {
      if (mask) score_ext_t(kt, key0, std::true_type{}, std::false_type{});
      else score_ext_t(kt, key0, std::false_type{}, std::false_type{});
    }
  };
  fetch(0, false);
  stash(0, false);
  __syncthreads();
  for (int t = 0; t < ntiles; ++t) {
    if (t + 1 < ntiles) fetch(t + 1, false);
    const char* kt = lds + (t & 1) * (AT_KBYTES + AT_VBYTES);
    if (wave_live && t * AT_KT < lim_hi) score_ext(kt, t * AT_KT);
    if (t + 1 < ntiles) stash((t + 1) & 1, false);
    __syncthreads();
  }
  {
    const int other = __shfl_xor(ext, 32, 64);  // the two lane halves hold different keys of the same row
    ext = want_max ? max(ext, other) : min(ext, other);
  }
  float cref;  // -(largest score * s2): the exponent's reference point of this lane's row
  {
    float v = (float)ext * p.qk_alpha;
    v = __builtin_amdgcn_fmed3f(v, -128.0f, 127.0f);
    cref = -(__builtin_rintf(v) * p.s2);
  }
  // Scores of one 64-key tile -> exponentials.  The tile's two 32-key blocks are two independent
  // MFMA chains, interleaved, with all fragment reads issued first; e[b][r] belongs to key
  // key0 + 32*b + 8*(r/4) + 4*lhi + r%4.  A block that lies wholly beyond the wave's last visible
  // key is computed too and masked to zero (at most one per wave and pass).
  auto score_exp_t = [&](const char* kt, int key0, float (&e)[2][16], auto mask_tag) {
    constexpr bool MASK = decltype(mask_tag)::value;
    v4i kf[2][4];
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
#pragma unroll
      for (int b = 0; b < 2; ++b) kf[b][ds] = *(const v4i*)(kt + (b * 32 + lrow) * AT_KP + ds * 32 + lhi * 16);
    v16i s[2];
    const v16i zero = {0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0};
#pragma unroll
    for (int ds = 0; ds < 4; ++ds)
#pragma unroll
      for (int b = 0; b < 2; ++b)
        s[b] = __builtin_amdgcn_mfma_i32_32x32x32_i8(kf[b][ds], qf[ds], ds == 0 ? zero : s[b], 0, 0, 0);  // rows of the result = keys
#pragma unroll
    for (int b = 0; b < 2; ++b) {
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        float v = (float)s[b][r] * p.qk_alpha;
        v = __builtin_amdgcn_fmed3f(v, -128.0f, 127.0f);
        const float x = __builtin_rintf(v);  // the int8 score, as a float (round half to even, like the BMM's)
        e[b][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(x, p.s2, cref));
      }
      if constexpr (MASK) {
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int key = key0 + 32 * b + 8 * (r >> 2) + 4 * lhi + (r & 3);
          e[b][r] = key < lim_lane ? e[b][r] : 0.0f;
        }
      }
    }
  };
  // Off the diagonal no row's limit falls inside or before the tile and the selects above must
  // cost nothing: two instantiations behind a wave-uniform branch (the MFMAs inside keep the
  // compiler from folding them back into one block of selects).
  auto score_exp = [&](const char* kt, int key0, float (&e)[2][16]) {
    if (key0 + AT_KT > lim_lo) score_exp_t(kt, key0, e, std::true_type{});
    else score_exp_t(kt, key0, e, std::false_type{});
  };

  // ================= pass 1: row sums (exact integers, see ti_common.h) =================
  unsigned long long sum = 0;
  fetch(0, false);
  stash(0, false);
  __syncthreads();
  for (int t = 0; t < ntiles; ++t) {
    if (t + 1 < ntiles) fetch(t + 1, false);
    const char* kt = lds + (t & 1) * (AT_KBYTES + AT_VBYTES);
    if (wave_live && t * AT_KT < lim_hi) {
      float e[2][16];
      score_exp(kt, t * AT_KT, e);
      unsigned s0 = 0, s1 = 0;
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        s0 += sm_unit_bits(e[0][r]);
        s1 += sm_unit_bits(e[1][r]);
      }
      sum += (unsigned)(s0 + s1 - 32u * SM_ONE_BITS);  // modulo 2^32: the tile's 32 units of this lane, below 2^29
    }
    if (t + 1 < ntiles) stash((t + 1) & 1, false);
    __syncthreads();
  }
  {
    // the two lane halves hold different keys of the same row
    const unsigned lo = (unsigned)__shfl_xor((int)(unsigned)sum, 32, 64);
    const unsigned hi = (unsigned)__shfl_xor((int)(unsigned)(sum >> 32), 32, 64);
    sum += ((unsigned long long)hi << 32) | lo;
  }
  const float rinv = sm_scale_from_sum(sum);

  // ================= pass 2: probabilities and P.V =================
  v16i o[4];
#pragma unroll
  for (int db = 0; db < 4; ++db)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[db][r] = 0;
  fetch(0, true);
  stash(0, true);
  __syncthreads();
  for (int t = 0; t < ntiles; ++t) {
    if (t + 1 < ntiles) fetch(t + 1, true);
    const char* kt = lds + (t & 1) * (AT_KBYTES + AT_VBYTES);
    const char* vt = kt + AT_KBYTES;
    if (wave_live && t * AT_KT < lim_hi) {
      float e[2][16];
      score_exp(kt, t * AT_KT, e);
      v4i vf[2][4];
#pragma unroll
      for (int db = 0; db < 4; ++db)
#pragma unroll
        for (int b = 0; b < 2; ++b) vf[b][db] = *(const v4i*)(vt + (db * 32 + lrow) * AT_VP + b * 32 + lhi * 16);
      v4i pf[2];  // 16 int8 probabilities of this lane's row per block, keys in accumulator order
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const unsigned b0 = __float_as_uint(__builtin_fmaf(e[b][4 * g + 0], rinv, MAGIC));
          const unsigned b1 = __float_as_uint(__builtin_fmaf(e[b][4 * g + 1], rinv, MAGIC));
          const unsigned b2 = __float_as_uint(__builtin_fmaf(e[b][4 * g + 2], rinv, MAGIC));
          const unsigned b3 = __float_as_uint(__builtin_fmaf(e[b][4 * g + 3], rinv, MAGIC));
          pf[b][g] = (int)(__builtin_amdgcn_perm(b1, b0, 0x0c0c0400u) | __builtin_amdgcn_perm(b3, b2, 0x04000c0cu));
        }
      // The accumulators hold a row's 32 keys of a block as alternate 4-key groups in the two lane
      // halves; two half-wave swaps give lane half h the keys 16h .. 16h+15 in order, which is how
      // the MFMA wants its 32-deep operand and how V^T lies in LDS.
#pragma unroll
      for (int b = 0; b < 2; ++b) {
        const auto s02 = __builtin_amdgcn_permlane32_swap((unsigned)pf[b][0], (unsigned)pf[b][2], false, false);
        const auto s13 = __builtin_amdgcn_permlane32_swap((unsigned)pf[b][1], (unsigned)pf[b][3], false, false);
        pf[b][0] = (int)s02[0]; pf[b][1] = (int)s02[1]; pf[b][2] = (int)s13[0]; pf[b][3] = (int)s13[1];
      }
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int db = 0; db < 4; ++db)
          o[db] = __builtin_amdgcn_mfma_i32_32x32x32_i8(vf[b][db], pf[b], o[db], 0, 0, 0);  // rows of the result = d
    }
    if (t + 1 < ntiles) stash((t + 1) & 1, true);
    __syncthreads();
  }

  // ---- context: o[db][r] is row lrow, d = 32*db + 8*(r/4) + 4*lhi + r%4 -> int8, 16 bytes per lane
  if (!wave_live) return;
  int8_t* ob = p.out + (int64_t)seq * p.sOb + (int64_t)head * p.sOh;
#pragma unroll
  for (int db = 0; db < 4; ++db) {
    unsigned X[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      unsigned b[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        float v = (float)o[db][4 * g + t] * p.pv_alpha;
        v = __builtin_amdgcn_fmed3f(v, -128.0f, 127.0f);
        b[t] = __float_as_uint(v + MAGIC);
      }
      X[g] = __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u) | __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);
    }
    // lanes l and l+32 hold alternate 4-byte groups of the row's 32 bytes: after the two swaps
    // lane l has bytes 0..15 and lane l+32 bytes 16..31
    const auto s02 = __builtin_amdgcn_permlane32_swap(X[0], X[2], false, false);
    const auto s13 = __builtin_amdgcn_permlane32_swap(X[1], X[3], false, false);
    v4u v;
    v[0] = s02[0]; v[1] = s02[1]; v[2] = s13[0]; v[3] = s13[1];
    if (row < p.S) *(v4u*)(ob + (int64_t)row * p.sOm + db * 32 + lhi * 16) = v;
  }
}


// ---- few query rows (decode, short chunks of a prompt): one workgroup per head and 16 rows ----------
//
// 16 query rows of a head's attention fit one workgroup: 16 waves, one pass.  Wave w computes the scores
// of the 16-key chunks w, w + 16, ... with 16x16x64 MFMAs (K rows
// loaded from memory straight into the operand layout: 16 rows x 64 bytes per instruction) and keeps
// them in registers; row maximum and sum go through LDS; the int8 probabilities are written to LDS in
// key order ([16 queries][T]), from where every wave reads them back as MFMA operands for P.V: wave w
// owns 16 of the 128 output columns (V^T rows, also loaded straight into the operand layout) and
// one half of the 64-key groups; the two halves meet in LDS.  The arithmetic is that of the three
// kernels (score quantisation, exponent against the row maximum, 127 / sum, context quantisation);
// only the order of a row's sum differs.  More rows are more workgroups, which share K and V^T in L2.
constexpr int AD_WAVES = 16;
constexpr int AD_MAXT = 4096;

// CPW: 16-key chunks per wave (T <= 256 * CPW), in steps of 256 keys up to 1536: chunks past the last key cost their loads' latency, scores and
// exponentials like any other.  us, 4 chunks at least and then 8 and 16 / these: 32 heads x 64 rows x 64 keys 6.2 / 4.5, x 128 x 128 7.1 / 5.3, x 64 x
// 1064 12.7 / 11.1, 64 x 140 x 437 27.7 / 19.9, 40 x 7 x 1200 11.5 / 10.1, 8 x 27 x 27 5.5 / 4.1.  3, 6 and 12 chunks alone against the
// next larger: 32 x 256 x 768 17.0 / 15.8, 40 x 16 x 600 7.7 / 7.3; 32 x 256 x 1400 31.4 / 28.0, 40 x 16 x 1400 13.0 / 11.7; 32 x 256 x 2500 49.7 / 47.4, 8 x 16 x 3072 19.7 / 18.5, 40 x 16 x
// 2500 20.9 / 21.1.  DBW: 16-column blocks of the output a workgroup
// produces (8: the whole head; fewer: the head is spread over 8 / DBW workgroups, each of which
// repeats the scores and the softmax and reads only its rows of V^T — a single CU fills its caches at
// about 30 GB/s, so a head's 512 KB of K and V^T through one CU alone would take 17 us).
// VANY: V^T rows without alignment, as in attention_i8_kernel.
template <int CPW, int DBW, bool VANY>
__global__ __launch_bounds__(AD_WAVES * 64, CPW <= 2 ? 8 : 4) void attention_decode_i8_kernel(AttnParams p) {
  constexpr int TMAX = 256 * CPW;
  constexpr int PP = TMAX + 16;             // LDS pitch of a query's probabilities
  constexpr int KPARTS = AD_WAVES / DBW;    // waves that share an output block and split the keys
  constexpr int GPW = (TMAX / 64 + KPARTS - 1) / KPARTS;  // 64-key groups per wave in P.V
  constexpr int HOIST = CPW >= 12 ? (GPW < 4 ? GPW : 4) : GPW;  // V^T operands fetched before the softmax reductions
  __shared__ __attribute__((aligned(16))) char p_lds[16 * PP];
  __shared__ float red_max[AD_WAVES][16];
  __shared__ unsigned red_sum[AD_WAVES][16];
  __shared__ __attribute__((aligned(16))) v4i ctx_red[AD_WAVES][64];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int n = lane & 15, kq = lane >> 4;  // operand row / 16-byte quarter of a 64-deep k-step
  // Grid: head; 16 query rows and block of output columns; sequence.  The workgroups of a head are p.heads apart: with
  // a multiple of 8 heads they run on the same XCD and share its L2 for K.  No division on the way to the first loads,
  // and no branch before all arguments are asked for: at 6 us a launch those are felt (head, sequence, rows and columns divided
  // out of one grid dimension, and the mask's period: 32 heads x 1 row x 64 keys 6.5 us, so 5.7; 40 x 1 x 512 7.4 / 7.0).
  constexpr int PARTS = 8 / DBW;
  const int head = blockIdx.x, seq = blockIdx.z;
  const int row0 = (int)blockIdx.y / PARTS * 16;  // this workgroup's 16 query rows
  const int dbase = (int)blockIdx.y % PARTS * DBW;
  const int OOB = 0x7ffffff0;
  const float MAGIC = 12582912.0f;
  const int8_t* vb = p.vt + (int64_t)seq * p.sVb + (int64_t)head * p.sVh;
  const __amdgpu_buffer_rsrc_t rQ = __builtin_amdgcn_make_buffer_rsrc((void*)(p.q + (int64_t)seq * p.sQb + (int64_t)head * p.sQh), 0,
                                                                      (int)((p.S - 1) * p.sQm + AT_D), 0x00020000);
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void*)(p.k + (int64_t)seq * p.sKb + (int64_t)head * p.sKh), 0,
                                                                      (int)((p.T - 1) * p.sKn + AT_D), 0x00020000);
  // the last chunk of an aligned row may cross T (see attention_i8_kernel)
  const __amdgpu_buffer_rsrc_t rV =
      __builtin_amdgcn_make_buffer_rsrc((void*)vb, 0, (int)((AT_D - 1) * p.sVd + ((p.T + 15) & ~15)), 0x00020000);
  const int db = dbase + wave % DBW, kh = wave / DBW;

  v4i qf[2];
#pragma unroll
  for (int ks = 0; ks < 2; ++ks)
    qf[ks] = __builtin_amdgcn_raw_buffer_load_b128(rQ, row0 + n < p.S ? (row0 + n) * (int)p.sQm + ks * 64 + kq * 16 : OOB, 0, 0);
  // keys that any of the rows sees (under a causal mask the later ones are not even loaded)
  const int rlast = min(row0 + 15, p.S - 1);
  const bool one_period = p.causal_q_len >= p.S;  // of the mask, as in every decoder layer: nothing to divide
  auto limit_of = [&](int row) { return one_period ? min(p.T, row + (p.T - p.causal_q_len) + 1) : attn_limit(p, row); };
  const int keys = one_period || (p.causal_q_len > 0 && row0 / p.causal_q_len == rlast / p.causal_q_len) ? limit_of(rlast) : p.T;
  auto load_v = [&](int d, int col) -> v4i {
    if constexpr (VANY) return load16_tail(vb + (int64_t)d * p.sVd, col, p.T);
    else return __builtin_amdgcn_raw_buffer_load_b128(rV, col < keys ? d * (int)p.sVd + col : OOB, 0, 0);
  };
  const int NCH = (keys + 15) >> 4;  // 16-key chunks; rows of K past T read as zeros and are masked
  const int NG = (keys + 63) >> 6;   // 64-key groups
  const int limit = limit_of(min(row0 + n, rlast));
  // ---- scores: f = the int8 score as a float, -inf where masked or beyond T
  const float NEG = -__builtin_inff();
  float f[CPW][4];
  constexpr int NB = CPW < 8 ? CPW : (CPW > 8 ? 4 : 8);  // chunks whose K operands are in flight together
#pragma unroll
  for (int b0 = 0; b0 < CPW; b0 += NB) {
    v4i kf[NB][2];
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int c = wave + AD_WAVES * (b0 + i);
      const int off = (c * 16 + n) * (int)p.sKn + kq * 16;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) kf[i][ks] = __builtin_amdgcn_raw_buffer_load_b128(rK, c < NCH ? off + ks * 64 : OOB, 0, 0);
    }
#pragma unroll
    for (int i = 0; i < NB; ++i) {
      const int c = wave + AD_WAVES * (b0 + i);
      v4i acc = {0, 0, 0, 0};
      acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf[i][0], qf[0], acc, 0, 0, 0);
      acc = __builtin_amdgcn_mfma_i32_16x16x64_i8(kf[i][1], qf[1], acc, 0, 0, 0);
      // acc[r]: key c*16 + 4*kq + r, query n
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        float v = (float)acc[r] * p.qk_alpha;
        v = __builtin_amdgcn_fmed3f(v, -128.0f, 127.0f);
        const int key = c * 16 + 4 * kq + r;
        f[b0 + i][r] = key < limit ? __builtin_rintf(v) : NEG;
      }
    }
  }
  // V^T operands of this wave's first groups: in flight during the reductions below
  v4i vf[HOIST];
#pragma unroll
  for (int i = 0; i < HOIST; ++i) {
    const int g = kh + KPARTS * i;
    const int col = 64 * g + 16 * kq;
    vf[i] = load_v(16 * db + n, col);
  }

  // ---- row maximum (exact: integers), exponentials, row sum
  float mx = NEG;
#pragma unroll
  for (int i = 0; i < CPW; ++i) mx = fmaxf(fmaxf(mx, fmaxf(f[i][0], f[i][1])), fmaxf(f[i][2], f[i][3]));
  mx = fmaxf(mx, __shfl_xor(mx, 16, 64));
  mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
  if (kq == 0) red_max[wave][n] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < AD_WAVES; ++w) mx = fmaxf(mx, red_max[w][n]);
  const float c0 = -(mx * p.s2);
  // exact integer row sum (see ti_common.h): a lane holds at most 64 scores (below 2^29 units), the
  // four lanes of a query below 2^31, the 16 waves meet in 64 bits
  unsigned bits = 0;
#pragma unroll
  for (int i = 0; i < CPW; ++i)
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      f[i][r] = __builtin_amdgcn_exp2f(__builtin_fmaf(f[i][r], p.s2, c0));
      bits += sm_unit_bits(f[i][r]);
    }
  bits -= (unsigned)(CPW * 4) * SM_ONE_BITS;  // modulo 2^32
  bits += (unsigned)__shfl_xor((int)bits, 16, 64);
  bits += (unsigned)__shfl_xor((int)bits, 32, 64);
  if (kq == 0) red_sum[wave][n] = bits;
  __syncthreads();
  unsigned long long sum = 0;
#pragma unroll
  for (int w = 0; w < AD_WAVES; ++w) sum += red_sum[w][n];
  const float rcp = sm_scale_from_sum(sum);

  // ---- int8 probabilities into LDS, key order; keys in [T, 64 * NG) get zeros (their f is -inf)
#pragma unroll
  for (int i = 0; i < CPW; ++i) {
    const int c = wave + AD_WAVES * i;
    if (c < 4 * NG) {
      const unsigned b0 = __float_as_uint(__builtin_fmaf(f[i][0], rcp, MAGIC)), b1 = __float_as_uint(__builtin_fmaf(f[i][1], rcp, MAGIC));
      const unsigned b2 = __float_as_uint(__builtin_fmaf(f[i][2], rcp, MAGIC)), b3 = __float_as_uint(__builtin_fmaf(f[i][3], rcp, MAGIC));
      *(unsigned*)(p_lds + n * PP + 16 * c + 4 * kq) =
          __builtin_amdgcn_perm(b1, b0, 0x0c0c0400u) | __builtin_amdgcn_perm(b3, b2, 0x04000c0cu);
    }
  }
  __syncthreads();

  // ---- P.V: D[d = 16*db + 4*kq + r][query n] over this wave's key groups
  v4i o = {0, 0, 0, 0};
#pragma unroll
  for (int i = 0; i < HOIST; ++i) {
    const int g = kh + KPARTS * i;
    if (g < NG) o = __builtin_amdgcn_mfma_i32_16x16x64_i8(vf[i], *(const v4i*)(p_lds + n * PP + 64 * g + 16 * kq), o, 0, 0, 0);
  }
#pragma unroll
  for (int i0 = HOIST; i0 < GPW; i0 += 4) {
    v4i vn[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int col = 64 * (kh + KPARTS * (i0 + i)) + 16 * kq;
      vn[i] = load_v(16 * db + n, col);
    }
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int g = kh + KPARTS * (i0 + i);
      if (g < NG) o = __builtin_amdgcn_mfma_i32_16x16x64_i8(vn[i], *(const v4i*)(p_lds + n * PP + 64 * g + 16 * kq), o, 0, 0, 0);
    }
  }
  if (kh > 0) ctx_red[wave][lane] = o;
  __syncthreads();
  if (kh == 0 && row0 + n < p.S) {
#pragma unroll
    for (int k2 = 1; k2 < KPARTS; ++k2) o += ctx_red[wave + k2 * DBW][lane];
    unsigned b[4];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      float v = (float)o[r] * p.pv_alpha;
      v = __builtin_amdgcn_fmed3f(v, -128.0f, 127.0f);
      b[r] = __float_as_uint(v + MAGIC);
    }
    *(unsigned*)(p.out + (int64_t)seq * p.sOb + (int64_t)head * p.sOh + (int64_t)(row0 + n) * p.sOm + 16 * db + 4 * kq) =
        __builtin_amdgcn_perm(b[1], b[0], 0x0c0c0400u) | __builtin_amdgcn_perm(b[3], b[2], 0x04000c0cu);
  }
}

// ---- one query row (a decode step): one workgroup per head, or several that share its V^T ----------------
//
// With one row the matrix units have nothing to do that the dot-product instructions do not do as well, and what their
// operand layout costs is the order of the reads: 16 rows x 64 bytes per instruction, of K as of V^T, and sixteen queries' worth
// of softmax for one.  Here a wave reads 1 KB of consecutive bytes per instruction: 8 rows of K (a lane one 16-byte piece, v_dot4, three
// additions across 8 lanes) and 64 x 16 keys of one row of V^T.  Scores end up one per lane, so the softmax of 1024 keys is one or two
// values a lane; int8 probabilities go through LDS once, and every lane keeps its 16 of each 1024 keys for all its rows of V^T.
// The loads of K and then V^T are one sequence with AR_WINDOW of them in flight, so V^T is on its way before the
// first reduction.  Sums are integers: the bits are those of the other kernels.
// Bound: HBM where the heads fill the chip, else what a CU takes in.  attention_decode_i8_kernel / this one, caches from HBM: 512
// heads x 1007 keys 30.7 / 24.9 us (5.3 TB/s), 640 x 2048 87 / 57.7 (5.8 TB/s), 40 x 1531 12.9 / 7.6, 32 x 64 5.6 / 4.2, rows of V^T at any
// byte 512 x 1007 36.9 / 23.6.  V^T (and K where one workgroup reads it) is loaded non-temporally: read once; 640 x 2048 60.6 -> 57.4.
// 24 loads in flight instead of 16: 1 - 3 % slower.
constexpr int AR_WINDOW = 16;
typedef v4i v4i_any __attribute__((aligned(1)));  // at any byte

// f(integral_constant i) for A <= i < B
template <int A, int B, class F>
__device__ __forceinline__ void static_for(F f) {
  if constexpr (A < B) {
    f(std::integral_constant<int, A>{});
    static_for<A + 1, B>(f);
  }
}

template <int CTRL>
__device__ __forceinline__ int dpp(int v) { return __builtin_amdgcn_update_dpp(v, v, CTRL, 0xf, 0xf, false); }

// lanes 0..31 of the result: a's sum over both halves of the wave; lanes 32..63: b's
__device__ __forceinline__ int merge32(int a, int b) {
  const auto s = __builtin_amdgcn_permlane32_swap((unsigned)a, (unsigned)b, false, false);
  return (int)s[0] + (int)s[1];
}
// the same with neighbouring rows of 16 lanes
__device__ __forceinline__ int merge16(int a, int b) {
  const auto s = __builtin_amdgcn_permlane16_swap((unsigned)a, (unsigned)b, false, false);
  return (int)s[0] + (int)s[1];
}
__device__ __forceinline__ int sum16(int v) {
  v += dpp<0x128>(v);
  v += dpp<0x124>(v);
  v += dpp<0x122>(v);
  return v + dpp<0x121>(v);
}
__device__ __forceinline__ float wave_max(float f) {
  const auto other = [&](int v) { f = fmaxf(f, __int_as_float(v)); };
  other(dpp<0x128>(__float_as_int(f)));
  other(dpp<0x124>(__float_as_int(f)));
  other(dpp<0x122>(__float_as_int(f)));
  other(dpp<0x121>(__float_as_int(f)));
  const auto a = __builtin_amdgcn_permlane16_swap(__float_as_uint(f), __float_as_uint(f), false, false);
  f = fmaxf(__uint_as_float(a[0]), __uint_as_float(a[1]));
  const auto b = __builtin_amdgcn_permlane32_swap(__float_as_uint(f), __float_as_uint(f), false, false);
  return fmaxf(__uint_as_float(b[0]), __uint_as_float(b[1]));
}

// NW waves; RW rows of V^T per wave (a workgroup has NW * RW of the 128); GR: T <= 64 * NW * GR.
// VANY: rows of V^T start at any byte (T >= 16): the lane with the row's end reads the row's last 16 bytes, against
// probabilities that lie the same way.
template <int NW, int RW, int GR, bool VANY>
__global__ __launch_bounds__(NW * 64, 4) void attention_row_i8_kernel(AttnParams p) {
  constexpr int KS = 8 * GR, SL = NW * GR * 64 / 1024, NV = RW * SL, W = AR_WINDOW, NT = 2;
  static_assert(SL * 1024 == NW * GR * 64 && NW * 64 * GR <= AD_MAXT && GR <= 4, "every probability has a slot; a wave's sum fits 32 bits");
  __shared__ __attribute__((aligned(16))) char p_lds[SL * 1024];
  __shared__ __attribute__((aligned(16))) char p_tail[16];
  __shared__ __attribute__((aligned(16))) float red_max[NW];
  __shared__ __attribute__((aligned(16))) unsigned red_sum[NW];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int head = blockIdx.x, seq = blockIdx.z;
  const int d0 = ((int)blockIdx.y * NW + wave) * RW;
  const float MAGIC = 12582912.0f, NEG = -__builtin_inff();
  const int8_t* qb = p.q + (int64_t)seq * p.sQb + (int64_t)head * p.sQh;
  const int8_t* vb = p.vt + (int64_t)seq * p.sVb + (int64_t)head * p.sVh;
  const __amdgpu_buffer_rsrc_t rK = __builtin_amdgcn_make_buffer_rsrc((void*)(p.k + (int64_t)seq * p.sKb + (int64_t)head * p.sKh), 0,
                                                                      (int)((p.T - 1) * p.sKn + AT_D), 0x00020000);
  const __amdgpu_buffer_rsrc_t rV =
      __builtin_amdgcn_make_buffer_rsrc((void*)vb, 0, (int)((AT_D - 1) * p.sVd + ((p.T + 15) & ~15)), 0x00020000);
  const v4i qf = *(const v4i*)(qb + (lane & 7) * 16);
  // keys from T on lie past K's descriptor and read as zeros
  const int koff = (wave * 8 + (lane >> 3)) * (int)p.sKn + (lane & 7) * 16, kstep = NW * 8 * (int)p.sKn;
  int voff[SL];
#pragma unroll
  for (int s = 0; s < SL; ++s) {
    const int col = s * 1024 + lane * 16;
    voff[s] = VANY ? min(col, p.T - 16) : (col < p.T ? col : 0x7ffffff0);
  }
  v4i slot[W];
  const auto issue = [&](auto at) {
    constexpr int i = decltype(at)::value;
    if constexpr (i < KS) {
      slot[i % W] = __builtin_amdgcn_raw_buffer_load_b128(rK, koff + i * kstep, 0, NW * RW == AT_D ? NT : 0);
    } else if constexpr (i < KS + NV) {
      constexpr int s = (i - KS) / RW, r = (i - KS) % RW;
      if constexpr (VANY) slot[i % W] = __builtin_nontemporal_load((const v4i_any*)(vb + (int64_t)(d0 + r) * p.sVd + voff[s]));
      else slot[i % W] = __builtin_amdgcn_raw_buffer_load_b128(rV, voff[s], (d0 + r) * (int)p.sVd, NT);
    }
  };
  static_for<0, W>(issue);
  if (VANY && tid < 16) p_tail[tid] = 0;

  // ---- scores: lane l keeps those of loads i with i % 8 == l % 8, key (i * NW + wave) * 8 + l / 8
  float f[GR];
  const int key0 = ((lane & 7) * NW + wave) * 8 + (lane >> 3);
  static_for<0, GR>([&](auto gt) {
    constexpr int g = decltype(gt)::value;
    int acc = 0;
    static_for<0, 8>([&](auto it) {
      constexpr int i = g * 8 + decltype(it)::value;
      int a = 0;
#pragma unroll
      for (int t = 0; t < 4; ++t) a = __builtin_amdgcn_sdot4(slot[i % W][t], qf[t], a, false);
      issue(std::integral_constant<int, i + W>{});
      a += dpp<0xB1>(a);   // neighbour
      a += dpp<0x4E>(a);   // pairs
      a += dpp<0x141>(a);  // halves of 8 lanes
      acc = (lane & 7) == decltype(it)::value ? a : acc;
    });
    float v = (float)acc * p.qk_alpha;
    v = __builtin_amdgcn_fmed3f(v, -128.0f, 127.0f);
    f[g] = key0 + g * 64 * NW < p.T ? __builtin_rintf(v) : NEG;
  });

  float mx = f[0];
#pragma unroll
  for (int g = 1; g < GR; ++g) mx = fmaxf(mx, f[g]);
  mx = wave_max(mx);
  if (lane == 0) red_max[wave] = mx;
  __syncthreads();
#pragma unroll
  for (int w = 0; w < NW; ++w) mx = fmaxf(mx, red_max[w]);
  const float c0 = -(mx * p.s2);
  unsigned bits = 0;
#pragma unroll
  for (int g = 0; g < GR; ++g) {
    f[g] = __builtin_amdgcn_exp2f(__builtin_fmaf(f[g], p.s2, c0));
    bits += sm_unit_bits(f[g]);
  }
  bits -= (unsigned)GR * SM_ONE_BITS;
  bits = (unsigned)sum16((int)bits);
  bits = (unsigned)merge16((int)bits, (int)bits);
  bits = (unsigned)merge32((int)bits, (int)bits);
  if (lane == 0) red_sum[wave] = bits;
  __syncthreads();
  unsigned long long sum = 0;
#pragma unroll
  for (int w = 0; w < NW; ++w) sum += red_sum[w];
  const float rcp = sm_scale_from_sum(sum);
#pragma unroll
  for (int g = 0; g < GR; ++g) {
    const int key = key0 + g * 64 * NW;
    const char b = (char)__float_as_uint(__builtin_fmaf(f[g], rcp, MAGIC));
    p_lds[key] = b;  // 0 from T on
    if (VANY && key >= (p.T & ~15) && key < p.T) p_tail[key - (p.T - 16)] = b;
  }
  __syncthreads();

  // ---- P.V
  int o[RW];
#pragma unroll
  for (int r = 0; r < RW; ++r) o[r] = 0;
  v4i pf[SL];
#pragma unroll
  for (int s = 0; s < SL; ++s) {
    const int col = s * 1024 + lane * 16;
    pf[s] = *(const v4i*)(VANY && col < p.T && col + 16 > p.T ? p_tail : p_lds + col);
  }
  static_for<0, NV>([&](auto it) {
    constexpr int i = KS + decltype(it)::value, s = decltype(it)::value / RW, r = decltype(it)::value % RW;
#pragma unroll
    for (int t = 0; t < 4; ++t) o[r] = __builtin_amdgcn_sdot4(slot[i % W][t], pf[s][t], o[r], false);
    issue(std::integral_constant<int, i + W>{});
  });
  // sums over the wave: two rows meet in the halves of a register, then four in its quarters
  constexpr int H = (RW + 1) / 2, Q = (H + 1) / 2;
  int q4[Q];
#pragma unroll
  for (int j = 0; j < Q; ++j) {
    const auto half = [&](int i) { return merge32(o[2 * i], o[RW > 1 ? 2 * i + 1 : 0]); };
    const int lo = half(2 * j);
    q4[j] = sum16(merge16(lo, H > 1 ? half(H > 1 ? 2 * j + 1 : 0) : lo));
  }
  // lane (half h, quarter q, i): row 4 i + 2 q + h
  const int i = lane & 15, h = lane >> 5, q = lane >> 4 & 1;
  int v = q4[0];
#pragma unroll
  for (int j = 1; j < Q; ++j) v = i == j ? q4[j] : v;
  const int r = 4 * i + (H > 1 ? 2 * q : 0) + (RW > 1 ? h : 0);
  float x = (float)v * p.pv_alpha;
  x = __builtin_amdgcn_fmed3f(x, -128.0f, 127.0f);
  if (i < Q && (H > 1 || q == 0) && (RW > 1 || h == 0))
    p.out[(int64_t)seq * p.sOb + (int64_t)head * p.sOh + d0 + r] = (int8_t)__float_as_uint(x + MAGIC);
}

// Groups of 16 query rows on attention_decode_i8_kernel where a head has one of them (a single row goes on to attention_row_i8_kernel).  Up to four
// rounds of the chip (256 workgroups each) on whichever kernel takes less: a round of groups walks the keys once, 0.2 us per 64 of them and
// 2.5 us besides, or as long as 4 TB/s take for the caches of the heads in it (up to 256: each is then read again in the
// next round); two workgroups on a CU fill a last round that is partly empty.  The blocks of 128 rows on attention_i8_kernel, all in one round,
// 1.8 us per 64 keys and 3 us besides however few their rows.  Rows of V^T of no whole 16-byte pieces: 0.5 us per 64 keys and 2 us, eight tenths of a last round's
// empty part, against 2.3 and 3.5.  128-row blocks beyond four rounds.
// Measured over 837 sizes of 17 .. 700 rows against 17 .. 4096 keys, with and without a mask: the choice is 1.1 % above the better kernel on average where rows
// of V^T are whole pieces (337 sizes; no launch of groups 3 % above the blocks), 0.6 % where they are not (500; by the first estimate 1.0 %).  us, groups / blocks, 40
// heads x 205 rows x 205 keys 9.1 / 15.2, 80 x 107 x 196 10.6 / 16.2, 32 x 371 x 371 13.7 / 20.3, 8 x 19 x 1103 10.1 / 46.9, 96 x 57 x 755 22.5 / 37.9; but 80 x 377 x 377
// 28.6 / 20.6, 160 x 232 x 434 58.8 / 32.0; V^T at any byte 40 x 207 x 207 12.4 / 15.8, 32 x 501 x 501 26.0 / 25.0, 40 x 377 x 763 46.4 / 35.5, 64 x 129 x 129 14.1 / 12.4.  Where it
// loses: 80 x 139 x 139 9.4 / 12.2, 32 x 516 x 516 (1056 groups) 20.4 / 25.9, at any byte 32 x 258 x 258 19.8 / 16.8.
// 16 rows and fewer, as many workgroups either way: 2560 x 16 x 2048 297 / 464.
static bool attn_groups_lead(int64_t heads, int S, int T, bool whole_pieces) {
  const int64_t groups = heads * ((S + 15) / 16);
  if (S <= 16) return true;
  if (groups > 1024) return false;
  const double walk = whole_pieces ? 2.5 + 0.2 * T / 64 : 2.0 + 0.5 * T / 64, fetch = (double)(heads < 256 ? heads : 256) * T * 2 * AT_D / 4.0e6;
  const double full = groups > 256 ? (double)groups / 256 : 1.0, empty = (double)((groups + 255) / 256) - full;
  const double rounds = whole_pieces ? full : full + 0.8 * empty;
  return rounds * (walk > fetch ? walk : fetch) <= (whole_pieces ? 3.0 + 1.8 * T / 64 : 3.5 + 2.3 * T / 64);
}

static bool attn_few_rows(int64_t heads, int S, int T, int64_t q_row_stride, int64_t k_row_stride, int64_t vt_row_stride) {
  const int64_t lim32 = (int64_t)1 << 31;  // descriptor extents and offsets
  return attn_groups_lead(heads, S, T, !(vt_row_stride & 15)) && T <= AD_MAXT && (int64_t)(T + 256) * k_row_stride < lim32 &&
         (int64_t)AT_D * vt_row_stride < lim32 && (int64_t)S * q_row_stride < lim32;
}

// One query row: what attention_row_i8_kernel takes of the calls for few rows.  An unaligned row of V^T needs 16 bytes; the
// offsets of all its score slots (up to AD_MAXT keys, those past T included) fit 32 bits.
static bool attn_one_row(int S, int T, bool vany, int64_t k_row_stride) {
  return S == 1 && (T >= 16 || !vany) && AD_MAXT * k_row_stride < (int64_t)1 << 31;
}

// A head is spread over as many workgroups (each reads K again, from L2) as fit one round of the 256 CUs; beyond one round K read
// once is worth more than an even last round.  us for 1 / 2 / 4 / 8 workgroups per head, caches from HBM: 8 heads x 1500 keys 7.9 / 7.7 /
// 6.4 / 6.0, 32 x 1000 5.7 / 6.4 / 5.3 / 4.9, 40 x 2047 10.0 / 10.0 / 7.4 / 10.3, 64 x 1500 10.1 / 9.7 / 8.3 / 11.0, 65 x 1500 10.0 / 10.0 / 15.1 / 21.0,
// 128 x 2047 14.2 / 13.7 / 16.8 / 21.9, 129 x 2047 13.9 / 22.0 / 31.0 / 49.0, 512 x 1000 25.0 / 35.0 / 52.7 / 89.3.  Up to 2048 keys
// 8 waves, which leave room for two workgroups on a CU; beyond, 16 (a wave's scores stay four registers): 3000 keys 1 / 2 / 4 per head, 40
// heads 16.5 / 15.0 / 12.5, 100 19.9 / 20.2 / 28.4.
static int launch_attention_row(const AttnParams& p, int seqs, bool vany, hipStream_t st) {
  const auto launch = [&](auto nw, auto rw, auto gr) {
    constexpr int NW = decltype(nw)::value, RW = decltype(rw)::value, GR = decltype(gr)::value;
    const dim3 grid((unsigned)p.heads, AT_D / (NW * RW), (unsigned)seqs), block(NW * 64);
    if (vany) attention_row_i8_kernel<NW, RW, GR, true><<<grid, block, 0, st>>>(p);
    else attention_row_i8_kernel<NW, RW, GR, false><<<grid, block, 0, st>>>(p);
  };
  const auto spread = [&](auto nw, auto gr) {
    constexpr int NW = decltype(nw)::value, RW = AT_D / NW;
    if (NW == 8 && p.batch <= 32) launch(nw, std::integral_constant<int, 2>{}, gr);
    else if (p.batch <= 64) launch(nw, std::integral_constant<int, RW / 4>{}, gr);
    else if (p.batch <= 128) launch(nw, std::integral_constant<int, RW / 2>{}, gr);
    else launch(nw, std::integral_constant<int, RW>{}, gr);
  };
  using W8 = std::integral_constant<int, 8>;
  if (p.T <= 1024) spread(W8{}, std::integral_constant<int, 2>{});
  else if (p.T <= 2048) spread(W8{}, std::integral_constant<int, 4>{});
  else spread(std::integral_constant<int, 16>{}, std::integral_constant<int, 4>{});
  return launch_status("attention_row_i8_kernel");
}

}  // namespace ti

extern "C" int ti_attention_i8_rows(int64_t heads, int S, int T, int64_t q_row_stride, int64_t k_row_stride, int64_t vt_row_stride) {
  return ti::attn_few_rows(heads, S, T, q_row_stride, k_row_stride, vt_row_stride) ? 16 : ti::AT_ROWS;
}

extern "C" int ti_attention_i8_heads(const int8_t* q, int64_t q_seq_stride, int64_t q_head_stride, int64_t q_row_stride,
                                     const int8_t* k, int64_t k_seq_stride, int64_t k_head_stride, int64_t k_row_stride,
                                     const int8_t* vt, int64_t vt_seq_stride, int64_t vt_head_stride, int64_t vt_row_stride,
                                     int8_t* out, int64_t out_seq_stride, int64_t out_head_stride, int64_t out_row_stride,
                                     int seqs, int heads, int S, int T, int D, float qk_alpha, float score_scale,
                                     float pv_alpha, int causal_q_len, void* stream) {
  using namespace ti;
  if (seqs < 0 || heads < 0 || S < 0 || T < 0 || causal_q_len < 0) return fail(TI_E_SHAPE, "negative size");
  if (seqs == 0 || heads == 0 || S == 0) return TI_OK;
  if (!q || !k || !vt || !out) return fail(TI_E_NULL, "q, k, vt and out are required");
  if (D != AT_D) return fail(TI_E_SHAPE, "head dimension %d: this kernel is built for %d", D, AT_D);
  if (T <= 0) return fail(TI_E_SHAPE, "T = %d must be positive", T);
  if ((int64_t)seqs * heads > 65535) return fail(TI_E_SHAPE, "%d x %d heads: more than 65535", seqs, heads);
  if (causal_q_len > T) return fail(TI_E_SHAPE, "causal_q_len %d > T %d", causal_q_len, T);
  if (causal_q_len > 0 && S % causal_q_len) return fail(TI_E_SHAPE, "S %d not a multiple of causal_q_len %d", S, causal_q_len);
  if (q_row_stride < D || k_row_stride < D || out_row_stride < D || vt_row_stride < T)
    return fail(TI_E_STRIDE, "row strides must cover a row");
  const uintptr_t align = (uintptr_t)q | (uintptr_t)k | (uintptr_t)out | (uintptr_t)q_seq_stride | (uintptr_t)q_head_stride |
                          (uintptr_t)q_row_stride | (uintptr_t)k_seq_stride | (uintptr_t)k_head_stride | (uintptr_t)k_row_stride |
                          (uintptr_t)out_seq_stride | (uintptr_t)out_head_stride | (uintptr_t)out_row_stride;
  if (align & 15) return fail(TI_E_STRIDE, "pointers and strides of q, k and out must be multiples of 16 bytes");
  const bool vany = (((uintptr_t)vt | (uintptr_t)vt_seq_stride | (uintptr_t)vt_head_stride | (uintptr_t)vt_row_stride) & 15) != 0;
  const float s2 = score_scale * 1.44269504088896340736f;
  if (!(score_scale > 0.0f) || !(score_scale <= SM_MAX_SCALE))
    return fail(TI_E_COMBO, "score_scale %g outside (0, %g]: the quantised softmax is exact in that range only", (double)score_scale, (double)SM_MAX_SCALE);
  const int64_t groups = (int64_t)seqs * heads * ((S + 15) / 16);
  const bool few_rows = attn_few_rows((int64_t)seqs * heads, S, T, q_row_stride, k_row_stride, vt_row_stride);
  int rc = check_device();
  if (rc != TI_OK) return rc;
  const int batch = seqs * heads;
  AttnParams p;
  p.q = q; p.k = k; p.vt = vt; p.out = out;
  p.sQb = q_seq_stride; p.sQh = q_head_stride; p.sQm = q_row_stride;
  p.sKb = k_seq_stride; p.sKh = k_head_stride; p.sKn = k_row_stride;
  p.sVb = vt_seq_stride; p.sVh = vt_head_stride; p.sVd = vt_row_stride;
  p.sOb = out_seq_stride; p.sOh = out_head_stride; p.sOm = out_row_stride;
  p.S = S; p.T = T; p.causal_q_len = causal_q_len;
  p.qk_alpha = qk_alpha; p.s2 = s2; p.pv_alpha = pv_alpha;
  p.nblk = (S + AT_ROWS - 1) / AT_ROWS;
  p.batch = batch; p.heads = heads;
  const hipStream_t st = (hipStream_t)stream;
  if (few_rows && attn_one_row(S, T, vany, k_row_stride)) return launch_attention_row(p, seqs, vany, st);
  if (few_rows) {
    // spread a head over as many workgroups as keep the launch within one round of the 256 CUs
    // (40 heads x 16 rows x 2048 keys: 18.9 / 15.3 / 13.6 us for 1 / 2 / 4 workgroups per head,
    // 24 us for 8, which no longer fit one round)
    int dbw = 8;
    while (dbw > 1 && groups * (16 / dbw) <= 256) dbw /= 2;
    const dim3 grid((unsigned)heads, (unsigned)((S + 15) / 16 * (8 / dbw)), (unsigned)seqs), block(AD_WAVES * 64);
#define TI_AD_LAUNCH(C, V) \
    (dbw == 8 ? attention_decode_i8_kernel<C, 8, V><<<grid, block, 0, st>>>(p) : dbw == 4 ? attention_decode_i8_kernel<C, 4, V><<<grid, block, 0, st>>>(p) \
     : dbw == 2 ? attention_decode_i8_kernel<C, 2, V><<<grid, block, 0, st>>>(p) : attention_decode_i8_kernel<C, 1, V><<<grid, block, 0, st>>>(p))
    if (T <= 256) vany ? TI_AD_LAUNCH(1, true) : TI_AD_LAUNCH(1, false);
    else if (T <= 512) vany ? TI_AD_LAUNCH(2, true) : TI_AD_LAUNCH(2, false);
    else if (T <= 768) vany ? TI_AD_LAUNCH(3, true) : TI_AD_LAUNCH(3, false);
    else if (T <= 1024) vany ? TI_AD_LAUNCH(4, true) : TI_AD_LAUNCH(4, false);
    else if (T <= 1280) vany ? TI_AD_LAUNCH(5, true) : TI_AD_LAUNCH(5, false);
    else if (T <= 1536) vany ? TI_AD_LAUNCH(6, true) : TI_AD_LAUNCH(6, false);
    else if (T <= 2048) vany ? TI_AD_LAUNCH(8, true) : TI_AD_LAUNCH(8, false);
    else if (T <= 3072) vany ? TI_AD_LAUNCH(12, true) : TI_AD_LAUNCH(12, false);
    else vany ? TI_AD_LAUNCH(16, true) : TI_AD_LAUNCH(16, false);
#undef TI_AD_LAUNCH
    return launch_status("attention_decode_i8_kernel");
  }
  const dim3 grid((unsigned)(p.nblk * batch));
  if (vany) attention_i8_kernel<true><<<grid, dim3(256), 0, st>>>(p);
  else attention_i8_kernel<false><<<grid, dim3(256), 0, st>>>(p);
  return launch_status("attention_i8_kernel");
}

extern "C" int ti_attention_i8(const int8_t* q, int64_t q_batch_stride, int64_t q_row_stride, const int8_t* k,
                               int64_t k_batch_stride, int64_t k_row_stride, const int8_t* vt,
                               int64_t vt_batch_stride, int64_t vt_row_stride, int8_t* out, int64_t out_batch_stride,
                               int64_t out_row_stride, int batch, int S, int T, int D, float qk_alpha,
                               float score_scale, float pv_alpha, int causal_q_len, void* stream) {
  return ti_attention_i8_heads(q, 0, q_batch_stride, q_row_stride, k, 0, k_batch_stride, k_row_stride, vt, 0, vt_batch_stride,
                               vt_row_stride, out, 0, out_batch_stride, out_row_stride, batch == 0 ? 0 : 1, batch, S, T, D,
                               qk_alpha, score_scale, pv_alpha, causal_q_len, stream);
}
