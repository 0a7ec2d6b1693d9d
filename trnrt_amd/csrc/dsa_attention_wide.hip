// Sparse MLA attention over many query rows for gfx950 (the arithmetic of dsa_attention.hip, for a prefill chunk's queries
// and batches of decode rows: attention_wide_splits below has the rule): one workgroup = one query row, or one split of
// its slots, x 64 heads, so each gathered row serves 64 heads; with splits combine_splits_kernel follows.
//
// What bounds it: both products on v_mfma_f32_32x32x16_bf16 are 68 products of 32 cycles per chunk of 64 slots and
// SIMD (2,176 cycles), with e4m3 -> bf16 conversions of the keys (144 per wave) and the values (64). A wave issues at
// most one instruction about every 5 cycles whatever its kind, so one wave per SIMD doing everything takes 690 x 5 =
// 3,400 cycles a chunk however it is scheduled, and 8 alike waves that meet at two barriers a chunk (the form before:
// scores, a barrier, softmax, a barrier, values) took 8,100: nothing overlapped. So the two waves of a SIMD (waves w and
// w + 4 share one) have different work, and a chunk's stages run an interval apart with one barrier per interval:
//   - scoring waves 0-3, interval c: chunk c's scores, wave (th, hh) tokens 32 th .. + 31 x heads 32 hh .. + 31 (S^T =
//     K . Q^T, its 32 heads' queries in 144 registers), then P = 2^(s - m) x kv scale in bf16 into LDS;
//   - value waves 4-7, interval c: chunk c - 1's O += V^T . P, wave w dims 128 w .. + 127 of all 64 heads (128
//     registers, heads as columns so that a lane holds 4 consecutive dims), and the gather: chunk c + 1's rows from
//     registers into LDS and chunk c + 2's loads, piece by piece in the shadow of the products.
// About 3,100 cycles a chunk. 2,048 rows x 64 heads x 2,048 of 67,584 tokens, 576-wide: 865 -> 529 us = 1.10 PFLOP/s (the chip then
// lowers its clock to about 1.7 GHz: the power limit that also holds large matrix products at 1.4 PFLOP/s here); 512-wide
// with 16,896 pools 800 -> 540 us; 1,001 rows 450 -> 281 us.
// The online softmax rescales lazily without waiting for the chunk's maximum: P is taken against the running maximum as
// it stands; a wave that meets a score past its slack raises a flag, and before the chunk's values are multiplied every
// wave sees the flags (the same for all) and, when one is up, the maxima are exchanged, P is taken again and O rescaled
// (chunk 0 always does, with O still zero).
// LDS: three tiles of 64 rows (chunk c's keys, chunk c - 1's values, chunk c + 1 being stored) at a 576-byte stride,
// 16-byte piece p of row r at piece p ^ ((r >> 1) & 3): the stores of 8 lanes (2 rows x 4 pieces) and the reads of one
// piece of 8 rows (key operand, ds_read_b128; value operand, ds_read_b64_tr_b8) then cover the 32 banks once.
// Slot forms: token (idx + cnt + table, with the pooled variant of PoolForm) and rows + cnt; no bias array.
#include "dsa_common.h"

namespace dsa {

int attention_default_splits(int B, int H, int keep, int num_cu);

constexpr int AW_DV = 512;
constexpr int AW_HEADS = 64;
constexpr int AW_CH = 64;         // slots per chunk
constexpr int AW_THREADS = 512;   // 8 waves: 4 that score, 4 that gather and multiply values, one of each per SIMD
constexpr int AW_ROLE = AW_THREADS / 2;
constexpr int AW_MAXSLOTS = 33 * AW_CH;  // 2,112: keep 2,048 plus a pooled tail
constexpr int AW_SPT = (AW_MAXSLOTS + AW_THREADS - 1) / AW_THREADS;
constexpr int AW_KROW = 576;             // LDS row stride of a tile
constexpr int AW_OROW = AW_DV + 8;       // staged output row (elements)
constexpr int AW_PROW = AW_CH + 8;       // P row stride (bf16)
constexpr float AW_SLACK = 11.5f;        // lazy rescaling (base 2): p = 2^(s - m) <= 2^11.5 between moves of m
constexpr float AW_LOG2E = 1.44269504088896341f;
constexpr float AW_LOG2E_LO = (float)(1.44269504088896341 - (double)AW_LOG2E);
constexpr int AW_KAHEAD = 3;  // score steps whose key reads are in flight
constexpr int AW_VAHEAD = 3;  // value steps whose operand reads are in flight
constexpr int AW_STORE = 5;   // the value step that begins storing the next chunk's rows

typedef int aw_v2i __attribute__((ext_vector_type(2)));

struct AwShared {
  alignas(16) uint8_t kt[3][AW_CH * AW_KROW];  // token-major e4m3 rows of three chunks (the queries before them)
  alignas(16) uint16_t p[2][AW_HEADS * AW_PROW];  // bf16 P[head][token] of two chunks
  int slot[AW_MAXSLOTS];
  alignas(16) float ksc[AW_MAXSLOTS];  // the slots' kv scales
  alignas(16) float kfac[AW_MAXSLOTS]; // kv scale x softmax scale x log2 e (0 in a row with no live slot: its scores
                                       // are all alike)
  float cmax[2][AW_HEADS];             // [token half][head]: a chunk's maxima when one moves
  float al[AW_HEADS];                  // and its rescale factors
  alignas(16) int flag[2][4];          // per chunk parity and wave: a score past the running maximum's slack
  float lsum[2][AW_HEADS];             // [token half][head]: final sums
  float mfin[AW_HEADS];                // and maxima
};

// Every wave of the workgroup, whichever its role: LDS accesses before it are visible after it; global loads stay in
// flight.
__device__ __forceinline__ void aw_barrier() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup");
}

template <int DQK>
__global__ __launch_bounds__(AW_THREADS, 1) void sparse_mla_wide_kernel(
    const uint16_t* __restrict__ q, const uint8_t* __restrict__ kv, const float* __restrict__ kvs,
    const int* __restrict__ idx, const int* __restrict__ cnt, const int* __restrict__ table,
    const int* __restrict__ rows, uint16_t* __restrict__ out, float* __restrict__ out_f32,
    float* __restrict__ lse_out, float* __restrict__ ws_o, float* __restrict__ ws_ml, int H, int keep, int max_pages,
    int page_size, int num_pages, float scale, int splits, int sps, PoolForm pf) {
  constexpr int PAIRS = DQK / 32;  // 32 dims: one 16-byte read of a key row per lane, two MFMAs
  constexpr int PPT = DQK / 64;    // 16-byte pieces per gathering thread and chunk (4 threads a row)
  constexpr int QROW = DQK + 8;    // staged query row (bf16)
  constexpr int QPIECES = AW_HEADS * DQK / 8, QPT = QPIECES / AW_THREADS;
  static_assert(QPIECES % AW_THREADS == 0 && AW_HEADS * QROW * 2 <= 3 * AW_CH * AW_KROW, "query staging");
  __shared__ AwShared sh;
  const int HB = H / AW_HEADS;
  int x = blockIdx.x;
  const int hb64 = x % HB;
  x /= HB;
  const int sp = x % splits, b = x / splits;
  if (pf.n_live && b >= *pf.n_live) return;  // a row past the run-time live count: left unwritten
  const int tid = threadIdx.x, lane = tid & (WAVE - 1);
  const int wave = __builtin_amdgcn_readfirstlane(tid / WAVE);
  const int j = lane & 31, h = lane >> 5;
  const size_t hrow = ((size_t)b * splits + sp) * H + AW_HEADS * hb64;  // (splits 1: the output row itself)

  // one round of loads (no branch between them): the split's slot list as it lies, the 64 heads' queries
  const bool token_form = rows == nullptr;
  const int* trow = table ? table + (size_t)b * max_pages : nullptr;
  const int k0 = sp * sps;
  const int* list = token_form ? idx : rows;
  const int per_row = pf.kp_shift ? pf.idx_stride : keep;
  int slot_r[AW_SPT];
#pragma unroll
  for (int i = 0; i < AW_SPT; ++i) {
    const int k = k0 + min(AW_THREADS * i + tid, sps - 1);
    slot_r[i] = list[(size_t)b * per_row + min(k >> pf.kp_shift, per_row - 1)];
  }
  u32x4 qv[QPT];
  {
    const u32x4* qsrc = reinterpret_cast<const u32x4*>(q + ((size_t)b * H + AW_HEADS * hb64) * DQK);
#pragma unroll
    for (int i = 0; i < QPT; ++i) qv[i] = qsrc[tid + AW_THREADS * i];
  }
  // live slots: cnt_b of keep, at least one (a row with none attends slot 0 fully masked); this split's are
  // k0 .. k0 + n - 1
  int cnt_b = cnt[b];
  int pools_b = 0, tail_pool = 0;
  if (pf.kp_shift) {
    pools_b = min(max(cnt_b, 0), pf.idx_stride);
    tail_pool = max(pf.npool[b], 0);
    const int tail = min(max(pf.positions[b] + 1 - (tail_pool << pf.kp_shift), 0), (1 << pf.kp_shift) - 1);
    cnt_b = (pools_b << pf.kp_shift) + tail;
  }
  const int n_eff = cnt_b < 1 ? min(max(pf.empty_n, 1), keep) : (cnt_b > keep ? keep : cnt_b);
  const bool masked = cnt_b < 1;
  const int n = min(n_eff - k0, sps);
  if (n <= 0) {  // only with splits: the combine reads no outputs of a split whose sum is 0
    if (tid < AW_HEADS) {
      ws_ml[2 * (hrow + tid)] = -INFINITY;
      ws_ml[2 * (hrow + tid) + 1] = 0.0f;
    }
    return;
  }
  const int nch = (n + AW_CH - 1) / AW_CH;
  // scale x log2 e to twice fp32's digits: rounded, its error would be the same for every score, and so the lse's
  const float sl2 = scale * AW_LOG2E, sl2_lo = fmaf(scale, AW_LOG2E, -sl2) + scale * AW_LOG2E_LO;
  // slot list entries -> cache slots, the table's loads again in one round
  if (token_form) {
    int pr[AW_SPT], pg[AW_SPT];
    const int ps_shift = (page_size & (page_size - 1)) == 0 ? 31 - __builtin_clz(page_size) : -1;
#pragma unroll
    for (int i = 0; i < AW_SPT; ++i) {
      const int k = k0 + min(AW_THREADS * i + tid, sps - 1);
      int pos = slot_r[i];
      if (pf.kp_shift) {
        pos = (k >> pf.kp_shift) < pools_b ? pos : tail_pool;
        pos = (pos << pf.kp_shift) + (k & ((1 << pf.kp_shift) - 1));
      }
      pos = pos < 0 ? 0 : pos;
      const int pi = ps_shift >= 0 ? pos >> ps_shift : pos / page_size;
      pr[i] = pos - pi * page_size;
      pg[i] = pi < max_pages ? pi : max_pages - 1;
    }
#pragma unroll
    for (int i = 0; i < AW_SPT; ++i) pg[i] = trow[pg[i]];
#pragma unroll
    for (int i = 0; i < AW_SPT; ++i) slot_r[i] = safe_page(pg[i], num_pages) * page_size + pr[i];
  } else {
    const size_t nslots_cache = (size_t)num_pages * page_size;
#pragma unroll
    for (int i = 0; i < AW_SPT; ++i) slot_r[i] = ((size_t)(unsigned)slot_r[i] < nslots_cache) ? slot_r[i] : 0;
  }
  float ksc_r[AW_SPT];
#pragma unroll
  for (int i = 0; i < AW_SPT; ++i) ksc_r[i] = kvs ? kvs[slot_r[i]] : 1.0f;  // null: the unscaled cache
  uint16_t* qs = reinterpret_cast<uint16_t*>(&sh.kt[0][0]);
#pragma unroll
  for (int i = 0; i < QPT; ++i) {
    const int pc = tid + AW_THREADS * i;
    *reinterpret_cast<u32x4*>(qs + (pc / (DQK / 8)) * QROW + 8 * (pc % (DQK / 8))) = qv[i];
  }
#pragma unroll
  for (int i = 0; i < AW_SPT; ++i) {
    const int k = AW_THREADS * i + tid;
    if (k < nch * AW_CH) {  // (past the row's slots: weight 0, and the gather takes its last slot)
      const float ksc = k < n ? ksc_r[i] : 0.0f;
      sh.slot[k] = slot_r[i];
      sh.ksc[k] = ksc;
      sh.kfac[k] = masked ? 0.0f : fmaf(ksc, sl2, ksc * sl2_lo);
    }
  }
  if (tid < 4) sh.flag[1][tid] = 0;
  aw_barrier();

  if (wave < 4) {
    // -- the scores: wave (th, hh) takes tokens 32 th .. + 31 of a chunk for heads 32 hh .. + 31 --
    const int th = wave >> 1, hh = wave & 1;
    bf16x8 qb[2 * PAIRS];  // head 32 hh + j: pair s holds dims 32 s + 16 h .. + 15
    {
      const uint16_t* qh = qs + (32 * hh + j) * QROW + 16 * h;
#pragma unroll
      for (int s = 0; s < PAIRS; ++s) {
        qb[2 * s] = as_bf16x8(*reinterpret_cast<const uint4*>(qh + 32 * s));
        qb[2 * s + 1] = as_bf16x8(*reinterpret_cast<const uint4*>(qh + 32 * s + 8));
      }
    }
    aw_barrier();  // the queries are read
    aw_barrier();  // tile 0 is in place
    float m_run = 0.0f;  // running max (base 2) of head 32 hh + j (the same in both token halves and lane halves);
                         // chunk 0's scores are taken against 0, and its flags are always up
    float l_run = 0.0f;  // this lane's share of its running sum
    float psum = 0.0f;   // and of the last chunk's, not yet in l_run
    f32x16 sv = {};      // the last chunk's scores - m_run: head 32 hh + j, tokens 32 th + 8 (r / 4) + 4 h + r % 4
    // byte offsets in a tile (16-byte piece p of row r at piece p ^ ((r >> 1) & 3)) at even and odd pairs
    const int kf = (j >> 1) & 3;
    const int koff[2] = {(32 * th + j) * AW_KROW + 16 * (h ^ kf), (32 * th + j) * AW_KROW + 16 * ((2 | h) ^ kf)};
    uint16_t* const pw = &sh.p[0][(32 * hh + j) * AW_PROW + 32 * th + 4 * h];
    auto k_scales = [&](int c, int g) __attribute__((always_inline)) {
      return *reinterpret_cast<const f32x4*>(&sh.ksc[c * AW_CH + 32 * th + 8 * g + 4 * h]);
    };
    auto k_factors = [&](int c, int g) __attribute__((always_inline)) {
      return *reinterpret_cast<const f32x4*>(&sh.kfac[c * AW_CH + 32 * th + 8 * g + 4 * h]);
    };
    // four tokens (group g of the lane's 16) of P from their scores and scales
    auto p_group = [&](int c, int g, const f32x4& ks) __attribute__((always_inline)) {
      float pv[4];
#pragma unroll
      for (int e = 0; e < 4; ++e) pv[e] = __builtin_amdgcn_exp2f(sv[4 * g + e]);
      psum += (pv[0] + pv[1]) + (pv[2] + pv[3]);
      *reinterpret_cast<uint2*>(pw + (c & 1) * AW_HEADS * AW_PROW + 8 * g) =
          make_uint2(bf16_pack(pv[0] * ks[0], pv[1] * ks[1]), bf16_pack(pv[2] * ks[2], pv[3] * ks[3]));
    };
    // a chunk whose flags (fl) are up: its maxima over both token halves, the moved running maxima, P again
    auto settle = [&](int c, const int4& fl) __attribute__((always_inline)) {
      if (__builtin_amdgcn_readfirstlane(fl.x | fl.y | fl.z | fl.w)) {
        float cm = sv[0];
#pragma unroll
        for (int r = 1; r < 16; ++r) cm = max_nonan(cm, sv[r]);
        cm = max_nonan(cm, __shfl_xor(cm, 32, WAVE));
        if (h == 0) sh.cmax[th][32 * hh + j] = cm;
        aw_barrier();
        cm = max_nonan(cm, sh.cmax[th ^ 1][32 * hh + j]);
        const float up = c == 0 || cm > AW_SLACK ? cm : 0.0f;  // how far the maximum moves
        // chunk 0 has nothing to rescale, and its factor would be infinite where every score is at or below -128
        const float alpha = c == 0 ? 0.0f : __builtin_amdgcn_exp2f(-up);
        m_run += up;
        l_run *= alpha;
        psum = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; ++r) sv[r] -= up;
#pragma unroll
        for (int g = 0; g < 4; ++g) p_group(c, g, k_scales(c, g));
        if (th == 0 && h == 0) sh.al[32 * hh + j] = alpha;
        aw_barrier();
      }
      l_run += psum;
      psum = 0.0f;
    };
    auto flags = [&](int c) __attribute__((always_inline)) { return *reinterpret_cast<const int4*>(sh.flag[c & 1]); };
    const uint8_t* tile = sh.kt[0];
    __builtin_amdgcn_s_setprio(1);  // these waves bound the interval: their products go before the value products
    for (int c = 0; c < nch; ++c) {
      auto k_read = [&](int s) __attribute__((always_inline)) {
        return *reinterpret_cast<const u32x4*>(tile + koff[s & 1] + 64 * (s >> 1));
      };
      const int4 fl = flags(c - 1);
      f32x16 sa = {};
      u32x4 kk[AW_KAHEAD + 1];
      bf16x8 ka[2], kb[2];
      f32x4 ks[2], kx[2];
#pragma unroll
      for (int s = 0; s < AW_KAHEAD; ++s) kk[s] = k_read(s);
      __builtin_amdgcn_sched_barrier(0);
      settle(c - 1, fl);
      ka[0] = fp8x8_to_bf16x8(kk[0][0], kk[0][1]);
      kb[0] = fp8x8_to_bf16x8(kk[0][2], kk[0][3]);
#pragma unroll
      for (int s = 0; s < PAIRS; ++s) {
        if (s + AW_KAHEAD < PAIRS) kk[(s + AW_KAHEAD) % (AW_KAHEAD + 1)] = k_read(s + AW_KAHEAD);
        sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(ka[s & 1], qb[2 * s], sa, 0, 0, 0);
        sa = __builtin_amdgcn_mfma_f32_32x32x16_bf16(kb[s & 1], qb[2 * s + 1], sa, 0, 0, 0);
        if (s + 1 < PAIRS) {
          const u32x4 k1 = kk[(s + 1) % (AW_KAHEAD + 1)];
          ka[(s + 1) & 1] = fp8x8_to_bf16x8(k1[0], k1[1]);
          kb[(s + 1) & 1] = fp8x8_to_bf16x8(k1[2], k1[3]);
        }
        if (s == PAIRS - 2) {
          ks[0] = k_scales(c, 0);
          kx[0] = k_factors(c, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      if (c == nch - 1) {  // the slots past the row's
        const int lim = n - c * AW_CH - 32 * th - 4 * h;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          kx[0] = k_factors(c, g);
#pragma unroll
          for (int e = 0; e < 4; ++e) sv[4 * g + e] = 8 * g + e < lim ? fmaf(sa[4 * g + e], kx[0][e], -m_run) : -INFINITY;
        }
      } else {
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if (g < 3) kx[(g + 1) & 1] = k_factors(c, g + 1);
#pragma unroll
          for (int e = 0; e < 4; ++e) sv[4 * g + e] = fmaf(sa[4 * g + e], kx[g & 1][e], -m_run);
        }
      }
      float cm = -INFINITY;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if (g < 3) ks[(g + 1) & 1] = k_scales(c, g + 1);
#pragma unroll
        for (int e = 0; e < 4; ++e) cm = max_nonan(cm, sv[4 * g + e]);
        p_group(c, g, ks[g & 1]);
      }
      const bool any = c == 0 || __ballot(cm > AW_SLACK) != 0;
      if (lane == 0) sh.flag[c & 1][wave] = any;
      aw_barrier();
      tile = tile == sh.kt[2] ? sh.kt[0] : tile + AW_CH * AW_KROW;
    }
    __builtin_amdgcn_s_setprio(0);
    settle(nch - 1, flags(nch - 1));
    const float lw = l_run + __shfl_xor(l_run, 32, WAVE);
    if (h == 0) sh.lsum[th][32 * hh + j] = lw;
    if (th == 0 && h == 0) sh.mfin[32 * hh + j] = m_run;
    aw_barrier();
  } else {
    // -- the gather and the values: wave w takes dims 128 w .. + 127 of all 64 heads --
    const int w = wave - 4, rt = tid - AW_ROLE;
    const int gr = rt >> 2, gp = 16 * (rt & 3);  // the gather: row gr of the chunk, bytes gp + 64 i .. + 15
    const int gs = gr * AW_KROW + 16 * ((rt & 3) ^ ((gr >> 1) & 3));  // and where they go in a tile
    // (a list entry past the row's count may name a cache row that was never written, whose NaN times weight 0 is NaN)
    auto gslot = [&](int c) __attribute__((always_inline)) { return sh.slot[min(c * AW_CH + gr, n - 1)]; };
    u32x4 r0[PPT];
    auto gload = [&](int slot) __attribute__((always_inline)) {
      const uint8_t* src = kv + (size_t)slot * DQK + gp;
#pragma unroll
      for (int i = 0; i < PPT; ++i) r0[i] = *reinterpret_cast<const u32x4*>(src + 64 * i);
    };
    auto lstore = [&](uint8_t* tile) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < PPT; ++i) *reinterpret_cast<u32x4*>(tile + gs + 64 * i) = r0[i];
    };
    f32x16 o[4][2];  // [dim block][head block]: lane (j, h) head 32 i + j, dims 128 w + 32 d + 8 (r / 4) + 4 h + r % 4
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int i = 0; i < 2; ++i) o[d][i] = f32x16{};
    const int vf = (lane >> 2) & 3, vb0 = (lane >> 4) & 1;
    const int vrow = (8 * (lane >> 5) + ((lane & 15) >> 1)) * AW_KROW + 128 * w + 8 * (lane & 1);
    const int voff[2] = {vrow + 16 * (vb0 ^ vf), vrow + 16 * ((2 | vb0) ^ vf)};
    const uint16_t* const pr = &sh.p[0][j * AW_PROW + 8 * h];
    // the value operand of step i (tokens 16 (i / 4) .. + 15, dims 128 w + 32 (i % 4) .. + 31), read transposed
    auto v_read = [&](const uint8_t* kt, int i) __attribute__((always_inline)) {
      return __builtin_amdgcn_ds_read_tr8_b64_v2i32(
          (__attribute__((address_space(3))) aw_v2i*)(kt + voff[i & 1] + 16 * (i >> 2) * AW_KROW + 64 * ((i & 3) >> 1)));
    };
    auto p_read = [&](int pb, int t, int i) __attribute__((always_inline)) {
      return as_bf16x8(*reinterpret_cast<const uint4*>(pr + pb * AW_HEADS * AW_PROW + 32 * i * AW_PROW + 16 * t));
    };
    // chunk c's weights are final after this (and O on their maxima)
    auto settle = [&](int c) __attribute__((always_inline)) {
      const int4 fl = *reinterpret_cast<const int4*>(sh.flag[c & 1]);
      if (__builtin_amdgcn_readfirstlane(fl.x | fl.y | fl.z | fl.w)) {
        aw_barrier();
        aw_barrier();
        if (c > 0) {  // O is zero before
          const float a0 = sh.al[j], a1 = sh.al[32 + j];
#pragma unroll
          for (int d = 0; d < 4; ++d)
#pragma unroll
            for (int r = 0; r < 16; ++r) {
              o[d][0][r] *= a0;
              o[d][1][r] *= a1;
            }
        }
      }
    };
    // a chunk's value product: 16 steps of two products, the next steps' operands read and converted ahead
    auto value = [&](const uint8_t* kt, int pb, auto side) __attribute__((always_inline)) {
      aw_v2i vr[AW_VAHEAD + 1];
      bf16x8 pa[2][2], vb[2];
#pragma unroll
      for (int i = 0; i < AW_VAHEAD; ++i) vr[i] = v_read(kt, i);
#pragma unroll
      for (int i = 0; i < 2; ++i) pa[0][i] = p_read(pb, 0, i);
      vb[0] = fp8x8_to_bf16x8((uint32_t)vr[0].x, (uint32_t)vr[0].y);
#pragma unroll
      for (int i = 0; i < 16; ++i) {
        const int t = i >> 2, d = i & 3;
        if (i + AW_VAHEAD < 16) vr[(i + AW_VAHEAD) % (AW_VAHEAD + 1)] = v_read(kt, i + AW_VAHEAD);
        if (d < 2 && t < 3) pa[(t + 1) & 1][d] = p_read(pb, t + 1, d);
        o[d][0] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vb[i & 1], pa[t & 1][0], o[d][0], 0, 0, 0);
        o[d][1] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(vb[i & 1], pa[t & 1][1], o[d][1], 0, 0, 0);
        if (i < 15) {
          const aw_v2i r = vr[(i + 1) % (AW_VAHEAD + 1)];
          vb[(i + 1) & 1] = fp8x8_to_bf16x8((uint32_t)r.x, (uint32_t)r.y);
        }
        side(i);
        __builtin_amdgcn_sched_barrier(0);
      }
    };
    gload(gslot(0));
    aw_barrier();  // the queries are read
    lstore(sh.kt[0]);
    gload(gslot(1));
    aw_barrier();  // tile 0 is in place
    const uint8_t* tp = sh.kt[0];  // chunk c - 1's tile
    uint8_t* tn = sh.kt[1];        // chunk c + 1's
    for (int c = 0; c < nch; ++c) {
      settle(c - 1);
      const int slot2 = gslot(c + 2);
      const uint8_t* src = kv + (size_t)slot2 * DQK + gp;
      // piece by piece: chunk c + 1's into its tile, chunk c + 2's load in its register (one interval in flight)
      auto piece = [&](int i) __attribute__((always_inline)) {
        *reinterpret_cast<u32x4*>(tn + gs + 64 * i) = r0[i];
        r0[i] = *reinterpret_cast<const u32x4*>(src + 64 * i);
      };
      if (c > 0) {
        value(tp, (c - 1) & 1, [&](int i) __attribute__((always_inline)) {
          if (i >= AW_STORE && i < AW_STORE + PPT) piece(i - AW_STORE);
        });
        tp = tp == sh.kt[2] ? sh.kt[0] : tp + AW_CH * AW_KROW;
      } else {
#pragma unroll
        for (int i = 0; i < PPT; ++i) piece(i);
      }
      aw_barrier();
      tn = tn == sh.kt[2] ? sh.kt[0] : tn + AW_CH * AW_KROW;
    }
    settle(nch - 1);
    value(tp, (nch - 1) & 1, [](int) {});
    aw_barrier();
    // the outputs through LDS (the tiles are free), scaled by the row's sums
    const float i0 = 1.0f / (sh.lsum[0][j] + sh.lsum[1][j]), i1 = 1.0f / (sh.lsum[0][32 + j] + sh.lsum[1][32 + j]);
    if (out) {
      uint16_t* st = reinterpret_cast<uint16_t*>(&sh.kt[0][0]) + j * AW_OROW + 128 * w + 4 * h;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float f = i ? i1 : i0;
            *reinterpret_cast<uint2*>(st + 32 * i * AW_OROW + 32 * d + 8 * g) =
                make_uint2(bf16_pack(o[d][i][4 * g] * f, o[d][i][4 * g + 1] * f),
                           bf16_pack(o[d][i][4 * g + 2] * f, o[d][i][4 * g + 3] * f));
          }
    }
    float* of = ws_o ? ws_o : out_f32;
    if (of) {
      float* p = of + (hrow + j) * AW_DV + 128 * w + 4 * h;
#pragma unroll
      for (int i = 0; i < 2; ++i)
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int g = 0; g < 4; ++g) {
            const float f = i ? i1 : i0;
            *reinterpret_cast<f32x4*>(p + 32 * i * AW_DV + 32 * d + 8 * g) =
                f32x4{o[d][i][4 * g] * f, o[d][i][4 * g + 1] * f, o[d][i][4 * g + 2] * f, o[d][i][4 * g + 3] * f};
          }
    }
  }
  if (tid < AW_HEADS) {
    const float l = sh.lsum[0][tid] + sh.lsum[1][tid];
    const float m = masked ? NEG_INF : sh.mfin[tid];
    if (ws_o) {  // base 2, as the combine of this form takes it
      ws_ml[2 * (hrow + tid)] = m;
      ws_ml[2 * (hrow + tid) + 1] = l;
    } else if (lse_out) {
      lse_out[hrow + tid] = lse_base2(m, l);
    }
  }
  if (out) {
    aw_barrier();
    const uint16_t* st = reinterpret_cast<const uint16_t*>(&sh.kt[0][0]);
#pragma unroll
    for (int i = 0; i < AW_HEADS * AW_DV / 8 / AW_THREADS; ++i) {
      const int u = tid + AW_THREADS * i, head = u / (AW_DV / 8), pc = u % (AW_DV / 8);
      *reinterpret_cast<u32x4*>(out + (hrow + head) * AW_DV + 8 * pc) =
          *reinterpret_cast<const u32x4*>(st + head * AW_OROW + 8 * pc);
    }
  }
}

// The splits this form takes a launch of B rows of up to keep + tail slots in (tail: a pooled row's tokens past its
// selected pools'), or 0 when it does not take it: 64-head workgroups, the token form or rows + cnt (no bias array), at
// most AW_MAXSLOTS slots a split. An asked split count of 1 takes it when the rows fill the GPU. Left to the library
// (splits 0), launches of more than 8 workgroups' rows take it, measured against the split form (16 heads a workgroup)
// with its combine, 64 heads, 576-byte rows, 9 to 255 workgroups' rows of 64 to 2,048 slots (us):
// - up to 10 chunks of slots, one split and no combine: 9 rows of 128 slots 9.6 (split form 13.6, this form in 2 splits
//   15.3), 64 rows of 256 13.0 (15.5; 4 splits 26.1), 20 rows of 512 17.3 (26.6; 8 splits 22.9), 32 of 640 19.9 (23.5; 5
//   splits 22.7); of 11 and 12 chunks from 24 rows on: 64 rows of 768 23.4 (28.5; 4 splits 28.8);
// - the split form instead for up to 16 rows of 8 to 24 chunks where its workgroups are all resident at once (a second
//   round of them costs it 7 us): 10 rows of 512 16.1 (17.3 here), 9 of 640 16.3 (18.2), 16 of 1,024 20.9 (22.0), 10 of
//   1,536 20.7 (21.3);
// - otherwise as many splits as keep one workgroup a CU, at most 8 (256 slots at keep 2,048: past that the fp32 split
//   outputs cost what the shorter splits gain; of 3 chunks at least past 16 rows, where they are more: 32 rows of 1,024
//   24.7 in 6 splits, 26.1 in 8): 12 rows of 1,024 28.0 -> 20.3, of 2,048 slots 12 rows 37.1 -> 23.0, 16
//   rows 26.5 -> 24.8, 48 rows 67.6 -> 32.6, 96 rows 115 -> 45, 200 rows 225 -> 58; 128 heads, 24 rows of 512-byte rows
//   65 -> 31. (8 rows of 2,048, 21.5 and 21.9, stay with the split form.)
int attention_wide_splits(int B, int H, int keep, int tail, bool has_bias, int splits, int num_cu) {
  if (B < 1 || H < AW_HEADS || H % AW_HEADS || has_bias || keep < 1 || splits > 1) return 0;
  const long units = (long)B * (H / AW_HEADS), slots = (long)keep + tail;
  if (splits == 1) return slots <= AW_MAXSLOTS && units >= num_cu ? 1 : 0;
  if (units <= 8) return 0;
  const long chunks = (slots + AW_CH - 1) / AW_CH;
  if (units <= 16 && chunks >= 8 && chunks <= 24) {
    const int sp = attention_default_splits(B, H, keep, num_cu);
    const int sps = ((keep + sp - 1) / sp + AW_CH - 1) / AW_CH * AW_CH;
    if (4 * units * ((keep + sps - 1) / sps) <= num_cu) return 0;
  }
  if (chunks <= 10 || (chunks <= 12 && units >= 24)) return 1;
  long s = num_cu / units;
  s = s < 1 ? 1 : s > 8 ? 8 : s;
  if (units > 16 && s > (chunks + 2) / 3) s = (chunks + 2) / 3;
  const long sps = ((slots + s - 1) / s + AW_CH - 1) / AW_CH * AW_CH;
  return sps <= AW_MAXSLOTS ? (int)((slots + sps - 1) / sps) : 0;
}

// Whether `keep` slots in this many splits fit the kernel's slot lists.
bool attention_wide_fits(int keep, int splits) {
  return splits > 0 && ((keep + splits - 1) / splits + AW_CH - 1) / AW_CH * AW_CH <= AW_MAXSLOTS;
}

hipError_t launch_sparse_mla_wide(const uint16_t* q, const uint8_t* kv, const float* kvs, const int* idx,
                                  const int* cnt, const int* table, const int* rows, uint16_t* out, float* out_f32,
                                  float* lse, float* ws_o, float* ws_ml, int B, int H, int Dqk, int keep,
                                  int max_pages, int page_size, int num_pages, float scale, int splits, int sps,
                                  const PoolForm& pf, hipStream_t s) {
  const dim3 grid(B * splits * (H / AW_HEADS));
  return Dqk == 512 ? launch("sparse_mla_wide_kernel", sparse_mla_wide_kernel<512>, grid, dim3(AW_THREADS), s, q, kv,
                             kvs, idx, cnt, table, rows, out, out_f32, lse, ws_o, ws_ml, H, keep, max_pages,
                             page_size, num_pages, scale, splits, sps, pf)
                    : launch("sparse_mla_wide_kernel", sparse_mla_wide_kernel<576>, grid, dim3(AW_THREADS), s, q, kv,
                             kvs, idx, cnt, table, rows, out, out_f32, lse, ws_o, ws_ml, H, keep, max_pages,
                             page_size, num_pages, scale, splits, sps, pf);
}

}  // namespace dsa
