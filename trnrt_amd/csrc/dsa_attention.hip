// Sparse MLA decode attention for gfx950 over the selected tokens of a paged FP8 latent cache (the arithmetic of
// trnrt/kernels/dsa_decode.py:26-37 and trnrt/kernels/dsa_slots.py:48-65, absorbed MLA, with a 576-wide key of
// 512 latent + 64 rope columns, or GLM's 512-wide NoPE latent, and the first 512 columns as the value; per-token FP8
// scales):
//
//   s[h, k] = scale * q[h, :] . K[k] + bias[k],  K[k] = kv_fp8[slot_k] * kv_scale[slot_k]
//   o[h, :] = sum_k softmax_k(s)[h, k] * K[k][:512],  lse[h] = max_k s + log sum_k exp(s - max)
//
// Work unit: one workgroup = one sequence, 16 query heads, one split of the selected slots (split-K), 8 waves.
// The split's slot ids and the queries come in one round of loads; then the rows of up to 256 slots (4 chunks of 64)
// are gathered straight into LDS by direct-to-LDS loads (global_load_lds_dwordx4: consecutive lanes read
// consecutive 16-byte pieces of a row, no register staging), all issued at once, so the workgroup waits for memory
// twice: slot ids, then rows. A chunk is token-major e4m3 with a 592-byte row stride (36 pieces and one padding
// piece, filled with a copy of piece 35), which spreads the operand reads over the LDS banks. Both products run on
// v_mfma_f32_16x16x32_bf16 with e4m3 -> bf16 conversions in registers (exact):
//   - scores: S^T[token, head] = K . Q^T; 16 tokens per wave, all 16 heads, the 576 dims in 18 steps of 32 (at each
//     step the four lane groups read consecutive 8-byte pieces of a row, so lanes 0-31 and 32-63 each cover every
//     LDS bank once; q staged once through LDS);
//   - online softmax in fp32 with the chunk maximum shared through LDS;
//   - value: O[head, dim] += P . V with P = exp(s - m) * kv_scale rounded to bf16 (the dequantisation of the value
//     folded into the weight), its operand read transposed from the token-major rows by ds_read_b64_tr_b8.
// The two halves of the workgroup (waves 0-3, 4-7) take alternate chunks, each with its own running max, sum and
// output, merged at the end; within a half, wave w takes tokens 16w .. 16w + 15 for the scores and dims
// 128w .. 128w + 127 for the value product.
// With one split the workgroup writes bf16 o and lse; with several it writes fp32 partial o (normalised) with its
// running max and sum, and a combine kernel merges them by log-sum-exp (trnrt/models/mla.py:853-856, 1152-1160).
#include "dsa_common.h"

namespace dsa {

constexpr int ATT_DV = 512;      // the value: the first 512 columns of a row (the latent)
constexpr int ATT_HPW = 16;       // heads per workgroup
constexpr int ATT_CH = 64;        // slots per chunk
constexpr int ATT_THREADS = 512;  // 8 waves: two halves of 4
constexpr int ATT_NCH = 4;        // chunks staged in LDS at once
constexpr int ATT_SUPER = ATT_NCH * ATT_CH;  // slots staged at once
// Rows of DQK = 576 (512 latent + 64 rope, 36 16-byte pieces) or 512 (a NoPE latent, 32 pieces) columns; in LDS
// both take 37 pieces (592 bytes: the data and one or five padding pieces), the stride that spreads the operand
// reads over the banks.
constexpr int ATT_KPIECES = 37;
constexpr int ATT_KROW = 16 * ATT_KPIECES;   // 592 bytes
constexpr int ATT_CHUNK_BYTES = ATT_CH * ATT_KROW;  // 37,888: 37 direct-to-LDS instructions of 1 KiB
constexpr int ATT_LOADS = ATT_NCH * ATT_KPIECES;    // 148 instructions per staged super-chunk
constexpr int ATT_PROW = ATT_CH + 8;         // P row stride (bf16 elements; 16-byte aligned rows)
constexpr int ATT_TAIL_BYTES = 3584;         // a pooled tail staged apart: 7 rows of 512 bytes or 6 of 576

typedef int att_v2i __attribute__((ext_vector_type(2)));

struct AttShared {
  uint8_t kt[ATT_NCH][ATT_CHUNK_BYTES];  // token-major e4m3 rows of the staged chunks (q before them)
  uint16_t p[2][ATT_HPW * ATT_PROW];     // per half: bf16 P[head][token]
  int slot[ATT_SUPER];
  float kscale[ATT_SUPER];
  float bias[ATT_SUPER];
  float red[2][4][ATT_HPW];
  float ml[2][ATT_HPW];  // the second half's final max and sum per head, for the merge
  int tslot[8];          // the pooled tail's cache slots (kpool <= 8: at most 7 tail tokens) and scales
  float tks[8];
  uint8_t trows[ATT_TAIL_BYTES];  // the pooled tail's rows, loaded with the first super-chunk's
};

// The value operand of v_mfma_f32_16x16x32_bf16 straight from the token-major tile: ds_read_b64_tr_b8 gives lane
// (a = i / 8, c = i % 8) of each 16-lane block byte c of the 8-byte rows addressed by the block's lanes 2j + a,
// j = 0..7. Lane p of block q addresses token 32 ks + 8 q + p / 2 at dims 16 n + 8 (p & 1), so lane l receives dim
// 16 n + l % 16 of tokens 32 ks + 8 (l / 16) + j: the B operand with k-slot 8 q + j = that token.
__device__ __forceinline__ bf16x8 value_operand(const uint8_t* kt, int ks, int n, int lane) {
  const int q = lane >> 4, p = lane & 15;
  const uint8_t* a = kt + (32 * ks + 8 * q + (p >> 1)) * ATT_KROW + 16 * n + 8 * (p & 1);
  const att_v2i r = __builtin_amdgcn_ds_read_tr8_b64_v2i32((__attribute__((address_space(3))) att_v2i*)(a));
  return fp8x8_to_bf16x8((uint32_t)r.x, (uint32_t)r.y);
}

// Slot forms: token (idx + cnt + table: positions through the page table, bias 0 below cnt), rows + bias (cache
// slots with an additive bias), rows + cnt (cache slots, bias 0 below cnt). The token form's pooled variant (pf.kp_shift
// > 0, kpool = 1 << kp_shift): idx [B, pf.idx_stride] selected pools, cnt their count; the row attends the kpool
// tokens of each selected pool and then the tail: tokens kpool npool .. pos of its incomplete pool npool (none when
// pos + 1 is a multiple of kpool), token slot k = pool slot k >> kp_shift, token k & (kpool - 1) of that pool -- the
// slots of trnrt/models/dsa_long.py:189-215 in the same order, with the masked ones left out.
template <int DQK>
__global__ __launch_bounds__(ATT_THREADS, 1) void sparse_mla_kernel(
    const uint16_t* __restrict__ q, const uint8_t* __restrict__ kv, const float* __restrict__ kvs,
    const int* __restrict__ idx, const int* __restrict__ cnt, const int* __restrict__ table,
    const int* __restrict__ rows, const float* __restrict__ bias, uint16_t* __restrict__ out,
    float* __restrict__ out_f32, float* __restrict__ lse_out, float* __restrict__ ws_o, float* __restrict__ ws_ml,
    int B, int H, int keep, int max_pages, int page_size, int num_pages, float scale, int splits,
    int slots_per_split, PoolForm pf) {
  constexpr int ATT_PIECES = DQK / 16;  // 16-byte data pieces per row
  constexpr int ATT_QROW = DQK + 8;     // staged query row stride (bf16 elements)
  constexpr int STEPS = DQK / 32;       // score steps of 32 dims
  static_assert(ATT_PIECES < ATT_KPIECES && STEPS % 2 == 0, "row width");
  __shared__ AttShared sh;
  const int HG = H / ATT_HPW;
  const int groups = B * splits;
  // XCD-aware order: workgroup x runs on XCD x % 8; the HG head groups of one (sequence, split) read the same rows,
  // so they get ids that are equal mod 8 (the same XCD, the same L2).
  const int x = blockIdx.x;
  const int blk = x / (8 * HG), rem = x - blk * 8 * HG;
  const int hg = rem / 8;
  const int gi = blk * 8 + (rem - hg * 8);
  if (gi >= groups) return;
  const int b = gi / splits, sp = gi - b * splits;
  if (pf.n_live && b >= *pf.n_live) return;  // a row past the run-time live count: left unwritten

  const int tid = threadIdx.x, wave = tid / WAVE, lane = tid & (WAVE - 1);
  const int half = wave >> 2, wh = wave & 3;  // the half (alternate chunks) and the wave within it
  const int l16 = lane & 15, q4 = lane >> 4;
  const bool token_form = rows == nullptr;
  int n_eff = keep;
  int cnt_b = keep;
  int pools_b = 0, tail_pool = 0;  // pooled form: selected pools, the tail pool
  int tail_apart = 0;              // pooled form with the tail apart: the row's tail tokens
  if (cnt) {
    cnt_b = cnt[b];
    if (pf.kp_shift) {
      // token slots: kpool per selected pool, then the tail's tokens
      pools_b = min(max(cnt_b, 0), pf.idx_stride);
      tail_pool = max(pf.npool[b], 0);
      const int tail = min(max(pf.positions[b] + 1 - (tail_pool << pf.kp_shift), 0), (1 << pf.kp_shift) - 1);
      cnt_b = pools_b << pf.kp_shift;
      if (pf.tail_apart)
        tail_apart = tail;
      else
        cnt_b += tail;
    }
    // cnt 0: attend slot 0 (or the first pf.empty_n slots), fully masked
    if (!bias) n_eff = cnt_b < 1 ? min(max(pf.empty_n, 1), keep) : (cnt_b > keep ? keep : cnt_b);
  }
  const int k_begin = sp * slots_per_split;
  const int k_end = min(k_begin + slots_per_split, n_eff);
  // the workgroup that holds the row's last slot (n_eff >= 1 here, so it has slots of its own) adds the tail as one
  // more chunk: rows 0 .. tail_n - 1 of a zeroed tile, loaded into registers with its first super-chunk's rows
  const int tail_n = (tail_apart > 0 && (n_eff - 1) / slots_per_split == sp) ? tail_apart : 0;
  const size_t nslots_cache = (size_t)num_pages * page_size;

  // the queries of the 16 heads (16 or 18 KiB), staged through LDS below
  const uint4* qsrc = reinterpret_cast<const uint4*>(q + ((size_t)b * H + ATT_HPW * hg) * DQK);
  constexpr int QPIECES = ATT_HPW * DQK / 8;  // 16-byte pieces: 1024 or 1152
  uint4 qv[3];
#pragma unroll
  for (int i = 0; i < 3; ++i) qv[i] = qsrc[min(tid + ATT_THREADS * i, QPIECES - 1)];

  bf16x8 qb[STEPS];
  f32x4 o[8];
#pragma unroll
  for (int n = 0; n < 8; ++n) o[n] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  float m_run = -INFINITY;  // running max of head l16 over this half's chunks (the same in its 4 waves)
  float l_run = 0.0f;       // this lane's share of the half's running sum of head l16

  const int* trow = table ? table + (size_t)b * max_pages : nullptr;
  // one pair of staged chunks: half h takes chunk c0 + h of the nch staged (tile c, slots 64 c .. of the super-chunk)
  auto chunk_pair = [&](int c0, int nch) __attribute__((always_inline)) {
    const int c = c0 + half;  // this half's chunk of the pair
    const bool live = c < nch;
    const int cb = c * ATT_CH;
    const uint8_t* kt = sh.kt[live ? c : 0];
    float s4[4];
    float alpha = 1.0f;
    if (live) {
      // scores of tokens 16 wh .. 16 wh + 15, heads l16 (two accumulators: independent MFMA chains); lane group q4
      // reads 16 bytes of its row per pair of steps (dims 64 j + 16 q4 ..: one ds_read_b128 for two MFMAs, 8 rows
      // at one column covering the 32 banks once at the 592-byte stride)
      f32x4 acc0 = {0.0f, 0.0f, 0.0f, 0.0f}, acc1 = {0.0f, 0.0f, 0.0f, 0.0f};
      const uint8_t* kr = kt + (16 * wh + l16) * ATT_KROW + 16 * q4;
#pragma unroll
      for (int st = 0; st < STEPS; st += 2) {
        const u32x4 kk = *reinterpret_cast<const u32x4*>(kr + 32 * st);
        acc0 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16x8(kk[0], kk[1]), qb[st], acc0, 0, 0, 0);
        acc1 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fp8x8_to_bf16x8(kk[2], kk[3]), qb[st + 1], acc1, 0, 0, 0);
      }
      // acc[r] = S^T[token 16 wh + 4 q4 + r][head l16]
      float mx = -INFINITY;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int tk = cb + 16 * wh + 4 * q4 + r;
        s4[r] = (acc0[r] + acc1[r]) * (sh.kscale[tk] * scale) + sh.bias[tk];
        mx = fmaxf(mx, s4[r]);
      }
      mx = fmaxf(mx, __shfl_xor(mx, 16, WAVE));
      mx = fmaxf(mx, __shfl_xor(mx, 32, WAVE));
      if (lane < ATT_HPW) sh.red[half][wh][lane] = mx;
    }
    __syncthreads();  // the chunk maxima
    if (live) {
      const float mc = fmaxf(fmaxf(sh.red[half][0][l16], sh.red[half][1][l16]),
                             fmaxf(sh.red[half][2][l16], sh.red[half][3][l16]));
      const float m_new = fmaxf(m_run, mc);
      alpha = __expf(m_run - m_new);
      m_run = m_new;
      float psum = 0.0f;
      uint32_t pk[2];
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        const int tk = cb + 16 * wh + 4 * q4 + r;
        const float p0 = __expf(s4[r] - m_new), p1 = __expf(s4[r + 1] - m_new);
        psum += p0 + p1;
        pk[r / 2] = (uint32_t)f32_to_bf16_bits(p0 * sh.kscale[tk]) |
                    ((uint32_t)f32_to_bf16_bits(p1 * sh.kscale[tk + 1]) << 16);
      }
      l_run = l_run * alpha + psum;
      *reinterpret_cast<uint2*>(&sh.p[half][l16 * ATT_PROW + 16 * wh + 4 * q4]) = make_uint2(pk[0], pk[1]);
    }
    __syncthreads();  // P complete (and every wave has read the maxima)
    if (live) {
      // rescale O (rows = heads 4 q4 + r) and accumulate P . V over the chunk's 64 tokens (dims 128 wh ..)
      float al[4];
#pragma unroll
      for (int r = 0; r < 4; ++r) al[r] = __shfl(alpha, 4 * q4 + r, WAVE);
#pragma unroll
      for (int n = 0; n < 8; ++n)
#pragma unroll
        for (int r = 0; r < 4; ++r) o[n][r] *= al[r];
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        // P operand: head l16, tokens 32 ks + 8 q4 .. + 7 (the value operand's k-slot order)
        const bf16x8 pop =
            as_bf16x8(*reinterpret_cast<const uint4*>(&sh.p[half][l16 * ATT_PROW + 32 * ks + 8 * q4]));
#pragma unroll
        for (int n = 0; n < 8; ++n)
          o[n] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(pop, value_operand(kt, ks, 8 * wh + n, lane), o[n], 0, 0,
                                                         0);
      }
    }
    // the next pair's maxima and P are written after its first barrier, which every wave reaches only after
    // this pair's P . V
  };
  for (int sc0 = k_begin; sc0 < k_end; sc0 += ATT_SUPER) {
    const int nslots = min(ATT_SUPER, k_end - sc0);
    const int nch = (nslots + ATT_CH - 1) / ATT_CH;
    const bool tail_thread = sc0 == k_begin && tid >= ATT_SUPER && tid - ATT_SUPER < tail_n;
    // slot ids and biases, one per thread of the first 256 (past the split: slot 0's row with weight exactly 0)
    if (tail_thread) {
      // the tail tokens' cache slots, with the first super-chunk's
      const int pos = (tail_pool << pf.kp_shift) + (tid - ATT_SUPER);
      int pi = pos / page_size;
      pi = pi < max_pages ? pi : max_pages - 1;
      sh.tslot[tid - ATT_SUPER] = safe_page(trow[pi], num_pages) * page_size + (pos - (pos / page_size) * page_size);
    }
    if (tid < ATT_SUPER) {
      const int k = min(sc0 + tid, keep - 1);
      int slot;
      float bs;
      if (token_form) {
        int pos;
        if (pf.kp_shift) {
          const int j = k >> pf.kp_shift;
          const int pool = j < pools_b ? idx[(size_t)b * pf.idx_stride + j] : tail_pool;
          pos = (pool << pf.kp_shift) + (k & ((1 << pf.kp_shift) - 1));
        } else {
          pos = idx[(size_t)b * keep + k];
        }
        pos = pos < 0 ? 0 : pos;
        int pi = pos / page_size;
        pi = pi < max_pages ? pi : max_pages - 1;
        slot = safe_page(trow[pi], num_pages) * page_size + (pos - (pos / page_size) * page_size);
        bs = (k < cnt_b) ? 0.0f : NEG_INF;
      } else {
        slot = rows[(size_t)b * keep + k];
        slot = ((size_t)(unsigned)slot < nslots_cache) ? slot : 0;
        bs = bias ? bias[(size_t)b * keep + k] : ((k < cnt_b) ? 0.0f : NEG_INF);
      }
      sh.slot[tid] = slot;
      sh.bias[tid] = tid < nslots ? bs : -INFINITY;
    }
    __syncthreads();
    if (sc0 == k_begin) {
      // query operand: head 16hg + l16, dims 32 st + 8 q4 .. + 7 at step st, through the rows' LDS (q rows padded
      // by 8 elements so the operand reads spread over the banks)
      uint16_t* qs = reinterpret_cast<uint16_t*>(sh.kt[ATT_NCH - 1]);
#pragma unroll
      for (int i = 0; i < 3; ++i) {
        const int pc = tid + ATT_THREADS * i;  // 16-byte piece: head pc / (DQK / 8), elements 8 (pc % (DQK / 8)) ..
        if (pc < QPIECES)
          *reinterpret_cast<uint4*>(qs + (pc / (DQK / 8)) * ATT_QROW + 8 * (pc % (DQK / 8))) = qv[i];
      }
      __syncthreads();
      // in the key operand's dim order: steps 2 j, 2 j + 1 give lane group q4 dims 64 j + 16 q4 + 8 (st % 2) .. + 7
      const uint16_t* qh = qs + l16 * ATT_QROW + 16 * q4;
#pragma unroll
      for (int st = 0; st < STEPS; ++st)
        qb[st] = as_bf16x8(*reinterpret_cast<const uint4*>(qh + 64 * (st >> 1) + 8 * (st & 1)));
      __syncthreads();  // every wave holds its operand before the rows overwrite it
    }
    // every staged row straight into LDS: instruction kk (chunk kk / 37, 1-KiB block j = kk % 37 of its tile) has
    // lane l load 16-byte unit u = 64 j + l of the tile: row u / 37, piece u % 37 (a padding piece re-reads the
    // last data piece);
    // the 148 instructions are spread over the 8 waves
    {
      int src_slot[(ATT_LOADS + 7) / 8];
#pragma unroll
      for (int i = 0; i < (ATT_LOADS + 7) / 8; ++i) {
        const int kk = min(wave + 8 * i, ATT_LOADS - 1);
        const int c = kk / ATT_KPIECES, j = kk - c * ATT_KPIECES;
        const int rr = c * ATT_CH + (WAVE * j + lane) / ATT_KPIECES;
        src_slot[i] = sh.slot[rr < nslots ? rr : 0];
      }
#pragma unroll
      for (int i = 0; i < (ATT_LOADS + 7) / 8; ++i) {
        const int kk = wave + 8 * i;
        const int c = kk / ATT_KPIECES, j = kk - c * ATT_KPIECES;
        if (kk < ATT_LOADS && c < nch) {
          const int u = WAVE * j + lane;
          const int pc = u - (u / ATT_KPIECES) * ATT_KPIECES;
          const uint8_t* src = kv + (size_t)src_slot[i] * DQK + 16 * (pc < ATT_PIECES ? pc : ATT_PIECES - 1);
          __builtin_amdgcn_global_load_lds(src, (__attribute__((address_space(3))) void*)&sh.kt[c][1024 * j], 16, 0,
                                           0);
        }
      }
    }
    // the tail rows straight into their own LDS (rows of DQK bytes), beside the first super-chunk's rows: lane l of
    // wave w < 4 loads piece 64 w + l of the tail
    if (sc0 == k_begin && wave < 4) {
      const int u = WAVE * wave + lane;
      if (u < tail_n * ATT_PIECES)
        __builtin_amdgcn_global_load_lds(kv + (size_t)sh.tslot[u / ATT_PIECES] * DQK + 16 * (u % ATT_PIECES),
                                         (__attribute__((address_space(3))) void*)&sh.trows[1024 * wave], 16, 0, 0);
    }
    // (kvs null: the reference's unscaled cache, scale 1)
    const float ksc = tid < ATT_SUPER ? (kvs ? kvs[sh.slot[tid < nslots ? tid : 0]] : 1.0f)
                                      : (tail_thread ? (kvs ? kvs[sh.tslot[tid - ATT_SUPER]] : 1.0f) : 0.0f);
    __builtin_amdgcn_s_waitcnt(0);  // this thread's rows are in LDS
    if (tid < ATT_SUPER)
      sh.kscale[tid] = ksc;
    else if (tail_thread)
      sh.tks[tid - ATT_SUPER] = ksc;
    __syncthreads();  // every wave's rows are in LDS
    for (int c0 = 0; c0 < nch; c0 += 2) chunk_pair(c0, nch);
    __syncthreads();  // the next super-chunk overwrites the staged rows and slots
  }
  if (tail_n > 0) {
    // the tail chunk: its rows copied into tile 0, every other row of the tile zero (finite operands where the
    // weight is 0), scales and biases for 64 slots
    for (int i = tid; i < ATT_CH * ATT_KPIECES; i += ATT_THREADS)
      if (i / ATT_KPIECES >= tail_n) *reinterpret_cast<u32x4*>(&sh.kt[0][16 * i]) = u32x4{0u, 0u, 0u, 0u};
    if (tid < tail_n * ATT_PIECES)
      *reinterpret_cast<u32x4*>(&sh.kt[0][(tid / ATT_PIECES) * ATT_KROW + 16 * (tid % ATT_PIECES)]) =
          *reinterpret_cast<const u32x4*>(&sh.trows[16 * tid]);
    if (tid < ATT_CH) {
      sh.kscale[tid] = tid < tail_n ? sh.tks[tid] : 0.0f;
      sh.bias[tid] = tid < tail_n ? 0.0f : -INFINITY;
    }
    __syncthreads();
    chunk_pair(0, 1);
  }

  // each half's row sums: lane shares -> per wave -> per half
  float lw = l_run;
  lw += __shfl_xor(lw, 16, WAVE);
  lw += __shfl_xor(lw, 32, WAVE);
  if (lane < ATT_HPW) sh.red[half][wh][lane] = lw;
  __syncthreads();
  const float l_half = sh.red[half][0][l16] + sh.red[half][1][l16] + sh.red[half][2][l16] + sh.red[half][3][l16];
  // merge the halves: the second half hands its max, sum and output to the first through LDS (the staged rows are
  // no longer needed)
  float* xo = reinterpret_cast<float*>(sh.kt[0]);  // [4 waves][32 values][64 lanes]
  if (half == 1) {
#pragma unroll
    for (int n = 0; n < 8; ++n)
#pragma unroll
      for (int r = 0; r < 4; ++r) xo[(wh * 32 + 4 * n + r) * WAVE + lane] = o[n][r];
    if (wh == 0 && lane < ATT_HPW) {
      sh.ml[0][lane] = m_run;
      sh.ml[1][lane] = l_half;
    }
  }
  __syncthreads();
  const bool writer = half == 0;  // the first half writes the merged result
  const float m1 = sh.ml[0][l16], l1 = sh.ml[1][l16];
  const float m_tot = fmaxf(m_run, m1);
  const float a0 = m_run == -INFINITY ? 0.0f : __expf(m_run - m_tot);
  const float a1 = m1 == -INFINITY ? 0.0f : __expf(m1 - m_tot);
  const float l_tot = a0 * l_half + a1 * l1;
  float lr[4], mr[4], a0r[4], a1r[4];
#pragma unroll
  for (int r = 0; r < 4; ++r) {
    lr[r] = __shfl(l_tot, 4 * q4 + r, WAVE);
    mr[r] = __shfl(m_tot, 4 * q4 + r, WAVE);
    a0r[r] = __shfl(a0, 4 * q4 + r, WAVE);
    a1r[r] = __shfl(a1, 4 * q4 + r, WAVE);
  }
#pragma unroll
  for (int n = 0; n < 8; ++n)
#pragma unroll
    for (int r = 0; r < 4; ++r) o[n][r] = a0r[r] * o[n][r] + a1r[r] * xo[(wh * 32 + 4 * n + r) * WAVE + lane];
  const bool empty = k_begin >= k_end;
  if (splits == 1) {
    if (writer) {
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const int head = ATT_HPW * hg + 4 * q4 + r;
        const float inv = 1.0f / lr[r];
#pragma unroll
        for (int n = 0; n < 8; ++n) {
          const int dim = 128 * wh + 16 * n + l16;
          const float v = o[n][r] * inv;
          const size_t oi = ((size_t)b * H + head) * ATT_DV + dim;
          if (out) out[oi] = f32_to_bf16_bits(v);
          if (out_f32) out_f32[oi] = v;
        }
        if (lse_out && wh == 0 && l16 == 0) lse_out[(size_t)b * H + head] = mr[r] + __logf(lr[r]);
      }
    }
    return;
  }
  if (writer) {
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int head = ATT_HPW * hg + 4 * q4 + r;
      const float inv = empty ? 0.0f : 1.0f / lr[r];
      const size_t base = (((size_t)b * splits + sp) * H + head) * ATT_DV;
#pragma unroll
      for (int n = 0; n < 8; ++n) ws_o[base + 128 * wh + 16 * n + l16] = o[n][r] * inv;
      // the split's running max and sum, not its lse: at a fully masked row lse = -1e30 + log(sum) rounds to -1e30
      // in fp32 and would lose the sums that weight the splits
      if (wh == 0 && l16 == 0) {
        const size_t mi = (((size_t)b * splits + sp) * H + head) * 2;
        ws_ml[mi] = empty ? -INFINITY : mr[r];
        ws_ml[mi + 1] = empty ? 0.0f : lr[r];
      }
    }
  }
}

// o = sum_s W_s o_s / sum_s W_s with W_s = l_s exp(m_s - M), M = max_s m_s, and lse = M + log sum_s W_s, per
// (sequence, head), from each split's normalised o_s, max m_s and sum l_s (the log-sum-exp combine of
// trnrt/models/mla.py:853-856 with lse_s = m_s + log l_s kept in two parts); 128 threads x 4 dims. Every load is
// issued before any is used (one memory round trip; unconditional, so the waits count exactly). An empty split of the
// split form has o_s 0 and weight 0. The many-row form (MANY) leaves its empty splits' o_s unwritten, so only o_0 is read
// before the sums are there; the others' loads follow them, a split with no slot repeating o_0's. That wait costs 0.1 to
// 0.2 us of a step whose splits are all full (13 rows, 128 heads: 42.45 -> 42.55 us); the zeros that it saves, 128 KiB a
// split written and read, cost 30 rows of 40 slots (keep 2,048, 8 splits, 64 heads) 22.1 us against 18.9, 16 rows of 300
// 20.6 against 19.5, a step of 17 rows of up to 300 tokens and 128 heads 37.8 against 30.9. S is the next of 2, 4 and 8:
// a thread's loads past the splits cost 128 rows in 2 splits 2 us.
template <int S, bool MANY>
__global__ __launch_bounds__(128) void combine_splits_kernel(const float* __restrict__ ws_o,
                                                             const float* __restrict__ ws_ml, int H, int splits,
                                                             uint16_t* __restrict__ out, float* __restrict__ out_f32,
                                                             float* __restrict__ lse_out,
                                                             const int* __restrict__ n_live) {
  // (the many-row form has at most 128 rows where it has splits: a grid of two dimensions, no division)
  const int b = MANY ? blockIdx.y : blockIdx.x / H, head = MANY ? blockIdx.x : blockIdx.x - b * H;
  if (!MANY && n_live && b >= *n_live) return;  // a row past the run-time live count: left unwritten
  const int d = 4 * threadIdx.x;
  // split s of the row: its o_s at o + s so, its (m_s, l_s) at m + s sm
  const size_t i0 = (size_t)b * splits * H + head;
  const float* o = ws_o + i0 * ATT_DV + d;
  const float* m = ws_ml + 2 * i0;
  const int so = H * ATT_DV, sm = 2 * H;
  float2 ml[S];
  float4 v[S];
  constexpr int FIRST = MANY ? 1 : S;  // split 0 always holds slots
#pragma unroll
  for (int s = 0; s < S; ++s) {
    ml[s] = *reinterpret_cast<const float2*>(m + (size_t)min(s, splits - 1) * sm);
    if (s < FIRST) v[s] = *reinterpret_cast<const float4*>(o + (size_t)min(s, splits - 1) * so);
  }
  if (MANY) __builtin_amdgcn_sched_barrier(0);
#pragma unroll
  for (int s = FIRST; s < S; ++s) {  // (as whole numbers: a scalar compare; l_s is +0 or not)
    const size_t at = (size_t)min(s, splits - 1) * so;
    v[s] = *reinterpret_cast<const float4*>(o + (__float_as_int(ml[s].y) ? at : 0));
  }
  if (MANY && n_live && b >= *n_live) return;
  float M = -INFINITY;
#pragma unroll
  for (int s = 0; s < S; ++s) M = s < splits ? fmaxf(M, ml[s].x) : M;
  float W = 0.0f;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
  for (int s = 0; s < S; ++s) {
    const float dm = ml[s].x - M;  // (MANY: base 2)
    const float wt = (s < splits && ml[s].y > 0.0f) ? ml[s].y * (MANY ? __builtin_amdgcn_exp2f(dm) : __expf(dm)) : 0.0f;
    W += wt;
    acc.x += wt * v[s].x;
    acc.y += wt * v[s].y;
    acc.z += wt * v[s].z;
    acc.w += wt * v[s].w;
  }
  const float inv = 1.0f / W;
  const size_t oi = ((size_t)b * H + head) * ATT_DV + d;
  if (out) {
    const uint32_t lo = f32_to_bf16_bits(acc.x * inv) | ((uint32_t)f32_to_bf16_bits(acc.y * inv) << 16);
    const uint32_t hi = f32_to_bf16_bits(acc.z * inv) | ((uint32_t)f32_to_bf16_bits(acc.w * inv) << 16);
    *reinterpret_cast<uint2*>(&out[oi]) = make_uint2(lo, hi);
  }
  if (out_f32)
    *reinterpret_cast<float4*>(&out_f32[oi]) = make_float4(acc.x * inv, acc.y * inv, acc.z * inv, acc.w * inv);
  if (lse_out && threadIdx.x == 0) lse_out[(size_t)b * H + head] = MANY ? lse_base2(M, W) : M + __logf(W);
}

// Token positions -> cache slots and biases (the kp = 1 form of trnrt/models/dsa_long.py:189-215).
__global__ void token_rows_kernel(const int* __restrict__ idx, const int* __restrict__ cnt,
                                  const int* __restrict__ table, int* __restrict__ rows, float* __restrict__ bias,
                                  int keep, int max_pages, int page_size, int num_pages) {
  const int b = blockIdx.y;
  const int k = blockIdx.x * blockDim.x + threadIdx.x;
  if (k >= keep) return;
  const bool live = k < cnt[b];
  int pos = live ? idx[(size_t)b * keep + k] : 0;
  pos = pos < 0 ? 0 : pos;
  int pi = pos / page_size;
  pi = pi < max_pages ? pi : max_pages - 1;
  const int page = safe_page(table[(size_t)b * max_pages + pi], num_pages);
  rows[(size_t)b * keep + k] = page * page_size + pos % page_size;
  if (bias) bias[(size_t)b * keep + k] = live ? 0.0f : NEG_INF;
}

// The attention's slots of query n (the arithmetic of trnrt/models/dsa_long.py:189-215 `slots` for any kpool kp):
// slot s < keep the selected pool pools[n, s] (taken when s < cnt[n]), slot keep the query's tail pool npool[n]
// (its tokens kp npool .. positions[n]), the rest pool 0 (masked); rows = the pool's row of the latent cache viewed
// as [slots / kp, kp R] through the query's table, bias 0 for every token to attend and NEG_INF otherwise.
__global__ void pool_slots_kernel(const int* __restrict__ pools, const int* __restrict__ cnt,
                                  const int* __restrict__ npool, const int* __restrict__ positions,
                                  const int* __restrict__ table, int table_shared, int* __restrict__ rows,
                                  float* __restrict__ bias, int keep, int n_slots, int table_pages, int ppp, int kp) {
  const int n = blockIdx.y;
  const int s = blockIdx.x * blockDim.x + threadIdx.x;
  if (s >= n_slots) return;
  const int last_pool = table_pages * ppp - 1;
  const int np = npool[n];
  int pl = s < keep ? pools[(size_t)n * keep + s] : (s == keep ? min(np, last_pool) : 0);
  pl = min(max(pl, 0), last_pool);  // in range whatever the inputs
  const int pg = pl / ppp;
  const int* tab = table + (table_shared ? 0 : (size_t)n * table_pages);
  rows[(size_t)n * n_slots + s] = tab[pg] * ppp + (pl - pg * ppp);
  const bool sel_ok = s < keep && s < cnt[n];
  const int pos = positions[n];
  for (int t = 0; t < kp; ++t) {
    const bool tail_ok = s == keep && (long)np * kp + t <= (long)pos;
    bias[((size_t)n * n_slots + s) * kp + t] = (sel_ok || tail_ok) ? 0.0f : NEG_INF;
  }
}

hipError_t launch_pool_slots(const int* pools, const int* cnt, const int* npool, const int* positions,
                             const int* table, int table_shared, int* rows, float* bias, int N, int keep, int n_slots,
                             int table_pages, int page_size, int kp, hipStream_t s) {
  return launch("pool_slots_kernel", pool_slots_kernel, dim3((n_slots + 255) / 256, N), dim3(256), s, pools, cnt,
                npool, positions, table, table_shared, rows, bias, keep, n_slots, table_pages, page_size / kp, kp);
}

int attention_default_splits(int B, int H, int keep, int num_cu) {
  const int wgs = B * (H / ATT_HPW);
  int max_splits = (keep + ATT_CH - 1) / ATT_CH;
  max_splits = max_splits > 32 ? 32 : max_splits;
  int s = (num_cu + wgs - 1) / (wgs > 0 ? wgs : 1);
  s = s < 1 ? 1 : s;
  return s > max_splits ? max_splits : s;
}

size_t attention_workspace_bytes(int B, int H, int splits) {
  if (splits <= 1) return 0;
  return (size_t)B * splits * H * ATT_DV * 4 + (size_t)B * splits * H * 8 + 256;
}

static hipError_t combine(const float* ws_o, const float* ws_ml, int B, int H, int splits, bool many, uint16_t* out,
                          float* out_f32, float* lse, const int* n_live, hipStream_t s) {
  const dim3 grid(B * H), block(128);
  if (many && splits > 8) return hipErrorInvalidValue;  // (attention_wide_splits)
  if (many) {
    const dim3 grid2(H, B);
    if (splits <= 2)
      return launch("combine_splits_kernel", combine_splits_kernel<2, true>, grid2, block, s, ws_o, ws_ml, H, splits,
                    out, out_f32, lse, n_live);
    if (splits <= 4)
      return launch("combine_splits_kernel", combine_splits_kernel<4, true>, grid2, block, s, ws_o, ws_ml, H, splits,
                    out, out_f32, lse, n_live);
    return launch("combine_splits_kernel", combine_splits_kernel<8, true>, grid2, block, s, ws_o, ws_ml, H, splits, out,
                  out_f32, lse, n_live);
  }
  if (splits <= 8)
    return launch("combine_splits_kernel", combine_splits_kernel<8, false>, grid, block, s, ws_o, ws_ml, H, splits, out,
                  out_f32, lse, n_live);
  if (splits <= 16)
    return launch("combine_splits_kernel", combine_splits_kernel<16, false>, grid, block, s, ws_o, ws_ml, H, splits,
                  out, out_f32, lse, n_live);
  return launch("combine_splits_kernel", combine_splits_kernel<32, false>, grid, block, s, ws_o, ws_ml, H, splits, out,
                out_f32, lse, n_live);
}

hipError_t launch_sparse_mla_wide(const uint16_t* q, const uint8_t* kv, const float* kvs, const int* idx,
                                  const int* cnt, const int* table, const int* rows, uint16_t* out, float* out_f32,
                                  float* lse, float* ws_o, float* ws_ml, int B, int H, int Dqk, int keep,
                                  int max_pages, int page_size, int num_pages, float scale, int splits, int sps,
                                  const PoolForm& pf, hipStream_t s);

// keep: slots per row; in the pooled form (pf.kp_shift > 0) kpool x pf.idx_stride, the selected pools' tokens, with
// the row's tail tokens on top.
hipError_t launch_sparse_mla(const uint16_t* q, const uint8_t* kv, const float* kvs, const int* idx, const int* cnt,
                             const int* table, const int* rows, const float* bias, uint16_t* out, float* out_f32,
                             float* lse, void* ws, int B, int H, int Dqk, int keep, int max_pages, int page_size,
                             int num_pages, float scale, int splits, hipStream_t s, PoolForm pf, bool wide) {
  if (wide) {
    // the many-row form takes the pooled tail among its slots: kpool more
    if (pf.kp_shift) keep += 1 << pf.kp_shift;
    pf.tail_apart = 0;
    const int sps = ((keep + splits - 1) / splits + ATT_CH - 1) / ATT_CH * ATT_CH;
    const int eff = (keep + sps - 1) / sps;
    float* ws_o = eff > 1 ? static_cast<float*>(ws) : nullptr;
    float* ws_ml = eff > 1 ? ws_o + (size_t)B * eff * H * ATT_DV : nullptr;
    const hipError_t e = launch_sparse_mla_wide(q, kv, kvs, idx, cnt, table, rows, eff > 1 ? nullptr : out,
                                                eff > 1 ? nullptr : out_f32, lse, ws_o, ws_ml, B, H, Dqk, keep,
                                                max_pages, page_size, num_pages, scale, eff, sps, pf, s);
    return e != hipSuccess || eff == 1 ? e : combine(ws_o, ws_ml, B, H, eff, true, out, out_f32, lse, pf.n_live, s);
  }
  // the split form adds the pooled tail apart from its keep slots when its rows fit their LDS (kpool 8 with 576-wide
  // rows: 7 x 576 bytes do not; the tail is then among the slots, keep + kpool of them)
  pf.tail_apart = pf.kp_shift && ((1 << pf.kp_shift) - 1) * Dqk <= ATT_TAIL_BYTES;
  if (pf.kp_shift && !pf.tail_apart) keep += 1 << pf.kp_shift;
  const int HG = H / ATT_HPW;
  // slots per split: a whole number of chunks
  int sps = (keep + splits - 1) / splits;
  sps = (sps + ATT_CH - 1) / ATT_CH * ATT_CH;
  const int eff_splits = (keep + sps - 1) / sps;
  const int groups = B * eff_splits;
  const int grid = (groups + 7) / 8 * 8 * HG;
  float* ws_o = nullptr;
  float* ws_ml = nullptr;
  if (eff_splits > 1) {
    ws_o = static_cast<float*>(ws);
    ws_ml = ws_o + (size_t)B * eff_splits * H * ATT_DV;  // [B, splits, H, 2]: max, sum
  }
  hipError_t e =
      Dqk == 512
          ? launch("sparse_mla_kernel", sparse_mla_kernel<512>, dim3(grid), dim3(ATT_THREADS), s, q, kv, kvs, idx, cnt,
                   table, rows, bias, out, out_f32, lse, ws_o, ws_ml, B, H, keep, max_pages, page_size, num_pages,
                   scale, eff_splits, sps, pf)
          : launch("sparse_mla_kernel", sparse_mla_kernel<576>, dim3(grid), dim3(ATT_THREADS), s, q, kv, kvs, idx, cnt,
                   table, rows, bias, out, out_f32, lse, ws_o, ws_ml, B, H, keep, max_pages, page_size, num_pages,
                   scale, eff_splits, sps, pf);
  return e != hipSuccess || eff_splits == 1 ? e
                                             : combine(ws_o, ws_ml, B, H, eff_splits, false, out, out_f32, lse,
                                                       pf.n_live, s);
}

hipError_t launch_token_rows(const int* idx, const int* cnt, const int* table, int* rows, float* bias, int B,
                             int keep, int max_pages, int page_size, int num_pages, hipStream_t s) {
  launch("token_rows_kernel", token_rows_kernel, dim3((keep + 255) / 256, B), dim3(256), s, idx, cnt, table, rows, bias,
                     keep, max_pages, page_size, num_pages);
  return hipGetLastError();
}

}  // namespace dsa
