// Token recurrence of the gated delta rule: recurrent_kernel (decode,
// spec-verify, short steps) and recurrent_tokens_kernel (sequences of many
// tokens, below).
//
// recurrent_kernel: one workgroup owns a [KD x VT] column slice of one (sequence, v-head)
// state (KD = 128 by default; 64 and 256 are also built, and any v head dim
// that is a multiple of VT) and keeps it in registers for all of the
// sequence's tokens: the
// state is read from HBM once and written once, so decode is a pure stream
// of the fp32 state (the HBM roofline).  Thread mapping (NT = 2*VT threads):
//   columns: 4 per thread (float4), TPR = VT/4 threads span the slice;
//   rows:    8 row groups, thread row group rg owns rows rg + 8r, r < KD / 8.
// Per token the two K-reductions k~^T S and q~^T S are done together: in
// registers over 16 rows, xor-shuffles across the row groups of a wave, and
// LDS across waves when VT > 32.  The output uses
//   o = q~^T (e^g S + k~ d^T) = e^g (q~^T S) + (q~ . k~) d,
// so no second reduction is needed after the rank-1 update.
//
// Semantics: transformers modeling_qwen3_5_moe.py:331-381 (the torch
// recurrence the reference imports at engine/runtime/cuda_graphs.py:126-135).
#include <algorithm>

#include "gdn_common.h"

namespace gdn {
namespace {

typedef __attribute__((ext_vector_type(4))) float f32x4;
typedef __attribute__((ext_vector_type(2))) float f32x2;
typedef __attribute__((ext_vector_type(4))) unsigned u32x4;

constexpr int KD_DEFAULT = 128;  // head dim of k (rows of the state) of the tuned build
constexpr int VD_DEFAULT = 128;  // head dim of v (columns of the state)

struct RecArgs {
  const void *q, *k, *v;
  int64_t qs, ks, vs;  // token strides (elements)
  GateArgs gate;
  const float *state_in;
  const int64_t *in_idx;
  int64_t in_rows;
  float *state_out;
  const int64_t *out_idx;
  int64_t out_rows;
  void *o;
  float *snap;
  const int32_t *cu;
  int n_seqs, T, Hk, Hv;
  int V;  // v head dim (a multiple of the workgroup's columns)
  int64_t total;
  float scale;
  int l2norm;
  int qkv_dt, o_dt;
  int head_major;  // workgroup order: v-head fastest (a capped decode grid) or column block fastest
};

// Workgroup shape: 32 state columns, 64 threads (one wave, 16 rows per
// thread, 149 VGPRs, 3 waves per SIMD; capped at 128 it spills and takes
// 64.3 us).  Measured at B=64 on MI355X, before the first token's inputs were
// requested ahead of the state: 56.0 us;
// 128 threads (8 rows per thread, 4 waves per SIMD) 58.5 us; 256 threads
// 62.7 us -- more waves per workgroup cost a cross-wave reduction per token.
constexpr int REC_VT = 32;
constexpr int REC_NT = 64;

// Resident workgroups per CU and their order.  The registers allow 12 of
// these one-wave workgroups per CU (3 waves per SIMD, 256 CUs: 3,072 at
// once).  A decode grid (one token per sequence) of more than 2,304
// workgroups (B > 18 at 32 v-heads) is launched
//   * with dynamic LDS reserved so that 6 share a CU: the state streams of
//     fewer resident workgroups reach HBM faster (B = 64, eager launches,
//     per CU: 3 / 4 / 5 / 6 / 7 / 8 / 12 workgroups 53.7 / 50.7 / 48.6 /
//     48.6 / 50.2 / 51.5 / 52.2 us with the order below);
//   * head-major: the v-heads of one (sequence, column block) in consecutive
//     workgroups, so that the 4 column blocks of a head are a multiple of 8
//     workgroups apart and run on one XCD (workgroups are dealt to the 8 XCDs
//     in turn): the two 64-byte halves of each 128-byte line of o meet in
//     that XCD's L2 and the head's q/k rows are fetched once (at 4 per CU:
//     49.9-50.3 us against 51.8-52.3 us column-block-major).
// From graphs: B = 20 / 24 / 25 / 32 / 64 17.7 / 20.4 / 21.9 / 26.4 / 48.7 us
// against 18.3 / 21.4 / 23.7 / 28.3 / 54.2 us at full occupancy, column-block-
// major.  A smaller grid (1.5 capped rounds or less) runs best with all of it
// resident and column-block-major (B = 16: 13.4 us; capped 15.4 us).
// A multi-token step that writes per-token snapshots (spec verify) is a
// write stream as much as a read stream: head-major with 4 per CU (B = 32 x
// T = 4: 66.4-67.9 us; full occupancy 71.4-71.6, head-major alone 69.4-70.3,
// at 3 / 5 / 6 per CU 81.0 / 71.6-72.3 / 68.9-69.5 us).  Without snapshots the
// tokens' arithmetic needs the resident waves: full occupancy, column-block-
// major (B = 32 / 64 x T = 4: 40.2-41.2 / 70.7-71.2 us; at 4 per CU 56.0-56.7 /
// 103.2-104.6 us).
constexpr int64_t REC_CAP_MIN_BLOCKS = 2304;   // 1.5 rounds of 6 per CU on 256 CUs
constexpr unsigned REC_CAP_LDS = 24 * 1024;    // + 1 KiB static: 6 per CU in 160 KiB
constexpr unsigned REC_SNAP_CAP_LDS = 36 * 1024;  // + 1 KiB static: 4 per CU

// KD: k head dim (64, 128 or 256); VDC: v head dim, or 0 for a.V
template <int VT, int NT, int KD, int VDC>
__global__ __launch_bounds__(NT) void recurrent_kernel(RecArgs a) {
  constexpr int NW = NT / 64;
  constexpr int TPR = VT / 4;     // threads per state row
  constexpr int NRG = NT / TPR;   // row groups
  constexpr int RPT = KD / NRG;   // rows per thread
  constexpr int QE = KD / 64;     // q and k elements per lane
  static_assert(KD % 64 == 0 && KD % NRG == 0, "k head dim");
  const int VD = VDC ? VDC : a.V;
  const int NSPLIT = VD / VT;

  __shared__ float qs_l[KD];
  __shared__ float ks_l[KD];
  __shared__ float red[NW > 1 ? NW : 1][2][VT];

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = tid >> 6;
  const int c4 = tid % TPR;
  const int rg = tid / TPR;

  int bid = blockIdx.x, vt, h;
  if (a.head_major) {
    h = bid % a.Hv;
    bid /= a.Hv;
    vt = bid % NSPLIT;
    bid /= NSPLIT;
  } else {
    vt = bid % NSPLIT;
    bid /= NSPLIT;
    h = bid % a.Hv;
    bid /= a.Hv;
  }
  const int n = bid;
  const int hk = h / (a.Hv / a.Hk);
  const int col0 = vt * VT + c4 * 4;

  int64_t t0;
  int len;
  seq_range(a.cu, n, a.T, a.total, &t0, &len);

  const int64_t in_row = a.state_in ? pool_row(a.in_idx, n, a.in_rows) : -1;
  int64_t out_row = a.state_out ? pool_row(a.out_idx, n, a.out_rows) : -1;

  // A token's inputs as raw bits: this lane's two elements of q and k, its
  // four columns of v, and the gates.
  struct TokIn {
    uint32_t q[QE], k[QE], v[4];
    GateRaw gate;
  };
  auto tok_load = [&](int64_t tok) {
    TokIn r;
    const int64_t qoff = tok * a.qs + (int64_t)hk * KD + QE * lane;
    const int64_t koff = tok * a.ks + (int64_t)hk * KD + QE * lane;
    const int64_t vo = tok * a.vs + (int64_t)h * VD + col0;
#pragma unroll
    for (int i = 0; i < QE; ++i) {
      r.q[i] = load_bits(a.q, qoff + i, a.qkv_dt);
      r.k[i] = load_bits(a.k, koff + i, a.qkv_dt);
    }
#pragma unroll
    for (int c = 0; c < 4; ++c) r.v[c] = load_bits(a.v, vo + c, a.qkv_dt);
    r.gate = load_gates_raw(a.gate, tok, h);
    return r;
  };

  // The first token's inputs and the earlier rows' slot ids are requested
  // before the state: vector loads complete in order, so the q/k prologue and
  // the repeated-slot test wait for these few loads only, while the state
  // stream is in flight, and nothing is left to fetch once the state is in.
  TokIn cur{};
  if (len > 0) cur = tok_load(t0);
  const int64_t in_lane_id = in_row >= 0 ? earlier_id_of_lane(a.in_idx, n, lane) : 0;
  const int64_t out_lane_id = out_row >= 0 ? earlier_id_of_lane(a.out_idx, n, lane) : 0;
  __builtin_amdgcn_sched_barrier(0);

  // The state is touched exactly once per launch: non-temporal loads and
  // stores keep it from displacing reusable lines in the caches.  One
  // (sequence, head) state is one 64 KiB buffer range; a thread's rows
  // rg + 8r sit 4 KiB apart, an offset carried in a scalar register, so the
  // 16 accesses share one vector offset.
  const int voff = (rg * VD + col0) * 4;
  const int ROW8 = NRG * VD * 4;  // bytes between a thread's rows
  // (a row with no slot gets an empty range: its loads read zeros without
  // touching memory, so the loads are issued on one path whatever the row)
  auto state_rsrc = [&](const float *pool, int64_t row) {
    return row >= 0 ? __builtin_amdgcn_make_buffer_rsrc(const_cast<float *>(pool) + (row * a.Hv + h) * (int64_t)(KD * VD),
                                                        0, KD * VD * 4, BUF_DWORD3)
                    : __builtin_amdgcn_make_buffer_rsrc(nullptr, 0, 0, BUF_DWORD3);
  };
  f32x4 s[RPT];
  {
    const auto rs = state_rsrc(a.state_in, in_row);
#pragma unroll
    for (int r = 0; r < RPT; ++r)
      s[r] = __builtin_bit_cast(f32x4, __builtin_amdgcn_raw_buffer_load_b128(rs, voff, r * ROW8, BUF_NT));
  }
  __builtin_amdgcn_sched_barrier(0);
  // A row whose slot id an earlier row already named: zero state, like a
  // padding row, and nothing written.
  const bool in_rep = in_row >= 0 && repeats_earlier_wave(a.in_idx, n, in_row, in_lane_id, lane);
  if (out_row >= 0 && repeats_earlier_wave(a.out_idx, n, out_row, out_lane_id, lane)) out_row = -1;

  for (int t = 0; t < len; ++t) {
    const int64_t tok = t0 + t;
    // ---- q/k prologue: every wave reduces the full KD-vectors itself
    float qv[QE], kv[QE], pqq = 0.f, pkk = 0.f, pqk = 0.f;
#pragma unroll
    for (int i = 0; i < QE; ++i) {
      qv[i] = bits_to_f32(cur.q[i], a.qkv_dt);
      kv[i] = bits_to_f32(cur.k[i], a.qkv_dt);
      pqq += qv[i] * qv[i];
      pkk += kv[i] * kv[i];
      pqk += qv[i] * kv[i];
    }
    const float sqq = wave_sum(pqq);
    const float skk = wave_sum(pkk);
    const float sqk = wave_sum(pqk);
    const float rq = a.l2norm ? rsqrtf(sqq + 1e-6f) : 1.f;
    const float rk = a.l2norm ? rsqrtf(skk + 1e-6f) : 1.f;
    const float qsc = rq * a.scale;
    if (wave == 0) {
#pragma unroll
      for (int i = 0; i < QE; ++i) {
        qs_l[QE * lane + i] = qv[i] * qsc;
        ks_l[QE * lane + i] = kv[i] * rk;
      }
    }
    const float qk = sqk * qsc * rk;
    float gl, bt;
    gates_from_raw(a.gate, cur.gate, &gl, &bt);
    const float eg = expf(gl);
    float vv[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) vv[c] = bits_to_f32(cur.v[c], a.qkv_dt);
    if (t + 1 < len) cur = tok_load(tok + 1);  // the next token's inputs, during this one's update
    if (t == 0 && in_rep) {
#pragma unroll
      for (int r = 0; r < RPT; ++r) s[r] = f32x4{0.f, 0.f, 0.f, 0.f};
    }
    __syncthreads();

    // ---- partial k~^T S and q~^T S over this thread's rows
    float pk[4] = {0.f, 0.f, 0.f, 0.f}, pq[4] = {0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const float kk = ks_l[rg + NRG * r], qq = qs_l[rg + NRG * r];
      pk[0] += kk * s[r].x; pk[1] += kk * s[r].y; pk[2] += kk * s[r].z; pk[3] += kk * s[r].w;
      pq[0] += qq * s[r].x; pq[1] += qq * s[r].y; pq[2] += qq * s[r].z; pq[3] += qq * s[r].w;
    }
#pragma unroll
    for (int m = TPR; m < 64; m <<= 1) {
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        pk[c] += __shfl_xor(pk[c], m, 64);
        pq[c] += __shfl_xor(pq[c], m, 64);
      }
    }
    if constexpr (NW > 1) {
      if (lane < TPR) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          red[wave][0][c4 * 4 + c] = pk[c];
          red[wave][1][c4 * 4 + c] = pq[c];
        }
      }
      __syncthreads();
#pragma unroll
      for (int c = 0; c < 4; ++c) {
        float sk = 0.f, sq = 0.f;
#pragma unroll
        for (int w = 0; w < NW; ++w) {
          sk += red[w][0][c4 * 4 + c];
          sq += red[w][1][c4 * 4 + c];
        }
        pk[c] = sk;
        pq[c] = sq;
      }
    }

    // ---- delta, rank-1 update, output
    float d[4], out[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      d[c] = bt * (vv[c] - eg * pk[c]);
      out[c] = eg * pq[c] + qk * d[c];
    }
#pragma unroll
    for (int r = 0; r < RPT; ++r) {
      const float kk = ks_l[rg + NRG * r];
      s[r].x = eg * s[r].x + kk * d[0];
      s[r].y = eg * s[r].y + kk * d[1];
      s[r].z = eg * s[r].z + kk * d[2];
      s[r].w = eg * s[r].w + kk * d[3];
    }
    if (rg == 0) {
      const int64_t ooff = (tok * a.Hv + h) * (int64_t)VD + col0;
#pragma unroll
      for (int c = 0; c < 4; ++c) store_elem(a.o, ooff + c, a.o_dt, out[c]);
    }
    // Snapshots take global stores: stores through a buffer range rebuilt
    // per token in this loop were compiled with a per-token term in the vector
    // offset and landed outside the range (dropped).  Non-temporal, as the
    // state stream: with ordinary stores the B = 32 x T = 4 verify step took
    // 75.2-75.6 us against 68.4-69.6 us.
    if (a.snap) {
      float *sb = a.snap + (((int64_t)n * a.T + t) * a.Hv + h) * (int64_t)(KD * VD) + col0;
#pragma unroll
      for (int r = 0; r < RPT; ++r)
        __builtin_nontemporal_store(s[r], reinterpret_cast<f32x4 *>(sb + (rg + NRG * r) * VD));
    }
    __syncthreads();
  }

  if (len <= 0 && in_rep) {
#pragma unroll
    for (int r = 0; r < RPT; ++r) s[r] = f32x4{0.f, 0.f, 0.f, 0.f};
  }
  if (out_row >= 0) {
    const auto rs = state_rsrc(a.state_out, out_row);
#pragma unroll
    for (int r = 0; r < RPT; ++r)
      __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u32x4, s[r]), rs, voff, r * ROW8, BUF_NT);
  }
}

// ------------------------------------------------------------ token blocks
// The same recurrence for sequences of many tokens (prefills in fp32 or fp16,
// or at head dims the chunk kernels are not built for).  recurrent_kernel's
// token step is a chain of memory and LDS round trips (the next token's inputs
// are waited for at each barrier, three wave sums go through LDS): 2.3 us per
// token whatever the batch.  Here a workgroup of 4 waves
//   * takes TB tokens at a time: their q and k rows, normalised and scaled,
//     their v columns and gates go into LDS once per block (the next block's
//     are requested into registers first), so a token step waits on no memory;
//   * holds few state elements per lane: LPC lanes share a column, lane r of
//     them owning rows 4 r + e + 4 LPC i (e < 4), CPL columns each, so that a
//     step is K / LPC * CPL * 4 multiply-adds per lane, the two K-reductions end
//     on DPP within the LPC lanes, and the outputs wait in LDS for the block's
//     end.
// Two tokens run together (step2), so that the chain from one pair to the next
// holds one reduction.  With 16 lanes per column and one column per lane a
// pair is about 100 vector instructions, one sequence of 32 v-heads has
// one wave on every SIMD, and the next pair's operands are read ahead; larger
// batches (several waves per SIMD) take 8 lanes and read nothing ahead.
// Bound: the vector ALUs' issue (one wave alone issues about every 9 cycles,
// two or more waves of a SIMD together about every 5).  Measured, fp32, 32
// v-heads of 128 x 128, from graphs, against recurrent_kernel: T = 256 at
// B = 1 / 4 / 8 55.7 / 98.2 / 171.9 against 598 / 624 / 648 us; T = 1024 at
// B = 1, eager calls, 193 against 2380.
constexpr int TOK_NT = 256;

// Sum over the LPC (8 or 16) lanes that share a column, in every lane.
template <int LPC>
__device__ __forceinline__ float col_sum(float x) {
  x += dpp_mov<0xB1>(x);                            // quad_perm [1,0,3,2]
  x += dpp_mov<0x4E>(x);                            // quad_perm [2,3,0,1]
  x += dpp_mov<0x141>(x);                           // row_half_mirror
  if constexpr (LPC == 16) x += dpp_mov<0x140>(x);  // row_mirror
  return x;
}

// 1 / sqrt(x), x > 0, rounded once: the hardware's value (off by up to 1 ulp,
// the same factor on a whole q or k row) and one Newton step whose residual is
// exact to fp32.  Once per row and block; fp32 outputs against 64 bits, 1 x 1024
// / 4 x 100 / 8 x 128 tokens: 1.000e-7 / 1.025e-7 / 1.023e-7 without it, 0.978e-7
// / 1.005e-7 / 1.001e-7 with it (recurrent_kernel 0.994e-7 / 1.001e-7 / 0.998e-7),
// for 190 -> 193 us at 1 x 1024.
__device__ __forceinline__ float rsqrt_once(float x) {
  const float r = rsqrtf(x), t = x * r;
  const float e = __builtin_fmaf(-__builtin_fmaf(x, r, -t), r, __builtin_fmaf(-t, r, 1.f));  // 1 - x r^2
  return x < __builtin_inff() ? __builtin_fmaf(0.5f * r, e, r) : r;
}

// ES: bytes of a q/k/v element (2 or 4); KD: k head dim; LPC, CPL: lanes per
// column, columns per lane
template <int ES, int KD, int LPC, int CPL>
__global__ __launch_bounds__(TOK_NT) void recurrent_tokens_kernel(RecArgs a) {
  constexpr bool AHEAD = LPC == 16 && KD <= 128 && CPL == 1;
  constexpr int TB = 4096 / KD;              // tokens per block
  constexpr int COLS = TOK_NT / LPC * CPL;   // state columns per workgroup
  constexpr int RPL = KD / LPC;              // state rows per lane
  constexpr int NI = RPL / 4;                // groups of 4 rows per lane
  constexpr int PER = KD / 16;               // q and k elements per lane of a row's 16 lanes
  constexpr int ROWS = TOK_NT / 16;          // q / k rows loaded per pass
  constexpr int NP = TB / ROWS;              // passes
  constexpr int VW = PER * ES / 4;           // 32-bit words of one lane's share of a row
  constexpr int VPT = TB * COLS / TOK_NT;    // v (and o) elements per thread
  __shared__ __align__(16) float kt[TB][KD], qt[TB][KD];
  __shared__ __align__(16) float gt[TB][4];  // e^g, beta, q~ . k~, beta e^g (written by two threads: a vector's elements would be stored as one)
  __shared__ __align__(8) float pt[TB][2];                 // odd tokens: k~ . (the even one before it)'s k~, q~ . that k~
  __shared__ __align__(16) float vt[TB][COLS], ot[TB][COLS];

  const int tid = threadIdx.x;
  const int r = tid & (LPC - 1);         // lane within the column
  const int cb = (tid / LPC) * CPL;      // this lane's first column within the workgroup's
  const int tiles = a.V / COLS;
  const int ratio = a.Hv / a.Hk;
  // the workgroups that read one (sequence, k-head)'s rows on one XCD (workgroups
  // are dealt to the 8 XCDs in turn)
  int n, h, tile;
  {
    const int per = ratio * tiles;
    int g = blockIdx.x / per, m = blockIdx.x % per;
    if ((a.n_seqs * a.Hk) % 8 == 0) {
      const int t = blockIdx.x >> 3;
      g = 8 * (t / per) + (blockIdx.x & 7);
      m = t % per;
    }
    n = g / a.Hk;
    h = (g % a.Hk) * ratio + m / tiles;
    tile = m % tiles;
  }
  const int hk = h / ratio;
  const int col0 = tile * COLS;

  int64_t t0;
  int len;
  seq_range(a.cu, n, a.T, a.total, &t0, &len);
  len = __builtin_amdgcn_readfirstlane(len);

  // ---- one block's inputs in registers
  const int row = tid >> 4, l16 = tid & 15;  // the q / k row of pass 0, and the lane's share of it
  uint32_t qu[NP][VW], ku[NP][VW], vu[VPT], gu[2];
  auto load_block = [&](int b0) {  // tokens b0 .. b0 + TB of the sequence (rows past its end: its last token)
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int64_t tok = t0 + min(b0 + row + ROWS * i, len - 1);
      const char *qp = static_cast<const char *>(a.q) + (tok * a.qs + (int64_t)hk * KD + l16 * PER) * ES;
      const char *kp = static_cast<const char *>(a.k) + (tok * a.ks + (int64_t)hk * KD + l16 * PER) * ES;
      if constexpr (VW % 4 == 0) {
#pragma unroll
        for (int w = 0; w < VW; w += 4) {
          const u32x4 x = *reinterpret_cast<const u32x4 *>(qp + 4 * w), y = *reinterpret_cast<const u32x4 *>(kp + 4 * w);
#pragma unroll
          for (int e = 0; e < 4; ++e) qu[i][w + e] = x[e], ku[i][w + e] = y[e];
        }
      } else {  // (K = 64 in 2-byte types: 8 bytes)
        typedef __attribute__((ext_vector_type(2))) unsigned u32x2;
        const u32x2 x = *reinterpret_cast<const u32x2 *>(qp), y = *reinterpret_cast<const u32x2 *>(kp);
        qu[i][0] = x.x, qu[i][1] = x.y, ku[i][0] = y.x, ku[i][1] = y.y;
      }
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int e = tid + TOK_NT * i;
      const int64_t tok = t0 + min(b0 + e / COLS, len - 1);
      vu[i] = load_bits(a.v, tok * a.vs + (int64_t)h * a.V + col0 + e % COLS, a.qkv_dt);
    }
    if (tid < TB) {
      const int64_t gi = (t0 + min(b0 + tid, len - 1)) * a.gate.stride + h;
      gu[0] = load_bits(a.gate.g_or_a, gi, a.gate.A_log ? a.gate.dt : GDN_DTYPE_F32);
      gu[1] = load_bits(a.gate.beta_or_b, gi, a.gate.dt);
    }
  };
  const float a_log = a.gate.A_log ? a.gate.A_log[h] : 0.f, dt_bias = a.gate.A_log ? a.gate.dt_bias[h] : 0.f;
  // ... and from them the block's operands in LDS
  auto elem = [&](const uint32_t (&u)[VW], int i) -> float {
    if constexpr (ES == 4)
      return __uint_as_float(u[i]);
    else
      return bits_to_f32((u[i / 2] >> (16 * (i & 1))) & 0xffffu, a.qkv_dt);
  };
  auto store_block = [&]() {
#pragma unroll
    for (int i = 0; i < NP; ++i) {
      const int t = row + ROWS * i;
      float qf[PER], kf[PER], sqq = 0.f, skk = 0.f, sqk = 0.f;
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        qf[e] = elem(qu[i], e);
        kf[e] = elem(ku[i], e);
        sqq += qf[e] * qf[e];
        skk += kf[e] * kf[e];
        sqk += qf[e] * kf[e];
      }
      sqq = row16_sum(sqq);
      skk = row16_sum(skk);
      sqk = row16_sum(sqk);
      const float rq = (a.l2norm ? rsqrt_once(sqq + 1e-6f) : 1.f) * a.scale;
      const float rk = a.l2norm ? rsqrt_once(skk + 1e-6f) : 1.f;
#pragma unroll
      for (int e = 0; e < PER; e += 4) {
        *reinterpret_cast<f32x4 *>(&qt[t][l16 * PER + e]) = f32x4{qf[e], qf[e + 1], qf[e + 2], qf[e + 3]} * rq;
        *reinterpret_cast<f32x4 *>(&kt[t][l16 * PER + e]) = f32x4{kf[e], kf[e + 1], kf[e + 2], kf[e + 3]} * rk;
      }
      if (l16 == 0) gt[t][2] = sqk * rq * rk;
      // (token t - 1 sits in the 16 lanes before these; ROWS is even)
      float pkk = 0.f, pqk = 0.f;
      const float rkp = __shfl_xor(rk, 16, 64);
#pragma unroll
      for (int e = 0; e < PER; ++e) {
        const float kp = __shfl_xor(kf[e], 16, 64);
        pkk += kf[e] * kp;
        pqk += qf[e] * kp;
      }
      pkk = row16_sum(pkk) * rk * rkp;
      pqk = row16_sum(pqk) * rq * rkp;
      if (l16 == 0 && (t & 1)) {
        pt[t][0] = pkk;
        pt[t][1] = pqk;
      }
    }
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int e = tid + TOK_NT * i;
      vt[e / COLS][e % COLS] = bits_to_f32(vu[i], a.qkv_dt);
    }
    if (tid < TB) {
      float gl, bt;
      gates_from_raw(a.gate, GateRaw{gu[0], gu[1], a_log, dt_bias}, &gl, &bt);
      const float eg = expf(gl);
      gt[tid][0] = eg;
      gt[tid][1] = bt;
      gt[tid][3] = bt * eg;
    }
  };

  if (len > 0) load_block(0);
  int64_t in_row = a.state_in ? pool_row_first(a.in_idx, n, a.in_rows) : -1;
  int64_t out_row = a.state_out ? pool_row_first(a.out_idx, n, a.out_rows) : -1;
  const int64_t soff = (int64_t)4 * r * a.V + col0 + cb;  // of this lane's row 0, column 0, within a head's state
  float s[RPL][CPL];
#pragma unroll
  for (int j = 0; j < RPL; ++j)
#pragma unroll
    for (int c = 0; c < CPL; ++c)
      s[j][c] = in_row >= 0 ? a.state_in[(in_row * a.Hv + h) * ((int64_t)KD * a.V) + soff +
                                         (int64_t)(j % 4 + 4 * LPC * (j / 4)) * a.V + c]
                            : 0.f;

  struct Tok {  // one token's operands of a lane
    f32x4 k[NI], q[NI];
    float v[CPL];
    f32x4 g;
  };
  auto read_tok = [&](Tok &x, int t) {
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      x.k[i] = *reinterpret_cast<const f32x4 *>(&kt[t][4 * r + 4 * LPC * i]);
      x.q[i] = *reinterpret_cast<const f32x4 *>(&qt[t][4 * r + 4 * LPC * i]);
    }
#pragma unroll
    for (int c = 0; c < CPL; ++c) x.v[c] = vt[t][cb + c];
    x.g = *reinterpret_cast<const f32x4 *>(gt[t]);
  };
  // k~^T S and q~^T S of one token over the whole column
  auto reduce = [&](const Tok &x, float (&pk)[CPL], float (&pq)[CPL]) {
#pragma unroll
    for (int c = 0; c < CPL; ++c) pk[c] = pq[c] = 0.f;
#pragma unroll
    for (int j = 0; j < RPL; ++j)
#pragma unroll
      for (int c = 0; c < CPL; ++c) {
        pk[c] = __builtin_fmaf(x.k[j / 4][j % 4], s[j][c], pk[c]);
        pq[c] = __builtin_fmaf(x.q[j / 4][j % 4], s[j][c], pq[c]);
      }
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      pk[c] = col_sum<LPC>(pk[c]);
      pq[c] = col_sum<LPC>(pq[c]);
    }
  };
  // Tokens t and t + 1 together: both reductions run over the state before
  // them, and token t's rank-1 update enters token t + 1's sums through the
  // dot products with k~_t, so the chain from one pair to the next holds one
  // reduction and the state is scaled once.
  auto step2 = [&](const Tok &x, const Tok &y, f32x2 yx, int t) {
    float pk0[CPL], pq0[CPL], pk1[CPL], pq1[CPL], d0[CPL], d1[CPL];
    reduce(x, pk0, pq0);
    reduce(y, pk1, pq1);
    const float e01 = x.g.x * y.g.x;
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      d0[c] = __builtin_fmaf(-x.g.w, pk0[c], x.g.y * x.v[c]);
      const float sk = __builtin_fmaf(yx.x, d0[c], x.g.x * pk1[c]);  // k~_{t+1}^T S after token t
      const float sq = __builtin_fmaf(yx.y, d0[c], x.g.x * pq1[c]);
      d1[c] = __builtin_fmaf(-y.g.w, sk, y.g.y * y.v[c]);
      if (r == 0) {
        ot[t][cb + c] = x.g.x * pq0[c] + x.g.z * d0[c];
        ot[t + 1][cb + c] = y.g.x * sq + y.g.z * d1[c];
      }
      d0[c] *= y.g.x;
    }
#pragma unroll
    for (int j = 0; j < RPL; ++j)
#pragma unroll
      for (int c = 0; c < CPL; ++c)
        s[j][c] = __builtin_fmaf(y.k[j / 4][j % 4], d1[c], __builtin_fmaf(x.k[j / 4][j % 4], d0[c], e01 * s[j][c]));
  };
  auto step1 = [&](const Tok &x, int t) {
    float pk[CPL], pq[CPL], d[CPL];
    reduce(x, pk, pq);
#pragma unroll
    for (int c = 0; c < CPL; ++c) {
      d[c] = __builtin_fmaf(-x.g.w, pk[c], x.g.y * x.v[c]);
      if (r == 0) ot[t][cb + c] = x.g.x * pq[c] + x.g.z * d[c];
    }
#pragma unroll
    for (int j = 0; j < RPL; ++j)
#pragma unroll
      for (int c = 0; c < CPL; ++c) s[j][c] = __builtin_fmaf(x.k[j / 4][j % 4], d[c], x.g.x * s[j][c]);
  };

  for (int b0 = 0; b0 < len; b0 += TB) {
    const int nb = min(TB, len - b0);
    store_block();
    __syncthreads();
    if (b0 + TB < len) load_block(b0 + TB);
    const int pairs = nb >> 1;
    Tok x0, x1, y0, y1;
    f32x2 p0, p1;
    auto read_pair = [&](Tok &x, Tok &y, f32x2 &yx, int t) {
      read_tok(x, t);
      read_tok(y, t + 1);
      yx = *reinterpret_cast<const f32x2 *>(pt[t + 1]);
    };
    if constexpr (AHEAD) {  // the next pair's operands are read while a pair runs (at the end: the last one again, unused)
      if (pairs > 0) read_pair(x0, y0, p0, 0);
      for (int i = 0; i < pairs; i += 2) {
        read_pair(x1, y1, p1, 2 * min(i + 1, pairs - 1));
        step2(x0, y0, p0, 2 * i);
        if (i + 1 < pairs) {
          read_pair(x0, y0, p0, 2 * min(i + 2, pairs - 1));
          step2(x1, y1, p1, 2 * i + 2);
        }
      }
    } else {
      for (int i = 0; i < pairs; ++i) {
        read_pair(x0, y0, p0, 2 * i);
        step2(x0, y0, p0, 2 * i);
      }
    }
    if (nb & 1) {
      read_tok(x0, nb - 1);
      step1(x0, nb - 1);
    }
    lds_barrier();  // the block's outputs are in LDS, its operands read
#pragma unroll
    for (int i = 0; i < VPT; ++i) {
      const int e = tid + TOK_NT * i;
      if (e / COLS < nb)
        store_elem(a.o, ((t0 + b0 + e / COLS) * a.Hv + h) * (int64_t)a.V + col0 + e % COLS, a.o_dt, ot[e / COLS][e % COLS]);
    }
  }

  if (out_row >= 0) {
    float *dst = a.state_out + (out_row * a.Hv + h) * ((int64_t)KD * a.V) + soff;
#pragma unroll
    for (int j = 0; j < RPL; ++j)
#pragma unroll
      for (int c = 0; c < CPL; ++c) dst[(int64_t)(j % 4 + 4 * LPC * (j / 4)) * a.V + c] = s[j][c];
  }
}

}  // namespace
}  // namespace gdn

namespace gdn {
namespace {

// Tokens per sequence (their average, with cu_seqlens) from which a call
// without snapshots takes recurrent_tokens_kernel.  Its token steps are much
// cheaper, its state accesses less contiguous (16 to 64 columns of a row per
// workgroup), so the line rises with the state a call moves.  Measured from
// graphs, this kernel against recurrent_kernel, us:
//   128 x 128, 32 v-heads, fp32: T = 4 at B = 1 / 4 / 8 7 / 10.6 / 15-17 against
//   12.2 / 13.5 / 15.8; T = 8 at B = 8 / 16 / 64 17.4 / 31-34 / 108-125 against
//   27.1 / 32.3 / 97.7; T = 16 at B = 16 / 64 38.6 / 129-146 against 54.3 / 156;
//   256 x 256, bf16: T = 4 at 32 / 64 / 128 pairs 0.76 / 1.20 / 1.28 of
//   recurrent_kernel's time, T = 6 at 64 / 128 0.97 / 1.08, T = 8 0.82 / 0.94
//   (256 x 128 at 96 / 128 pairs: T = 4 0.89 / 1.20, T = 6 0.68 / 0.95);
//   128 x 256, bf16: T = 4 at 64 / 96 pairs 0.85 / 1.13, T = 6 at 96 0.90; T = 8 at
//   160 / 256 pairs 1.11 / 1.09, T = 12 0.89 / 0.91;
//   64 x 64, bf16: T = 16 at 1,024 / 2,048 pairs 0.81 / 1.14, T = 24 0.63 / 0.92 (fp32,
//   T = 16: 0.64 / 0.89).
inline int64_t tokens_min(int64_t pairs, int K, int V, int64_t es) {
  const int64_t cols = pairs * V;
  const int64_t few = pairs <= 128 ? 4 : pairs <= 256 ? 8 : 16;
  int64_t wide = 0;
  if (K == 256)
    wide = cols > 96 * 128 ? 8 : 0;
  else if (K == 128)
    wide = cols > 256 * 128 ? 12 : cols > 128 * 128 ? 6 : 0;
  else
    wide = es == 2 && cols > 512 * 128 ? 24 : 0;
  return std::max(few, wide);
}

// State columns (pairs x V) from which more rows per lane pay: below
// REC_TOKENS_MID_COLS a wave per SIMD is all there is and the shortest step
// wins (16 lanes per column, 1 column per lane); then 8 lanes and, for K = 128,
// from REC_TOKENS_WIDE_COLS 2 columns per lane (fewer reduction steps and LDS
// reads per element).  fp32, T = 256, 32 v-heads of 128 x 128, (16, 1) / (8, 1)
// / (8, 2) lanes and columns: B = 1 55.7 / 75.0 / 116.9 us; B = 2 70.5 / 76.1 /
// 117.4; B = 4 136 / 98 / 124; B = 8 264 / 195 / 172.  K = 64 at B = 8, T = 128:
// 56 / 41 / 51; K = 256: 236 / 233 with one column per lane, (16, 2) 199.
constexpr int64_t REC_TOKENS_MID_COLS = 96 * 128;
constexpr int64_t REC_TOKENS_WIDE_COLS = 192 * 128;

template <int ES, int KD, int LPC, int CPL>
void launch_tokens_as(const RecArgs &a, hipStream_t st) {
  const int64_t blocks = static_cast<int64_t>(a.n_seqs) * a.Hv * (a.V / (TOK_NT / LPC * CPL));
  hipLaunchKernelGGL((recurrent_tokens_kernel<ES, KD, LPC, CPL>), dim3(static_cast<unsigned>(blocks)), dim3(TOK_NT), 0,
                     st, a);
}
template <int ES, int KD>
void launch_tokens(const RecArgs &a, hipStream_t st) {  // (V is a multiple of 32)
  const int64_t cols = static_cast<int64_t>(a.n_seqs) * a.Hv * a.V;
  if constexpr (KD == 256) {
    if (cols >= REC_TOKENS_WIDE_COLS) return launch_tokens_as<ES, KD, 16, 2>(a, st);
  } else {
    if (KD == 128 && cols >= REC_TOKENS_WIDE_COLS && a.V % 64 == 0) return launch_tokens_as<ES, KD, 8, KD / 64>(a, st);
    if (cols >= REC_TOKENS_MID_COLS) return launch_tokens_as<ES, KD, 8, 1>(a, st);
  }
  launch_tokens_as<ES, KD, 16, 1>(a, st);
}

int recurrent_fwd(const void *q, const void *k, const void *v, int qkv_dtype,
                  int64_t q_stride_t, int64_t k_stride_t, int64_t v_stride_t, const GateArgs &gate,
                  const float *state_in, const int64_t *state_in_idx, int64_t state_in_rows,
                  float *state_out, const int64_t *state_out_idx, int64_t state_out_rows,
                  void *o, int o_dtype, float *snapshots,
                  const int32_t *cu_seqlens, int32_t n_seqs, int32_t T,
                  int32_t Hk, int32_t Hv, int32_t K, int32_t V,
                  float scale, int l2norm_qk, void *stream, const char *name) {
  if ((K != 64 && K != 128 && K != 256) || V <= 0 || V % REC_VT)
    return fail(GDN_ERR_UNSUPPORTED, "%s: K=%d V=%d; K must be 64, 128 or 256 and V a positive multiple of %d",
                name, K, V, REC_VT);
  if (n_seqs < 0 || T < 0 || Hk <= 0 || Hv <= 0 || Hv % Hk)
    return fail(GDN_ERR_INVALID_ARGUMENT, "%s: bad sizes n_seqs=%d T=%d Hk=%d Hv=%d", name, n_seqs, T, Hk, Hv);
  if (!valid_dtype(qkv_dtype) || !valid_dtype(gate.dt) || !valid_dtype(o_dtype))
    return fail(GDN_ERR_INVALID_ARGUMENT, "%s: bad dtype", name);
  if (n_seqs == 0) return ok();
  if (!q || !k || !v || !gate.g_or_a || !gate.beta_or_b || !o)
    return fail(GDN_ERR_INVALID_ARGUMENT, "%s: null q/k/v/gate/o", name);
  if (gate.A_log && !gate.dt_bias) return fail(GDN_ERR_INVALID_ARGUMENT, "%s: null dt_bias", name);
  if (gate.stride < Hv) return fail(GDN_ERR_INVALID_ARGUMENT, "%s: gate token stride smaller than Hv", name);
  if (snapshots && cu_seqlens)
    return fail(GDN_ERR_INVALID_ARGUMENT, "%s: snapshots need equal-length sequences", name);
  if (!rows_cover(state_in, state_in_idx, state_in_rows, n_seqs) ||
      !rows_cover(state_out, state_out_idx, state_out_rows, n_seqs))
    return fail(GDN_ERR_INVALID_ARGUMENT, "%s: state rows (%lld in, %lld out) do not cover %d sequences", name,
                static_cast<long long>(state_in_rows), static_cast<long long>(state_out_rows), n_seqs);
  if (q_stride_t < Hk * K || k_stride_t < Hk * K || v_stride_t < Hv * V)
    return fail(GDN_ERR_INVALID_ARGUMENT, "%s: token stride smaller than a row", name);
  const int64_t n_blocks = static_cast<int64_t>(n_seqs) * Hv * (V / REC_VT);
  if (n_blocks > 0x7fffffff) return fail(GDN_ERR_INVALID_ARGUMENT, "%s: grid too large", name);

  RecArgs a{q, k, v, q_stride_t, k_stride_t, v_stride_t, gate, state_in, state_in_idx, state_in_rows,
            state_out, state_out_idx, state_out_rows, o, snapshots, cu_seqlens, n_seqs, T, Hk, Hv, V,
            cu_seqlens ? static_cast<int64_t>(T) : static_cast<int64_t>(n_seqs) * T,
            scale, l2norm_qk, qkv_dtype, o_dtype};
  const hipStream_t st = static_cast<hipStream_t>(stream);
  // q / k rows are read in 16-byte pieces there
  const int64_t es = static_cast<int64_t>(dtype_size(qkv_dtype));
  const bool aligned = (reinterpret_cast<uintptr_t>(q) | reinterpret_cast<uintptr_t>(k)) % 16 == 0 &&
                       (q_stride_t * es) % 16 == 0 && (k_stride_t * es) % 16 == 0;
  if (!snapshots && aligned && n_blocks * 2 <= 0x7fffffff &&
      a.total >= tokens_min(static_cast<int64_t>(n_seqs) * Hv, K, V, es) * n_seqs) {
    if (es == 2)
      K == 64 ? launch_tokens<2, 64>(a, st) : K == 128 ? launch_tokens<2, 128>(a, st) : launch_tokens<2, 256>(a, st);
    else
      K == 64 ? launch_tokens<4, 64>(a, st) : K == 128 ? launch_tokens<4, 128>(a, st) : launch_tokens<4, 256>(a, st);
    return check_launch(name);
  }
  const bool capped = n_blocks > REC_CAP_MIN_BLOCKS && (T == 1 || snapshots);
  a.head_major = capped;
  const unsigned lds = !capped ? 0u : T == 1 ? REC_CAP_LDS : REC_SNAP_CAP_LDS;
  const dim3 grid(static_cast<unsigned>(n_blocks)), block(REC_NT);
  if (K == KD_DEFAULT && V == VD_DEFAULT)
    hipLaunchKernelGGL((recurrent_kernel<REC_VT, REC_NT, KD_DEFAULT, VD_DEFAULT>), grid, block, lds, st, a);
  else if (K == 64)
    hipLaunchKernelGGL((recurrent_kernel<REC_VT, REC_NT, 64, 0>), grid, block, lds, st, a);
  else if (K == 128)
    hipLaunchKernelGGL((recurrent_kernel<REC_VT, REC_NT, 128, 0>), grid, block, lds, st, a);
  else
    hipLaunchKernelGGL((recurrent_kernel<REC_VT, REC_NT, 256, 0>), grid, block, lds, st, a);
  return check_launch(name);
}

}  // namespace
}  // namespace gdn

extern "C" int gdn_recurrent_fwd(const void *q, const void *k, const void *v, int qkv_dtype,
                                 int64_t q_stride_t, int64_t k_stride_t, int64_t v_stride_t,
                                 const float *g, const void *beta, int beta_dtype,
                                 const float *state_in, const int64_t *state_in_idx, int64_t state_in_rows,
                                 float *state_out, const int64_t *state_out_idx, int64_t state_out_rows,
                                 void *o, int o_dtype, float *snapshots,
                                 const int32_t *cu_seqlens, int32_t n_seqs, int32_t T,
                                 int32_t Hk, int32_t Hv, int32_t K, int32_t V,
                                 float scale, int l2norm_qk, void *stream) {
  const gdn::GateArgs gate{g, beta, beta_dtype, Hv, nullptr, nullptr};
  return gdn::recurrent_fwd(q, k, v, qkv_dtype, q_stride_t, k_stride_t, v_stride_t, gate, state_in, state_in_idx,
                            state_in_rows, state_out, state_out_idx, state_out_rows, o, o_dtype, snapshots, cu_seqlens, n_seqs, T, Hk, Hv, K, V,
                            scale, l2norm_qk, stream, "gdn_recurrent_fwd");
}

extern "C" int gdn_recurrent_fwd_gated(const void *q, const void *k, const void *v, int qkv_dtype,
                                       int64_t q_stride_t, int64_t k_stride_t, int64_t v_stride_t,
                                       const void *a, const void *b, int ab_dtype, int64_t ab_stride_t,
                                       const float *A_log, const float *dt_bias,
                                       const float *state_in, const int64_t *state_in_idx, int64_t state_in_rows,
                                       float *state_out, const int64_t *state_out_idx, int64_t state_out_rows,
                                       void *o, int o_dtype, float *snapshots,
                                       const int32_t *cu_seqlens, int32_t n_seqs, int32_t T,
                                       int32_t Hk, int32_t Hv, int32_t K, int32_t V,
                                       float scale, int l2norm_qk, void *stream) {
  if (!A_log) return gdn::fail(GDN_ERR_INVALID_ARGUMENT, "gdn_recurrent_fwd_gated: null A_log");
  const gdn::GateArgs gate{a, b, ab_dtype, ab_stride_t, A_log, dt_bias};
  return gdn::recurrent_fwd(q, k, v, qkv_dtype, q_stride_t, k_stride_t, v_stride_t, gate, state_in, state_in_idx,
                            state_in_rows, state_out, state_out_idx, state_out_rows, o, o_dtype, snapshots, cu_seqlens, n_seqs, T, Hk, Hv, K, V,
                            scale, l2norm_qk, stream, "gdn_recurrent_fwd_gated");
}
