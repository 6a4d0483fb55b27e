// zg_attn_prefill.hip -- causal attention of the batched prefill on the fp32
// matrix cores.
//
// No reference counterpart as a batch: the reference prefills token by token
// (kernel/src/inference.rs:1188-1330) and attends per head
// (kernel/src/inference_avx512.rs:1744-1800, softmax attention.rs:48-84).
//
// A workgroup owns 32 query columns of one KV head, two halves of 16 (16
// prompt rows of two query heads that share it, or 32 rows of one).  Its
// eight waves take the context's 16-key tiles in turn (tile t: wave t mod 8);
// per tile a wave forms S^T = K Q^T and O^T += V^T P^T with
// v_mfma_f32_16x16x4_f32:
//   S^T   A = K: lane (key l % 16, slot j = l / 16) holds its row's float4
//         columns 16 c + 4 j, so step (c, r) contracts d = 16 c + 4 j + r;
//         B = Q in the same order, read from LDS
//   P     element r of a lane is (key 4 j + r, query l % 16): step r of P.V
//         takes it as its B operand as it stands
//   O^T   A = V: lane (i = l % 16, j) holds dims DT i .. DT i + DT - 1 of key
//         4 j + r (whole rows, coalesced); accumulator dt, row i is dim
//         DT i + dt, so a lane ends with HD / 4 consecutive dims of its query
// The next tile's K loads are issued after S^T and this tile's V loads
// before it, so both are in flight under matrix work.  The softmax runs per
// column and wave with the running max (the column's four lanes swap their
// maxima), and the waves' (O, max, sum) meet in LDS once at the end.
//
// A row's result depends on its own position and keys only (masked scores
// give exactly 0, a later tile rescales by exactly 1), not on the chunk it
// is computed in, nor on the form: launches of few workgroups spread the same
// sums over more of them (attn_prefill_half_kernel, attn_prefill_split_kernel).
//
// Bound: the fp32 matrix rate (32 cycles per MFMA, 128 MFMAs per tile at
// head_dim 128; 157 TFLOP/s for the chip; the matrix cores are busy 51 % of
// the cycles of 1,800 rows), then each workgroup's own prologue and merge
// (7.4 us for 16 rows; one workgroup fits a CU), the masked half of the
// diagonal tiles and the last workgroups of a chunk.  K and V come from L2:
// 16 KB per tile and wave.  16 query and 8 KV heads of 128, graph replays: 150
// rows 15.5 us, 512 rows at position 0 28 us, at 1024 67 us (80 TFLOP/s), 1,800
// rows 162 us.  The form before it, one workgroup per query head and row that
// re-read K and V for every row: prefill of 1,800 tokens in 512-row chunks 50.4
// ms in all, 22.1 ms with this one.  Measured and not used: 32-key tiles with
// v_mfma_f32_32x32x2_f32 (22.6 ms), V loaded a tile ahead as K is (512 rows at
// 1024: 74 us); without the exponentials or without the loads the time hardly
// moved (72 and 70 us, of 69 then).
#include <type_traits>

#include "zg_device.h"
#include "zg_prefill.h"

namespace zg {

typedef float v4f __attribute__((ext_vector_type(4)));

constexpr int kPaWaves = 8;  // waves per workgroup: the tiles' stride
constexpr int kPaCols = 32;  // query columns per workgroup
constexpr int kPaKeys = 16;  // keys per tile

// Max over the four 16-lane rows, lane by lane.
__device__ __forceinline__ float rows_max(float v) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = fmaxf(__uint_as_float(h[0]), __uint_as_float(h[1]));
  const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}
__device__ __forceinline__ float rows_sum(float v) {
  const auto h = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  v = __uint_as_float(h[0]) + __uint_as_float(h[1]);
  const auto q = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false, false);
  return __uint_as_float(q[0]) + __uint_as_float(q[1]);
}

// Element e of a lane is (key kPaKeys t + 4 j + e, its column): scores to
// exp(score - running max) in place, the running state updated; returns the
// factor for the column's earlier sums.
__device__ __forceinline__ float pa_soften(v4f& s, float scale, int t, int j, bool masked, int pos, float& m, float& l,
                                           bool& nan_score) {
  float tm = -INFINITY;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    float v = s[e] * scale;
    if (masked && kPaKeys * t + 4 * j + e > pos) v = -INFINITY;
    nan_score = nan_score || v != v;
    tm = fmaxf(tm, v);
    s[e] = v;
  }
  const float mn = fmaxf(m, rows_max(tm));
  const float alpha = m == -INFINITY ? 0.0f : expf(m - mn);
  m = mn;
  float ls = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; e++) {
    const float p = s[e] == -INFINITY ? 0.0f : expf(s[e] - mn);
    ls += p;
    s[e] = p;
  }
  l = fmaf(l, alpha, ls);
  return alpha;
}

// A non-finite V row must not reach (as 0 * NaN) the columns that do not
// attend to it: in a tile with masked keys it enters as zeros, and the
// columns that do attend to it end as NaN.  Returns the tile's first such
// key, or 64.
template <int DT>
__device__ __forceinline__ int pa_clean(v4f (&vr)[4][DT / 4]) {
  float z = 0.0f;
#pragma unroll
  for (int e = 0; e < 4; e++)
#pragma unroll
    for (int d = 0; d < DT; d++) z = fmaf(vr[e][d / 4][d % 4], 0.0f, z);
  int first = 64;
  if (__any(z != z)) {
#pragma unroll
    for (int e = 0; e < 4; e++) {
      bool b = false;
#pragma unroll
      for (int d = 0; d < DT; d++) {
        const bool f = isfinite(vr[e][d / 4][d % 4]);
        b = b || !f;
        vr[e][d / 4][d % 4] = f ? vr[e][d / 4][d % 4] : 0.0f;
      }
      const uint64_t bm = __ballot(b);
#pragma unroll
      for (int x = 0; x < 4; x++)
        if ((bm >> (16 * x)) & 0xFFFFu) first = min(first, 4 * x + e);
    }
  }
  return first;
}

// A wave's partials of one half (O [column][dim], max and sum per column); the
// lane holds dims DT (4 j + r) + d of its column.  op: the column's row, mw /
// lw / nw: the column's entries.  store: the column is wanted.
template <int HD>
__device__ __forceinline__ void pa_put(float* op, float* mw, float* lw, uint8_t* nw, int col, int j, bool store,
                                       const v4f (&o)[HD / 16], float m, float l, bool nan_score, bool poison) {
  constexpr int DT = HD / 16;
  const float lt = rows_sum(l);
  uint64_t bad = __ballot(nan_score);
  bad |= bad >> 32;
  bad |= bad >> 16;  // any of the column's four lanes
  if (!store) return;
#pragma unroll
  for (int r = 0; r < 4; r++)
#pragma unroll
    for (int x = 0; x < DT / 4; x++)
      *reinterpret_cast<v4f*>(op + 4 * DT * j + DT * r + 4 * x) =
          v4f{o[4 * x][r], o[4 * x + 1][r], o[4 * x + 2][r], o[4 * x + 3][r]};
  if (j == 0) {
    *mw = m;
    *lw = (bad >> col) & 1 ? __builtin_nanf("") : lt;
    *nw = poison;
  }
}

// Tile t for one half's 16 columns, every operand loaded up front; qrow and qh:
// this lane's column's row and query head, the partials to op / mw / lw / nw.
template <int HD>
__device__ __forceinline__ void pa_one_tile(const PrefillAttnArgs& a, int kvh, int t, int col, int j, int qrow, int qh,
                                            bool masked, float* op, float* mw, float* lw, uint8_t* nw) {
  constexpr int C4 = HD / 16, DT = HD / 16;
  const size_t qd = (size_t)a.nq * HD, kvd = (size_t)a.nkv * HD;
  const int pos = a.pos0 + qrow;
  const v4f* qg = reinterpret_cast<const v4f*>(a.q + (size_t)qrow * qd + (size_t)qh * HD) + j;
  const uint32_t rowb = (uint32_t)kvd * 4;
  const uint8_t* kt = reinterpret_cast<const uint8_t*>(a.kcache + (size_t)kvh * HD) + (size_t)(kPaKeys * t) * rowb;
  const uint8_t* vt = reinterpret_cast<const uint8_t*>(a.vcache + (size_t)kvh * HD) + (size_t)(kPaKeys * t) * rowb;
  const uint32_t koff = (uint32_t)col * rowb + 16u * (uint32_t)j;
  const uint32_t voff = 4u * (uint32_t)j * rowb + (uint32_t)(4 * DT * col);
  v4f qr[C4], kr[C4], vr[4][DT / 4];
#pragma unroll
  for (int c = 0; c < C4; c++) {
    qr[c] = qg[4 * c];
    kr[c] = *reinterpret_cast<const v4f*>(kt + koff + 64 * c);
  }
#pragma unroll
  for (int e = 0; e < 4; e++)
#pragma unroll
    for (int x = 0; x < DT / 4; x++) vr[e][x] = *reinterpret_cast<const v4f*>(vt + (size_t)(e * rowb) + voff + 16 * x);
  __builtin_amdgcn_sched_barrier(0);
  v4f s = {0.0f, 0.0f, 0.0f, 0.0f}, s2 = s;
#pragma unroll
  for (int c = 0; c < C4 / 2; c++)
#pragma unroll
    for (int r = 0; r < 4; r++) {
      s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c][r], qr[c][r], s, 0, 0, 0);
      s2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[C4 / 2 + c][r], qr[C4 / 2 + c][r], s2, 0, 0, 0);
    }
  s += s2;
  float m = -INFINITY, l = 0.0f;
  bool nan_score = false, poison = false;
  pa_soften(s, a.scale, t, j, masked, pos, m, l, nan_score);
  if (masked) {
    const int first = pa_clean<DT>(vr);
    poison = first < 64 && kPaKeys * t + first <= pos;
  }
  v4f o[DT];
#pragma unroll
  for (int d = 0; d < DT; d++) o[d] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int e = 0; e < 4; e++)
#pragma unroll
    for (int d = 0; d < DT; d++) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[e][d / 4][d % 4], s[e], o[d], 0, 0, 0);
  pa_put<HD>(op, mw, lw, nw, col, j, true, o, m, l, nan_score, poison);
}

// The merge of a workgroup's slots (the partial sums of wave w of the long
// form) into the rows of its NC columns from c0 on, by eight waves: HD / 4
// lanes hold one column as float4 pieces, eight lanes a Q8_0 block.
// op [slot][column][pitch], mw_ / lw_ / nw_ [slot][column].
template <int HD, int NS, int NC = kPaCols>
__device__ __forceinline__ void pa_finish(const PrefillAttnArgs& a, int h0, int row0, int rpt, int wave, int lane,
                                          const float* op, int pitch, const float* mw_, const float* lw_,
                                          const uint8_t* nw_, int c0 = 0) {
  const size_t qd = (size_t)a.nq * HD;
  constexpr int LPC = HD / 4, CPP = 64 / LPC;  // lanes per column, columns per pass
  constexpr int CPW = NC / kPaWaves > CPP ? NC / kPaWaves : CPP;  // columns per wave
  if (wave * CPW >= NC) return;
#pragma unroll
  for (int i = 0; i < CPW; i += CPP) {
    const int cl = wave * CPW + i + lane / LPC, c = c0 + cl, d = 4 * (lane % LPC);
    const int row = row0 + c % rpt;
    float M = -INFINITY;
#pragma unroll
    for (int w = 0; w < NS; w++) M = fmaxf(M, mw_[w * NC + cl]);
    float L = 0.0f;
    v4f v = {0.0f, 0.0f, 0.0f, 0.0f};
    bool nan = false;
#pragma unroll
    for (int w = 0; w < NS; w++) {
      // no tile or masked keys only: (0, -inf, 0); a NaN sum always counts
      const float mw = mw_[w * NC + cl], lw = lw_[w * NC + cl];
      const float f = mw == -INFINITY ? 0.0f : expf(mw - M);
      L += lw != lw ? lw : f * lw;
      nan = nan || nw_[w * NC + cl];
      const v4f ow = *reinterpret_cast<const v4f*>(op + (size_t)(w * NC + cl) * pitch + d);
#pragma unroll
      for (int x = 0; x < 4; x++) v[x] = f != 0.0f ? fmaf(f, ow[x], v[x]) : v[x];
    }
    if (d == 0 && row < a.n && !(isfinite(M) && isfinite(L))) atomicOr(a.err, 4u);
    const float inv = nan ? __builtin_nanf("") : 1.0f / L;
#pragma unroll
    for (int x = 0; x < 4; x++) v[x] *= inv;
    const size_t o0 = (size_t)row * qd + (size_t)(h0 + c / rpt) * HD + d;
    if (a.out) {
      if (row < a.n) *reinterpret_cast<v4f*>(a.out + o0) = v;
    } else {
      // q8_0_encode_lane's arithmetic, four values per lane
      float amax = fmaxf(fmaxf(fabsf(v.x), fabsf(v.y)), fmaxf(fabsf(v.z), fabsf(v.w)));
      float bad = isfinite(v.x) && isfinite(v.y) && isfinite(v.z) && isfinite(v.w) ? 0.0f : 1.0f;
      amax = fmaxf(amax, dpp_f32<0xB1>(amax));   // quad_perm [1,0,3,2]
      amax = fmaxf(amax, dpp_f32<0x4E>(amax));   // quad_perm [2,3,0,1]
      amax = fmaxf(amax, dpp_f32<0x141>(amax));  // row_half_mirror: the block's 8 lanes
      bad = fmaxf(bad, dpp_f32<0xB1>(bad));
      bad = fmaxf(bad, dpp_f32<0x4E>(bad));
      bad = fmaxf(bad, dpp_f32<0x141>(bad));
      uint32_t dbits = bad != 0.0f ? 0x7E00u : 0u, q4 = 0;
      if (bad == 0.0f && amax != 0.0f) {
        const double dd = (double)amax / 127.0;
        const double dinv = 1.0 / dd;
#pragma unroll
        for (int x = 0; x < 4; x++) {
          const double r = fmin(127.0, fmax(-127.0, rint((double)v[x] * dinv)));
          q4 |= ((uint32_t)(int)r & 0xFFu) << (8 * x);
        }
        dbits = f64_to_f16_rne(fmin(dd, 65504.0));
      }
      if (row < a.n) {
        *reinterpret_cast<uint32_t*>(a.qs + o0) = q4;
        if ((lane & 7) == 0) a.qsd[o0 / 32] = (uint16_t)dbits;
      }
    }
  }
}

template <int HD>
__global__ __launch_bounds__(kPaWaves * 64) void attn_prefill_kernel(PrefillAttnArgs a, int hp) {
  constexpr int C4 = HD / 16;  // float4 columns per lane of a K row
  constexpr int DT = HD / 16;  // dims per lane of a V row
  constexpr int P = HD + 4;    // LDS row pitch (floats)
  __shared__ __attribute__((aligned(16))) float Qs[kPaCols * P];
  __shared__ __attribute__((aligned(16))) float Op[kPaWaves][kPaCols * P];
  __shared__ float Mw[kPaWaves][kPaCols], Lw[kPaWaves][kPaCols];
  __shared__ uint8_t Nw[kPaWaves][kPaCols];  // the column attends to a non-finite V row
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int col = lane & 15, j = lane >> 4;
  const int rpt = kPaCols / hp;                              // prompt rows per workgroup
  const int h0 = blockIdx.x * hp;                            // first query head
  const int kvh = h0 / (a.nq / a.nkv);
  const int row0 = (int)(gridDim.y - 1 - blockIdx.y) * rpt;  // the longest contexts first
  const size_t qd = (size_t)a.nq * HD, kvd = (size_t)a.nkv * HD;
  // column c: head h0 + c / rpt, row row0 + c % rpt (clamped past the
  // chunk); half h holds columns 16 h ..
  const int pos0h = a.pos0 + min(row0 + col, a.n - 1);
  const int pos1h = a.pos0 + min(row0 + (16 + col) % rpt, a.n - 1);
  const int pos_min = a.pos0 + row0, pos_max = a.pos0 + min(row0 + rpt, a.n) - 1;
  const int ntiles = pos_max / kPaKeys + 1;
  // byte offsets from a tile's first row: this lane's K row, its V piece
  const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.kcache + (size_t)kvh * HD);
  const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.vcache + (size_t)kvh * HD);
  const uint32_t rowb = (uint32_t)kvd * 4;
  const uint32_t koff = (uint32_t)col * rowb + 16u * (uint32_t)j;
  const uint32_t voff = 4u * (uint32_t)j * rowb + (uint32_t)(4 * DT * col);

  if (ntiles <= kPaWaves / 2) {
    // Short contexts: a wave takes one tile for one half, with every operand
    // loaded up front (Q too, from memory): one round trip and half the
    // matrix work of a tile on the way.  The sums are the long form's, so a
    // row's bits are too.
    const int t = wave & 3, h = wave >> 2;
    if (t < ntiles) {
      pa_one_tile<HD>(a, kvh, t, col, j, min(row0 + (16 * h + col) % rpt, a.n - 1), h0 + (16 * h + col) / rpt,
                      kPaKeys * t + kPaKeys - 1 > pos_min, &Op[t][(16 * h + col) * P], &Mw[t][16 * h + col],
                      &Lw[t][16 * h + col], &Nw[t][16 * h + col]);
    } else if (j == 0) {
      Mw[t][16 * h + col] = -INFINITY;
      Lw[t][16 * h + col] = 0.0f;
      Nw[t][16 * h + col] = 0;
    }
  } else {
  for (int i = tid; i < kPaCols * (HD / 4); i += kPaWaves * 64) {
    const int c = i / (HD / 4), f = i % (HD / 4);
    const int row = min(row0 + c % rpt, a.n - 1);
    *reinterpret_cast<v4f*>(Qs + c * P + 4 * f) =
        reinterpret_cast<const v4f*>(a.q + (size_t)row * qd + (size_t)(h0 + c / rpt) * HD)[f];
  }

  v4f kr[C4];
  // rows past the last position are read too (the cache ends in a tile of
  // padding rows); their scores are masked
  auto load_k = [&](int t) {
    const uint8_t* kt = kbase + (size_t)(kPaKeys * t) * rowb;
#pragma unroll
    for (int c = 0; c < C4; c++) kr[c] = *reinterpret_cast<const v4f*>(kt + koff + 64 * c);
  };
  if (wave < ntiles) load_k(wave);
  __syncthreads();

  v4f o[2][DT];
#pragma unroll
  for (int h = 0; h < 2; h++)
#pragma unroll
    for (int d = 0; d < DT; d++) o[h][d] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  float m[2] = {-INFINITY, -INFINITY}, l[2] = {0.0f, 0.0f};
  bool nan_score[2] = {false, false}, poison[2] = {false, false};

  auto tile = [&](int t, auto more) {
    v4f vr[4][DT / 4];
    const uint8_t* vt = vbase + (size_t)(kPaKeys * t) * rowb;
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int x = 0; x < DT / 4; x++)
        vr[e][x] = *reinterpret_cast<const v4f*>(vt + (size_t)(e * rowb) + voff + 16 * x);
    __builtin_amdgcn_sched_barrier(0);
    // per half two chains, one per half of the head dim (half the additions
    // on a chain: smaller rounding errors, and shorter dependent runs)
    v4f s[2] = {v4f{0.0f, 0.0f, 0.0f, 0.0f}, v4f{0.0f, 0.0f, 0.0f, 0.0f}}, s2[2] = {s[0], s[0]};
    // Q is read from LDS per tile, one column ahead (hoisted out of the tile
    // loop its 64 registers would spill)
    const auto* q4 = (const __attribute__((address_space(3))) v4f*)(Qs + col * P + 4 * j);
    asm volatile("" : "+v"(q4));
    v4f q0 = q4[0], q1 = q4[4 * P];
#pragma unroll
    for (int c = 0; c < C4; c++) {
      // keeps the steps in this order, and the reads whole
      asm volatile("" : "+v"(s[0]), "+v"(s[1]), "+v"(s2[0]), "+v"(s2[1]), "+v"(q0), "+v"(q1));
      const v4f p0 = q0, p1 = q1;
      if (c + 1 < C4) {
        q0 = q4[4 * (c + 1)];
        q1 = q4[4 * P + 4 * (c + 1)];
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int r = 0; r < 4; r++) {
        v4f(&sc)[2] = c >= C4 / 2 ? s2 : s;
        sc[0] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c][r], p0[r], sc[0], 0, 0, 0);
        sc[1] = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c][r], p1[r], sc[1], 0, 0, 0);
      }
    }
    s[0] += s2[0];
    s[1] += s2[1];
    __builtin_amdgcn_sched_barrier(0);
    if (decltype(more)::value) load_k(t + kPaWaves);
    __builtin_amdgcn_sched_barrier(0);
    const bool masked = kPaKeys * t + kPaKeys - 1 > pos_min;  // uniform: some column ends inside the tile
#pragma unroll
    for (int h = 0; h < 2; h++) {
      const float alpha = pa_soften(s[h], a.scale, t, j, masked, h ? pos1h : pos0h, m[h], l[h], nan_score[h]);
#pragma unroll
      for (int d = 0; d < DT; d++) o[h][d] *= alpha;
    }
    if (masked) {
      const int first = pa_clean<DT>(vr);
      poison[0] = poison[0] || (first < 64 && kPaKeys * t + first <= pos0h);
      poison[1] = poison[1] || (first < 64 && kPaKeys * t + first <= pos1h);
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int d = 0; d < DT; d++) {
        o[0][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[e][d / 4][d % 4], s[0][e], o[0][d], 0, 0, 0);
        o[1][d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[e][d / 4][d % 4], s[1][e], o[1][d], 0, 0, 0);
      }
  };
  if (wave < ntiles) {
    int t = wave;
    for (; t + kPaWaves < ntiles; t += kPaWaves) tile(t, std::true_type{});
    tile(t, std::false_type{});
#pragma unroll
    for (int h = 0; h < 2; h++)
      pa_put<HD>(&Op[wave][(16 * h + col) * P], &Mw[wave][16 * h + col], &Lw[wave][16 * h + col], &Nw[wave][16 * h + col], col,
                 j, true, o[h], m[h], l[h], nan_score[h], poison[h]);
  } else if (lane < kPaCols) {
    Mw[wave][lane] = -INFINITY;
    Lw[wave][lane] = 0.0f;
    Nw[wave][lane] = 0;
  }
  }
  __syncthreads();
  if (ntiles <= kPaWaves / 2)
    pa_finish<HD, kPaWaves / 2>(a, h0, row0, rpt, wave, lane, &Op[0][0], P, &Mw[0][0], &Lw[0][0], &Nw[0][0]);
  else
    pa_finish<HD, kPaWaves>(a, h0, row0, rpt, wave, lane, &Op[0][0], P, &Mw[0][0], &Lw[0][0], &Nw[0][0]);
}

// Five to eight tiles of few units: a workgroup per half, each wave one tile of
// it with every operand loaded up front as in the short form (the long form's
// waves take both halves and read Q through LDS).  The sums are the long
// form's.  16 query and 8 KV heads of 128: 16 rows at position 64 12.4 -> 8.0 us,
// at 112 12.8 -> 8.8, 100 rows at 0 12.6 -> 8.2 us.
template <int HD>
__global__ __launch_bounds__(kPaWaves * 64) void attn_prefill_half_kernel(PrefillAttnArgs a, int hp) {
  constexpr int P = HD + 4, NC = kPaCols / 2;
  __shared__ __attribute__((aligned(16))) float Op[kPaWaves][NC * P];
  __shared__ float Mw[kPaWaves][NC], Lw[kPaWaves][NC];
  __shared__ uint8_t Nw[kPaWaves][NC];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, j = lane >> 4, h = blockIdx.z;
  const int rpt = kPaCols / hp, h0 = blockIdx.x * hp, kvh = h0 / (a.nq / a.nkv);
  const int row0 = (int)(gridDim.y - 1 - blockIdx.y) * rpt;
  const int qrow = min(row0 + (16 * h + col) % rpt, a.n - 1);
  const int pos_min = a.pos0 + row0, ntiles = (a.pos0 + min(row0 + rpt, a.n) - 1) / kPaKeys + 1;
  float* op = &Op[wave][col * P];
  if (wave < ntiles) {
    pa_one_tile<HD>(a, kvh, wave, col, j, qrow, h0 + (16 * h + col) / rpt, kPaKeys * wave + kPaKeys - 1 > pos_min, op,
                    &Mw[wave][col], &Lw[wave][col], &Nw[wave][col]);
  } else if (j == 0) {
    Mw[wave][col] = -INFINITY;
    Lw[wave][col] = 0.0f;
    Nw[wave][col] = 0;
  }
  __syncthreads();
  pa_finish<HD, kPaWaves, NC>(a, h0, row0, rpt, wave, lane, &Op[0][0], P, &Mw[0][0], &Lw[0][0], &Nw[0][0], 16 * h);
}

// Few rows at a long context (a short turn of a long conversation): a launch
// of nq / hp workgroups leaves most CUs idle while each walks the whole
// context.  Here four workgroups share a (heads, rows) unit: wave w of
// workgroup z takes half w % 2 of slot 2 z + w / 2, whose tiles are that slot's
// of the long form (slot, slot + 8, ...), one wave per SIMD; the partials go
// to memory and attn_prefill_merge_kernel finishes the rows.  Every sum is the
// long form's, so a row's bits are too.  16 query and 8 KV heads of 128, 16 rows,
// with the merge's launch: at position 128 15.1 -> 13.2 us, 400 25.2 -> 15.9, 2,000
// 85.7 -> 32.5 us (a model's prefill of 16 rows there 4.65 -> 3.25 ms, 3.60 ms
// with one workgroup per head and row).
constexpr int kPaSplit = 4;      // workgroups per unit
constexpr int kPaSplitWgs = 64;  // units of a split launch at most: a workgroup per CU
struct PaPart {  // one unit's partials in memory
  float* op;
  float *mw, *lw;
  uint8_t* nw;
};
template <int HD>
__device__ __forceinline__ PaPart pa_part(const PrefillAttnArgs& a) {
  constexpr size_t SC = (size_t)kPaWaves * kPaCols;
  const size_t u = blockIdx.y * gridDim.x + blockIdx.x, nu = (size_t)gridDim.x * gridDim.y;
  float* mw = a.part + nu * SC * HD;
  return {a.part + u * SC * HD, mw + u * SC, mw + (nu + u) * SC, reinterpret_cast<uint8_t*>(mw + 2 * nu * SC) + u * SC};
}

template <int HD>
__global__ __launch_bounds__(kPaSplit * 64) void attn_prefill_split_kernel(PrefillAttnArgs a, int hp) {
  constexpr int C4 = HD / 16, DT = HD / 16;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int col = lane & 15, j = lane >> 4;
  const int rpt = kPaCols / hp, h0 = blockIdx.x * hp, kvh = h0 / (a.nq / a.nkv);
  const int row0 = (int)(gridDim.y - 1 - blockIdx.y) * rpt;
  const size_t qd = (size_t)a.nq * HD, kvd = (size_t)a.nkv * HD;
  const int slot = 2 * (int)blockIdx.z + (wave >> 1), h = wave & 1;
  const int row = row0 + (16 * h + col) % rpt, qrow = min(row, a.n - 1), pos = a.pos0 + qrow;
  const int pos_min = a.pos0 + row0, pos_max = a.pos0 + min(row0 + rpt, a.n) - 1;
  const int ntiles = pos_max / kPaKeys + 1;
  const PaPart part = pa_part<HD>(a);
  const int at = slot * kPaCols + 16 * h + col;
  if (slot >= ntiles) {
    if (j == 0) {
      part.mw[at] = -INFINITY;
      part.lw[at] = 0.0f;
      part.nw[at] = 0;
    }
    return;
  }
  const uint32_t rowb = (uint32_t)kvd * 4;
  const uint8_t* kbase = reinterpret_cast<const uint8_t*>(a.kcache + (size_t)kvh * HD);
  const uint8_t* vbase = reinterpret_cast<const uint8_t*>(a.vcache + (size_t)kvh * HD);
  const uint32_t koff = (uint32_t)col * rowb + 16u * (uint32_t)j;
  const uint32_t voff = 4u * (uint32_t)j * rowb + (uint32_t)(4 * DT * col);
  const v4f* qg = reinterpret_cast<const v4f*>(a.q + (size_t)qrow * qd + (size_t)(h0 + (16 * h + col) / rpt) * HD) + j;
  v4f qr[C4], kr[C4];
  auto load_k = [&](int t) {
    const uint8_t* kt = kbase + (size_t)(kPaKeys * t) * rowb;
#pragma unroll
    for (int c = 0; c < C4; c++) kr[c] = *reinterpret_cast<const v4f*>(kt + koff + 64 * c);
  };
#pragma unroll
  for (int c = 0; c < C4; c++) qr[c] = qg[4 * c];
  load_k(slot);
  v4f o[DT];
#pragma unroll
  for (int d = 0; d < DT; d++) o[d] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
  float m = -INFINITY, l = 0.0f;
  bool nan_score = false, poison = false;
  for (int t = slot; t < ntiles; t += kPaWaves) {
    v4f vr[4][DT / 4];
    const uint8_t* vt = vbase + (size_t)(kPaKeys * t) * rowb;
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int x = 0; x < DT / 4; x++)
        vr[e][x] = *reinterpret_cast<const v4f*>(vt + (size_t)(e * rowb) + voff + 16 * x);
    __builtin_amdgcn_sched_barrier(0);
    v4f s = {0.0f, 0.0f, 0.0f, 0.0f}, s2 = s;
#pragma unroll
    for (int c = 0; c < C4 / 2; c++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        s = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[c][r], qr[c][r], s, 0, 0, 0);
        s2 = __builtin_amdgcn_mfma_f32_16x16x4f32(kr[C4 / 2 + c][r], qr[C4 / 2 + c][r], s2, 0, 0, 0);
      }
    s += s2;
    __builtin_amdgcn_sched_barrier(0);
    load_k(min(t + kPaWaves, ntiles - 1));  // (the last tile's again past the end: not used)
    __builtin_amdgcn_sched_barrier(0);
    const bool masked = kPaKeys * t + kPaKeys - 1 > pos_min;
    const float alpha = pa_soften(s, a.scale, t, j, masked, pos, m, l, nan_score);
#pragma unroll
    for (int d = 0; d < DT; d++) o[d] *= alpha;
    if (masked) {
      const int first = pa_clean<DT>(vr);
      poison = poison || (first < 64 && kPaKeys * t + first <= pos);
    }
#pragma unroll
    for (int e = 0; e < 4; e++)
#pragma unroll
      for (int d = 0; d < DT; d++) o[d] = __builtin_amdgcn_mfma_f32_16x16x4f32(vr[e][d / 4][d % 4], s[e], o[d], 0, 0, 0);
  }
  pa_put<HD>(part.op + (size_t)at * HD, part.mw + at, part.lw + at, part.nw + at, col, j, row < a.n, o, m, l, nan_score, poison);
}

template <int HD>
__global__ __launch_bounds__(kPaWaves * 64) void attn_prefill_merge_kernel(PrefillAttnArgs a, int hp) {
  const int rpt = kPaCols / hp;
  const PaPart part = pa_part<HD>(a);
  pa_finish<HD, kPaWaves>(a, (int)blockIdx.x * hp, (int)(gridDim.y - 1 - blockIdx.y) * rpt, rpt,
                          __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), threadIdx.x & 63, part.op, HD, part.mw, part.lw,
                          part.nw);
}

// Units of a launch: grid x (heads in groups of hp), grid y (rows).
static dim3 pa_grid(int nq, int nkv, int n, int& hp) {
  // two query heads of a KV head per workgroup where it has an even number
  hp = (nq / nkv) % 2 == 0 ? 2 : 1;
  return dim3((unsigned)(nq / hp), (unsigned)((n + kPaCols / hp - 1) / (kPaCols / hp)));
}

size_t attn_prefill_scratch(int nq, int nkv, int head_dim, int n) {
  int hp;
  const dim3 g = pa_grid(nq, nkv, n, hp);
  const size_t nu = (size_t)g.x * g.y;
  return nu <= kPaSplitWgs ? nu * kPaWaves * kPaCols * ((size_t)head_dim * 4 + 9) : 0;
}

template <int HD>
static void launch_pa(const PrefillAttnArgs& a, hipStream_t st) {
  int hp;
  dim3 grid = pa_grid(a.nq, a.nkv, a.n, hp);
  const int tiles = (a.pos0 + a.n - 1) / kPaKeys + 1;  // of the longest context
  const bool few = grid.x * grid.y <= (unsigned)kPaSplitWgs;
  if (few && tiles > kPaWaves / 2 && tiles <= kPaWaves) {
    grid.z = 2;
    hipLaunchKernelGGL(attn_prefill_half_kernel<HD>, grid, dim3(kPaWaves * 64), 0, st, a, hp);
    return;
  }
  // from nine tiles on some slot has two (64 units of head_dim 64, 128 rows at
  // position 128, gain the least: 9.4 / 9.5 us)
  if (!(few && tiles > kPaWaves && a.part && a.part_bytes >= attn_prefill_scratch(a.nq, a.nkv, HD, a.n))) {
    hipLaunchKernelGGL(attn_prefill_kernel<HD>, grid, dim3(kPaWaves * 64), 0, st, a, hp);
    return;
  }
  grid.z = kPaSplit;
  hipLaunchKernelGGL(attn_prefill_split_kernel<HD>, grid, dim3(kPaSplit * 64), 0, st, a, hp);
  grid.z = 1;
  hipLaunchKernelGGL(attn_prefill_merge_kernel<HD>, grid, dim3(kPaWaves * 64), 0, st, a, hp);
}

hipError_t launch_attn_prefill(const PrefillAttnArgs& a, int head_dim, hipStream_t st) {
  if (a.n <= 0) return hipSuccess;
  if (head_dim == 128) launch_pa<128>(a, st);
  else if (head_dim == 64) launch_pa<64>(a, st);
  else return hipErrorInvalidValue;
  return hipGetLastError();
}

}  // namespace zg
