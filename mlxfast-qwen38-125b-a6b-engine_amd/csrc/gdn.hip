// Gated-deltanet (GDN) sublayer core of the target's linear-attention layers
// for a window of S <= 8 positions: causal depthwise conv + SiLU, q/k RMS
// norms and scales, decay/beta gates, the delta-rule recurrence with a
// Kahan-compensated key product, and the gated output RMS norm -- one launch,
// four workgroups per value head (each owns a quarter of the head's state
// rows; the head's last one to finish, by a ticket, runs the gated norm over
// the rows' outputs the others published at device scope).
//
// Window state.  The reference keeps the recurrent state after every window
// position so the engine can roll back to any of them (Runner/FastModel/
// TrackFastModel.swift:726-731, stageCaptured).  Here a window writes a
// journal instead -- its conv input rows, the normalised keys, and per
// (head, value row) the delta and per head the decay of every position, about
// 50 KB per position against 3.1 MB of state -- and leaves the committed state
// alone.  Committing n positions only records n; the next window first replays
// those n steps (the same float operations, so the same bits) onto the
// committed state and stores it, then runs its own positions.  Journal and conv
// base are double-buffered (slot `cur` read, slot `nxt` written) so no
// workgroup overwrites what another still reads; each recurrent state row is
// read and written by the one workgroup that owns it.
//
// Lane structure (fixes the float order): every 128-element reduction is 32
// lanes x 4 consecutive elements, each lane in element order, then an xor
// butterfly over the 32 lanes (half a wave).
// Reference: FM/TrackFastKernels.swift:48-117 (prep), :486-605 (recurrence,
// peeled Kahan form), FM/TrackFastKernels2.swift:325-352 (gated RMS),
// FM/TrackFastGDNDecode.swift:50-274 (the fused decode form this follows),
// FM/TrackFastKernels2.swift:48-58 (logaddexp).
#include "mtpx_kernels.h"

namespace mtpx {

constexpr int GDN_THREADS = 512;  // 16 half-waves
constexpr int GDN_D = 128;
constexpr int GDN_SPLIT = 4;      // workgroups per value head, each owning 128 / GDN_SPLIT state rows
constexpr int GDN_BSPLIT = 16;    // the batch kernel's workgroups per value head
constexpr int GDN_BTHREADS = 256; // and their threads: a state row per half-wave
constexpr int GDN_BWIN = 16;      // positions it stages at once

// log1p(y), y in [0, 1]: 2 atanh(s), s = y / (2 + y), odd series to s^15.
__device__ __forceinline__ float log1p_det(float y) {
  if (y != y) return y;
  const float t = 2.0f + y;
  const float s = y / t;
  const float s2 = s * s;
  float r = 1.0f / 15.0f;
  r = 1.0f / 13.0f + s2 * r;
  r = 1.0f / 11.0f + s2 * r;
  r = 1.0f / 9.0f + s2 * r;
  r = 1.0f / 7.0f + s2 * r;
  r = 1.0f / 5.0f + s2 * r;
  r = 1.0f / 3.0f + s2 * r;
  r = s2 * r;
  const float h = s + s * r;
  return h + h;
}

// MLX logaddexp(x, 0) in bf16 arithmetic.
__device__ __forceinline__ float logaddexp0_bf16(float x) {
  if (x != x) return x;
  const float inf = __uint_as_float(0x7f800000u);
  const float mx = x > 0.0f ? x : 0.0f;
  const float mn = x < 0.0f ? x : 0.0f;
  if (mn == -inf || mx == inf) return mx;
  const float d = round_bf(mn - mx);
  const float e = round_bf(expf_det(d));
  const float l = round_bf(log1p_det(e));
  return round_bf(mx + l);
}

// MLX Sigmoid in f32.
__device__ __forceinline__ float sigmoid_f32(float x) {
  const float e = expf_det(__builtin_fabsf(x));
  const float y = 1.0f / (1.0f + e);
  return (x < 0.0f) ? y : 1.0f - y;
}

__device__ __forceinline__ float half_wave_sum(float v) {
  return fold_sum<16>(v);
}

// Element c of four bf16 packed in two words (little-endian), as a float.
__device__ __forceinline__ float kjournal(uint2 w, int c) {
  const uint32_t v = c < 2 ? w.x : w.y;
  return __uint_as_float((c & 1) ? (v & 0xffff0000u) : (v << 16));
}

// Row r of the virtual input sequence conv_cur (KC-1 rows) ++ the P committed
// journal rows ++ the window's projection rows.
__device__ __forceinline__ float gdn_row(const GdnArgs& a, int r, int ch) {
  const int KM1 = a.kc - 1;
  if (r < KM1) return bf2f(a.conv_cur[(size_t)r * a.cd + ch]);
  r -= KM1;
  if (r < a.P) return bf2f(a.win_cur[(size_t)r * a.cd + ch]);
  r -= a.P;
  return bf2f(a.proj[(size_t)r * a.pw + ch]);
}

// Row r of the same virtual sequence as a pointer to its channel 0 (r is uniform).
__device__ __forceinline__ const bf16* gdn_row_ptr(const GdnArgs& a, int r) {
  const int KM1 = a.kc - 1;
  if (r < KM1) return a.conv_cur + (size_t)r * a.cd;
  r -= KM1;
  if (r < a.P) return a.win_cur + (size_t)r * a.cd;
  return a.proj + (size_t)(r - a.P) * a.pw;
}

// JP: journal steps the launch can replay (P <= JP), so the replay's loads issued up front are its
// own, not clamped duplicates up to MAX_TOKENS ahead of the prep's loads.
template <int KC, int JP>
__global__ __launch_bounds__(GDN_THREADS) void k_gdn_step(GdnArgs a) {
  static_assert(JP >= 1 && JP <= MAX_TOKENS, "journal steps");
  __shared__ float qs[MAX_TOKENS][GDN_D], ks[MAX_TOKENS][GDN_D], vs[MAX_TOKENS][GDN_D], ys[MAX_TOKENS][GDN_D];
  __shared__ float dec[MAX_TOKENS], bet[MAX_TOKENS];
  __shared__ bf16 gated[MAX_TOKENS][GDN_D];
  const int h = blockIdx.x, ratio = a.hv / a.hk, hk = h / ratio;
  const int r0 = blockIdx.y * (GDN_D / GDN_SPLIT);  // this workgroup's state rows r0 .. r0 + 128/GDN_SPLIT - 1
  const bool w0 = blockIdx.y == 0;                  // writes the head's journal rows (conv, keys, decay)
  const bool lead = (h % ratio) == 0 && w0;         // writes the q/k channels' journal and conv rows
  const int hw = threadIdx.x >> 5, l = threadIdx.x & 31;
  const int S = a.S, P = a.P, KM1 = a.kc - 1;
  const float inv_scale = 1.0f / sqrtf((float)GDN_D);
  const float q_mul = round_bf(inv_scale * inv_scale), k_mul = round_bf(inv_scale);

  // The state rows of this half-wave's recurrence (r = r0 + hw + 16 i) and the journal steps it replays,
  // loaded before the prep so their latency hides behind it.
  constexpr int RPH = GDN_D / GDN_SPLIT / (GDN_THREADS / 32);
  float s[RPH][4];
#pragma unroll
  for (int i = 0; i < RPH; ++i) {
    const float4 s4 = *reinterpret_cast<const float4*>(a.ssm + ((size_t)h * GDN_D + r0 + hw + 16 * i) * GDN_D + 4 * l);
    s[i][0] = s4.x;
    s[i][1] = s4.y;
    s[i][2] = s4.z;
    s[i][3] = s4.w;
  }
  float gdp[JP], dlp[JP][RPH];
  uint2 kpw[JP];  // the journal keys' four bf16 (raw until the replay, so no wait for them here)
  if (P > 0) {
#pragma unroll
    for (int p = 0; p < JP; ++p) {
      const int pc = p < P ? p : P - 1;  // clamped: loads beyond P are issued but not used
      gdp[p] = a.decay_cur[(size_t)pc * a.hv + h];
      kpw[p] = *reinterpret_cast<const uint2*>(a.key_cur + ((size_t)pc * a.hk + hk) * GDN_D + 4 * l);
#pragma unroll
      for (int i = 0; i < RPH; ++i) dlp[p][i] = a.delta_cur[((size_t)pc * a.hv + h) * GDN_D + r0 + hw + 16 * i];
    }
  }

  // The inputs of the prep's last steps, loaded now so their latency hides behind the loads above
  // and the conv's: the positions' gate inputs (position t: thread GDN_THREADS - S + t, the last
  // wave, which has no conv task up to five positions) and, in a head's first workgroup, the conv
  // rows R[P .. P+KC-1) that become the next window's base (element i = (j, kind, d)).
  // (every thread loads, position 0 outside the gate threads, no branch; raw bf16 bits until the
  // use, so nothing waits for them here)
  const int gt = (int)threadIdx.x - (GDN_THREADS - S);  // this thread's gate position, or < 0
  const uint16_t* prow = reinterpret_cast<const uint16_t*>(a.proj) + (size_t)(gt >= 0 ? gt : 0) * a.pw;
  const uint32_t g_b = prow[a.b_off + h], g_a = prow[a.a_off + h];
  const uint32_t g_dt = reinterpret_cast<const uint16_t*>(a.dt_bias)[h];
  const float g_al = a.neg_exp_alog[h];
  constexpr int CN = ((KC - 1) * 3 * GDN_D + GDN_THREADS - 1) / GDN_THREADS;
  bf16 cb[CN];
#pragma unroll
  for (int q = 0; q < CN; ++q) {
    const int i = (int)threadIdx.x + q * GDN_THREADS;
    const int j = i / (3 * GDN_D), kind = (i / GDN_D) % 3, d = i % GDN_D;
    const int vec = kind == 0 ? hk : (kind == 1 ? a.hk + hk : 2 * a.hk + h);
    cb[q] = (w0 && i < KM1 * 3 * GDN_D && (kind == 2 || lead)) ? gdn_row_ptr(a, P + j)[vec * GDN_D + d] : (bf16)0;
  }
  asm volatile("" ::: "memory");

  // ---- prep: (q, k, v) vectors x positions, 32 lanes x 4 channels each; a lane's KC input rows
  // (4 channels each) and its 4 x KC conv taps are loaded before the first multiply
  for (int task = hw; task < 3 * S; task += GDN_THREADS / 32) {
    const int t = task / 3, kind = task % 3;
    const int vec = kind == 0 ? hk : (kind == 1 ? a.hk + hk : 2 * a.hk + h);
    const int ch0 = vec * GDN_D + 4 * l;
    uint2 xin[KC];
#pragma unroll
    for (int j = 0; j < KC; ++j) xin[j] = *reinterpret_cast<const uint2*>(gdn_row_ptr(a, P + t + j) + ch0);
    uint32_t wt[2 * KC];  // conv_w[ch0 .. ch0+3][0 .. KC-1]: 4*KC bf16, contiguous
#pragma unroll
    for (int q = 0; q < 2 * KC; ++q) wt[q] = reinterpret_cast<const uint32_t*>(a.conv_w + (size_t)ch0 * KC)[q];
    auto hbf = [](uint32_t w, int odd) { return __uint_as_float(odd ? (w & 0xffff0000u) : (w << 16)); };
    float xs[4], acc = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float c = 0.0f;
#pragma unroll
      for (int j = 0; j < KC; ++j) {
        const float xv = hbf(i < 2 ? xin[j].x : xin[j].y, i & 1);
        const int e = i * KC + j;
        c = c + xv * hbf(wt[e >> 1], e & 1);
      }
      const float x = silu_bf16(round_bf(c));
      xs[i] = x;
      acc = __builtin_fmaf(x, x, acc);
    }
    if ((kind == 2 && w0) || lead)  // this position's conv input row (row P + t + KC-1 is projection row t)
      *reinterpret_cast<uint2*>(a.win_nxt + (size_t)t * a.cd + ch0) = xin[KC - 1];
    if (kind < 2) {
      const float inv = 1.0f / sqrtf(half_wave_sum(acc) / 128.0f + 1e-6f);
      const float mul = kind == 0 ? q_mul : k_mul;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float val = round_bf(mul * round_bf(xs[i] * inv));
        if (kind == 0) {
          qs[t][4 * l + i] = val;
        } else {
          ks[t][4 * l + i] = val;
          if (lead) a.key_nxt[((size_t)t * a.hk + hk) * GDN_D + 4 * l + i] = f2bf(val);
        }
      }
    } else {
#pragma unroll
      for (int i = 0; i < 4; ++i) vs[t][4 * l + i] = xs[i];
    }
  }
  if (gt >= 0) {
    const int t = gt;
    const float b = sigmoid_bf16(__uint_as_float(g_b << 16));
    const float ax = round_bf(__uint_as_float(g_a << 16) + __uint_as_float(g_dt << 16));
    const float d = expf_det(g_al * logaddexp0_bf16(ax));
    dec[t] = d;
    bet[t] = b;
    if (w0) a.decay_nxt[(size_t)t * a.hv + h] = d;
  }
  // the committed conv rows R[P .. P+KC-1) become the next window's base
#pragma unroll
  for (int q = 0; q < CN; ++q) {
    const int i = (int)threadIdx.x + q * GDN_THREADS;
    const int j = i / (3 * GDN_D), kind = (i / GDN_D) % 3, d = i % GDN_D;
    const int vec = kind == 0 ? hk : (kind == 1 ? a.hk + hk : 2 * a.hk + h);
    if (w0 && i < KM1 * 3 * GDN_D && (kind == 2 || lead)) a.conv_nxt[(size_t)j * a.cd + vec * GDN_D + d] = cb[q];
  }
  __syncthreads();

  // ---- recurrence: RPH value rows per half-wave (r = r0 + hw + 16 i), lane l owns key elements 4l..4l+3
  if (P > 0) {  // committed steps of the previous window, in order
#pragma unroll
    for (int p = 0; p < JP; ++p) {
      if (p < P) {
#pragma unroll
        for (int i = 0; i < RPH; ++i)
#pragma unroll
          for (int c = 0; c < 4; ++c) {
            s[i][c] = s[i][c] * gdp[p];
            s[i][c] = __builtin_fmaf(kjournal(kpw[p], c), dlp[p][i], s[i][c]);
          }
      }
    }
#pragma unroll
    for (int i = 0; i < RPH; ++i)
      *reinterpret_cast<float4*>(a.ssm + ((size_t)h * GDN_D + r0 + hw + 16 * i) * GDN_D + 4 * l) =
          make_float4(s[i][0], s[i][1], s[i][2], s[i][3]);
  }
  // position by position, this thread's RPH state rows side by side (independent chains)
  for (int t = 0; t < S; ++t) {
    const float gd = dec[t], bt = bet[t];
    const float k0 = ks[t][4 * l], k1 = ks[t][4 * l + 1], k2 = ks[t][4 * l + 2], k3 = ks[t][4 * l + 3];
    const float q0 = qs[t][4 * l], q1 = qs[t][4 * l + 1], q2 = qs[t][4 * l + 2], q3 = qs[t][4 * l + 3];
#pragma unroll
    for (int i = 0; i < RPH; ++i) {
      const int r = r0 + hw + 16 * i;
      s[i][0] = s[i][0] * gd;
      float kv = 0.0f + s[i][0] * k0;
      float comp = 0.0f;
      {
        s[i][1] = s[i][1] * gd;
        const float prod = s[i][1] * k1, corr = prod - comp, next = kv + corr;
        comp = (next - kv) - corr;
        kv = next;
      }
      {
        s[i][2] = s[i][2] * gd;
        const float prod = s[i][2] * k2, corr = prod - comp, next = kv + corr;
        comp = (next - kv) - corr;
        kv = next;
      }
      {
        s[i][3] = s[i][3] * gd;
        const float prod = s[i][3] * k3, corr = prod - comp, next = kv + corr;
        kv = next;
      }
      const float kvm = half_wave_sum(kv);
      const float delta = (vs[t][r] - kvm) * bt;
      if (l == 0) a.delta_nxt[((size_t)t * a.hv + h) * GDN_D + r] = delta;
      float o = 0.0f;
      s[i][0] = __builtin_fmaf(k0, delta, s[i][0]);
      o = __builtin_fmaf(s[i][0], q0, o);
      s[i][1] = __builtin_fmaf(k1, delta, s[i][1]);
      o = __builtin_fmaf(s[i][1], q1, o);
      s[i][2] = __builtin_fmaf(k2, delta, s[i][2]);
      o = __builtin_fmaf(s[i][2], q2, o);
      s[i][3] = __builtin_fmaf(k3, delta, s[i][3]);
      o = __builtin_fmaf(s[i][3], q3, o);
      const float y = half_wave_sum(o);
      if (l == 0) st_pub(a.ypub + ((size_t)t * a.hv + h) * GDN_D + r, round_bf(y));
    }
  }
  // the head's last workgroup to finish gathers every row's output and runs the gated norm
  if (!ticket_last(a.tickets + h, GDN_SPLIT - 1)) return;
  for (int i = threadIdx.x; i < S * GDN_D; i += GDN_THREADS)
    ys[i / GDN_D][i % GDN_D] = ld_pub(a.ypub + ((size_t)(i / GDN_D) * a.hv + h) * GDN_D + i % GDN_D);
  __syncthreads();

  // ---- gated RMS norm per position
  for (int t = hw; t < S; t += GDN_THREADS / 32) {
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_fmaf(ys[t][4 * l + i], ys[t][4 * l + i], acc);
    const float inv = 1.0f / sqrtf(half_wave_sum(acc) / 128.0f + a.eps);
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int d = 4 * l + i;
      const float n = round_bf(bf2f(a.norm_w[d]) * round_bf(ys[t][d] * inv));
      const float z = bf2f(a.proj[(size_t)t * a.pw + a.z_off + h * GDN_D + d]);
      const bf16 out = f2bf(sigmoid_f32(z) * n);
      gated[t][d] = out;
      if (a.gated) a.gated[(size_t)t * a.hv * GDN_D + h * GDN_D + d] = out;
    }
  }
  __syncthreads();

  // ---- prepared blocks of the gated rows for the output projection (4 per head and position)
  if (a.xp)
    for (int task = hw; task < 4 * S; task += GDN_THREADS / 32) {
      const int t = task >> 2, blk = task & 3;
      xprep_lanes_direct(gated[t][blk * 32 + l], l, a.xp + ((size_t)t * a.hv * 4 + h * 4 + blk) * XP_DW);
    }
}

// A prefill batch through the core (S positions, any count), three launches.
//   k_gdn_prep_batch: one workgroup per position: the conv, SiLU and q/k norms of every key head's
//     q and k and every value head's v (a half-wave per 128-channel vector, as the step kernel
//     does them), and every head's decay and beta gates, into the batch's prep buffers;
//   k_gdn_batch: each value head's recurrence, the P committed steps of the previous window replayed
//     onto the state, then the batch's positions in order, the next positions' prepped vectors loaded
//     while the current ones' recurrence runs; every position committed: the state is stored after the
//     last one, the batch's last kc-1 conv input rows become the conv base (slot nxt), no journal is
//     written; the outputs go to ypub [hv][128][S rounded up to 32] as f32;
//   k_gdn_norm_batch: the gated norm and the prepared output blocks of every position.
// The float operations of every position are a verify window's, so the bits are the same.
template <int KC>
__global__ __launch_bounds__(GDN_THREADS) void k_gdn_prep_batch(GdnArgs a, GdnBatch b) {
  const int t = blockIdx.x, hw = threadIdx.x >> 5, l = threadIdx.x & 31;
  const int P = a.P;
  const float inv_scale = 1.0f / sqrtf((float)GDN_D);
  const float q_mul = round_bf(inv_scale * inv_scale), k_mul = round_bf(inv_scale);
  const int ntask = 2 * a.hk + a.hv;  // q of every key head, k of every key head, v of every value head
  for (int task = hw; task < ntask; task += GDN_THREADS / 32) {
    const int kind = task < a.hk ? 0 : (task < 2 * a.hk ? 1 : 2);
    const int vec = task;  // channel block: q heads, then k heads, then v heads
    const int ch0 = vec * GDN_D + 4 * l;
    uint2 xin[KC];
#pragma unroll
    for (int j = 0; j < KC; ++j) xin[j] = *reinterpret_cast<const uint2*>(gdn_row_ptr(a, P + t + j) + ch0);
    uint32_t wt[2 * KC];
#pragma unroll
    for (int q = 0; q < 2 * KC; ++q) wt[q] = reinterpret_cast<const uint32_t*>(a.conv_w + (size_t)ch0 * KC)[q];
    auto hbf = [](uint32_t w, int odd) { return __uint_as_float(odd ? (w & 0xffff0000u) : (w << 16)); };
    float xs[4], acc = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      float c = 0.0f;
#pragma unroll
      for (int j = 0; j < KC; ++j) {
        const float xv = hbf(i < 2 ? xin[j].x : xin[j].y, i & 1);
        const int e = i * KC + j;
        c = c + xv * hbf(wt[e >> 1], e & 1);
      }
      const float x = silu_bf16(round_bf(c));
      xs[i] = x;
      acc = __builtin_fmaf(x, x, acc);
    }
    float4 o;
    if (kind < 2) {
      const float inv = 1.0f / sqrtf(half_wave_sum(acc) / 128.0f + 1e-6f);
      const float mul = kind == 0 ? q_mul : k_mul;
      o = make_float4(round_bf(mul * round_bf(xs[0] * inv)), round_bf(mul * round_bf(xs[1] * inv)),
                      round_bf(mul * round_bf(xs[2] * inv)), round_bf(mul * round_bf(xs[3] * inv)));
    } else {
      o = make_float4(xs[0], xs[1], xs[2], xs[3]);
    }
    *reinterpret_cast<float4*>(b.vecs + ((size_t)t * ntask + vec) * GDN_D + 4 * l) = o;
  }
  for (int h = threadIdx.x; h < a.hv; h += GDN_THREADS) {
    const bf16* prow = a.proj + (size_t)t * a.pw;
    const float bt = sigmoid_bf16(bf2f(prow[a.b_off + h]));
    const float ax = round_bf(bf2f(prow[a.a_off + h]) + bf2f(a.dt_bias[h]));
    b.gates[((size_t)t * a.hv + h) * 2] = expf_det(a.neg_exp_alog[h] * logaddexp0_bf16(ax));
    b.gates[((size_t)t * a.hv + h) * 2 + 1] = bt;
  }
}

// Sixteen workgroups of four waves per value head, one state row per half-wave (768 workgroups at 48
// heads: three per CU, three waves per SIMD).  A step is about 45 vector instructions per row pair, at four
// cycles each and three waves 540 cycles a position: what it takes (575 measured).  So the rows' output sums
// of two positions share their fold (the first level puts one position in the lower, the other in the upper
// 16 lanes), the outputs stay in registers until 32 of them go out as one 128-byte store, and the gated norm
// is a launch of its own.  1003 positions, 48 heads: 333 us with a fold per position and the staged rows in
// an array (the compiler kept it in scratch, so the prefetch waited for its loads) -> 275 us; two rows per
// half-wave, sharing the k and q reads and both folds, 315 us (1.5 waves per SIMD do not spread evenly).
__global__ __launch_bounds__(GDN_BTHREADS) void k_gdn_batch(GdnArgs a, GdnBatch b) {
  constexpr int W = GDN_BWIN, RW = GDN_D / GDN_BSPLIT;  // staged positions; state rows of a workgroup
  static_assert(RW == GDN_BTHREADS / 32 && 2 * GDN_BWIN == 32, "a row per half-wave, two windows per output store");
  __shared__ float qs[2][W][GDN_D], ks[2][W][GDN_D];
  __shared__ float vs[2][W][RW], dec[2][W], bet[2][W];
  const int h = blockIdx.x, ratio = a.hv / a.hk, hk = h / ratio;
  const int r0 = blockIdx.y * RW;               // this workgroup's state rows
  const bool w0 = blockIdx.y == 0;
  const bool lead = (h % ratio) == 0 && w0;     // writes the q/k channels' conv base rows
  const int tid = threadIdx.x, hw = tid >> 5, l = tid & 31, r = r0 + hw;
  const int S = a.S, P = a.P, KM1 = a.kc - 1;
  const size_t pstride = (size_t)(2 * a.hk + a.hv) * GDN_D;
  // staged per window: q and k [W][128] as float4 units (thread -> position tid / 32 + 8 k, float4 l),
  // v of this workgroup's rows [W][RW] and the gates [W][2] (position clamped: past S loaded, not used)
  constexpr int TP = GDN_BTHREADS / 32;
  static_assert(W == 2 * TP, "two positions per half-wave (named registers: an array of them went to scratch)");
  const float* qsrc = b.vecs + (size_t)hk * GDN_D + 4 * l;
  const float* ksrc = qsrc + (size_t)a.hk * GDN_D;
  const float* vsrc = b.vecs + (size_t)(2 * a.hk + h) * GDN_D + r0 + (tid & (RW - 1));
  float4 pq0, pq1, pk0, pk1;
  float pv, pg;
  auto fetch = [&](int t0) {
    const size_t ta = (size_t)min(t0 + hw, S - 1) * pstride, tb = (size_t)min(t0 + hw + TP, S - 1) * pstride;
    pq0 = *reinterpret_cast<const float4*>(qsrc + ta);
    pk0 = *reinterpret_cast<const float4*>(ksrc + ta);
    pq1 = *reinterpret_cast<const float4*>(qsrc + tb);
    pk1 = *reinterpret_cast<const float4*>(ksrc + tb);
    pv = vsrc[(size_t)min(t0 + (tid / RW) % W, S - 1) * pstride];
    pg = b.gates[((size_t)min(t0 + (tid >> 1) % W, S - 1) * a.hv + h) * 2 + (tid & 1)];
  };
  auto store = [&](int buf) {
    *reinterpret_cast<float4*>(&qs[buf][hw][4 * l]) = pq0;
    *reinterpret_cast<float4*>(&ks[buf][hw][4 * l]) = pk0;
    *reinterpret_cast<float4*>(&qs[buf][hw + TP][4 * l]) = pq1;
    *reinterpret_cast<float4*>(&ks[buf][hw + TP][4 * l]) = pk1;
    if (tid < W * RW) vs[buf][tid / RW][tid % RW] = pv;
    if (tid < 2 * W) (tid & 1 ? bet : dec)[buf][tid >> 1] = pg;
  };
  fetch(0);
  float s[4];
  {
    const float4 s4 = *reinterpret_cast<const float4*>(a.ssm + ((size_t)h * GDN_D + r) * GDN_D + 4 * l);
    s[0] = s4.x;
    s[1] = s4.y;
    s[2] = s4.z;
    s[3] = s4.w;
  }
  // the previous window's committed steps, in order
  for (int p = 0; p < P; ++p) {
    const float gd = a.decay_cur[(size_t)p * a.hv + h];
    const uint2 kw = *reinterpret_cast<const uint2*>(a.key_cur + ((size_t)p * a.hk + hk) * GDN_D + 4 * l);
    const float kp[4] = {__uint_as_float(kw.x << 16), __uint_as_float(kw.x & 0xffff0000u),
                         __uint_as_float(kw.y << 16), __uint_as_float(kw.y & 0xffff0000u)};
    const float dl = a.delta_cur[((size_t)p * a.hv + h) * GDN_D + r];
#pragma unroll
    for (int c = 0; c < 4; ++c) {
      s[c] = s[c] * gd;
      s[c] = __builtin_fmaf(kp[c], dl, s[c]);
    }
  }
  // one position: the step kernel's operations in its order, the row's q dot before its sum over the lanes
  auto step = [&](int buf, int t) -> float {
    const float gd = dec[buf][t], bt = bet[buf][t], v = vs[buf][t][hw];
    const float4 k = *reinterpret_cast<const float4*>(&ks[buf][t][4 * l]);
    const float4 q = *reinterpret_cast<const float4*>(&qs[buf][t][4 * l]);
    s[0] = s[0] * gd;
    s[1] = s[1] * gd;
    s[2] = s[2] * gd;
    s[3] = s[3] * gd;
    float kv = 0.0f + s[0] * k.x;
    float corr = s[1] * k.y, next = kv + corr;
    float comp = (next - kv) - corr;
    kv = next;
    corr = s[2] * k.z - comp;
    next = kv + corr;
    comp = (next - kv) - corr;
    kv = next;
    corr = s[3] * k.w - comp;
    kv = kv + corr;
    const float kvm = half_wave_sum(kv);
    const float delta = (v - kvm) * bt;
    s[0] = __builtin_fmaf(k.x, delta, s[0]);
    s[1] = __builtin_fmaf(k.y, delta, s[1]);
    s[2] = __builtin_fmaf(k.z, delta, s[2]);
    s[3] = __builtin_fmaf(k.w, delta, s[3]);
    float o = __builtin_fmaf(s[0], q.x, 0.0f);
    o = __builtin_fmaf(s[1], q.y, o);
    o = __builtin_fmaf(s[2], q.z, o);
    return __builtin_fmaf(s[3], q.w, o);
  };
  // half_wave_sum of two positions' dots: the first level puts x in the lower 16 lanes, y in the upper
  auto fold2 = [](float x, float y) {
    const auto p = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
    return fold_sum<8>(__uint_as_float(p[0]) + __uint_as_float(p[1]));
  };
  const int sp = (S + 31) & ~31;  // padded positions of an output row
  float* yrow = a.ypub + ((size_t)h * GDN_D + r) * sp;
  store(0);
  __syncthreads();
  float yb = 0.0f;  // lane l of a row: position 2 (l & 15) + l / 16 of 32
  for (int t0 = 0, buf = 0; t0 < S; t0 += W, buf ^= 1) {
    const bool more = t0 + W < S;
    if (more) fetch(t0 + W);  // in flight during this window's recurrence
    const int base = (t0 & W) / 2;  // the window's pairs: 0 .. 7 or 8 .. 15
    if (t0 + W <= S) {
#pragma unroll 2
      for (int t = 0; t < W; t += 2) {
        const float o0 = step(buf, t), o1 = step(buf, t + 1);
        const float y = fold2(o0, o1);
        yb = (l & 15) == base + t / 2 ? y : yb;
      }
    } else {
      for (int t = 0; t < S - t0; t += 2) {
        const float o0 = step(buf, t);
        const float o1 = t + 1 < S - t0 ? step(buf, t + 1) : 0.0f;  // (a position past S: the row's pad)
        const float y = fold2(o0, o1);
        yb = (l & 15) == base + t / 2 ? y : yb;
      }
    }
    if (base != 0 || !more) yrow[(t0 & ~31) + 2 * (l & 15) + (l >> 4)] = yb;
    if (more) store(buf ^ 1);  // the other buffer: last read in the previous window, before its barrier
    __syncthreads();
  }
  *reinterpret_cast<float4*>(a.ssm + ((size_t)h * GDN_D + r) * GDN_D + 4 * l) = make_float4(s[0], s[1], s[2], s[3]);
  // the batch's last kc-1 input rows become the conv base
  for (int i = tid; i < (w0 ? KM1 * 3 * GDN_D : 0); i += GDN_BTHREADS) {
    const int j = i / (3 * GDN_D), kind = (i / GDN_D) % 3, d = i % GDN_D;
    if (kind < 2 && !lead) continue;
    const int vec = kind == 0 ? hk : (kind == 1 ? a.hk + hk : 2 * a.hk + h);
    const int ch = vec * GDN_D + d;
    a.conv_nxt[(size_t)j * a.cd + ch] = f2bf(gdn_row(a, P + S + j, ch));
  }
}

// The batch's gated norm: one workgroup per 32 positions of a value head.  The outputs [128 rows][32
// positions] are turned through LDS (rounded to bf16 as the step kernel publishes them), then a
// half-wave per position runs the step kernel's norm.
__global__ __launch_bounds__(256) void k_gdn_norm_batch(GdnArgs a) {
  __shared__ float ys[32][GDN_D + 4];
  __shared__ bf16 gated[32][GDN_D];
  const int t0 = blockIdx.x * 32, h = blockIdx.y, S = a.S, sp = (S + 31) & ~31;
  const int hw = threadIdx.x >> 5, l = threadIdx.x & 31, n = min(32, S - t0);
  const float* src = a.ypub + (size_t)h * GDN_D * sp + t0 + l;
  float v[GDN_D / 8];
#pragma unroll
  for (int k = 0; k < GDN_D / 8; ++k) v[k] = src[(size_t)(hw + 8 * k) * sp];
#pragma unroll
  for (int k = 0; k < GDN_D / 8; ++k) ys[l][hw + 8 * k] = round_bf(v[k]);
  __syncthreads();
  for (int t = hw; t < n; t += 8) {
    const size_t row = (size_t)(t0 + t);
    const uint32_t* zp = reinterpret_cast<const uint32_t*>(a.proj + row * a.pw + a.z_off + h * GDN_D + 4 * l);
    const uint2 zw = make_uint2(zp[0], zp[1]);  // a row starts at an even element
    const float4 y4 = *reinterpret_cast<const float4*>(&ys[t][4 * l]);
    const float y[4] = {y4.x, y4.y, y4.z, y4.w};
    float acc = 0.0f;
#pragma unroll
    for (int i = 0; i < 4; ++i) acc = __builtin_fmaf(y[i], y[i], acc);
    const float inv = 1.0f / sqrtf(half_wave_sum(acc) / 128.0f + a.eps);
    uint32_t out[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const float nv = round_bf(bf2f(a.norm_w[4 * l + i]) * round_bf(y[i] * inv));
      out[i] = f2bf(sigmoid_f32(kjournal(zw, i)) * nv);
    }
    const uint2 o2 = make_uint2(out[0] | (out[1] << 16), out[2] | (out[3] << 16));
    *reinterpret_cast<uint2*>(&gated[t][4 * l]) = o2;
    if (a.gated) *reinterpret_cast<uint2*>(a.gated + (row * a.hv + h) * GDN_D + 4 * l) = o2;
  }
  if (!a.xp) return;
  __syncthreads();
  for (int task = hw; task < 4 * n; task += 8) {
    const int t = task >> 2, blk = task & 3;
    xprep_lanes_direct(gated[t][blk * 32 + l], l, a.xp + ((size_t)(t0 + t) * a.hv * 4 + h * 4 + blk) * XP_DW);
  }
}

// Committed state without modifying it: the P journal steps replayed onto the
// state rows into ssm_dst, and the committed conv rows into conv_dst.
__global__ __launch_bounds__(GDN_THREADS) void k_gdn_replay(GdnArgs a, float* ssm_dst, bf16* conv_dst) {
  const int h = blockIdx.x, ratio = a.hv / a.hk, hk = h / ratio;
  const bool lead = (h % ratio) == 0;
  const int hw = threadIdx.x >> 5, l = threadIdx.x & 31;
  const int P = a.P, KM1 = a.kc - 1;
  for (int r = hw; r < GDN_D; r += GDN_THREADS / 32) {
    const float* srow = a.ssm + ((size_t)h * GDN_D + r) * GDN_D + 4 * l;
    const float4 s4 = *reinterpret_cast<const float4*>(srow);
    float s[4] = {s4.x, s4.y, s4.z, s4.w};
    for (int p = 0; p < P; ++p) {
      const float gd = a.decay_cur[(size_t)p * a.hv + h];
      const float dl = a.delta_cur[((size_t)p * a.hv + h) * GDN_D + r];
      const bf16* kp = a.key_cur + ((size_t)p * a.hk + hk) * GDN_D + 4 * l;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        s[i] = s[i] * gd;
        s[i] = __builtin_fmaf(bf2f(kp[i]), dl, s[i]);
      }
    }
    *reinterpret_cast<float4*>(ssm_dst + ((size_t)h * GDN_D + r) * GDN_D + 4 * l) = make_float4(s[0], s[1], s[2], s[3]);
  }
  for (int i = threadIdx.x; i < KM1 * 3 * GDN_D; i += GDN_THREADS) {
    const int j = i / (3 * GDN_D), kind = (i / GDN_D) % 3, d = i % GDN_D;
    if (kind < 2 && !lead) continue;
    const int vec = kind == 0 ? hk : (kind == 1 ? a.hk + hk : 2 * a.hk + h);
    const int ch = vec * GDN_D + d;
    conv_dst[(size_t)j * a.cd + ch] = f2bf(gdn_row(a, P + j, ch));
  }
}

template <int KC>
static hipError_t gdn_step_kc(const GdnArgs& a, hipStream_t st) {
  if (!a.tickets || !a.ypub || a.P < 0 || a.P > MAX_TOKENS) return hipErrorInvalidValue;
  const dim3 grid(a.hv, GDN_SPLIT);
  if constexpr (KC == 4) {  // the model's conv: the replay sized to the journal (1, 2, 4 or 8 steps)
    if (a.P <= 1) {
      hipLaunchKernelGGL((k_gdn_step<KC, 1>), grid, dim3(GDN_THREADS), 0, st, a);
    } else if (a.P <= 2) {
      hipLaunchKernelGGL((k_gdn_step<KC, 2>), grid, dim3(GDN_THREADS), 0, st, a);
    } else if (a.P <= 4) {
      hipLaunchKernelGGL((k_gdn_step<KC, 4>), grid, dim3(GDN_THREADS), 0, st, a);
    } else {
      hipLaunchKernelGGL((k_gdn_step<KC, MAX_TOKENS>), grid, dim3(GDN_THREADS), 0, st, a);
    }
    return hipGetLastError();
  }
  hipLaunchKernelGGL((k_gdn_step<KC, MAX_TOKENS>), grid, dim3(GDN_THREADS), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_gdn_step(const GdnArgs& a, hipStream_t st) {
  switch (a.kc) {
    case 2: return gdn_step_kc<2>(a, st);
    case 3: return gdn_step_kc<3>(a, st);
    case 4: return gdn_step_kc<4>(a, st);
    case 5: return gdn_step_kc<5>(a, st);
    case 6: return gdn_step_kc<6>(a, st);
    case 7: return gdn_step_kc<7>(a, st);
    case 8: return gdn_step_kc<8>(a, st);
    default: return hipErrorInvalidValue;
  }
}

template <int KC>
static hipError_t gdn_batch_kc(const GdnArgs& a, const GdnBatch& b, hipStream_t st) {
  if (!a.ypub || !b.vecs || !b.gates || a.S < 1) return hipErrorInvalidValue;
  hipLaunchKernelGGL(k_gdn_prep_batch<KC>, dim3(a.S), dim3(GDN_THREADS), 0, st, a, b);
  hipLaunchKernelGGL(k_gdn_batch, dim3(a.hv, GDN_BSPLIT), dim3(GDN_BTHREADS), 0, st, a, b);
  hipLaunchKernelGGL(k_gdn_norm_batch, dim3((a.S + 31) / 32, a.hv), dim3(256), 0, st, a);
  return hipGetLastError();
}

hipError_t launch_gdn_batch(const GdnArgs& a, const GdnBatch& b, hipStream_t st) {
  switch (a.kc) {
    case 2: return gdn_batch_kc<2>(a, b, st);
    case 3: return gdn_batch_kc<3>(a, b, st);
    case 4: return gdn_batch_kc<4>(a, b, st);
    case 5: return gdn_batch_kc<5>(a, b, st);
    case 6: return gdn_batch_kc<6>(a, b, st);
    case 7: return gdn_batch_kc<7>(a, b, st);
    case 8: return gdn_batch_kc<8>(a, b, st);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_gdn_replay(const GdnArgs& a, float* ssm_dst, bf16* conv_dst, hipStream_t st) {
  hipLaunchKernelGGL(k_gdn_replay, dim3(a.hv), dim3(GDN_THREADS), 0, st, a, ssm_dst, conv_dst);
  return hipGetLastError();
}

}  // namespace mtpx
