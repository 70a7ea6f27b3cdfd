// The operations around the cell of a float32 sLSTM layer, forward and backward: causal depthwise convolution + SiLU, the
// four block-diagonal gate projections, and the gradients of both; the per-head group norm (forward).  Everything is held and
// summed in float32 (the products on v_mfma_f32_16x16x4_f32).  Included by slstm_hip.hip only (one translation unit),
// after slstm_device_common.h.
#pragma once

namespace {

struct LayerConvParams {
  const float *x;
  long long x_sb, x_st;
  const float *state;  // [B, KS-1, D] or null; rows state_sb elements apart (forward)
  long long state_sb;
  const float *w;      // [D, KS]
  const float *bias;   // [D] or null
  const unsigned char *reset;
  long long reset_sb;
  float *out;          // [B, T, D]: the forward's result
  const float *d_out;  // [B, T, D]: gradient of that result (backward)
  float *d_x;          // [B, T, D]: on entry the gradient that reaches x past the convolution (backward); null: not wanted
  float *partial;      // [workgroups over tokens][D][KS+1]: sums over a workgroup's tokens (backward); null: not wanted
  int B, T, D;
};

__device__ __forceinline__ f32x4 load4(const float *p) { return *reinterpret_cast<const f32x4 *>(p); }
__device__ __forceinline__ f32x4 zero4() { return f32x4{0.0f, 0.0f, 0.0f, 0.0f}; }

// The weights of 4 channels, tap by tap (KS consecutive floats a channel in memory)
template <int KS>
__device__ __forceinline__ void load_taps(const float *w, f32x4 (&taps)[KS]) {
  float v[4 * KS];
#pragma unroll
  for (int i = 0; i < KS; ++i) {
    const f32x4 q = load4(w + 4 * i);
#pragma unroll
    for (int e = 0; e < 4; ++e) v[4 * i + e] = q[e];
  }
#pragma unroll
  for (int j = 0; j < KS; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) taps[j][e] = v[e * KS + j];
}

// Bit i of the result: a document starts at token t_first + i (i < n; tokens outside the row: none)
template <int N>
__device__ __forceinline__ uint32_t starts_of(const unsigned char *row, int t_first, int T) {
  uint32_t bits = 0;
#pragma unroll
  for (int i = 0; i < N; ++i) {
    const int t = t_first + i;
    if (t >= 0 && t < T && row[t] != 0) bits |= 1u << i;
  }
  return bits;
}

// silu(bias + sum over the taps); a tap in front of the token's document reads nothing.  One thread: 4 channels of kConvRun
// tokens, so that a token is read once and not KS times; every load of a thread is asked for at once.
constexpr int kConvRun = 4;
template <int KS>
__global__ __launch_bounds__(256) void layer_conv_f32_kernel(LayerConvParams p) {
  constexpr int R = kConvRun, W = R + KS - 1;
  const int pieces = p.D >> 2, runs = (p.T + R - 1) / R;
  const long long idx = (long long)blockIdx.x * 256 + threadIdx.x;
  if (idx >= (long long)p.B * runs * pieces) return;
  const int c0 = (int)(idx % pieces) * 4;
  const long long br = idx / pieces;
  const int t0 = (int)(br % runs) * R, b = (int)(br / runs);

  f32x4 x[W];  // x[i]: token t0 - (KS - 1) + i
#pragma unroll
  for (int i = 0; i < W; ++i) {
    const int t = t0 - (KS - 1) + i;
    x[i] = zero4();
    if (t >= 0) {
      if (t < p.T) x[i] = load4(p.x + b * p.x_sb + t * p.x_st + c0);
    } else if (p.state) {
      x[i] = load4(p.state + b * p.state_sb + (long long)(KS - 1 + t) * p.D + c0);
    }
  }
  f32x4 taps[KS];
  load_taps<KS>(p.w + (long long)c0 * KS, taps);
  const f32x4 bias = p.bias ? load4(p.bias + c0) : zero4();
  const uint32_t starts = p.reset ? starts_of<W>(p.reset + b * p.reset_sb, t0 - (KS - 1), p.T) : 0u;
#pragma unroll
  for (int r = 0; r < R; ++r) {
    if (t0 + r >= p.T) break;
    f32x4 a = bias;
    bool alive = true;
#pragma unroll
    for (int back = 0; back < KS; ++back) {
      const int i = r + KS - 1 - back;
      if (back > 0) alive = alive && !((starts >> (i + 1)) & 1u);
      if (alive) a += taps[KS - 1 - back] * x[i];
    }
    f32x4 o;
#pragma unroll
    for (int e = 0; e < 4; ++e) o[e] = a[e] / (1.0f + expf(-a[e]));
    *reinterpret_cast<f32x4 *>(p.out + ((long long)b * p.T + t0 + r) * p.D + c0) = o;
  }
}

// Its gradients.  A thread owns 4 channels of kConvBackRun tokens: it makes their pre-activations again (four multiply-adds,
// against a tensor more to keep) and those of the KS - 1 tokens behind, whose gradient reaches its tokens, and adds what
// reaches x through the convolution to what is in d_x already.  A workgroup (32 channel pieces x 8 runs) adds up its
// tokens' share of the gradients of the weights and the bias and leaves it for layer_reduce_kernel.
constexpr int kConvBackRun = 8;
template <int KS>
__global__ __launch_bounds__(256) void layer_conv_backward_f32_kernel(LayerConvParams p, int piece_blocks) {
  constexpr int R = kConvBackRun, H = KS - 1, N = R + H;  // N: tokens whose pre-activation is made
  constexpr int G = KS + 1;
  __shared__ float sums[8][32 * 4 * G];
  const int pieces = p.D >> 2, runs = (p.T + R - 1) / R;
  const int pb = blockIdx.x % piece_blocks, rb = blockIdx.x / piece_blocks;
  const int lp = threadIdx.x & 31, lr = threadIdx.x >> 5;
  const int piece = pb * 32 + lp;
  const long long br = (long long)rb * 8 + lr;
  const bool active = piece < pieces && br < (long long)p.B * runs;
  f32x4 dw[G];  // gradients of the taps, then of the bias
#pragma unroll
  for (int j = 0; j < G; ++j) dw[j] = zero4();
  if (active) {
    const int c0 = piece * 4, t0 = (int)(br % runs) * R, b = (int)(br / runs);
    const float *xrow = p.x + b * p.x_sb + c0;
    const float *drow = p.d_out + (long long)b * p.T * p.D + c0;
    float *dxrow = p.d_x + (long long)b * p.T * p.D + c0;
    f32x4 x[N + H];  // x[i]: token t0 - H + i
#pragma unroll
    for (int i = 0; i < N + H; ++i) {
      const int t = t0 - H + i;
      x[i] = t >= 0 && t < p.T ? load4(xrow + t * p.x_st) : zero4();
    }
    f32x4 d[N];  // of token t0 + i
#pragma unroll
    for (int i = 0; i < N; ++i) d[i] = t0 + i < p.T ? load4(drow + (long long)(t0 + i) * p.D) : zero4();
    f32x4 dx[R];
#pragma unroll
    for (int i = 0; i < R; ++i) dx[i] = p.d_x && t0 + i < p.T ? load4(dxrow + (long long)(t0 + i) * p.D) : zero4();
    f32x4 taps[KS];
    load_taps<KS>(p.w + (long long)c0 * KS, taps);
    const f32x4 bias = p.bias ? load4(p.bias + c0) : zero4();
    const uint32_t starts = p.reset ? starts_of<N + H>(p.reset + b * p.reset_sb, t0 - H, p.T) : 0u;
#pragma unroll
    for (int i = 0; i < N; ++i) {
      f32x4 a = bias;
      bool alive[KS];
      alive[0] = true;
#pragma unroll
      for (int back = 0; back < KS; ++back) {
        if (back > 0) alive[back] = alive[back - 1] && !((starts >> (i + H - back + 1)) & 1u);
        if (alive[back]) a += taps[KS - 1 - back] * x[i + H - back];
      }
      f32x4 g;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const float s = 1.0f / (1.0f + expf(-a[e]));
        g[e] = d[i][e] * (s * (1.0f + a[e] * (1.0f - s)));
      }
      if (t0 + i >= p.T) continue;  // (its gradient is no tensor's)
#pragma unroll
      for (int back = 0; back < KS; ++back) {
        if (!alive[back]) continue;
        if (i < R) dw[KS - 1 - back] += g * x[i + H - back];
        if (i - back >= 0 && i - back < R) dx[i - back] += taps[KS - 1 - back] * g;
      }
      if (i < R) dw[KS] += g;
    }
#pragma unroll
    for (int i = 0; i < R; ++i)
      if (p.d_x && t0 + i < p.T) *reinterpret_cast<f32x4 *>(dxrow + (long long)(t0 + i) * p.D) = dx[i];
  }
  if (!p.partial) return;
#pragma unroll
  for (int j = 0; j < G; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) sums[lr][(lp * 4 + e) * G + j] = dw[j][e];
  __syncthreads();
  float *out = p.partial + ((long long)rb * p.D + pb * 128) * G;
  const int n = (p.D - pb * 128 < 128 ? p.D - pb * 128 : 128) * G;
  for (int i = threadIdx.x; i < n; i += 256) {
    float s = sums[0][i];
#pragma unroll
    for (int r = 1; r < 8; ++r) s += sums[r][i];
    out[i] = s;
  }
}

// ---------------------------------------------------------------------------
// The projections as products in float32, H = NH*dh, M = B*T tokens, slots g = i, f, z, o with operand A_g = x_conv (i, f)
// or x (z, o):
//   PROJECT   out[m, g*H + h*dh + o]    = sum_d  A_g[m, h*dh + d] * w_g[h, o, d]
//   INPUTS    d_A[m, h*dh + d]          = sum over the two slots of A and o of  d_out[m, g*H + h*dh + o] * w_g[h, o, d]
//   WEIGHTS   d_w_g[h, o, d]            = sum_m  d_out[m, g*H + h*dh + o] * A_g[m, h*dh + d]
// A workgroup makes 64 x 64 outputs in slabs of 32 of the summed index, through two LDS buffers (the next slab's loads are
// asked for in front of the products of this one), four waves of 32 x 32.  An operand lies in LDS as it lies in memory:
// with the summed index running along a row (rows of 36 floats: a lane's four values are one 16-byte read without bank
// conflicts), or with it counting rows (rows of 68 floats: 4-byte reads, the four lane groups on banks 16 apart).
// v_mfma_f32_16x16x4_f32 takes 32 cycles, so that the LDS reads are hidden either way; what bounds the kernel is the
// matrix cores (157 TFLOP/s at their peak in float32), short of it the fill and drain of a tile's few slabs: 6732 tokens x
// 8 heads of 256 take 329, 271 and 303 us (86, 104 and 93 TFLOP/s; the library's products, which need a copy of their
// operand per slot, 348, 280 and 399), 4096 x 4 of 128 31, 26 and 29 us (53, 41 and 103).  128 x 64 outputs a workgroup
// are 3 to 8 % slower.  The sums over m are cut into `slices`, each with its own partial result, where the outputs alone
// would leave compute units idle; layer_reduce_kernel adds them up in a fixed order.
// ---------------------------------------------------------------------------
enum class LayerProduct { PROJECT, INPUTS, WEIGHTS };
struct LayerProductParams {
  const float *a[2];       // x_conv, x
  long long a_sb[2], a_st[2];  // strides of a row and of a token
  const float *w[4];
  const float *d_wx;       // [M, 4H]
  float *wx;               // [M, 4H] (PROJECT)
  float *d_a[2];           // [M, H] (INPUTS)
  float *d_w[4];           // [NH, dh, dh] (WEIGHTS; written here with one slice), null: not wanted
  float *partial;          // [slices][4][NH][dh][dh] (WEIGHTS, several)
  int M, T, NH, dh, slices, slice_tokens;
  int m_tiles, tiles, pairs, pairs_per_xcd;
};

constexpr int kProductK = 32, kAlongPitch = 36, kAcrossPitch = 68;

template <LayerProduct MODE>
__global__ __launch_bounds__(256) void layer_product_f32_kernel(LayerProductParams p) {
  constexpr bool kRowsAcross = MODE == LayerProduct::WEIGHTS;   // the operand of the output's rows: summed index counts rows
  constexpr bool kColsAcross = MODE != LayerProduct::PROJECT;   // the operand of the output's columns likewise
  __shared__ __attribute__((aligned(16))) float rows_lds[2][kRowsAcross ? kProductK * kAcrossPitch : 64 * kAlongPitch];
  __shared__ __attribute__((aligned(16))) float cols_lds[2][kColsAcross ? kProductK * kAcrossPitch : 64 * kAlongPitch];

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int q = lane >> 4, r16 = lane & 15;
  const int wm = (wave >> 1) * 32, wn = (wave & 1) * 32;
  const int dh = p.dh, up = (dh + 63) >> 6;  // tiles of 64 over a head's units
  const long long H = (long long)p.NH * dh;

  // Which tile.  Tiles that share operands - of one (head, block of tokens), WEIGHTS: (slice, head) - are neighbours on one
  // XCD (workgroup i runs on XCD i % 8), and an XCD has a contiguous range of those pairs: the weights of a head are read
  // into its L2 once, a block of tokens too.
  int m0, n0, slot, head, slice = 0;
  {
    const int pair = (blockIdx.x & 7) * p.pairs_per_xcd + (blockIdx.x >> 3) / p.tiles;
    if (pair >= p.pairs) return;  // (the whole workgroup, in front of any barrier)
    int tile = (blockIdx.x >> 3) % p.tiles;
    n0 = (tile % up) * 64; tile /= up;
    if constexpr (MODE == LayerProduct::WEIGHTS) {
      m0 = (tile % up) * 64; tile /= up;
      slice = pair / p.NH;
      head = pair % p.NH;
    } else {
      head = pair / p.m_tiles;
      m0 = pair % p.m_tiles * 64;
    }
    slot = tile;  // INPUTS: the operand instead (0: x_conv, slots i and f; 1: x, slots z and o)
  }
  if constexpr (MODE == LayerProduct::WEIGHTS) {
    if (!p.d_w[slot]) return;
  }
  const int which = MODE == LayerProduct::INPUTS ? slot : slot >> 1;
  const int k_first = MODE == LayerProduct::WEIGHTS ? slice * p.slice_tokens : 0;
  const int k_end = MODE == LayerProduct::WEIGHTS ? (k_first + p.slice_tokens < p.M ? k_first + p.slice_tokens : p.M) : dh;
  const int per_slot = (k_end - k_first + kProductK - 1) / kProductK;
  const int slabs = MODE == LayerProduct::INPUTS ? 2 * per_slot : per_slot;

  auto token = [&](int m) { return p.a[which] + (m / p.T) * p.a_sb[which] + (m % p.T) * p.a_st[which] + (long long)head * dh; };
  // a thread stages 2 pieces of 4 floats of each operand.  Summed index along a row: row tid/8 + 32 i, piece tid%8;
  // counting rows: row tid/16 + 16 i, piece tid%16
  f32x4 rr[2], cr[2];
  const float *fixed[2];  // PROJECT: this thread's tokens; INPUTS: its rows of d_out
  if constexpr (!kRowsAcross) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int m = m0 + (tid >> 3) + 32 * i;
      fixed[i] = m >= p.M ? nullptr : (MODE == LayerProduct::PROJECT ? token(m) : p.d_wx + m * 4 * H + 2 * which * H + (long long)head * dh);
    }
  }
  auto load = [&](int s) {
    const int ss = MODE == LayerProduct::INPUTS && s >= per_slot ? 1 : 0;  // which of the two slots
    const int k0 = k_first + (s - ss * per_slot) * kProductK;
    const int along_k = k0 + (tid & 7) * 4, across_c = (tid & 15) * 4;
    if constexpr (!kRowsAcross) {
#pragma unroll
      for (int i = 0; i < 2; ++i) rr[i] = fixed[i] && along_k < dh ? load4(fixed[i] + ss * H + along_k) : zero4();
    }
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int across_k = k0 + (tid >> 4) + 16 * i;
      cr[i] = zero4();
      if constexpr (kRowsAcross) {
        rr[i] = zero4();
        if (across_k < k_end) {
          if (m0 + across_c < dh) rr[i] = load4(p.d_wx + across_k * 4 * H + slot * H + (long long)head * dh + m0 + across_c);
          if (n0 + across_c < dh) cr[i] = load4(token(across_k) + n0 + across_c);
        }
      } else {
        if constexpr (kColsAcross) {
          if (across_k < dh && n0 + across_c < dh) cr[i] = load4(p.w[2 * which + ss] + ((long long)head * dh + across_k) * dh + n0 + across_c);
        } else {
          const int n = n0 + (tid >> 3) + 32 * i;
          if (n < dh && along_k < dh) cr[i] = load4(p.w[slot] + ((long long)head * dh + n) * dh + along_k);
        }
      }
    }
  };
  auto store = [&](int buf) {
    auto at = [&](bool across, int i) {
      return across ? ((tid >> 4) + 16 * i) * kAcrossPitch + (tid & 15) * 4 : ((tid >> 3) + 32 * i) * kAlongPitch + (tid & 7) * 4;
    };
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4 *>(&rows_lds[buf][at(kRowsAcross, i)]) = rr[i];
#pragma unroll
    for (int i = 0; i < 2; ++i) *reinterpret_cast<f32x4 *>(&cols_lds[buf][at(kColsAcross, i)]) = cr[i];
  };

  f32x4 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = zero4();
  load(0);
  store(0);
  __syncthreads();
  for (int s = 0; s < slabs; ++s) {
    if (s + 1 < slabs) load(s + 1);
    const float *rb = rows_lds[s & 1], *cb = cols_lds[s & 1];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks) {
      // lane (r16, q) brings 4 consecutive values of the summed index, one to each of four products: value 4 q + e to product e
      f32x4 rv[2], cv[2];
      const int k = 16 * ks + 4 * q;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int r = wm + 16 * i + r16;
        if constexpr (kRowsAcross) {
#pragma unroll
          for (int e = 0; e < 4; ++e) rv[i][e] = rb[(k + e) * kAcrossPitch + r];
        } else {
          rv[i] = load4(rb + r * kAlongPitch + k);
        }
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int c = wn + 16 * i + r16;
        if constexpr (kColsAcross) {
#pragma unroll
          for (int e = 0; e < 4; ++e) cv[i][e] = cb[(k + e) * kAcrossPitch + c];
        } else {
          cv[i] = load4(cb + c * kAlongPitch + k);
        }
      }
      // (the output's columns on the M side, so that a lane ends with 4 consecutive columns of one row)
#pragma unroll
      for (int e = 0; e < 4; ++e)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x4f32(cv[j][e], rv[i][e], acc[i][j], 0, 0, 0);
    }
    if (s + 1 < slabs) store((s + 1) & 1);
    __syncthreads();
  }

  // lane (r16, q): row wm + 16 i + r16, columns wn + 16 j + 4 q .. +3
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int m = m0 + wm + 16 * i + r16;
    float *row;
    if constexpr (MODE == LayerProduct::PROJECT) row = m < p.M ? p.wx + m * 4 * H + slot * H + (long long)head * dh : nullptr;
    else if constexpr (MODE == LayerProduct::INPUTS) row = m < p.M ? p.d_a[which] + m * H + (long long)head * dh : nullptr;
    else row = m >= dh ? nullptr : (p.slices > 1 ? p.partial + (((long long)slice * 4 + slot) * p.NH + head) * dh * dh : p.d_w[slot] + (long long)head * dh * dh) + (long long)m * dh;
    if (!row) continue;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const int n = n0 + wn + 16 * j + 4 * q;
      if (n < dh) *reinterpret_cast<f32x4 *>(row + n) = acc[i][j];
    }
  }
}

// ---------------------------------------------------------------------------
// the per-head group norm: (y - mean) / sqrt(var + eps) * (1 + w) over the units of a head.  L lanes hold a group, 4 units a
// lane and piece; one read and one write of the tensor bound it (4096 tokens x 4 heads of 128: 5.4 us, the library's
// copies, moments and products 50).
// ---------------------------------------------------------------------------
struct LayerNormParams {
  const float *y;       // [T, B, H]
  const float *weight;  // [H] or null
  float *out;           // [B, T, H]
  float eps;
  int B, T, NH, dh;
};

template <int L, int P>
__global__ __launch_bounds__(256) void layer_norm_f32_kernel(LayerNormParams p) {
  auto total = [](float s) {
#pragma unroll
    for (int o = L / 2; o > 0; o >>= 1) s += __shfl_xor(s, o, 64);
    return s;
  };
  const int lane = threadIdx.x % L;
  const long long i = (long long)blockIdx.x * (256 / L) + threadIdx.x / L;  // (b, t, head)
  const bool active = i < (long long)p.B * p.T * p.NH;
  const long long at = active ? i : 0;
  const int head = (int)(at % p.NH), t = (int)(at / p.NH % p.T), b = (int)(at / p.NH / p.T);
  const long long H = (long long)p.NH * p.dh;
  const float *src = p.y + ((long long)t * p.B + b) * H + head * p.dh;
  f32x4 v[P];
  float s = 0.0f;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int u = (lane + L * j) * 4;
    v[j] = u < p.dh ? load4(src + u) : zero4();
    s += (v[j][0] + v[j][1]) + (v[j][2] + v[j][3]);
  }
  const float mean = total(s) / (float)p.dh;
  s = 0.0f;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    if ((lane + L * j) * 4 < p.dh) {
      v[j] -= mean;
      s += (v[j][0] * v[j][0] + v[j][1] * v[j][1]) + (v[j][2] * v[j][2] + v[j][3] * v[j][3]);
    }
  }
  const float rstd = 1.0f / sqrtf(total(s) / (float)p.dh + p.eps);
  if (!active) return;
  float *dst = p.out + ((long long)b * p.T + t) * H + head * p.dh;
#pragma unroll
  for (int j = 0; j < P; ++j) {
    const int u = (lane + L * j) * 4;
    if (u >= p.dh) continue;
    f32x4 scale = {1.0f, 1.0f, 1.0f, 1.0f};
    if (p.weight) scale += load4(p.weight + head * p.dh + u);
    *reinterpret_cast<f32x4 *>(dst + u) = v[j] * rstd * scale;
  }
}

// The partial sums of the kernels above, added up in a fixed order: a workgroup takes 64 results, four waves a quarter of the
// parts each.  Two regions in one launch (a launch costs more than either of them).
struct LayerReduceParams {
  struct Region { const float *partial; long long n; int parts, blocks; } region[2];  // gate weights, convolution
  float *d_w[4], *d_conv_w, *d_conv_b;  // null: not wanted
  long long per_gate;
  int taps;
};
__global__ __launch_bounds__(256) void layer_reduce_kernel(LayerReduceParams p) {
  __shared__ float sums[3][64];
  const int which = (int)blockIdx.x >= p.region[0].blocks ? 1 : 0, block = blockIdx.x - (which ? p.region[0].blocks : 0);
  const LayerReduceParams::Region r = p.region[which];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long long i = (long long)block * 64 + lane;
  const int per_wave = (r.parts + 3) / 4, first = wave * per_wave, end = first + per_wave < r.parts ? first + per_wave : r.parts;
  float s = 0.0f;
  if (i < r.n) {
#pragma unroll 8
    for (int k = first; k < end; ++k) s += r.partial[k * r.n + i];
  }
  if (wave) sums[wave - 1][lane] = s;
  __syncthreads();
  if (wave || i >= r.n) return;
  s = (s + sums[0][lane]) + (sums[1][lane] + sums[2][lane]);
  if (which == 0) {
    if (float *d_w = p.d_w[i / p.per_gate]) d_w[i % p.per_gate] = s;
  } else {
    const long long c = i / (p.taps + 1);
    const int j = (int)(i % (p.taps + 1));
    if (j < p.taps) {
      if (p.d_conv_w) p.d_conv_w[c * p.taps + j] = s;
    } else if (p.d_conv_b) {
      p.d_conv_b[c] = s;
    }
  }
}

}  // namespace
