// Small heads: a whole head in ONE compute unit.  Included by slstm_hip.hip only, behind slstm_backward_kernels.h.
//
// Up to head dim 128 (bf16; 64 in float32) the recurrent matrix of a head is small enough for one compute unit (bf16: 128 KiB of 512 of registers), and
// then nothing has to cross between compute units: the exchange of h that takes two thirds of a step of
// slstm_seq_kernel (0.5 us of 0.75) becomes a pass through LDS, and so does the exchange of the gate deltas in the
// reverse pass.  A workgroup owns four batch rows of one head; wave w owns the 16 units 16 w .. 16 w + 15 with all four
// gates, a lane one element (batch row b, unit 16 w + n).  Workgroups do not wait for each other, so any number of them
// may be launched, nothing can give up, and what does not fit the device at once simply follows.
//
//   slstm_local_kernel       forward, one launch for all T steps: h_{t-1} out of LDS as the MFMA operand, one product per gate (the
//                            wave's 16 units are the columns, so a lane ends with the four gates of its own element
//                            and no shuffles), gating, h_t into the other of two LDS buffers, one barrier.
//                            bf16: v_mfma_f32_16x16x32, batch row b at MFMA row 4 b.  float32: v_mfma_f32_4x4x1 with
//                            its 16 blocks as 4 groups of columns x 4 quarters of K - a tile of four rows without
//                            padding, a quarter of the cycles of v_mfma_f32_16x16x4 - whose four quarter sums come
//                            together in a 4 x 4 transpose across the lane groups (v_permlane32_swap, v_permlane16_swap).
//                            K is accumulated in the quarters of every other kernel and folded in their order: the same bits.
//   slstm_local_bwd_kernel   the reverse pass: a wave multiplies ITS gate deltas (16 units x 4 gates = 64 of K) by
//                            their rows of R, which gives partial sums for all units of the head; the partial sums of
//                            the waves go through LDS to the lanes that own them (two buffers, one barrier per step).
//
// What bounds a step is a chain again - LDS read, MFMAs, gating (some 300 cycles), LDS write, barrier - of 0.28 us at head dim
// 16 to 0.60 at 128.  Measured, us per step at T 512, 4 heads, B 16 (slstm_seq_kernel and slstm_bwd_split / quad_kernel before
// it): forward bf16 head dim 64 0.38 (0.73), 128 0.60 (0.75), float32 head dim 64 0.59 (1.20); reverse pass bf16 head dim
// 64 0.72 (0.90, and 0.25 for the forward walk in front of it).  float32 beyond 64 is bound by the matrix instructions of one
// compute unit (1,024 cycles per wave and step at head dim 128: 1.57 forward, 1.70 reverse at 96, against 0.79 and 1.00 over
// several).  Large batches are bound by the coefficients' 36 bytes per element.
//
// W.x (the coefficients, d_h) is fetched by the lanes that use it, kLocalAhead (kLocalBwdAhead) steps ahead into a ring
// of registers; without polls there is nothing that these misses could hold up.
#pragma once

namespace {

constexpr int kLocalAhead = 8;     // steps of W.x in flight (5 loads, 1 to 4 stores a step: a wave counts 63 at most)
constexpr int kLocalBwdAhead = 6;  // steps of coefficients and d_h in flight (5 loads, 4 stores a step)
constexpr int kLocalMaxHeadDim = 128;

struct LocalParams {
  const void *wx;
  long long wx_sb, wx_st;
  const void *r;
  int r_bf16;
  const float *bias;
  const float *s0;
  const unsigned char *reset;
  long long reset_sb;
  void *h_out;
  float *s_out;
  xs_slstm_status *status;   // or null
  float *coef;               // COEF: [T][ceil(B/4)][NH][waves][{64 lanes x 4}, {64 x 4}, {64 x 1}]: coefficients 0-3, 4-7, 8
  int B, T, NH, dh;
  int heads;                 // of this launch: the last ones, whose first one every pointer but coef and status names
};

struct LocalBwdParams {
  const float *coef;
  const void *d_h;           // element (t, b, h*dh + a) at t d_h_st + b d_h_sb + ..., in the type of the operands
  long long d_h_sb, d_h_st;
  const float *d_s_final;    // [4,B,H] or null
  const void *r;             // [NH,4 dh,dh], the forward's layout
  int r_bf16;
  const unsigned char *reset;
  long long reset_sb;
  void *d_wx;
  long long d_wx_sb, d_wx_st;
  float *d_s0;
  int cut;
  float clip;
  int B, T, NH, dh;
};

// workgroup i runs on XCD i % 8: a contiguous range of (row tile, head) pairs, heads fastest, on each XCD, so that heads
// that share a line of W.x (64 units of bf16) find it in one L2
__device__ __forceinline__ bool local_place(int n, int NH, int &head, int &tile) {
  const int per = (int)gridDim.x >> 3, idx = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  head = idx % NH; tile = idx / NH;
  return idx < n;
}

template <bool BF16, int W, bool COEF>
__global__ __launch_bounds__(64 * W) void slstm_local_kernel(LocalParams p) {
  typedef typename std::conditional<BF16, uint16_t, float>::type elem_t;
  static_assert(BF16 || W <= 4, "float32: head dims up to 64");
  constexpr int KS = BF16 ? (W + 1) / 2 : 1;            // bf16: MFMA k-steps of 32
  constexpr int KW = 16 * KS;                           // (float32) inputs per quarter of K
  // elements between the rows of the h tile in LDS: bf16 16 bytes of padding; float32 16 words beyond a multiple of 64
  // (the 16 lanes of a quarter of K read 4 rows x 16 words: all banks once)
  constexpr int HS = BF16 ? KS * 32 + 8 : 4 * KW + (4 * KW % 64 == 0 ? 16 : 80 - 4 * KW % 64);
  constexpr int PD = kLocalAhead;
  __shared__ __attribute__((aligned(16))) elem_t htile[2][4 * HS];

  int head, tile;
  const int ntiles = (p.B + 3) >> 2;
  if (!local_place(ntiles * p.heads, p.heads, head, tile)) return;  // the whole workgroup leaves before any barrier
  const int tid = threadIdx.x, lane = tid & 63, wave = (int)uniform((uint32_t)(tid >> 6));
  const int b = lane >> 4, n = lane & 15;
  const int dh = p.dh, H = p.NH * dh;
  const long long BH = (long long)p.B * H;
  const int a = 16 * wave + n, brow = 4 * tile + b;
  const bool mine = a < dh && brow < p.B;
  const int ac = a < dh ? a : dh - 1, bc = brow < p.B ? brow : p.B - 1;
  const long long so = (long long)bc * H + head * dh + ac;
  if (p.status && blockIdx.x == 0 && tid < 16) {
    uint32_t *const word = reinterpret_cast<uint32_t *>(p.status) + tid;
    if (p.heads == p.NH) *word = tid == 5 ? 1u : (tid == 7 ? 4u : 0u);
    else if (tid == 5) *word += 1u;  // (behind the launches of the heads in front: what they said stays)
    else if (tid == 7) *word = 4u;
  }

  // ---- R: bf16: column n of gate g is unit 16 w + n, k-step ks, lane group q = b: inputs 32 ks + 8 q .. + 7
  //      float32: lane (quarter kq = b, column n): inputs kq KW .. + KW - 1 of its unit's row
  uint4 rb[4][BF16 ? KS : 1];
  float rf[4][BF16 ? 1 : KW];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const long long row = ((long long)head * 4 * dh + (long long)g * dh + ac) * dh;
    if constexpr (BF16) {
#pragma unroll
      for (int ks = 0; ks < KS; ++ks) {
        const int k = 32 * ks + 8 * b;
        rb[g][ks] = make_uint4(0, 0, 0, 0);
        if (a < dh && k < dh) {
          if (p.r_bf16) {
            rb[g][ks] = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(p.r) + row + k);
          } else {
            const float4 lo = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p.r) + row + k);
            const float4 hi = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p.r) + row + k + 4);
            rb[g][ks] = uint4{pack_bf16x2(lo.x, lo.y), pack_bf16x2(lo.z, lo.w), pack_bf16x2(hi.x, hi.y), pack_bf16x2(hi.z, hi.w)};
          }
        }
      }
    } else {
#pragma unroll
      for (int k4 = 0; k4 < KW / 4; ++k4) {
        const int k = b * KW + 4 * k4;
        float4 v = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
        if (a < dh && k < dh) v = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p.r) + row + k);
        rf[g][4 * k4] = v.x; rf[g][4 * k4 + 1] = v.y; rf[g][4 * k4 + 2] = v.z; rf[g][4 * k4 + 3] = v.w;
      }
    }
  }
  float bias_g[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) bias_g[g] = p.bias[((long long)head * 4 + g) * dh + ac];
  CellState st{0.0f, 0.0f, 0.0f, 0.0f};
  if (p.s0) { st.y = p.s0[so]; st.c = p.s0[BH + so]; st.n = p.s0[2 * BH + so]; st.m = p.s0[3 * BH + so]; }

  // ---- the h tile in front of step 0 (buffer 1): the y of the initial state; units past the head dim stay zero for good
  for (int i = tid; i < 2 * 4 * HS; i += 64 * W) reinterpret_cast<elem_t *>(htile)[i] = 0;
  __syncthreads();
  elem_t *const hw[2] = {&htile[0][b * HS + a], &htile[1][b * HS + a]};
  if (a < dh) {
    if constexpr (BF16) *hw[1] = (uint16_t)float_to_bf16_bits(st.y);
    else *hw[1] = st.y;
  }

  // ---- W.x and the reset flags, PD steps ahead
  const char *wxp = reinterpret_cast<const char *>(p.wx) + ((long long)bc * p.wx_sb + head * dh + ac) * (long long)sizeof(elem_t);
  const long long wx_step = p.wx_st * (long long)sizeof(elem_t), wx_gate = (long long)H * sizeof(elem_t);
  const unsigned char *flp = p.reset ? p.reset + (long long)bc * p.reset_sb : nullptr;
  const int Tl = p.T - 1;
  elem_t ring[PD][4];
  unsigned char flag[PD];
  auto fetch = [&](int u, int t) {
    const char *src = wxp + (long long)(t < Tl ? t : Tl) * wx_step;
#pragma unroll
    for (int g = 0; g < 4; ++g) ring[u][g] = *reinterpret_cast<const elem_t *>(src + g * wx_gate);
    flag[u] = flp ? flp[t < Tl ? t : Tl] : (unsigned char)0;
  };
#pragma unroll
  for (int u = 0; u < PD; ++u) fetch(u, u);

  // COEF: what the coefficients of a step are made of, kept until the operands of the next one are on their way
  GateValues kept{0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
  float kept_y = 0.0f, kept_c = 0.0f, kept_n = 0.0f, kept_f = 0.0f;
  float *cfp = nullptr;
  long long coef_step = 0;
  if constexpr (COEF) {
    coef_step = (long long)ntiles * p.NH * W * 576;
    cfp = p.coef + (((long long)tile * p.NH + head) * W + wave) * 576;
  }
  elem_t *hop = reinterpret_cast<elem_t *>(p.h_out) + so;
  elem_t h_bits = 0;
  auto leave = [&](int t) {  // step t's output and coefficients to memory
    if (mine) __builtin_nontemporal_store(h_bits, hop + (long long)t * BH);
    if constexpr (COEF) {
      const float omf = __builtin_amdgcn_rcpf(1.0f + __expf(kept_f));  // 1 - sigmoid(f)
      store_coefficients(cfp + t * coef_step, lane, kept, kept_y, kept_c, kept_n, omf);
    }
  };

  // operand addresses: bf16: MFMA row n is batch row n / 4, lane group q = b: inputs 8 q ..; float32: lane (kq = b, c = n / 4,
  // row n % 4): inputs kq KW + 4 c .. + 3 of chunk 0
  const int ho = BF16 ? (n >> 2) * HS + 8 * b : (n & 3) * HS + b * KW + 4 * (n >> 2);
  for (int t0 = 0; t0 < p.T; t0 += PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      const int t = t0 + u;
      if (t >= p.T) break;
      lds_barrier();  // h_{t-1} is in LDS; everybody has read h_{t-2}
      const elem_t *hsrc = htile[(t + 1) & 1] + ho;
      float raw[4];
      float wxv[4];
      const bool start = flag[u] != 0;
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        if constexpr (BF16) wxv[g] = bf16_bits_to_float(ring[u][g]);
        else wxv[g] = ring[u][g];
      }
      float ry[4];
      if constexpr (BF16) {
        uint4 areg[KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks) areg[ks] = *reinterpret_cast<const uint4 *>(hsrc + 32 * ks);
        if (t > 0) leave(t - 1);
        fetch(u, t + PD);
        f32x4 acc[4][KS];
#pragma unroll
        for (int ks = 0; ks < KS; ++ks)
#pragma unroll
          for (int g = 0; g < 4; ++g)
            acc[g][ks] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, areg[ks]), __builtin_bit_cast(bf16x8, rb[g][ks]),
                                                                 f32x4{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0);
#pragma unroll
        for (int g = 0; g < 4; ++g) {  // (a quarter of K is one k-step here: the quarters in order)
          ry[g] = acc[g][0][0];
#pragma unroll
          for (int ks = 1; ks < KS; ++ks) ry[g] += acc[g][ks][0];
        }
      } else {
        f32x4 hv[KS];
#pragma unroll
        for (int c = 0; c < KS; ++c) hv[c] = *reinterpret_cast<const f32x4 *>(hsrc + 16 * c);
        if (t > 0) leave(t - 1);
        fetch(u, t + PD);
        f32x4 acc[4];
#pragma unroll
        for (int g = 0; g < 4; ++g) acc[g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        // inputs in the order v_mfma_f32_16x16x4 takes them in the other kernels: element e of the four 16-byte pieces of a chunk
#pragma unroll
        for (int c = 0; c < KS; ++c)
#pragma unroll
          for (int e = 0; e < 4; ++e) {
#define XS_LOCAL_MFMA(piece)                                                                                            \
            _Pragma("unroll") for (int g = 0; g < 4; ++g)                                                               \
              acc[g] = __builtin_amdgcn_mfma_f32_4x4x1f32(hv[c][e], rf[g][16 * c + 4 * piece + e], acc[g], 2, piece, 0);
            XS_LOCAL_MFMA(0) XS_LOCAL_MFMA(1) XS_LOCAL_MFMA(2) XS_LOCAL_MFMA(3)
#undef XS_LOCAL_MFMA
          }
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          float x0 = acc[g][0], x1 = acc[g][1], x2 = acc[g][2], x3 = acc[g][3];
          transpose_lane_groups(x0, x1, x2, x3);
          ry[g] = ((x0 + x1) + x2) + x3;
        }
      }
      if (start) {  // (a row that starts a document: R.0 = +0 exactly, a zero state)
        st = CellState{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int g = 0; g < 4; ++g) ry[g] = 0.0f;
      }
#pragma unroll
      for (int g = 0; g < 4; ++g) raw[g] = (wxv[g] + ry[g]) + bias_g[g];
      if constexpr (COEF) {
        kept_c = st.c; kept_n = st.n; kept_f = raw[1];
        slstm_pointwise_keep(raw[0], raw[1], raw[2], raw[3], st, kept);
        kept_y = st.y;
      } else {
        slstm_pointwise(raw[0], raw[1], raw[2], raw[3], st);
      }
      if constexpr (BF16) h_bits = (uint16_t)float_to_bf16_bits(st.y);
      else h_bits = st.y;
      if (a < dh) *hw[t & 1] = h_bits;
    }
  }
  if (p.T > 0) leave(p.T - 1);
  if (mine) {
    p.s_out[so] = st.y; p.s_out[BH + so] = st.c; p.s_out[2 * BH + so] = st.n; p.s_out[3 * BH + so] = st.m;
  }
}

template <bool BF16, int W, bool DWX16>
__global__ __launch_bounds__(64 * W) void slstm_local_bwd_kernel(LocalBwdParams p) {
  typedef typename std::conditional<BF16, uint16_t, float>::type elem_t;
  constexpr int DHP = 16 * W;                 // columns of the partial sums
  constexpr int CG = (DHP + 63) / 64;         // (float32) groups of 64 columns
  constexpr int LR = 64 + 8;                  // (bf16) elements between the rows of a wave's deltas in LDS
  constexpr int PD = kLocalBwdAhead;
  __shared__ float part[2][W][4][BF16 ? DHP : 64 * CG];
  __shared__ __attribute__((aligned(16))) uint16_t delt[BF16 ? W : 1][BF16 ? 4 * LR : 1];

  int head, tile;
  const int ntiles = (p.B + 3) >> 2;
  if (!local_place(ntiles * p.NH, p.NH, head, tile)) return;
  const int tid = threadIdx.x, lane = tid & 63, wave = (int)uniform((uint32_t)(tid >> 6));
  // a lane's element: bf16 (row lane / 16, unit lane % 16) as in the forward; float32 (unit lane / 4, row lane % 4): the
  // four deltas of a lane are then MFMA operands as they are (block = unit)
  const int b = BF16 ? lane >> 4 : lane & 3, n = BF16 ? lane & 15 : lane >> 2;
  const int dh = p.dh, H = p.NH * dh;
  const long long BH = (long long)p.B * H;
  const int a = 16 * wave + n, brow = 4 * tile + b;
  const bool mine = a < dh && brow < p.B;
  const int ac = a < dh ? a : dh - 1, bc = brow < p.B ? brow : p.B - 1;
  const long long so = (long long)bc * H + head * dh + ac;

  // ---- R: this wave's 64 rows k = (unit 16 w + k / 4, gate k % 4) of every column d.  bf16: k-step ks, lane group q: k = 32
  //      ks + 8 q + i, columns 16 j + lane % 16.  float32: block = lane / 4: columns 64 cg + lane.
  auto r_at = [&](int k, int d) -> float {
    const int u = 16 * wave + (k >> 2), g = k & 3;
    if (u >= dh || d >= dh) return 0.0f;
    const long long o = ((long long)head * 4 * dh + (long long)g * dh + u) * dh + d;
    return p.r_bf16 ? bf16_bits_to_float(reinterpret_cast<const uint16_t *>(p.r)[o]) : reinterpret_cast<const float *>(p.r)[o];
  };
  uint4 rb[BF16 ? W : 1][2];
  float rf[BF16 ? 1 : CG][BF16 ? 1 : 64];
  if constexpr (BF16) {
#pragma unroll
    for (int j = 0; j < W; ++j)
#pragma unroll
      for (int ks = 0; ks < 2; ++ks) {
        uint32_t w4[4];
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int k = 32 * ks + 8 * (lane >> 4) + 2 * i, d = 16 * j + (lane & 15);
          w4[i] = pack_bf16x2(r_at(k, d), r_at(k + 1, d));
        }
        rb[j][ks] = uint4{w4[0], w4[1], w4[2], w4[3]};
      }
  } else {
#pragma unroll
    for (int cg = 0; cg < CG; ++cg)
#pragma unroll
      for (int k = 0; k < 64; ++k) rf[cg][k] = r_at(k, 64 * cg + lane);
  }

  // ---- the step's inputs, PD steps ahead of the reverse walk
  const long long coef_step = (long long)ntiles * p.NH * W * 576;
  const int clane = BF16 ? lane : (b << 4) | n;  // (the lane of the forward kernel that left this element's coefficients)
  const float *cfp = p.coef + (((long long)tile * p.NH + head) * W + wave) * 576;
  const elem_t *dhp = reinterpret_cast<const elem_t *>(p.d_h) + (long long)bc * p.d_h_sb + head * dh + ac;
  const unsigned char *flp = p.reset ? p.reset + (long long)bc * p.reset_sb : nullptr;
  f32x4 cA[PD], cB[PD];
  float cC[PD];
  elem_t dhr[PD];
  unsigned char flag[PD];
  auto fetch = [&](int u, int t) {
    t = t > 0 ? t : 0;
    const float *src = cfp + t * coef_step;
    cA[u] = *reinterpret_cast<const f32x4 *>(src + 4 * clane);
    cB[u] = *reinterpret_cast<const f32x4 *>(src + 256 + 4 * clane);
    cC[u] = src[512 + clane];
    dhr[u] = dhp[(long long)t * p.d_h_st];
    flag[u] = flp ? flp[t] : (unsigned char)0;
  };
#pragma unroll
  for (int u = 0; u < PD; ++u) fetch(u, p.T - 1 - u);
  float dy = 0.0f, dc = 0.0f, dn = 0.0f;
  if (p.d_s_final) { dy = p.d_s_final[so]; dc = p.d_s_final[BH + so]; dn = p.d_s_final[2 * BH + so]; }
  const long long wo = (long long)bc * p.d_wx_sb + head * dh + ac;

  auto reduce = [&](int buf) {  // what reached this lane's y through the recurrence: the waves' partial sums in order
    float s = part[buf][0][b][a];
#pragma unroll
    for (int w = 1; w < W; ++w) s += part[buf][w][b][a];
    return s;
  };
  bool after = false;  // a document starts at step t + 1: it took nothing from this one
  for (int t0 = p.T - 1; t0 >= 0; t0 -= PD) {
#pragma unroll
    for (int u = 0; u < PD; ++u) {
      const int t = t0 - u;
      if (t < 0) break;
      const bool first = t == p.T - 1;
      if (!first && !p.cut) {
        lds_barrier();  // the partial sums of step t + 1 are in LDS
        dy = reduce((t + 1) & 1);
      } else if (!first) {
        dy = 0.0f;
      }
      if (after) dy = 0.0f;
      const float dh_in = [&] { if constexpr (BF16) return bf16_bits_to_float(dhr[u]); else return dhr[u]; }();
      const float dyt = dh_in + bwd_recurrent_dy(dy, p.clip, first);
      const float dct = dc + dyt * cA[u][0], dnt = dn - dyt * cA[u][1];
      float delta[4] = {cA[u][2] * dct + cA[u][3] * dnt, cB[u][0] * dct + cB[u][1] * dnt, cB[u][2] * dct, cB[u][3] * dyt};
      const bool start = flag[u] != 0;
      dc = start ? 0.0f : cC[u] * dct;
      dn = start ? 0.0f : cC[u] * dnt;
      after = start;
      if (!mine) delta[0] = delta[1] = delta[2] = delta[3] = 0.0f;
      if constexpr (BF16) {
        if (!p.cut) {
          uint16_t *const dl = delt[wave];
          *reinterpret_cast<uint2 *>(dl + b * LR + 4 * n) = uint2{pack_bf16x2(delta[0], delta[1]), pack_bf16x2(delta[2], delta[3])};
          asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the wave's own corner of LDS: no barrier)
          uint4 av[2];
#pragma unroll
          for (int ks = 0; ks < 2; ++ks) av[ks] = *reinterpret_cast<const uint4 *>(dl + (n >> 2) * LR + 32 * ks + 8 * b);
          f32x4 acc[W];
#pragma unroll
          for (int j = 0; j < W; ++j) acc[j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
          for (int ks = 0; ks < 2; ++ks)
#pragma unroll
            for (int j = 0; j < W; ++j)
              acc[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av[ks]), __builtin_bit_cast(bf16x8, rb[j][ks]), acc[j], 0, 0, 0);
#pragma unroll
          for (int j = 0; j < W; ++j) part[t & 1][wave][b][16 * j + n] = acc[j][0];
        }
      } else {
        if (!p.cut) {
          f32x4 acc[CG];
#pragma unroll
          for (int cg = 0; cg < CG; ++cg) acc[cg] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
          // block `unit` of the deltas to all sixteen blocks of columns
#define XS_LOCAL_MFMA(unit)                                                                                             \
          _Pragma("unroll") for (int g = 0; g < 4; ++g) _Pragma("unroll") for (int cg = 0; cg < CG; ++cg)               \
            acc[cg] = __builtin_amdgcn_mfma_f32_4x4x1f32(delta[g], rf[cg][4 * unit + g], acc[cg], 4, unit, 0);
          XS_LOCAL_MFMA(0) XS_LOCAL_MFMA(1) XS_LOCAL_MFMA(2) XS_LOCAL_MFMA(3) XS_LOCAL_MFMA(4) XS_LOCAL_MFMA(5) XS_LOCAL_MFMA(6) XS_LOCAL_MFMA(7)
          XS_LOCAL_MFMA(8) XS_LOCAL_MFMA(9) XS_LOCAL_MFMA(10) XS_LOCAL_MFMA(11) XS_LOCAL_MFMA(12) XS_LOCAL_MFMA(13) XS_LOCAL_MFMA(14) XS_LOCAL_MFMA(15)
#undef XS_LOCAL_MFMA
#pragma unroll
          for (int cg = 0; cg < CG; ++cg)
#pragma unroll
            for (int r = 0; r < 4; ++r) part[t & 1][wave][r][64 * cg + lane] = acc[cg][r];
        }
      }
      // ---- off the chain: the deltas to d_wx, the inputs of the step PD further back
      if (mine) {
        const long long o = wo + (long long)t * p.d_wx_st;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if constexpr (DWX16) reinterpret_cast<uint16_t *>(p.d_wx)[o + (long long)g * H] = (uint16_t)(pack_bf16x2(delta[g], 0.0f) & 0xFFFFu);
          else reinterpret_cast<float *>(p.d_wx)[o + (long long)g * H] = delta[g];
        }
      }
      fetch(u, t - PD);
    }
  }
  // ---- the gradient of the initial state
  if (p.T > 0 && !p.cut) {
    lds_barrier();
    dy = reduce(0);  // (step 0's partial sums)
  } else if (p.T > 0) {
    dy = 0.0f;
  }
  if (after) dy = 0.0f;
  if (mine) {
    p.d_s0[so] = dy; p.d_s0[BH + so] = dc; p.d_s0[2 * BH + so] = dn; p.d_s0[3 * BH + so] = 0.0f;
  }
}

}  // namespace
