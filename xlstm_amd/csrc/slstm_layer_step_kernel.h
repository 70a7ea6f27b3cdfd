// One decoded token of a bfloat16 sLSTM layer up to its hidden state in ONE kernel: convolution + SiLU, the four gate
// projections, R.h and the gating.  Included by slstm_hip.hip only, behind slstm_step_small_kernel.h.
#pragma once

namespace {

struct LayerStepParams {
  StepParams step;          // (wx is not read; row tiles of 16 rows, unit tiles of 16 UT units)
  const uint16_t *x;        // [B, D] contiguous
  const uint16_t *state;    // [B, 3, D]: the inputs before x, oldest first, rows state_sb apart; or null
  long long state_sb;
  const uint16_t *conv_w;   // [D, 4]
  const uint16_t *conv_b;   // [D] or null
  const uint16_t *gate_w[4];  // each [NH, dh, dh]
  uint16_t *ring_out;       // [B, 4, D]: the inputs before x, then x
  uint16_t *x_out;          // [B, D]: x, or null
  int row_tiles;            // of the batch; step.n_row_tiles: of the grid, a workgroup takes every n_row_tiles-th
};

constexpr int layer_step_row_bytes(int nq) { return 2 * 128 * nq + 16; }  // a row of an operand in LDS: K range and 16 bytes of padding
constexpr int layer_step_lds_bytes(int nq) { return 2 * 16 * layer_step_row_bytes(nq); }

// Everything a layer does to a token stays within a head (the convolution is depthwise, the projections and R are block
// diagonal), so the 16 rows x 16 units of a workgroup of slstm_step_small_kernel need nothing of any other
// workgroup if each makes the convolution of its rows' whole head again: 16 x dh values of four taps against four kernels
// one behind the other, of which each costs 2.4 us and more for the launch alone.
// The waves first make a share of the head's x_conv each and leave it in LDS beside x; then wave g of the four of 16 units
// multiplies all of it by its 16 columns of gate g's weights (K in order, one chain: the bits of the projection kernels), and
// each wave a quarter of the previous h by R for all gates (as slstm_step_small_kernel does, its bits).  Weights, R and h are
// asked for in front of the convolution's arithmetic.  W.x is rounded to bfloat16 where the kernels in a row store it.
// UT 2: 32 units, eight waves; the convolution is made half as often, which counts where a compute unit has more than one
// workgroup of UT 1.  LOOP: a workgroup keeps its weights and R in registers for several row tiles, the rows of the next one
// on their way while this one is multiplied and gated.
// What bounds it, 8 heads of 256 with the norm behind it, us a token at 256 / 64 rows: 20.6 / 10.9; without the convolution's arithmetic (150
// instructions a wave and k-step) 20.0 / 10.6, without the products and the reads of their weights 16.4 / 8.1, without either 15.5 / 7.6.  So
// most of it is the way in and out: a latency of memory in front of each row tile's work, x and the taps read once per unit tile, 34 MB
// of states, ring and weights.  The times of both sides stand at layer_step_split.
template <int NQ, int UT, bool HB, bool LOOP>  // NQ: MFMA k-steps of a quarter of K; HB: the recurrent operand comes from h_prev, in bf16
__global__ __launch_bounds__(256 * UT, UT == 2 ? (NQ == 1 && !LOOP ? 4 : 2) : (NQ >= 4 ? 1 : 2)) void slstm_layer_step_kernel(LayerStepParams p) {
  constexpr int QS = 20;  // (see slstm_step_small_kernel)
  constexpr int KS = 4 * NQ, RB = layer_step_row_bytes(NQ);
  constexpr int CV = NQ < UT ? 1 : NQ / UT;  // k-steps of the convolution a wave makes (the waves behind the last of them: none)
  __shared__ f32x4 sums[UT][5][4][4 * QS];  // [quarter of R.h, then W.x][gate][lane group][row]: units 4 q .. + 3
  extern __shared__ __attribute__((aligned(16))) unsigned char layer_step_lds[];  // [x_conv, x][16 rows][RB]
  const StepParams &c = p.step;
  int head, unit_tile, row_tile;
  step_tile_of(c, blockIdx.x, head, unit_tile, row_tile);
  const int lane = threadIdx.x & 63, any_wave = (int)uniform((uint32_t)(threadIdx.x >> 6)), q = lane >> 4, r16 = lane & 15;
  const int wave = any_wave & 3, ut = any_wave >> 2, tid = threadIdx.x & 255;  // of the 16 units
  const int dh = c.dh, H = c.NH * dh, a0 = (unit_tile * UT + ut) * 16;
  const long long BH = (long long)c.B * H;
  if (blockIdx.x == 0 && threadIdx.x < 16) reinterpret_cast<uint32_t *>(c.status)[threadIdx.x] = (threadIdx.x == 5 || threadIdx.x == 6) ? 1u : 0u;  // (see slstm_step_tile_kernel)
  auto in_head = [&](int k) { return k < dh ? k : 0; };  // (inputs past the head: any; zeroed below)

  // ---- what a row tile takes: lane (q, r16) holds inputs 32 k + 8 q .. + 7 of row r16, thread (tid / 16, tid % 16) gates an element
  constexpr int HL = HB ? 1 : 2, HSZ = HB ? 2 : 4;
  struct Rows { uint4 x[CV], taps[CV][3], h[NQ][HL]; float c, n, m; };
  auto fetch_rows = [&](int rt, Rows &o) {
    const int row = rt * 16 + r16, rowc = row < c.B ? row : c.B - 1;
    const uint16_t *xrow = p.x + (long long)rowc * H + head * dh;
    const uint16_t *trow = p.state ? p.state + (long long)rowc * p.state_sb + head * dh : nullptr;
    const char *hrow = HB ? reinterpret_cast<const char *>(reinterpret_cast<const uint16_t *>(c.h_prev) + (long long)rowc * H + head * dh)
                          : reinterpret_cast<const char *>(c.s0 + (long long)rowc * H + head * dh);
#pragma unroll
    for (int s = 0; s < CV; ++s) {
      const int k = in_head((any_wave * CV + s) * 32 + 8 * q);
      o.x[s] = *reinterpret_cast<const uint4 *>(xrow + k);
#pragma unroll
      for (int j = 0; j < 3; ++j) o.taps[s][j] = trow ? *reinterpret_cast<const uint4 *>(trow + (long long)j * H + k) : uint4{0u, 0u, 0u, 0u};
    }
#pragma unroll
    for (int s = 0; s < NQ; ++s) {
      const int k = in_head((wave * NQ + s) * 32 + 8 * q);
#pragma unroll
      for (int i = 0; i < HL; ++i) o.h[s][i] = *reinterpret_cast<const uint4 *>(hrow + k * HSZ + 16 * i);
    }
    const int erow = rt * 16 + (tid >> 4), er = erow < c.B ? erow : c.B - 1;
    const long long eo = (long long)er * H + (long long)head * dh + a0 + (tid & 15);
    o.c = c.s0[BH + eo]; o.n = c.s0[2 * BH + eo]; o.m = c.s0[3 * BH + eo];
  };
  Rows rows, next;
  fetch_rows(row_tile, rows);

  // ---- what stays: the taps' weights, R and the gate's weights (unit r16 of lane (q, r16)), the bias of the element's unit
  constexpr int CH = CV < 4 ? CV : 2;  // k-steps whose convolution is made at once
  uint4 cw[CH][4], cb[CH];
  auto fetch_taps = [&](int s0) {
#pragma unroll
    for (int s = 0; s < CH; ++s) {
      const int ch = head * dh + in_head((any_wave * CV + s0 + s) * 32 + 8 * q);
#pragma unroll
      for (int j = 0; j < 4; ++j) cw[s][j] = *reinterpret_cast<const uint4 *>(p.conv_w + (long long)ch * 4 + 8 * j);
      cb[s] = p.conv_b ? *reinterpret_cast<const uint4 *>(p.conv_b + ch) : uint4{0u, 0u, 0u, 0u};
    }
  };
  fetch_taps(0);
  const uint16_t *wrow = p.gate_w[wave] + ((long long)head * dh + a0 + r16) * dh;
  const uint16_t *rrow = reinterpret_cast<const uint16_t *>(c.r) + ((long long)head * 4 * dh + a0 + r16) * dh;
  uint4 rv[NQ][4], wv[KS];
#pragma unroll
  for (int s = 0; s < NQ; ++s)
#pragma unroll
    for (int g = 0; g < 4; ++g) rv[s][g] = *reinterpret_cast<const uint4 *>(rrow + (long long)g * dh * dh + in_head((wave * NQ + s) * 32 + 8 * q));
#pragma unroll
  for (int s = 0; s < KS; ++s) wv[s] = *reinterpret_cast<const uint4 *>(wrow + in_head(32 * s + 8 * q));
  float bias[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) bias[g] = c.bias[((long long)head * 4 + g) * dh + a0 + (tid & 15)];

  for (;;) {
    const int row0 = row_tile * 16;
    if constexpr (LOOP) {
      if (row_tile + c.n_row_tiles < p.row_tiles) fetch_rows(row_tile + c.n_row_tiles, next);
    }
    // ---- convolution + SiLU of the wave's share (the arithmetic of causal_conv_silu_kernel, tap by tap back in time)
#pragma unroll
    for (int s0 = 0; s0 < CV; s0 += CH) {
      if (s0) fetch_taps(s0);
#pragma unroll
      for (int s = 0; s < CH; ++s) {
        const int k = (any_wave * CV + s0 + s) * 32 + 8 * q;
        if (NQ < UT && any_wave >= 4 * NQ) break;
        const uint32_t bw[4] = {cb[s].x, cb[s].y, cb[s].z, cb[s].w};
        float a[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) a[e] = bf16_bits_to_float((bw[e >> 1] >> (16 * (e & 1))) & 0xFFFFu);
#pragma unroll
        for (int back = 0; back < 4; ++back) {
          if (back && !p.state) break;  // (nothing in front of x)
          const uint4 v = back ? rows.taps[s0 + s][3 - back] : rows.x[s0 + s];
          const uint32_t d[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
          for (int e = 0; e < 8; ++e) {  // weight (channel e, tap 3 - back): 16 bits 4 e + 3 - back of the lane's 64 bytes
            const int i = 4 * e + 3 - back;
            const uint4 &wq = cw[s][i >> 3];
            const uint32_t ww = ((i >> 1) & 3) == 0 ? wq.x : (((i >> 1) & 3) == 1 ? wq.y : (((i >> 1) & 3) == 2 ? wq.z : wq.w));
            a[e] += bf16_bits_to_float((ww >> (16 * (i & 1))) & 0xFFFFu) * bf16_bits_to_float((d[e >> 1] >> (16 * (e & 1))) & 0xFFFFu);
          }
        }
        uint32_t o[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const float u = a[2 * e], w = a[2 * e + 1];
          o[e] = pack_bf16x2(u * __builtin_amdgcn_rcpf(1.0f + __expf(-u)), w * __builtin_amdgcn_rcpf(1.0f + __expf(-w)));
        }
        // the workgroup's piece of the next ring, from the lanes that hold it
        if (k >= unit_tile * (16 * UT) && k < (unit_tile + 1) * (16 * UT) && row0 + r16 < c.B) {
          uint16_t *ring = p.ring_out + (long long)(row0 + r16) * 4 * H + head * dh + k;
#pragma unroll
          for (int j = 0; j < 4; ++j) *reinterpret_cast<uint4 *>(ring + (long long)j * H) = j == 3 ? rows.x[s0 + s] : rows.taps[s0 + s][j];
          if (p.x_out) *reinterpret_cast<uint4 *>(p.x_out + (long long)(row0 + r16) * H + head * dh + k) = rows.x[s0 + s];
        }
        const bool there = k < dh;
        unsigned char *dst = layer_step_lds + r16 * RB + 2 * k;
        *reinterpret_cast<uint4 *>(dst) = there ? uint4{o[0], o[1], o[2], o[3]} : uint4{0u, 0u, 0u, 0u};
        *reinterpret_cast<uint4 *>(dst + 16 * RB) = there ? rows.x[s0 + s] : uint4{0u, 0u, 0u, 0u};
      }
    }
    // ---- R.h of the wave's quarter of K
    const bool dead = row0 + r16 >= c.B;
    f32x4 acc[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) acc[g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < NQ; ++s) {
      const bool there = (wave * NQ + s) * 32 + 8 * q < dh;
      uint4 h = rows.h[s][0];
      if constexpr (!HB) {
        const uint4 l = rows.h[s][0], m = rows.h[s][HL - 1];
        h = uint4{pack_bf16x2(__uint_as_float(l.x), __uint_as_float(l.y)), pack_bf16x2(__uint_as_float(l.z), __uint_as_float(l.w)),
                  pack_bf16x2(__uint_as_float(m.x), __uint_as_float(m.y)), pack_bf16x2(__uint_as_float(m.z), __uint_as_float(m.w))};
      }
      if (dead || !there) h = uint4{0u, 0u, 0u, 0u};
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        const uint4 r = there ? rv[s][g] : uint4{0u, 0u, 0u, 0u};
        acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, r), __builtin_bit_cast(bf16x8, h), acc[g], 0, 0, 0);
      }
    }
#pragma unroll
    for (int g = 0; g < 4; ++g) sums[ut][wave][g][q * QS + r16] = acc[g];
    lds_barrier();
    // ---- W.x of gate `wave` over all of K (slots i, f: x_conv; z, o: x)
    f32x4 wx4 = {0.0f, 0.0f, 0.0f, 0.0f};
    const unsigned char *operand = layer_step_lds + (wave >= 2 ? 16 * RB : 0) + r16 * RB + 16 * q;
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      if (32 * s < dh) {
        const uint4 v = *reinterpret_cast<const uint4 *>(operand + 64 * s);
        wx4 = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, wv[s]), __builtin_bit_cast(bf16x8, v), wx4, 0, 0, 0);
      }
    }
    sums[ut][4][wave][q * QS + r16] = wx4;
    lds_barrier();
    float raw[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const int place = ((tid & 15) >> 2) * QS + (tid >> 4), e = tid & 3;
      auto at = [&](int part) { return reinterpret_cast<const float *>(&sums[ut][part][g][place])[e]; };
      float s = at(0);
#pragma unroll
      for (int w = 1; w < 4; ++w) s += at(w);
      raw[g] = (bf16_bits_to_float(pack_bf16x2(at(4), 0.0f) & 0xFFFFu) + s) + bias[g];
    }
    CellState st{0.0f, rows.c, rows.n, rows.m};
    slstm_pointwise(raw[0], raw[1], raw[2], raw[3], st);
    if (row0 + (tid >> 4) < c.B) {
      const long long eo = (long long)(row0 + (tid >> 4)) * H + (long long)head * dh + a0 + (tid & 15);
      c.s_out[eo] = st.y; c.s_out[BH + eo] = st.c; c.s_out[2 * BH + eo] = st.n; c.s_out[3 * BH + eo] = st.m;
      reinterpret_cast<uint16_t *>(c.h_out)[eo] = (uint16_t)float_to_bf16_bits(st.y);
    }
    if constexpr (!LOOP) return;
    row_tile += c.n_row_tiles;
    if (row_tile >= p.row_tiles) return;  // (the same for all waves)
    rows = next;
    lds_barrier();  // (the sums of this row tile have been read)
  }
}

typedef void (*LayerStepKernel)(LayerStepParams);
template <bool HB>
LayerStepKernel pick_layer_step(int nch, int ut, bool loop) {
  if (nch == 1) return loop ? slstm_layer_step_kernel<1, 2, HB, true> : (ut == 2 ? slstm_layer_step_kernel<1, 2, HB, false> : slstm_layer_step_kernel<1, 1, HB, false>);
  if (nch == 2) return loop ? slstm_layer_step_kernel<2, 2, HB, true> : (ut == 2 ? slstm_layer_step_kernel<2, 2, HB, false> : slstm_layer_step_kernel<2, 1, HB, false>);
  return ut == 2 ? slstm_layer_step_kernel<4, 2, HB, false> : slstm_layer_step_kernel<4, 1, HB, false>;
}

}  // namespace
