// The decode step (T = 1) of small batches.  Included by slstm_hip.hip only, behind slstm_step_kernel.h.
//
// slstm_step_tile_kernel gives a workgroup 64 rows x 32 units: 16 rows of 4 heads of 256 are 32 workgroups on 256 compute
// units, each of which brings 64 KiB of R to LDS and multiplies 48 rows that are not there.  Here a workgroup owns 16 rows x 16
// units of a head, and its four waves a quarter of K each, so that every compute unit has little to fetch and everything is
// asked for at once, straight into MFMA operand registers: a lane's pieces of R (16 bytes of each gate per k-step), of the
// previous h, and what the gating of its element takes (W.x, bias, c, n, m).  One latency of memory, the quarter's MFMAs, the
// four quarters through LDS in the order every kernel adds them (the same bits), one element (row, unit) per thread.
//
// us a step replayed from a graph, before -> after: bf16 4 heads of 128, 1 row 5.6 -> 3.3, 4 heads of 256, 16 rows 7.7 -> 4.1, 4
// heads of 1024, 1 row 9.8 -> 6.8; float32 4 heads of 256, 16 rows 13.2 -> 5.9, 4 heads of 512, 16 rows 21.7 -> 9.7.
// Bound by that one latency behind the launch; with more than a few row tiles by R, which every row tile reads once more.
#pragma once

namespace {

template <bool BF16, int NQ, bool HB>  // NQ: MFMA k-steps of a quarter of K; HB: the operand comes from h_prev, in bf16
__global__ __launch_bounds__(256, NQ == 8 ? 1 : 2) void slstm_step_small_kernel(StepParams p) {
  static_assert(!HB || BF16, "h_prev is a bf16 operand");
  constexpr int EPC = BF16 ? 8 : 4, CHK = 4 * EPC, ESZ = BF16 ? 2 : 4;
  constexpr int QS = 20;  // 16-byte places per lane group in LDS: 16 and 4 of padding, so that a gating wave's reads hit all banks once
  __shared__ f32x4 sums[4][4][4 * QS];  // [quarter][gate][lane group][row]: units 4 q .. + 3
  int head, unit_tile, row_tile;
  step_tile_of(p, blockIdx.x, head, unit_tile, row_tile);
  const int tid = threadIdx.x, lane = tid & 63, wave = (int)uniform((uint32_t)(tid >> 6)), q = lane >> 4, r16 = lane & 15;
  const int dh = p.dh, H = p.NH * dh, a0 = unit_tile * 16, row0 = row_tile * 16;
  const long long BH = (long long)p.B * H;
  if (blockIdx.x == 0 && tid < 16) reinterpret_cast<uint32_t *>(p.status)[tid] = (tid == 5 || tid == 6) ? 1u : 0u;  // (see slstm_step_tile_kernel)

  // ---- operands: lane (q, r16) holds inputs CHK ch + EPC q .. of unit r16 (R, on the MFMA M axis) and of row r16 (h)
  const int u = a0 + r16, uc = u < dh ? u : dh - 1;
  const int row = row0 + r16, rowc = row < p.B ? row : p.B - 1;
  const bool live = row < p.B && p.s0 != nullptr;
  const char *rp = reinterpret_cast<const char *>(p.r) + ((long long)head * 4 * dh + uc) * dh * ESZ;
  const char *hp = HB ? reinterpret_cast<const char *>(reinterpret_cast<const uint16_t *>(p.h_prev) + (long long)rowc * H + head * dh)
                      : (live ? reinterpret_cast<const char *>(p.s0 + (long long)rowc * H + head * dh) : rp);
  constexpr int HSZ = HB ? 2 : 4;
  constexpr int HL = BF16 && !HB ? 2 : 1;  // 16-byte loads of h per k-step
  uint4 hv[NQ][HL], rv[NQ][4];
#pragma unroll
  for (int c = 0; c < NQ; ++c) {
    const int k = (wave * NQ + c) * CHK + EPC * q, kc = k < dh ? k : 0;  // (inputs past the head: any, zeroed below)
#pragma unroll
    for (int i = 0; i < HL; ++i) hv[c][i] = *reinterpret_cast<const uint4 *>(hp + ((HB || live) ? kc * HSZ : 0) + 16 * i);
#pragma unroll
    for (int g = 0; g < 4; ++g) rv[c][g] = *reinterpret_cast<const uint4 *>(rp + ((long long)g * dh * dh + kc) * ESZ);
  }
  bool zero = !live;
  if (p.reset && live) zero = p.reset[(long long)rowc * p.reset_sb] != 0;

  // ---- the thread's element
  const int erow = row0 + (tid >> 4), eu = a0 + (tid & 15);
  const bool mine = erow < p.B && eu < dh;
  const int er = erow < p.B ? erow : p.B - 1, ec = eu < dh ? eu : dh - 1;
  const long long eo = (long long)er * H + (long long)head * dh + ec;
  float wx[4], bias[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const long long o = (long long)er * p.wx_sb + (long long)g * H + (long long)head * dh + ec;
    if constexpr (BF16) wx[g] = bf16_bits_to_float(reinterpret_cast<const uint16_t *>(p.wx)[o]);
    else wx[g] = reinterpret_cast<const float *>(p.wx)[o];
    bias[g] = p.bias[((long long)head * 4 + g) * dh + ec];
  }
  CellState st{0.0f, 0.0f, 0.0f, 0.0f};
  if (p.s0) {
    st.c = p.s0[BH + eo]; st.n = p.s0[2 * BH + eo]; st.m = p.s0[3 * BH + eo];
    if (p.reset && p.reset[(long long)er * p.reset_sb]) st = CellState{0.0f, 0.0f, 0.0f, 0.0f};
  }

  f32x4 acc[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) acc[g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int c = 0; c < NQ; ++c) {
    const bool there = (wave * NQ + c) * CHK + EPC * q < dh;
    uint4 h = hv[c][0];
    if constexpr (BF16 && !HB) {
      const uint4 l = hv[c][0], m = hv[c][HL - 1];
      h = uint4{pack_bf16x2(__uint_as_float(l.x), __uint_as_float(l.y)), pack_bf16x2(__uint_as_float(l.z), __uint_as_float(l.w)),
                pack_bf16x2(__uint_as_float(m.x), __uint_as_float(m.y)), pack_bf16x2(__uint_as_float(m.z), __uint_as_float(m.w))};
    }
    if (zero || !there) h = uint4{0u, 0u, 0u, 0u};
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      const uint4 r = there ? rv[c][g] : uint4{0u, 0u, 0u, 0u};
      if constexpr (BF16) {
        acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, r), __builtin_bit_cast(bf16x8, h), acc[g], 0, 0, 0);
      } else {
        const uint32_t rw[4] = {r.x, r.y, r.z, r.w}, hw[4] = {h.x, h.y, h.z, h.w};
#pragma unroll
        for (int e = 0; e < 4; ++e) acc[g] = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(rw[e]), __uint_as_float(hw[e]), acc[g], 0, 0, 0);
      }
    }
  }
#pragma unroll
  for (int g = 0; g < 4; ++g) sums[wave][g][q * QS + r16] = acc[g];
  __syncthreads();
  float raw[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) {
    const int place = ((tid & 15) >> 2) * QS + (tid >> 4), e = tid & 3;
    float s = reinterpret_cast<const float *>(&sums[0][g][place])[e];
#pragma unroll
    for (int w = 1; w < 4; ++w) s += reinterpret_cast<const float *>(&sums[w][g][place])[e];
    raw[g] = (wx[g] + s) + bias[g];
  }
  slstm_pointwise(raw[0], raw[1], raw[2], raw[3], st);
  if (mine) {
    p.s_out[eo] = st.y; p.s_out[BH + eo] = st.c; p.s_out[2 * BH + eo] = st.n; p.s_out[3 * BH + eo] = st.m;
    if constexpr (BF16) reinterpret_cast<uint16_t *>(p.h_out)[eo] = (uint16_t)float_to_bf16_bits(st.y);
    else reinterpret_cast<float *>(p.h_out)[eo] = st.y;
  }
}

template <bool BF16, bool HB>
void (*pick_step_small(int nch))(StepParams) {
  switch (nch) {
    case 1: return slstm_step_small_kernel<BF16, 1, HB>;
    case 2: return slstm_step_small_kernel<BF16, 2, HB>;
    case 4: return slstm_step_small_kernel<BF16, 4, HB>;
    default: return slstm_step_small_kernel<BF16, 8, HB>;
  }
}

}  // namespace
