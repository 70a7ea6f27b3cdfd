// The persistent sequence kernel with two workgroups per compute unit (bf16): heads of more than 512 units, whose group it keeps on ONE
// XCD, and batches of smaller heads that fill the device.  Included by slstm_hip.hip only, after slstm_seq_kernel.h (same parameters, same exchange ring, same bits).
//
// At 16 units a workgroup such a head has 33 to 64 members.  With one workgroup per compute unit they sit on an XCD pair, half of
// every poll crosses the fabric between the two (the exchange alone: 1.72 us a step against 0.58 inside an XCD), and four
// groups fill the device.  The 128 KiB of R of a workgroup take a quarter of a compute unit's registers, so two fit: here a workgroup
// is FOUR waves of up to 256 registers that do everything themselves, 64 of them share the 32 compute units of an XCD, and
// eight groups fill the device, each with half of the batch rows that an XCD pair would get.  The two workgroups of a compute unit know
// nothing of each other; one multiplies while the other gates or waits.
//
//   MFMA     a wave owns a quarter of K for the 64 columns (128 registers of R), 32 MFMAs per row tile; the four partial sums meet
//            in LDS (one barrier per tile) and are added in the order of the other kernels: the same bits.
//   gating   rows 4 wave .. + 3 of a tile, one element per lane, by the wave itself.
//   W.x      one load per wave and tile, four tiles ahead, into registers; to the lanes that gate it through a private corner of LDS.
//   polls    with two row tiles a wave asks for the other tile's h behind its own gating, in front of its stores (behind the
//            barrier: 3.12 against 3.05 us a step at head dim 1024; behind the stores: 3.64).  With one row tile it asks
//            behind a pause after its own publication.  Row tiles of 4 and 8 rows fill the MFMA rows that they leave empty with other chunks of K
//            (2 and 4 loads a wave instead of 8) and shift them into place with DPP: B 1 / 8 / 16 x 4 heads of 1024 1.87 / 1.90 / 2.23 ->
//            1.47 / 1.51 / 2.01 us a step.
//   training COEF: the nine coefficients leave the registers they were formed in as 16-byte stores (a wave's 64 elements are one
//            576-float set): no staging.  Two row tiles are possible, so a batch takes fewer launches.
//
// Measured, us a step, the kernels of one workgroup per compute unit -> this one: 4 heads of 1024 at B 64 3.33 -> 3.00 (512 steps
// and more), B 32 3.35 -> 2.29, B 16 2.40 -> 1.87, B 1 1.91 -> 1.38; 4 x 768 B 64 3.78 -> 2.96, B 16 2.29 -> 1.71; training 3 x 768
// B 200 T 52 87 -> 63 with the backward pass.
//
// Smaller heads (NCH 2 and 4: head dims 136 to 512) come here where two workgroups per compute unit make one row tile per workgroup of two, or
// fewer launches; see the dispatch for both sides.
//
// Bound, at B 64 x 4 heads of 1024: a tile goes round once in two iterations of 3,400 cycles.  By its counters a SIMD's matrix unit is busy for
// 1,023 of them and its vector unit issues for 1,200 (141 instructions a wave, arrival tests, sums and gating of two workgroups), and the data path of
// the texture unit has something under way for 2,860 (64 KiB of operand a compute unit, waiting included): latencies, one behind the other.  The
// later of two workgroups on a compute unit has no slack (300 arrival test, 900 MFMA, 850 sums and gating with the request, 650 stores and
// W.x, 300 to 600 at the barrier), the earlier waits for its h.  Dropped: ONE workgroup of eight waves and 32 units with the operand
// polled once and shared through LDS (half the texture traffic): 3.83 at B 64, 2.14 at B 16, because all eight waves then multiply,
// and gate, at the same time; priorities between the two workgroups: no change; the request in two halves: 3.48.
#pragma once

namespace {

constexpr int kPairThreads = 256;
template <int NCH, int MT, int RT, int COEF>  // NCH: 16-byte chunks of an operand row per lane and wave
__global__ __launch_bounds__(kPairThreads, 2) void slstm_seq_pair_kernel(SeqParams p) {
  constexpr int KW = NCH * 32;           // input units per wave
  constexpr int PK = 16 / RT;            // chunks per load: the MFMA rows of batch rows that do not exist bring other chunks of those that do
  constexpr int NL = NCH / PK;           // loads per wave and tile
  constexpr int D = 4;                   // iterations W.x is fetched ahead
  static_assert(RT == 4 || RT == 8 || RT == 16, "rows of a tile");
  static_assert(MT == 1 || RT == 16, "two row tiles are of 16 rows");
  static_assert(NCH % PK == 0, "whole loads");
  static_assert(D % MT == 0, "the ring of W.x turns over in whole steps");
  __shared__ float part[2][4][4][kTileFloats];  // [buffer][wave][gate][unit*stride + row]
  __shared__ __attribute__((aligned(16))) uint16_t wxt[4][16][16];  // [wave][row * 4 + gate][unit]
  __shared__ uint32_t cross_s;

  const int wg = blockIdx.x;
  const int ngroups = p.NHL * p.NBT;
  int gi, member;
  seq_place(p, wg, gi, member);
  if (gi >= ngroups) return;
  const int head = p.head0 + gi / p.NBT;
  const int bt = gi % p.NBT;
  const int tid = threadIdx.x;
  const int wave = (int)uniform((uint32_t)(tid >> 6));
  const int lane = tid & 63;
  const long long spin_limit = p.spin_limit > 0 ? p.spin_limit : kDefaultSpinLimit;
  if (tid < 64) {
    const uint32_t verdict = seq_handshake(p, wg, gi, spin_limit);
    if (tid == 0) cross_s = verdict;
  }

  const int dh = p.dh;
  const int H = p.NH * dh;
  const int a0 = member * 16;
  const int rowbase = p.b0 + bt * p.rows_per_wg;
  const int rend = (rowbase + p.rows_per_wg < p.bend) ? rowbase + p.rows_per_wg : p.bend;
  const long long BH = (long long)p.B * H;
  const int NIT = p.T * MT;
  constexpr int XTILE = 16 * 16 * 2;                 // bytes one member publishes per row tile
  const int xslot = p.G * MT * XTILE;                // bytes one group publishes per step
  char *const xbase = reinterpret_cast<char *>(p.xbuf) + (long long)gi * kRing * xslot;
  const int q = lane >> 4;     // MFMA: lane group
  const int r16 = lane & 15;   // MFMA: row (A) / column (B, C)

  // ---- R slice -> registers (once).  B operand: column n = unit a0 + r16 of gate g, K chunk c of this wave / lane group.
  uint4 rreg[4][NCH];
#pragma unroll
  for (int g = 0; g < 4; ++g)
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const int a = a0 + r16, k0 = wave * KW + c * 32 + q * 8;
      uint4 v = make_uint4(0, 0, 0, 0);
      if (a < dh && k0 < dh) {
        const long long off = ((long long)head * 4 * dh + (long long)g * dh + a) * dh + k0;
        if (p.r_bf16) {
          v = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(p.r) + off);
        } else {
          const float4 lo = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p.r) + off);
          const float4 hi = *reinterpret_cast<const float4 *>(reinterpret_cast<const float *>(p.r) + off + 4);
          v.x = pack_bf16x2(lo.x, lo.y); v.y = pack_bf16x2(lo.z, lo.w);
          v.z = pack_bf16x2(hi.x, hi.y); v.w = pack_bf16x2(hi.z, hi.w);
        }
      }
      rreg[g][c] = v;
    }

  // ---- gating role: rows 4 wave .. + 3 of every tile, one element per lane
  const bool gates = 4 * wave < RT;
  const int pa = lane & 15, pb = 4 * wave + (lane >> 4);
  const int ua = a0 + pa;
  const bool unit_ok = gates && ua < dh;
  const int col = head * dh + (unit_ok ? ua : a0);
  float bias_g[4];
#pragma unroll
  for (int g = 0; g < 4; ++g) bias_g[g] = unit_ok ? p.bias[((long long)head * 4 + g) * dh + ua] : 0.0f;
  CellState st[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int brow = rowbase + mt * 16 + pb;
    st[mt] = CellState{0.0f, 0.0f, 0.0f, 0.0f};
    if (p.s0 && unit_ok && brow < rend) {
      const long long o = (long long)brow * H + col;
      st[mt].y = p.s0[o]; st[mt].c = p.s0[BH + o]; st[mt].n = p.s0[2 * BH + o]; st[mt].m = p.s0[3 * BH + o];
    }
  }

  // ---- W.x and the reset flags: D iterations ahead, one load per wave: lane l fetches units 4 (l & 3) .. + 3 of gate
  //      (l >> 2) & 3 for row l >> 4 of the wave's four rows.  What does not exist lies past the descriptor's end: zeros.
  constexpr int kNone = (int)0xFFFFFF00u;
  auto descriptor = [&](const void *base, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void *>(base), 0, (int)bytes, 0x00020000);
  };
  int wx_off[MT], flag_off[MT], h_off[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int row0 = rowbase + mt * 16 + 4 * wave;
    const bool there = gates && row0 + (lane >> 4) < rend;
    wx_off[mt] = there && a0 + 4 * (lane & 3) < dh ? (int)(uint32_t)(((lane >> 4) * p.wx_sb + (long long)((lane >> 2) & 3) * H + 4 * (lane & 3)) * 2) : kNone;
    flag_off[mt] = there ? (int)(uint32_t)((lane >> 4) * p.reset_sb) : kNone;
    h_off[mt] = there && unit_ok ? (int)(uint32_t)(((lane >> 4) * (long long)H + pa) * 2) : kNone;
  }
  typedef uint32_t wxq_t __attribute__((ext_vector_type(2)));
  wxq_t wxq[D];
  uint32_t flq[D];
  auto fetch = [&](int t, int mt, wxq_t &dst, uint32_t &flag) {
    const int tc = t < p.T ? t : p.T - 1;  // (what is fetched past the end is never looked at)
    const long long row0 = rowbase + mt * 16 + 4 * wave;
    const __amdgpu_buffer_rsrc_t rs = descriptor(reinterpret_cast<const uint16_t *>(p.wx) + row0 * p.wx_sb + (long long)tc * p.wx_st + (long long)head * dh + a0, 0xFFFFFF00u);
    dst = __builtin_bit_cast(wxq_t, __builtin_amdgcn_raw_buffer_load_b64(rs, wx_off[mt], 0, 0));
    if (p.reset) flag = __builtin_amdgcn_raw_buffer_load_b8(descriptor(p.reset + row0 * p.reset_sb + tc, 0xFFFFFF00u), flag_off[mt], 0, 0);
  };
#pragma unroll
  for (int u = 0; u < D; ++u) {
    flq[u] = 0u;
    fetch(u / MT, u % MT, wxq[u], flq[u]);
  }

  bool aborted = false;
  uint32_t max_spins = 0;
  lds_barrier();  // the placement verdict is in LDS
  const bool cross = cross_s != 0u;

  // ---- the exchange: load j brings chunk PK j + r16 / RT of batch row r16 % RT.  Unit k of row r of row tile mt lives at
  //      [mt][k/16][r][k%16] of a slot.  A descriptor ends with its row tile: units past the last workgroup are zeros, as are rows that do not exist.
  const int xtile = p.G * XTILE;
  const int xrow = r16 % RT;
  int xlane[MT];
#pragma unroll
  for (int mt = 0; mt < MT; ++mt)
    xlane[mt] = rowbase + mt * 16 + xrow < rend ? ((wave * KW + q * 8) >> 4) * XTILE + (r16 / RT) * 2 * XTILE + xrow * 32 + ((q * 8) & 15) * 2 : 0x7FFFFF00;
  auto ring = [&](int slot, int mt) { return descriptor(xbase + (slot % kRing) * xslot + mt * xtile, (uint32_t)xtile); };
  uint4 op[NL];
  auto request = [&](int t, int mt) {
    const __amdgpu_buffer_rsrc_t rs = ring(t + kRing - 1, mt);
#pragma unroll
    for (int j = 0; j < NL; ++j) op[j] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, xlane[mt], j * PK * 2 * XTILE, 16));
  };
  auto any_missing = [&]() {
    uint32_t mark = 0u;
#pragma unroll
    for (int j = 0; j < NL; ++j) mark = mark_join<true>(mark, chunk_mark<true>(op[j]));
    return __builtin_amdgcn_ballot_w64(mark_has_sentinel<true>(mark)) != 0ull;
  };
  // the MFMA operand of chunk c: its rows lie in lanes r16 = RT (c % PK) .. of load c / PK
  auto chunk = [&](int c) {
    const uint4 v = op[c / PK];
    auto rows = [&](uint32_t w) {
      const int s = RT * (c % PK);
      if (s == 4) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x104, 0xF, 0xF, true);   // row_shl
      if (s == 8) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x108, 0xF, 0xF, true);
      if (s == 12) return (uint32_t)__builtin_amdgcn_update_dpp(0, (int)w, 0x10C, 0xF, 0xF, true);
      return w;
    };
    return __builtin_bit_cast(bf16x8, uint4{rows(v.x), rows(v.y), rows(v.z), rows(v.w)});
  };
#ifdef XS_PROFILE
  long long prof[8] = {0, 0, 0, 0, 0, 0, 0, 0};
  long long tick = clock64();
#define XS_PTICK(i) do { const long long now_ = clock64(); prof[i] += now_ - tick; tick = now_; } while (0)
#else
#define XS_PTICK(i) do { } while (0)
#endif

  auto iteration = [&](auto uc, auto first_c, int t) {
    constexpr int u = decltype(uc)::value, mt = u % MT, buf = u & 1;
    constexpr bool initial = decltype(first_c)::value && u < MT;
    XS_PTICK(7);
    // ---- 1. the operand: h_{t-1} of batch row rowbase + mt * 16 + r16, this wave's quarter of K
    if constexpr (initial) {
#pragma unroll
      for (int j = 0; j < NL; ++j) {
        const int k0 = wave * KW + (j * PK + r16 / RT) * 32 + q * 8, row = rowbase + mt * 16 + xrow;
        op[j] = make_uint4(0, 0, 0, 0);
        if (p.s0 && row < rend && k0 < dh) {
          const float *src = p.s0 + (long long)row * H + head * dh + k0;
          const float4 lo = *reinterpret_cast<const float4 *>(src), hi = *reinterpret_cast<const float4 *>(src + 4);
          op[j].x = pack_bf16x2(lo.x, lo.y); op[j].y = pack_bf16x2(lo.z, lo.w);
          op[j].z = pack_bf16x2(hi.x, hi.y); op[j].w = pack_bf16x2(hi.z, hi.w);
        }
      }
    } else {
#pragma unroll
      for (int j = 0; j < NL; ++j) asm volatile("" : "+v"(op[j].x), "+v"(op[j].y), "+v"(op[j].z), "+v"(op[j].w));
      XS_PTICK(0);
      if (!aborted && any_missing()) {
        uint32_t spins = 0;
        for (;;) {
          ++spins;
          if ((spins & 1023u) == 0u && __hip_atomic_load(&p.status->aborted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u) {
            aborted = true;
            break;
          }
          if ((long long)spins >= spin_limit) {
            aborted = true;
            if (atomicExch(&p.status->aborted, 1u) == 0u) {
              p.status->abort_wg = (uint32_t)wg;
              p.status->abort_step = (uint32_t)t;
            }
            break;
          }
          request(t, mt);
          if (!any_missing()) break;
        }
        max_spins = spins > max_spins ? spins : max_spins;
#ifdef XS_PROFILE
        prof[6] += spins;
#endif
      }
    }
    XS_PTICK(1);
    if (MT > 1) __builtin_amdgcn_s_setprio(2);  // (1 % at B 64; with one row tile 1 % the other way)
    // ---- 2. partial R.h over this wave's quarter of K, all four gates
    f32x4 acc[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) acc[g] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      const bf16x8 av = chunk(c);
#pragma unroll
      for (int g = 0; g < 4; ++g) acc[g] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(av, __builtin_bit_cast(bf16x8, rreg[g][c]), acc[g], 0, 0, 0);
    }
    // W.x of this iteration to the lanes that gate it (same wave: no barrier, LDS keeps a wave's order)
    float wxf[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    bool restart = false;
    if (RT == 16 || gates) {
      *reinterpret_cast<wxq_t *>(&wxt[wave][lane >> 2][4 * (lane & 3)]) = wxq[u];
#pragma unroll
      for (int g = 0; g < 4; ++g) wxf[g] = bf16_bits_to_float(wxt[wave][(lane >> 4) * 4 + g][pa]);
      // a row that starts a document: zero state, and R.h counts as the +0 a zero operand row gives
      restart = (flq[u] & 0xFFu) != 0u;
      asm volatile("" : "+v"(wxf[0]), "+v"(wxf[1]), "+v"(wxf[2]), "+v"(wxf[3]));
    }
#pragma unroll
    for (int g = 0; g < 4; ++g)
      if (RT == 16 || 4 * q < RT) *reinterpret_cast<f32x4 *>(&part[buf][wave][g][r16 * kTileStride + 4 * q]) = acc[g];
    XS_PTICK(2);
    lds_barrier();
    if (MT > 1) __builtin_amdgcn_s_setprio(0);
    XS_PTICK(3);
    constexpr int nmt = (mt + 1) % MT;
    const int nt = t + (nmt == 0 ? 1 : 0);
    if (RT < 16 && !gates) {
      __builtin_amdgcn_s_sleep(RT == 4 ? 16 : 18);
      if (nt < p.T) request(nt, 0);
      return;
    }
    // ---- 3. the gating of element (row pb, unit pa)
    float raw[4];
#pragma unroll
    for (int g = 0; g < 4; ++g) {
      // fixed summation order: wave 0 + wave 1 + wave 2 + wave 3
      float ry = part[buf][0][g][pa * kTileStride + pb];
      ry += part[buf][1][g][pa * kTileStride + pb];
      ry += part[buf][2][g][pa * kTileStride + pb];
      ry += part[buf][3][g][pa * kTileStride + pb];
      if (restart) ry = 0.0f;
      raw[g] = (wxf[g] + ry) + bias_g[g];
    }
    if (restart) st[mt] = CellState{0.0f, 0.0f, 0.0f, 0.0f};
    GateValues kept{0.0f, 0.0f, 0.0f, 0.0f, 0.0f};
    const float kept_c = st[mt].c, kept_n = st[mt].n;
    if constexpr (COEF != 0) slstm_pointwise_keep(raw[0], raw[1], raw[2], raw[3], st[mt], kept);
    else slstm_pointwise(raw[0], raw[1], raw[2], raw[3], st[mt]);
    if (MT > 1 && !(decltype(first_c)::value && u + 1 < MT) && nt < p.T) request(nt, nmt);
    const uint16_t hbits = (uint16_t)float_to_bf16_bits(st[mt].y);
    XS_PTICK(4);
    // ---- 4. h_t to the peers, the words of h_{t-2} re-armed (lanes outside the batch or the head write words of their own block that
    //      nobody polls), then what nobody waits for
    {
      const int off = member * XTILE + (pb * 16 + pa) * 2;
      const __amdgpu_buffer_rsrc_t now = ring(t, mt), old = ring(t + kRing - 2, mt);
      if (cross) {
        __builtin_amdgcn_raw_buffer_store_b16(hbits, now, off, 0, 16);
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)kSentinel16, old, off, 0, 16);
      } else {
        __builtin_amdgcn_raw_buffer_store_b16(hbits, now, off, 0, 0);
        __builtin_amdgcn_raw_buffer_store_b16((uint16_t)kSentinel16, old, off, 0, 0);
      }
    }
    if (MT == 1) {
      // (units of 64 cycles; a poll that comes back incomplete costs a whole one: B 32 / 16 / 8 with 2: 2.36 / 1.99 / 1.50 us a step, with 6:
      // 2.37 / 1.94 / 1.45, with 8: 2.40 / 1.91 / 1.47, with 12: 2.33 / 1.93 / 1.56)
      __builtin_amdgcn_s_sleep(RT == 4 ? 6 : (RT == 8 ? 8 : 12));
      if (nt < p.T) request(nt, 0);
    }
    const long long row0 = rowbase + mt * 16 + 4 * wave;
    __builtin_amdgcn_raw_buffer_store_b16(hbits, descriptor(reinterpret_cast<uint16_t *>(p.h_out) + (long long)t * BH + row0 * H + (long long)head * dh + a0, 0xFFFFFF00u), h_off[mt], 0, 0);
    if constexpr (COEF != 0) {
      if (row0 < rend) {  // (576 floats per 4 rows, head and workgroup)
        const long long set = (long long)p.NH * p.G * 576;
        store_coefficients(p.coef_out + ((long long)t * ((p.B + 3) >> 2) + (row0 >> 2)) * set + ((long long)head * p.G + member) * 576,
                           lane, kept, st[mt].y, kept_c, kept_n, __builtin_amdgcn_rcpf(1.0f + __expf(raw[1])));
      }
    }
    fetch(t + D / MT, mt, wxq[u], flq[u]);  // iteration it + D, into the slot of this one
    XS_PTICK(5);
  };
  auto round = [&](auto first_c, int t0) {  // D iterations
    iteration(std::integral_constant<int, 0>{}, first_c, t0);
    if (t0 * MT + 1 < NIT) iteration(std::integral_constant<int, 1>{}, first_c, t0 + 1 / MT);
    if (t0 * MT + 2 < NIT) iteration(std::integral_constant<int, 2>{}, first_c, t0 + 2 / MT);
    if (t0 * MT + 3 < NIT) iteration(std::integral_constant<int, 3>{}, first_c, t0 + 3 / MT);
  };
  round(std::true_type{}, 0);
  for (int t0 = D / MT; t0 < p.T; t0 += D / MT) round(std::false_type{}, t0);
#ifdef XS_PROFILE
  if (lane == 0 && member == 0 && gi == 0) {
    long long *dst = reinterpret_cast<long long *>(p.wg_xcc + kStampWord) + wave * 8;
    for (int i = 0; i < 8; ++i) dst[i] = prof[i];
  }
#endif
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");

  // ---- final state; NaN all over this workgroup's outputs when a bounded wait ran out anywhere in the call
  const bool poisoned = __hip_atomic_load(&p.status->aborted, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
  if (poisoned) report_abort(p.abort_host);
#pragma unroll
  for (int mt = 0; mt < MT; ++mt) {
    const int brow = rowbase + mt * 16 + pb;
    if (unit_ok && brow < rend) {
      const long long o = (long long)brow * H + col;
      if (poisoned) st[mt] = CellState{kPoison, kPoison, kPoison, kPoison};
      p.s_out[o] = st[mt].y; p.s_out[BH + o] = st[mt].c; p.s_out[2 * BH + o] = st[mt].n; p.s_out[3 * BH + o] = st[mt].m;
      if (poisoned)
        for (int t = 0; t < p.T; ++t) reinterpret_cast<uint16_t *>(p.h_out)[(long long)t * BH + o] = (uint16_t)0x7FC0u;
    }
  }
  if (lane == 0 && max_spins) atomicMax(&p.status->max_spins, max_spins);
}

}  // namespace
