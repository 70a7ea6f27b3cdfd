// The reverse pass for the head dims that no compute unit holds alone: float32 beyond head dim 64 (up to 512), bf16 beyond
// 128 (up to 1024), from the coefficients that the training forward left.  Included by slstm_hip.hip only, behind
// slstm_local_kernel.h.
//
// slstm_bwd_split_kernel gives a compute unit 64 output units, so that float32 at head dim 256 has 128 KiB of R per wave
// set and 64 to 128 MFMAs per wave and step, and head dims beyond 512 (256 in float32) do not fit the registers at all;
// they ran one launch per step, with R read from memory every step.  Here a head is spread like in the forward: workgroup
// `member` owns 16 CT output units of a tile of RT = 4, 8 or 16 batch rows: SIXTEEN with four compute waves (CT 1), or in
// bf16 32 with eight (CT 2), which keeps a head of 1024 on one XCD and halves what a larger batch polls.  Per step:
//   - the lanes that own an element (row, unit) add up the waves' partial sums of what reached its y from the step
//     behind, form the step's gradient and publish the four gate deltas in the group's slot of an exchange ring, in the order
//     in which a look's lanes take them (unit_bwd_word; K is ordered (unit, gate));
//   - wave w polls the deltas of a quarter (CT 2: an eighth) of the members straight into MFMA operand registers (a word is
//     data or the "not written yet" pattern; the publisher re-arms its words of two steps ago, as in the forward's ring),
//     multiplies them by its share of R transposed and leaves its partial sums in LDS (two sets of tiles, one barrier a step).
// float32 multiplies with v_mfma_f32_4x4x1 (4 column groups x 4 pieces of K, see slstm_local_kernel.h), one pass per four
// rows; bf16 with v_mfma_f32_16x16x32, the batch rows spread over the 16 MFMA rows (RT 4: rows 0, 4, 8, 12).
// A feeder wave (CT 2: the compute waves between them) brings the steps' coefficients, d_h and reset flags to LDS in
// bursts of several steps: a compute unit returns its loads in the order they were issued, so a miss to memory holds up
// the polls behind it, and in bursts that happens once in unit_bwd_burst steps.  The members of a group sit on one XCD and
// publish with plain stores.  Waits are bounded; one that runs out sets the call's abort word and d_s0 becomes NaN.
//
// Bound by the chain of a step (publish, poll, MFMA, barrier: about 1 us); us a step at NH heads x head dim, batch, the
// forward's coefficients included, against the walk and the reverse kernel before: float32 4x256 B16 1.5 (9.0), bf16
// 4x192 B16 1.0, 4x512 B8 1.3, 4x512 B64 3.5, 4x1024 B16 3.8 (18.0).  Polls whose lanes are all rows that are there (row tiles
// of 4 and 8 rows in bf16: below), us a training call before -> after: 4x1024 B16 T512 3609 -> 2997 (the reverse pass 3.8 -> 2.6 a
// step), 8x384 B8 T300 785 -> 660, 4x256 B6 T300 601 -> 557, 4x512 B16 T256 815 -> 763.
#pragma once

namespace {

struct UnitBwdParams {
  const float *coef;         // [T][ceil(B/4)][NH][members][576]: what slstm_local_kernel describes
  const void *d_h;           // element (t, b, ..) at t d_h_st + b d_h_sb, in the type of the operands
  long long d_h_sb, d_h_st;
  const float *d_s_final;    // [4,B,H] or null
  const void *r;             // [NH,4 dh,dh]
  int r_bf16;
  const unsigned char *reset;
  long long reset_sb;
  void *d_wx;
  long long d_wx_sb, d_wx_st;
  float *d_s0;
  char *xch;                 // exchange ring [kBwdRing][groups of the launch][slot]: unit_bwd_slot_members() x RT rows x 16 CT units x 4 gates
  unsigned int *abort_word, *placement;
  unsigned int *abort_host;  // a pinned host word that a wait that ran out is reported in, or null
  long long spin_limit;
  int cut;
  float clip;
  int B, T, NH, dh;
  int G, W;                  // members of a group (at most 32: they sit on one XCD); the head's 16 units of coefficients
  int b0, bend, head0, NHL, NBT;  // rows and heads of this launch, row tiles per head
};

constexpr int unit_bwd_threads(int ct) { return ct == 1 ? 320 : 512; }  // 4 compute waves and a feeder wave; 8 waves that do both
constexpr int unit_part_stride(int ct) { return 16 * ct + 4; }          // floats between the rows of a partial tile
constexpr int unit_bwd_burst(int rt, int ct) { return rt * ct <= 4 ? 8 : (rt * ct <= 16 ? 4 : 2); }
constexpr int unit_bwd_slot(int rt, int ct, bool bf16) { return rt / 4 * ct * 2304 + rt * 16 * ct * (bf16 ? 2 : 4) + rt * 4; }
constexpr int unit_bwd_lds_bytes(int rt, int ct, bool bf16) {
  return 2 * 4 * ct * rt * unit_part_stride(ct) * 4 + 2 * unit_bwd_burst(rt, ct) * unit_bwd_slot(rt, ct, bf16);
}

// A slot of the exchange ring: pieces of 1 KiB, each what ONE load of a look brings, lane after lane.  (With the words as [member][row]
// [unit][gate] the lanes of a load lay 256 bytes apart, and a compute unit's address path, which takes a line a cycle, was what a
// step waited for: float32 at 8 x 512, 10 rows, looks of 10,200 of 14,600 cycles, 6,300 now.  us a training call, that order -> this one: bf16
// 4 x 1024 B 16 T 512 2,724 -> 2,585, 4 x 768 B 20 T 384 3,046 -> 2,295, 3 x 768 B 200 T 52 3,149 -> 2,418, float32 8 x 512 B 10 T 384 4,264 -> 3,561,
// 3 x 256 B 4 T 130 381 -> 327, 4 x 96 B 6 T 250 459 -> 434, of these two 128 and 64 cycles a step by the second chain of MFMAs.)  bf16: a piece of K is 8 units = an MFMA's 32
// inputs, PK = 16 / RT of them share a load: lane (unit pair q, row x PK + piece % PK), 16 bytes.  float32: 16 units of a set of
// four rows: lane (unit / 4, unit % 4, row), 16 bytes.
__host__ __device__ constexpr int unit_bwd_slot_members(int members, int rt, int ct, bool bf16) {
  return bf16 && rt * ct == 4 ? members + (members & 1) : members;  // (a load brings two members there: an odd last one has an empty neighbour)
}
template <bool BF16, int RT, int CT>
__device__ __forceinline__ int unit_bwd_word(int member, int row, int pu) {  // where the deltas of (row, unit pu of a member) lie in a slot
  if constexpr (BF16) {
    constexpr int PK = 16 / RT;
    const int piece = member * 2 * CT + (pu >> 3);
    return piece / PK * 1024 + (((pu >> 1) & 3) * 16 + row * PK + piece % PK) * 16 + (pu & 1) * 8;
  } else {
    return (member * (RT / 4) + (row >> 2)) * 1024 + (pu * 4 + (row & 3)) * 16;
  }
}

// s_sleep units (64 cycles each) in front of a wave's first look at the step's deltas: of the waves that have just published,
// and of the others.  A look that comes back incomplete costs its whole round trip.  Head dim 1024 in row tiles of 8 rows has
// the longest step (us a training call; B 16 x T 512 x 4 heads: (2, 8) 3006, (2, 12) 2924, (4, 12) 2917, (6, 16) 2881, (9, 16) 2883,
// (6, 20) 2905, (9, 24) 2933; other batches, lengths and head dims that run in this form, (2, 8) / (4, 12) / (6, 16) / (9, 24): B 16 T 128 872 / 857 /
// 847 / 862, B 9 T 300 1630 / 1593 / 1563 / 1597, 4 heads of 768 B 16 T 512 2506 / 2476 / 2455 / 2542); the others lose with more than (2, 8):
// 4 heads of 256, 6 rows, T 300 (2, 8) 558, (4, 10) 570, (6, 16) 597.
constexpr int unit_bwd_sleep(int rt, int ct, int gq, bool published) { return rt == 8 && ct == 2 && gq == 4 ? (published ? 6 : 16) : (published ? 2 : 8); }

// Whether a wave's own publication has to have reached the L2 before it looks, and a look that came back incomplete clears the compute
// unit's vector cache.  A look that is under way while a store of the same compute unit goes through the same lines can leave
// the old ones there, and looks that follow find those again: measured in row tiles of 16 rows at head dims beyond 512 (16 loads a
// look), where such a wave went on until its 256th look read the abort word, 420 us (1,740 with that read every 1,024th, 60
// every 32nd), in one of some hundred steps.  us a backward call of 128 steps, without / with both (the wait alone prevents it, the
// clearing alone ends it with the next look): 4 heads of 1024 B 32 1452-1911 / 977-1000, B 128 5463-8569 / 3580-3640, 8 of 640 B 12
// 4889-9293 / 700-720.  No other form showed it, and with both they gain nothing.
constexpr bool unit_bwd_settles(bool bf16, int gq, int rt) { return bf16 && gq == 4 && rt == 16; }

template <bool BF16, int GQ, int RT, int CT, bool DWX16>  // GQ: members of a wave's share of K (rounded up)
__global__ __launch_bounds__(unit_bwd_threads(CT)) void slstm_bwd_unit_kernel(UnitBwdParams p) {
  static_assert(RT == 4 || (RT == 16 && BF16 == (CT == 2)) || (RT == 8 && CT == 2), "row tiles of 4, 8 (bf16) or 16 rows");
  static_assert(CT == 1 || (CT == 2 && BF16), "32 units per workgroup: bf16");
  typedef typename std::conditional<BF16, uint16_t, float>::type elem_t;
  constexpr int ESZ = BF16 ? 2 : 4;
  constexpr int NW = 4 * CT;                  // compute waves
  constexpr int UW = 16 * CT;                 // units of a member
  constexpr int MB = RT * UW * 4 * ESZ;       // bytes a member publishes a step
  constexpr int SETS = RT / 4;
  constexpr int BL = unit_bwd_burst(RT, CT), SLOTB = unit_bwd_slot(RT, CT, BF16);
  constexpr int PSTRIDE = unit_part_stride(CT), PWAVE = RT * PSTRIDE;
  constexpr int COEFS = SETS * CT * 2304;     // bytes of a step's coefficients: [set of 4 rows][16 units][576 floats]
  constexpr int NLD = BF16 ? 2 * CT * GQ : GQ;  // 16-byte pieces of deltas a lane polls per step (float32: per set of four rows)
  // bf16, row tiles of fewer than 16 rows: PK MFMA rows per batch row, each of which takes another piece, so that a load has
  // no lane without a row; NPL loads for the NLD pieces
  constexpr int PK = BF16 ? 16 / RT : 1, NPL = NLD / PK;
  static_assert(NLD % PK == 0, "whole loads");
  constexpr int BATCH = NPL < 16 ? NPL : 16;  // ... in one go
  constexpr int NPASS = BF16 ? 1 : SETS;
  extern __shared__ __attribute__((aligned(1024))) unsigned char unit_lds[];
  float *const part = reinterpret_cast<float *>(unit_lds);          // [2][NW waves][RT][PSTRIDE]
  unsigned char *const feed = unit_lds + 2 * NW * PWAVE * 4;

  // ---- role of the workgroup
  const int wg = blockIdx.x, local = wg >> 3, place = local / p.G;
  const int member = local - place * p.G, gi = place * 8 + (wg & 7);
  const int ngroups = p.NHL * p.NBT;
  if (gi >= ngroups) return;
  const int head = p.head0 + gi / p.NBT, row0 = p.b0 + (gi % p.NBT) * RT;
  const int tid = threadIdx.x, lane = tid & 63, wave = (int)uniform((uint32_t)(tid >> 6));
  const int q = lane >> 4, r16 = lane & 15;
  const int dh = p.dh, H = p.NH * dh, a0 = member * UW;
  const long long BH = (long long)p.B * H;
  if (tid == 0) atomicOr(p.placement + gi, 1u << (__builtin_amdgcn_s_getreg(20 | (3 << 11)) & 0xFu));  // XCC_ID, bits [3:0]
  const int ntiles4 = (p.B + 3) >> 2;
  const long long coef_set = (long long)p.NH * p.W * 576, coef_step = (long long)ntiles4 * coef_set;

  // ---- feeding: burst k (steps k BL ...) into half k & 1 of the ring.  It has landed in front of barrier A(k BL - 2),
  //      behind which the compute waves read its first step; the next burst is asked for behind that barrier (the last
  //      step of the burst before has been read in front of it).  `f` of `nf` waves takes every nf-th load.
  const uint32_t feed_lds = (uint32_t)(unsigned long long)((__attribute__((address_space(3))) unsigned char *)feed);
  const int rows_there = p.bend - row0 < RT ? p.bend - row0 : RT;
  constexpr int LPR = CT * ESZ;  // lanes per row of d_h: the member's units in pieces of 16 bytes
  constexpr int DROWS = 64 / LPR < RT ? 64 / LPR : RT;  // rows of d_h per load
  const unsigned long long fb = reinterpret_cast<unsigned long long>(p.reset ? p.reset + (long long)row0 * p.reset_sb : reinterpret_cast<const unsigned char *>(p.coef));
  const u32x4_t frs = {uniform((uint32_t)fb), uniform((uint32_t)(fb >> 32) & 0xFFFFu), p.reset ? 0x7FFFFFFFu : 0u, 0x00020000u};
  const uint32_t fvo = (uint32_t)((lane < rows_there ? lane : 0) * p.reset_sb);
  auto request = [&](int k, int f, int nf) {
    int turn = 0;
    for (int i = 0; i < BL; ++i) {
      const int n = k * BL + i;
      if (n >= p.T) break;
      const int t = p.T - 1 - n;
      const uint32_t slot = feed_lds + (uint32_t)((k & 1) * BL + i) * SLOTB;
#pragma unroll
      for (int sc = 0; sc < SETS * CT; ++sc) {
        if (turn++ % nf != f) continue;
        const int s = sc / CT, m16 = member * CT + sc % CT;
        if ((row0 >> 2) + s >= ntiles4 || m16 >= p.W) continue;
        const unsigned long long cb = reinterpret_cast<unsigned long long>(p.coef + t * coef_step + ((row0 >> 2) + s) * coef_set + ((long long)head * p.W + m16) * 576);
        const u32x4_t crs = {uniform((uint32_t)cb), uniform((uint32_t)(cb >> 32) & 0xFFFFu), 2304u, 0x00020000u};
        bwd_fetch_to_lds_b128(crs, uniform(slot + sc * 2304), (uint32_t)lane * 16u);
        bwd_fetch_to_lds_b128(crs, uniform(slot + sc * 2304 + 1024), 1024u + (uint32_t)lane * 16u);
        if (lane < 16) bwd_fetch_to_lds_b128(crs, uniform(slot + sc * 2304 + 2048), 2048u + (uint32_t)lane * 16u);
      }
      if (turn++ % nf != f) continue;
      const unsigned long long db = reinterpret_cast<unsigned long long>(reinterpret_cast<const elem_t *>(p.d_h) + (long long)t * p.d_h_st + (long long)row0 * p.d_h_sb + head * dh + a0);
      const u32x4_t drs = {uniform((uint32_t)db), uniform((uint32_t)(db >> 32) & 0xFFFFu), 0x7FFFFFFFu, 0x00020000u};
#pragma unroll
      for (int r = 0; r < RT; r += DROWS) {
        const int dr = r + lane / LPR, drow = dr < rows_there ? dr : 0;
        // (a member that the head dim ends inside: the pieces behind the head's units are not fetched)
        if (lane < DROWS * LPR && a0 + (lane % LPR) * (16 / ESZ) < dh)
          bwd_fetch_to_lds_b128(drs, uniform(slot + COEFS + r * UW * ESZ), (uint32_t)(drow * p.d_h_sb * ESZ + (lane % LPR) * 16));
      }
      if (lane < RT) bwd_fetch_to_lds_u8(frs, uniform(slot + COEFS + RT * UW * ESZ), fvo + (uint32_t)t);
    }
  };
  if (CT == 1 && wave == NW) {  // the feeder wave
    request(0, 0, 1);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    request(1, 0, 1);
    lds_barrier();  // P
    for (int m = 0; m < p.T; ++m) {
      const bool turn = (m + 2) % BL == 0;
      if (turn) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();  // A(m)
      if (turn) request((m + 2) / BL + 1, 0, 1);
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    return;
  }

  // ---- R transposed: this wave's share of K for the workgroup's columns (units past the head: past the end of the descriptor)
  uint4 rb[BF16 ? NLD : 1][CT];
  float rf[BF16 ? 1 : 16 * GQ];
  const int u_first = wave * GQ * UW;
  auto load_r = [&](auto rbits) {
    constexpr bool RBITS = decltype(rbits)::value;
    constexpr int RSZ = RBITS ? 2 : 4;
    const long long head_elems = 4ll * dh * dh;
    const __amdgpu_buffer_rsrc_t rr = __builtin_amdgcn_make_buffer_rsrc(
        const_cast<char *>(reinterpret_cast<const char *>(p.r)) + head * head_elems * RSZ, 0, (int)(head_elems * RSZ), 0x00020000);
    auto at = [&](int u, int g, int d) -> float {
      const int o = (u < dh && d < dh) ? ((g * dh + u) * dh + d) * RSZ : 0x7FFFFFF0;
      if constexpr (RBITS) return bf16_bits_to_float((uint16_t)__builtin_amdgcn_raw_buffer_load_b16(rr, o, 0, 0));
      else return __uint_as_float(__builtin_amdgcn_raw_buffer_load_b32(rr, o, 0, 0));
    };
#pragma unroll
    for (int c = 0; c < (BF16 ? NLD : GQ); ++c) {
      if constexpr (BF16) {
#pragma unroll
        for (int ct = 0; ct < CT; ++ct) {
          const int u = u_first + c * 8 + 2 * q, d = a0 + 16 * ct + r16;
          rb[c][ct] = uint4{pack_bf16x2(at(u, 0, d), at(u, 1, d)), pack_bf16x2(at(u, 2, d), at(u, 3, d)),
                            pack_bf16x2(at(u + 1, 0, d), at(u + 1, 1, d)), pack_bf16x2(at(u + 1, 2, d), at(u + 1, 3, d))};
        }
      } else {
#pragma unroll
        for (int pc = 0; pc < 4; ++pc)
#pragma unroll
          for (int g = 0; g < 4; ++g) rf[16 * c + 4 * pc + g] = at(u_first + c * 16 + 4 * q + pc, g, a0 + r16);
      }
      if (c % 4 == 3) asm volatile("" ::: "memory");  // (some chunks' loads at a time: all in flight would take registers the loop needs)
    }
  };
  if (p.r_bf16) load_r(std::true_type{});
  else load_r(std::false_type{});
  // ---- the lane's element: the first SETS CT waves form gradients: 16 units each of a set of four rows, row q, unit r16
  const bool grad_wave = wave < SETS * CT;
  const int set = grad_wave ? wave / CT : 0, prow = 4 * set + q, pu = 16 * (wave % CT) + r16;
  const int row = row0 + prow, a = a0 + pu;
  const bool mine = grad_wave && row < p.bend && a < dh;
  const long long so = (long long)(row < p.B ? row : p.B - 1) * H + head * dh + (a < dh ? a : dh - 1);
  float dy = 0.0f, dc = 0.0f, dn = 0.0f;
  if (mine && p.d_s_final) { dy = p.d_s_final[so]; dc = p.d_s_final[BH + so]; dn = p.d_s_final[2 * BH + so]; }
  const long long wo = (long long)(row < p.B ? row : p.B - 1) * p.d_wx_sb + head * dh + (a < dh ? a : dh - 1);

  const int xslot = unit_bwd_slot_members(p.G, RT, CT, BF16) * MB;
  char *const ring = p.xch + (long long)gi * xslot;
  const long long ring_stride = (long long)ngroups * xslot;
  const int pub = unit_bwd_word<BF16, RT, CT>(member, prow, pu);
  // poll: bf16: load i: pieces PK i, + 1, ... of the wave's share, MFMA row r16 holds piece r16 % PK of batch row r16 / PK; float32: piece c of
  // set s: member wave GQ + c, unit 4 q + r16 / 4 of row r16 % 4.  Members past the last one lie past the end of the descriptor: zeros
  const int vo = wave * GQ * MB + lane * 16;
  if (BF16 && unit_bwd_slot_members(p.G, RT, CT, BF16) != p.G && member == p.G - 1 && grad_wave) {
    // (the empty neighbour's words are polled like the others: zeros)
#pragma unroll
    for (int i = 0; i < kBwdRing; ++i) *reinterpret_cast<unsigned long long *>(ring + i * ring_stride + unit_bwd_word<BF16, RT, CT>(p.G, prow, pu)) = 0ull;
  }

  f32x4 cA{0, 0, 0, 0}, cB{0, 0, 0, 0};
  float cC = 0.0f, dht = 0.0f;
  bool start = false;
  auto read_inputs = [&](int n) {
    const unsigned char *slot = feed + ((n / BL & 1) * BL + n % BL) * SLOTB;
    const float *cs = reinterpret_cast<const float *>(slot + (grad_wave ? wave : 0) * 2304);
    cA = *reinterpret_cast<const f32x4 *>(cs + 4 * lane);
    cB = *reinterpret_cast<const f32x4 *>(cs + 256 + 4 * lane);
    cC = cs[512 + lane];
    const elem_t d = reinterpret_cast<const elem_t *>(slot + COEFS)[prow * UW + pu];
    if constexpr (BF16) dht = bf16_bits_to_float(d);
    else dht = d;
    start = (reinterpret_cast<const uint32_t *>(slot + COEFS + RT * UW * ESZ)[prow] & 0xFFu) != 0u;
  };
  auto add_up = [&](int n) {
    const float *t = part + (n & 1) * (NW * PWAVE) + prow * PSTRIDE + pu;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < NW; ++w) sum += t[w * PWAVE];
    return sum;
  };
  bool gave_up = false, after = false;
  if constexpr (CT == 2) {
    request(0, wave, NW);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    request(1, wave, NW);
  }
  lds_barrier();  // P
  if (grad_wave) read_inputs(0);
  for (int n = 0; n < p.T; ++n) {
    const int t = p.T - 1 - n;
    if (grad_wave) {
      if (n > 0) dy = (p.cut || after) ? 0.0f : add_up(n - 1);
      const float dyt = dht + bwd_recurrent_dy(dy, p.clip, n == 0);
      const float dct = dc + dyt * cA[0], dnt = dn - dyt * cA[1];
      float delta[4] = {cA[2] * dct + cA[3] * dnt, cB[0] * dct + cB[1] * dnt, cB[2] * dct, cB[3] * dyt};
      dc = start ? 0.0f : cC * dct;  // (a row that starts a document at t took nothing from the step before)
      dn = start ? 0.0f : cC * dnt;
      after = start;
      if (!mine) delta[0] = delta[1] = delta[2] = delta[3] = 0.0f;
      if (!p.cut) {
        char *const now = ring + (n % kBwdRing) * ring_stride + pub, *const old = ring + ((n + kBwdRing - 2) % kBwdRing) * ring_stride + pub;
        unsigned long long w0, w1 = 0ull;
        if constexpr (BF16) {  // (a half of all ones, which only a NaN can give, becomes 0xFFFE, a NaN as well)
          const u16x2_t lo = __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, pack_bf16x2(delta[0], delta[1])), u16x2_t{0xFFFE, 0xFFFE});
          const u16x2_t hi = __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, pack_bf16x2(delta[2], delta[3])), u16x2_t{0xFFFE, 0xFFFE});
          w0 = (unsigned long long)__builtin_bit_cast(uint32_t, lo) | ((unsigned long long)__builtin_bit_cast(uint32_t, hi) << 32);
        } else {
          uint32_t v[4];
#pragma unroll
          for (int g = 0; g < 4; ++g) v[g] = __float_as_uint(delta[g]) == kSentinel32 ? 0x7FC00000u : __float_as_uint(delta[g]);
          w0 = (unsigned long long)v[0] | ((unsigned long long)v[1] << 32);
          w1 = (unsigned long long)v[2] | ((unsigned long long)v[3] << 32);
        }
        if constexpr (BF16) {
          *reinterpret_cast<unsigned long long *>(now) = w0;
          *reinterpret_cast<unsigned long long *>(old) = ~0ull;
        } else {
          *reinterpret_cast<uint4 *>(now) = uint4{(uint32_t)w0, (uint32_t)(w0 >> 32), (uint32_t)w1, (uint32_t)(w1 >> 32)};
          *reinterpret_cast<uint4 *>(old) = uint4{kSentinel32, kSentinel32, kSentinel32, kSentinel32};
        }
      }
      if constexpr (unit_bwd_settles(BF16, GQ, RT)) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (mine) {
        const long long o = wo + (long long)t * p.d_wx_st;
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          if constexpr (DWX16) reinterpret_cast<uint16_t *>(p.d_wx)[o + (long long)g * H] = (uint16_t)(pack_bf16x2(delta[g], 0.0f) & 0xFFFFu);
          else reinterpret_cast<float *>(p.d_wx)[o + (long long)g * H] = delta[g];
        }
      }
      if (n + 1 < p.T) read_inputs(n + 1);
      if (!p.cut) __builtin_amdgcn_s_sleep(unit_bwd_sleep(RT, CT, GQ, true));
    } else {
      if (!p.cut) __builtin_amdgcn_s_sleep(unit_bwd_sleep(RT, CT, GQ, false));
    }
    if (!p.cut) {
      const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(ring + (n % kBwdRing) * ring_stride, 0, xslot, 0x00020000);
      float *const tiles = part + (n & 1) * (NW * PWAVE) + wave * PWAVE;
#pragma unroll
      for (int ps = 0; ps < NPASS; ++ps) {
        // bf16: a chain per column tile and MFMA row of a batch row (RT 16: four chains, CT 2: two per column tile)
        constexpr int CH = PK == 1 ? 4 / CT : PK;
        // (float32: two, a v_mfma_f32_4x4x1 behind one that it adds to issues after 12 cycles instead of 8)
        f32x4 acc[BF16 ? CT * CH : 2];
#pragma unroll
        for (int i = 0; i < (BF16 ? CT * CH : 2); ++i) acc[i] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
        for (int b0 = 0; b0 < NPL; b0 += BATCH) {
          uint4 areg[BATCH];
          long long spins = 0;
          for (;;) {
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
              const int off = BF16 ? (b0 + i) * 1024 : (b0 + i) * MB + ps * 1024;
              areg[i] = __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(rs, vo + off, 0, 16));
            }
            uint32_t mark = 0u;
#pragma unroll
            for (int i = 0; i < BATCH; ++i) mark = mark_join<BF16>(mark, chunk_mark<BF16>(areg[i]));
            if ((__builtin_amdgcn_ballot_w64(mark_has_sentinel<BF16>(mark)) == 0ull && p.spin_limit >= 0) || gave_up) break;
            if constexpr (unit_bwd_settles(BF16, GQ, RT)) asm volatile("buffer_inv sc0" ::: "memory");
            if (++spins > p.spin_limit || ((spins & 255) == 0 && __hip_atomic_load(p.abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
              __hip_atomic_store(p.abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
              gave_up = true;
            }
          }
          if constexpr (BF16) {
#pragma unroll
            for (int i = 0; i < BATCH; ++i)
#pragma unroll
              for (int j = 0; j < PK; ++j)
#pragma unroll
                for (int ct = 0; ct < CT; ++ct) {
                  const int piece = (b0 + i) * PK + j;
                  if (piece >= NLD) continue;
                  f32x4 &c = acc[ct * CH + (PK == 1 ? i % CH : j)];
                  c = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, areg[i]), __builtin_bit_cast(bf16x8, rb[piece][ct]), c, 0, 0, 0);
                }
          } else {
#pragma unroll
            for (int i = 0; i < BATCH; ++i) {
              const float dv[4] = {__uint_as_float(areg[i].x), __uint_as_float(areg[i].y), __uint_as_float(areg[i].z), __uint_as_float(areg[i].w)};
              const float *const rr = rf + 16 * (b0 + i);
#pragma unroll
              for (int g = 0; g < 4; ++g) {
                acc[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(dv[g], rr[g], acc[0], 2, 0, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(dv[g], rr[4 + g], acc[1], 2, 1, 0);
                acc[0] = __builtin_amdgcn_mfma_f32_4x4x1f32(dv[g], rr[8 + g], acc[0], 2, 2, 0);
                acc[1] = __builtin_amdgcn_mfma_f32_4x4x1f32(dv[g], rr[12 + g], acc[1], 2, 3, 0);
              }
            }
          }
        }
        if constexpr (BF16) {
          // lane group q holds MFMA rows 4 q .. 4 q + 3: batch rows (4 q + i) / PK, the sums of chain j in row j of the PK
#pragma unroll
          for (int ct = 0; ct < CT; ++ct)
#pragma unroll
            for (int i = 0; i < 4; i += PK) {
              float sum = acc[ct * CH][i];
              if constexpr (PK == 1) {
                if constexpr (CH == 4) sum = (sum + acc[1][i]) + (acc[2][i] + acc[3][i]);
                else sum += acc[ct * CH + 1][i];
              } else {
#pragma unroll
                for (int j = 1; j < PK; ++j) sum += acc[ct * CH + j][i + j];
              }
              tiles[(4 * q + i) / PK * PSTRIDE + 16 * ct + r16] = sum;
            }
        } else {
          float x0 = acc[0][0] + acc[1][0], x1 = acc[0][1] + acc[1][1], x2 = acc[0][2] + acc[1][2], x3 = acc[0][3] + acc[1][3];
          transpose_lane_groups(x0, x1, x2, x3);
          tiles[(4 * ps + q) * PSTRIDE + r16] = ((x0 + x1) + x2) + x3;
        }
      }
    }
    if constexpr (CT == 2) {
      const bool turn = (n + 2) % BL == 0;
      if (turn) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      lds_barrier();  // A(n)
      if (turn) request((n + 2) / BL + 1, wave, NW);
    } else {
      lds_barrier();  // A(n)
    }
  }
  if constexpr (CT == 2) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // ---- the gradient of the initial state (the stabiliser's part is zero by the rule; NaN when a wait ran out)
  if (grad_wave) {
    const unsigned int seen = __hip_atomic_load(p.placement + gi, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    const bool mixed = bwd_exchange_torn(p.G, p.cut != 0, seen);
    if (mixed && tid == 0) __hip_atomic_store(p.abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
    dy = (p.cut || after) ? 0.0f : add_up(p.T - 1);
    const bool poisoned = mixed || __hip_atomic_load(p.abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
    if (poisoned && p.abort_host && lane == 0) __hip_atomic_store(p.abort_host, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    if (mine) {
      p.d_s0[so] = poisoned ? kPoison : dy;
      p.d_s0[BH + so] = poisoned ? kPoison : dc;
      p.d_s0[2 * BH + so] = poisoned ? kPoison : dn;
      p.d_s0[3 * BH + so] = 0.0f;
    }
  }
}

}  // namespace
