// The reverse pass of the sLSTM backward for row tiles of 4 batch rows (bf16, head dims 64, 128, 256).  Included by
// slstm_hip.hip only (one translation unit), after slstm_backward_kernels.h, whose parameter block, exchange ring
// protocol, arm kernel and prefetching workgroups it shares.
//
// slstm_bwd_split_kernel walks 16 rows per workgroup: two elements per thread in the gradient of a step, 32 KiB of gate
// deltas per workgroup and poll round, partial tiles of 16 rows through LDS, two barriers.  A batch of few rows (16 at
// four heads, say) then keeps 16 compute units busy and the step is as long as its longest wave.  Here a workgroup
// owns 4 rows x UW units, and each of its waves has one role:
//   - UW / 8 matrix waves, each holding its share of K of the slice of R transposed in registers for the whole call: they poll
//     the group's deltas straight into MFMA operand registers, multiply and leave partial tiles of 4 rows in LDS;
//   - UW / 16 gradient waves, one element per lane: they add the partial tiles up, form the step's gradient and publish its deltas;
//   - feeder waves, which bring the steps' inputs and write d_wx.
// ONE barrier per step; words that are data or the all-ones pattern, the publisher re-arming its words of two steps ago, bounded waits.
//
// A step is the way round: barrier, sums and gradient, publication, the look that finds all of it, MFMAs, partial tiles, barrier.  What
// bounds it is that chain, so nothing that is not on it stands in a wave that is (with the gradient formed by waves that poll and
// multiply as well, their first look left 280 cycles after the others'), and the MFMAs, of which a tile of 4 rows leaves three quarters
// empty, are split over twice the workgroups (UW 32) where these fit: 128 of 16 cycles a step and workgroup at head dim 256 with UW 64.
// ms a training call at 4 heads of 256, one form of wave and UW 64 -> these roles and UW 64 -> UW 32: B 16 x T 1024 1.757 -> 1.751 -> 1.694, B 8 x T 512
// 0.904 -> 0.866 -> 0.816, 2 heads B 5 x T 600 1.010 -> 0.967 -> 0.910, 3 heads B 16 x T 400 0.766 -> 0.736 -> 0.720.  (Each pair with the
// prefetch of then; with its pace, its threads and the waits as they are now 1.567, 0.818, 0.909, 0.700.  Where the coefficients always are in
// the L2, B 16 x T 1024 takes 1.56.)
//
// K is ordered (unit of the head, gate): the four deltas of an element are 8 bytes and a thread publishes them with one store.  Matrix
// wave w multiplies KS k-steps (of 32 inputs, 8 units) of the head.  Batch row b takes the MFMA rows 4 b .. 4 b + 3, each with another of
// PK k-steps, so that no lane of a poll is a row that is not there; the sum of (row b, column n) over k-step j arrives in lane group b, lane n,
// element j.  A slot of the ring is pieces of PK k-steps, each what a load of a look brings, lane after lane; the units of a
// workgroup are UW / (8 PK) pieces in a row, which its gradient waves write in the same order.
#pragma once

namespace {

constexpr int kBwdQuadSlots = 8;
constexpr int kBwdQuadFeeders = 4;                 // feeder wave f brings the inputs of the steps n = f (mod 4)
constexpr int kBwdQuadDepth = 6;                   // steps the feeder waves request ahead
// Threads of a prefetching workgroup that do so, whatever a computing one has: what many waves touch at once stands in front of the
// polls and requests of the other compute units.  us of the reverse kernel with 64 / 128 / 192 / 256 / 512 / all (704 with 32 units a
// workgroup, 1,024 with 64) threads: 4 heads of 256, B 16 x T 2048 1,820 / 1,608 / 1,568 / 1,636 / 1,710 / 1,762, T 512, B 8 441 / 384 / 384 /
// 384 / 386 / 385, B 28 466 / 477 / 467 / 495 / 519 / 565, B 48 552 / 545 / 541 / 554 / 562 / 604, B 56 (no room for more than four per XCD)
// 622 / 617 / 615 / 613 / 613 / 617; 8 of 128, B 28 422 / 419 / 439 / 425 / 448 / 478.
constexpr int kBwdQuadPrefetchThreads = 192;
static_assert(kBwdQuadDepth >= 3 && kBwdQuadDepth <= kBwdQuadSlots && kBwdQuadDepth <= kBwdQuadFeeders + 2, "feeder depth");
// a slot of the feeder waves: the coefficients [4 rows][9][UW] in whole loads, d_h (4 rows in a landing zone of 1 KiB), the reset
// flags of the 4 rows as words (in a landing zone of 256 bytes)
constexpr int bwd_quad_coef_loads(int uw) { return (9 * uw + 63) / 64; }
constexpr int bwd_quad_slot(int uw) { return bwd_quad_coef_loads(uw) * 1024 + 1024 + 256; }
constexpr bool bwd_quad_drains(int uw) { return uw == 32; }  // a wave of its own writes d_wx (where one is left: a workgroup has 16)
constexpr int bwd_quad_threads(int uw) { return (uw / 8 + uw / 16 + kBwdQuadFeeders + bwd_quad_drains(uw)) * 64; }
constexpr int bwd_quad_part_stride(int uw) { return uw == 64 ? 68 : 48; }  // floats between the rows of a wave's partial tile (writes without bank conflicts)
constexpr int bwd_quad_tiles(int uw) { return 2 * (uw / 8) * 4 * bwd_quad_part_stride(uw) * 4; }
constexpr int bwd_quad_stash(int uw) { return 4 * uw * 16; }  // a step's deltas on their way to d_wx: four values per element
constexpr int bwd_quad_lds_bytes(int uw) {
  const int bytes = bwd_quad_tiles(uw) + kBwdQuadSlots * bwd_quad_slot(uw) + 2 * bwd_quad_stash(uw);
  return bytes < 84 * 1024 ? 84 * 1024 : bytes;  // (more than half of a compute unit's: no two workgroups share one)
}

// s_sleep units (64 cycles each) between the barrier and a matrix wave's first look at the step's deltas.  A look that comes back
// incomplete costs its whole round trip, and so does every cycle slept past the arrival.  (ms a training call at 4 heads of 256, B 16 x T 1024 /
// B 8 x T 512: 6 1.857 / 0.836, 7 1.746 / 0.835, 9 1.728 / 0.824, 11 1.745 / 0.837, 12 1.698 / 0.828 against 1.694 / 0.816 with 9, 14 1.714 / 0.860:
// several states of the kernel, each pair to be read by itself.  Raised priorities of the matrix or the gradient waves: no difference.)
constexpr int kBwdQuadSleep = 9;

// What a wave has asked for in front of its loop is there, and the compiler knows it (it reads this builtin, not a wait in inline assembly).  All
// roles are one function to it: left open, the loads of R at the head of the matrix waves were waited for in the loop of the feeder waves,
// where another use of the registers stands, that is, every step waited for the requests just made (64 units a workgroup).
// us of the reverse kernel at 4 heads of 256, T 512, B 25 / 32 / 48 / 64: 615 / 643 / 665 / 740 -> 550 / 580 / 607 / 668.
__device__ __forceinline__ void settle_loads() { __builtin_amdgcn_s_waitcnt(0x0F70); }  // vmcnt(0)

template <int S, int UW, bool DWX16 = false>  // dh = 64 S; UW units a workgroup; DWX16: d_wx takes the gate deltas rounded to bf16
__global__ __launch_bounds__(bwd_quad_threads(UW)) void slstm_bwd_quad_kernel(BwdSplitParams p) {
  constexpr int dh = S * 64;
  constexpr int M = dh / UW;                  // workgroups per group
  constexpr int K = 4 * dh;
  constexpr int NMW = UW / 8, NGW = UW / 16;  // matrix and gradient waves
  constexpr int KS = K / 32 / NMW;            // MFMA k-steps of a matrix wave
  constexpr int PK = KS < 4 ? KS : 4;         // ... of a load
  constexpr int LOADS = KS / PK;
  constexpr int CB = UW / 16;                 // column tiles of a workgroup
  constexpr int K8 = K / 8 / 32;              // k-steps of an eighth of K (the order of p.r_ts)
  constexpr int SLOT = 4 * K * 2;             // bytes of a group's slot
  constexpr int PSTRIDE = bwd_quad_part_stride(UW), PART = 4 * PSTRIDE;
  constexpr int FSLOT = bwd_quad_slot(UW), COEFZ = bwd_quad_coef_loads(UW) * 1024;
  constexpr int kPiece = 4 * 9 * 64 * 4;      // bytes of the coefficients of 64 units and 4 rows
  extern __shared__ __attribute__((aligned(16))) float part[];  // [2][NMW waves][4 rows][PSTRIDE], the feeder's slots, the stash
  const int H = p.NH * dh;
  const long long BH = (long long)p.B * H;
  const int ntiles = (p.B + 3) >> 2;
  const int ngroups = p.NH * ntiles;
  const int xcd = blockIdx.x & 7, local = blockIdx.x >> 3;
#ifdef XS_PROFILE
  const long long wg_start = wall_clock64();
#endif
  if (local >= p.main_locals) {
    if (threadIdx.x < kBwdQuadPrefetchThreads)  // (the others end here: a barrier waits for the waves that are left)
      bwd_tile_prefetch<true, S, 4, kBwdQuadDepth, kBwdQuadPrefetchThreads>(p, xcd, local - p.main_locals, (int)(gridDim.x >> 3) - p.main_locals);
    return;
  }
  const int group = (local / M) * 8 + xcd, member = local % M;
  if (group >= ngroups) return;
  const int head = group % p.NH;
  const int row0 = (group / p.NH) * 4;
  const int tid = threadIdx.x, wave = tid >> 6, lane = tid & 63, q = lane >> 4, r16 = lane & 15;
  char *const feed = reinterpret_cast<char *>(part + 2 * NMW * PART);
  // the deltas of the step before, for the drainer wave (or the feeder waves) to write to d_wx: [2][row][UW units][4 gates].  (Stores of the waves
  // that form the gradient stood in front of their look at the peers' deltas, which waits for their acknowledgement.)
  typedef typename std::conditional<DWX16, uint16_t, float>::type wx_t;
  wx_t *const stash = reinterpret_cast<wx_t *>(feed + kBwdQuadSlots * FSLOT);
  bwd_note_placement(p, group);
  // look_step[w]: 1 + the step of the call whose first look matrix wave w has issued (for the feeder waves, see there)
  __shared__ volatile int look_step[NMW];
  if (tid < NMW) look_step[tid] = 0;
  const int rows_there = p.B - row0 < 4 ? p.B - row0 : 4;
  constexpr bool DRAINS = bwd_quad_drains(UW);
  if (DRAINS && wave == NMW + NGW + kBwdQuadFeeders) {
    // ---- the drainer wave: the step's deltas to d_wx, and the group's progress.  (Nothing waits for its stores; from the feeder waves,
    //      whose waits for their loads were waits for these stores too, they held up the requests.)
    __syncthreads();  // P
    typedef wx_t pair_t __attribute__((ext_vector_type(2)));
    const int unit = 2 * (lane & 15), g = lane >> 4;
    for (int m = 0; m < p.T; ++m) {
      lds_barrier();  // A(m)
      if (member == 0 && lane == 0 && m + 1 < p.T) p.progress[group] = (unsigned int)(m + 1);
      const wx_t *const mine = stash + ((m & 1) * 4 * UW + unit) * 4 + g;
      wx_t *const to = reinterpret_cast<wx_t *>(p.d_wx) + row0 * p.d_wx_sb + (long long)(p.T - 1 - m) * p.d_wx_st + (long long)g * H + head * dh + member * UW + unit;
#pragma unroll
      for (int r = 0; r < 4; ++r)
        if (r < rows_there) *reinterpret_cast<pair_t *>(to + r * p.d_wx_sb) = pair_t{mine[r * UW * 4], mine[(r * UW + 1) * 4]};
    }
#ifdef XS_PROFILE
    __syncthreads();
#endif
    return;
  }
  if (wave >= NMW + NGW) {
    // ---- the feeder waves: the inputs of step n into slot n % 8, kBwdQuadDepth steps ahead, with loads that write LDS
    //      directly (no registers; their waits are written by hand)
    const uint32_t feed_lds = (uint32_t)(unsigned long long)((__attribute__((address_space(3))) unsigned char *)feed);
    const long long coef_piece0 = (((long long)(row0 >> 2) * p.NH + head) * S + member * UW / 64) * kPiece;  // + t * coef_step
    const long long coef_step = (long long)ntiles * p.NH * S * kPiece;
    const uint32_t dh_records = (uint32_t)(((long long)(rows_there - 1) * H + UW) * 2);
    const int dh_voff = (lane / (UW / 8)) * H * 2 + (lane % (UW / 8)) * 16;  // (rows 4 and up lie past the records: zeros into the landing zone)
    const unsigned long long fb = reinterpret_cast<unsigned long long>(p.reset ? p.reset + (long long)row0 * p.reset_sb : reinterpret_cast<const uint8_t *>(p.coef));
    const uint32_t flag_records = p.reset ? (uint32_t)((long long)(rows_there - 1) * p.reset_sb + p.T) : 0u;  // (no mask: every flag reads zero)
    const u32x4_t frs = {uniform((uint32_t)fb), uniform((uint32_t)(fb >> 32) & 0xFFFFu), uniform(flag_records), 0x00020000u};
    const uint32_t flag_lane = lane < rows_there ? (uint32_t)(lane * p.reset_sb) : 0x7FFFFF00u;
    auto request = [&](int n) {
      const int t = p.T - 1 - n;
      const unsigned long long cb = reinterpret_cast<unsigned long long>(p.coef) + (unsigned long long)(coef_piece0 + t * coef_step);
      const u32x4_t crs = {uniform((uint32_t)cb), uniform((uint32_t)(cb >> 32) & 0xFFFFu), (uint32_t)kPiece, 0x00020000u};
      const uint32_t slot = feed_lds + (n & (kBwdQuadSlots - 1)) * FSLOT;
#pragma unroll
      for (int k = 0; k < bwd_quad_coef_loads(UW); ++k) {
        const int i = k * 64 + lane;  // 16 bytes of run (row, coefficient) i / (UW / 4)
        const uint32_t off = UW == 64 ? (uint32_t)(i * 16)
                                      : (i < 9 * UW ? (uint32_t)(i / (UW / 4) * 256 + member * UW % 64 * 4 + i % (UW / 4) * 16) : 0x7FFFFF00u);
        bwd_fetch_to_lds_b128(crs, uniform(slot + k * 1024), off);
      }
      const unsigned long long db = reinterpret_cast<unsigned long long>(p.d_h) + (unsigned long long)((((long long)t * p.B + row0) * H + (long long)head * dh + member * UW) * 2);
      const u32x4_t drs = {uniform((uint32_t)db), uniform((uint32_t)(db >> 32) & 0xFFFFu), dh_records, 0x00020000u};
      bwd_fetch_to_lds_b128(drs, uniform(slot + COEFZ), (uint32_t)dh_voff);
      bwd_fetch_to_lds_u8(frs, uniform(slot + COEFZ + 1024), lane < rows_there ? flag_lane + (uint32_t)t : 0x7FFFFF00u);
    };
    // Feeder wave f owns the steps n = f (mod kBwdQuadFeeders): it asks for step n's inputs behind barrier A(n - depth)
    // and waits for them - for everything it has in flight - in front of barrier A(n - 2), behind which the gradient
    // waves read them; its next request goes out behind that barrier at the earliest (depth <= feeders + 2), so it never
    // has two requests in flight and no wait needs a count.  (One wave with several requests in flight and counted
    // waits, `s_waitcnt vmcnt(33)` for "all but the last three requests", waited a request's whole latency every step:
    // the wait counter of a wave has 6 bits, and these loads seem to weigh more than one each.)
    const int f = wave - (NMW + NGW);
#ifdef XS_PROFILE
    long long fprof[6] = {0, 0, 0, 0, 0, 0}, ftick = clock64();
#endif
    for (int n = f; n < kBwdQuadDepth && n < p.T; n += kBwdQuadFeeders) request(n);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (among them the inputs of steps 0 and 1)
    __syncthreads();           // P: the gradient waves read the inputs of steps 0 and 1 behind it
    for (int m = 0; m < p.T; ++m) {
      // in front of barrier A(m) the inputs of step m + 2 are in place: the gradient waves read them behind it
      if ((m + 2) % kBwdQuadFeeders == f) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#ifdef XS_PROFILE
      fprof[4] += clock64() - ftick;  // (the wait, if it was this wave's turn)
#endif
      lds_barrier();  // A(m)
      // (without a drainer wave) feeder wave f writes the step's deltas of row f, and the first the group's progress
      if (!DRAINS && member == 0 && f == 0 && lane == 0 && m + 1 < p.T) p.progress[group] = (unsigned int)(m + 1);
      if (!DRAINS && f < rows_there) {
        const int unit = lane % UW, gate0 = lane / UW;
        const long long wo = (long long)(row0 + f) * p.d_wx_sb + (long long)(p.T - 1 - m) * p.d_wx_st + (long long)head * dh + member * UW + unit;
        const wx_t *const mine = stash + (((m & 1) * 4 + f) * UW + unit) * 4 + gate0;
#pragma unroll
        for (int g = 0; g < 4; g += 64 / UW) reinterpret_cast<wx_t *>(p.d_wx)[wo + (long long)(g + gate0) * H] = mine[g];
      }
#ifdef XS_PROFILE
      fprof[5] += clock64() - ftick;  // (the step)
      ftick = clock64();
#endif
      const int n = m + kBwdQuadDepth;  // (into the slot of step n - 8, read in front of A(n - 9))
      if (n % kBwdQuadFeeders == f && n < p.T) {
        // The request goes out behind the matrix waves' looks at the next step's deltas: a compute unit returns its
        // loads in the order they were issued, and these take longer than a look.  (A bounded wait: nobody depends on it.  ms a training
        // call at B 16 x T 1024 x 4 heads of 256: 1.69; right behind the barrier 1.85, behind the looks' return 1.81 to 1.84; a third of the
        // loads behind each of three barriers 1.70.)
        if (p.cut == 0 && m + 1 < p.T) {
          for (int spin = 0; spin < 512; ++spin) {
            const int seen = lane < NMW ? look_step[lane] : 0x7FFFFFFF;
            if (__builtin_amdgcn_ballot_w64(seen < m + 2) == 0ull) break;
            __builtin_amdgcn_s_sleep(1);
          }
        }
#ifdef XS_PROFILE
        fprof[2] += clock64() - ftick;  // (the matrix waves' looks are out)
        if ((m & 63) >= 32 && (m & 63) < 36) {  // (measurement: how long a request takes; sampled, every wait below is in the way)
          const long long f0 = clock64();
          request(n);
          asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
          fprof[0] += clock64() - f0; fprof[1] += 1;
        } else
#endif
        request(n);
      }
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
#ifdef XS_PROFILE
    __syncthreads();  // (the gradient waves have cleared the m plane of d_s0)
    if (group == 0 && member == 0 && lane == 0 && f == 0 && p.B >= 4) {
      long long *out = reinterpret_cast<long long *>(p.d_s0 + 3 * BH + 3 * H);
      for (int i = 0; i < 6; ++i) out[i] = fprof[i];
    }
#endif
    return;
  }
  char *const ring = reinterpret_cast<char *>(p.xch) + (long long)group * SLOT;
  const long long ring_stride = (long long)ngroups * SLOT;
  const bool cut = p.cut != 0;
#ifdef XS_PROFILE
  // measurement build: when a wave passes fixed points of the loop, in cycles since it left the step's barrier, summed over the
  // steps; the first gradient wave and the first and last matrix wave of the first workgroup leave theirs in rows of the m plane of d_s0
  long long bprof[8] = {0, 0, 0, 0, 0, 0, 0, 0}, btick = clock64(), blook = 0;
#define XS_BTICK(i) do { const long long now_ = clock64(); bprof[i] += now_ - btick; if ((i) == 5) btick = now_; } while (0)
#else
#define XS_BTICK(i) do { } while (0)
#endif
  if (wave < NMW) {
    // ---- the matrix waves: this wave's share of the workgroup's slice of R transposed -> registers, once
    const int wave_u = (int)uniform((uint32_t)wave);
    uint4 bq[KS][CB];
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      const int kk = wave * KS + ks;  // k-step of the head
      const char *base = reinterpret_cast<const char *>(p.r_ts) +
                         (((((long long)(head * S + member * UW / 64) * 8 + kk / K8) * K8 + kk % K8) * 4 + member * UW % 64 / 16) * 64 << 4);
#pragma unroll
      for (int cb = 0; cb < CB; ++cb) bq[ks][cb] = *reinterpret_cast<const uint4 *>(base + ((cb * 64 + lane) << 4));
    }
    settle_loads();
    // MFMA row r16 holds k-step r16 % 4 (+ 4 a load) of batch row r16 / 4: a load brings PK k-steps, no lane of it is a row that
    // is not there (one k-step a load, its rows at MFMA rows 0, 4, 8, 12: 2.11 ms at B 16 x T 2048 x 4 heads of 256, 2.01 with this)
    const int poll_off = (r16 & 3) < PK ? ((q * 4 + (r16 >> 2)) * PK + (r16 & 3)) * 16 : 0x7FFFFF00;
    bool gave_up = false;
    __syncthreads();  // P
    for (int n = 0; n < p.T; ++n) {
      if (!cut) {
        __builtin_amdgcn_s_sleep(kBwdQuadSleep);
        XS_BTICK(2);
        u32x4_t a[LOADS];
        const __amdgpu_buffer_rsrc_t rs = __builtin_amdgcn_make_buffer_rsrc(ring + (n % kBwdRing) * ring_stride, 0, SLOT, 0x00020000);
        constexpr int kPastL1 = 16;  // (the load's scope bits: served by the L2)
        if (lane == 0) look_step[wave] = n + 1;
        // (two looks in flight half a round trip apart, so that an incomplete one is followed sooner: 0.15 to 0.4 ms slower,
        // as was every variant that asks more often)
        for (long long spins = 0;;) {
#ifdef XS_PROFILE
          blook = clock64() - btick;
#endif
          uint32_t mark = 0u;
#pragma unroll
          for (int i = 0; i < LOADS; ++i)
            a[i] = __builtin_bit_cast(u32x4_t, __builtin_amdgcn_raw_buffer_load_b128(rs, poll_off, (wave_u * LOADS + i) * PK * 256, kPastL1));
#pragma unroll
          for (int i = 0; i < LOADS; ++i) mark = mark_join<true>(mark, chunk_mark<true>(__builtin_bit_cast(uint4, a[i])));
          // (a negative spin limit is the host's way to make every wait run out at its first look: the error path, forced)
          if ((__builtin_amdgcn_ballot_w64(mark_has_sentinel<true>(mark)) == 0ull && p.spin_limit >= 0) || gave_up) break;
#ifdef XS_PROFILE
          bprof[6] += 1;
#endif
          if (++spins > p.spin_limit || ((spins & 255) == 0 && __hip_atomic_load(p.abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))) {
            __hip_atomic_store(p.abort_word, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // (the gradient waves read it behind the last barrier)
            gave_up = true;
          }
        }
#ifdef XS_PROFILE
        bprof[7] += blook;
#endif
        XS_BTICK(3);
        // ---- delta [4 rows x K share] . R^T [K share x UW]: the wave's partial result, to LDS.  Two sets of tiles, used in turn: the
        //      gradient waves have read those of step n in front of barrier A(n + 1), behind which they are written again.
        float *const tiles = part + (n & 1) * NMW * PART + wave * PART + q * PSTRIDE + r16;
#pragma unroll
        for (int cb = 0; cb < CB; ++cb) {
          f32x4 acc[PK];  // a chain per MFMA row of a batch row: its sums arrive in register j of lane group q
#pragma unroll
          for (int ks = 0; ks < KS; ++ks)
            acc[ks % PK] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a[ks / PK]), __builtin_bit_cast(bf16x8, bq[ks][cb]),
                                                                   ks < PK ? f32x4{0.0f, 0.0f, 0.0f, 0.0f} : acc[ks % PK], 0, 0, 0);
          float sum = acc[0][0];
#pragma unroll
          for (int j = 1; j < PK; ++j) sum += acc[j][j];
          tiles[cb * 16] = sum;
        }
      }
      XS_BTICK(4);
      lds_barrier();  // A(n)
      XS_BTICK(5);
    }
    bwd_placement_mixed(p, group, M);  // (thread 0 flags the call)
#ifdef XS_PROFILE
    __syncthreads();
    if (tid == 0 && member == 0) p.progress[group] = 0x40000000u + (unsigned int)(wall_clock64() - wg_start);  // (how long the group took, in 10 ns)
    if (group == 0 && member == 0 && lane == 0 && (wave == 0 || wave == NMW - 1) && p.B >= 4) {
      long long *out = reinterpret_cast<long long *>(p.d_s0 + 3 * BH + (wave == 0 ? 1 : 2) * H);
      for (int i = 0; i < 8; ++i) out[i] = bprof[i];
    }
#endif
    return;
  }
  // ---- the gradient waves: one element a lane, in the order of the ring's words: [piece][unit pair of 8][row][k-step of the piece][unit of the pair]
  const int e = (wave - NMW) * 64 + lane;
  const int prow = (e / (2 * PK)) & 3;
  const int pu = (e / (32 * PK) * PK + (e >> 1) % PK) * 8 + ((e / (8 * PK)) & 3) * 2 + (e & 1);
  const int row = row0 + prow;
  const bool there = row < p.B;
  const long long ecol = (long long)head * dh + member * UW + pu;
  float dy = 0.0f, dc = 0.0f, dn = 0.0f;
  if (there && p.d_s_final) {
    const long long o = (long long)row * H + ecol;
    dy = p.d_s_final[o]; dc = p.d_s_final[BH + o]; dn = p.d_s_final[2 * BH + o];
  }
  settle_loads();
  const int pub_off = member * (UW * 32) + e * 8;
  float c9[9], dht = 0.0f;
  bool restart = false, zero_dy = false;
  auto read_inputs = [&](int n) {  // the inputs of step n of the call, from the feeder's slot
    const char *slot = feed + (n & (kBwdQuadSlots - 1)) * FSLOT;
    const float *src = reinterpret_cast<const float *>(slot) + prow * (9 * UW) + pu;
#pragma unroll
    for (int j = 0; j < 9; ++j) c9[j] = src[j * UW];
    dht = __uint_as_float((uint32_t)*reinterpret_cast<const uint16_t *>(slot + COEFZ + prow * (UW * 2) + pu * 2) << 16);
    restart = *reinterpret_cast<const uint32_t *>(slot + COEFZ + 1024 + prow * 4) != 0u;
  };
  auto add_up = [&](int n) {  // what reaches y of the lane's element from step n of the call: the partial results, in the order of the waves
    const float *tiles = part + (n & 1) * NMW * PART + prow * PSTRIDE + pu;
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < NMW; ++w) sum += tiles[w * PART];
    return sum;
  };
  __syncthreads();  // P
  read_inputs(0);
  for (int n = 0; n < p.T; ++n) {
    if (n > 0) dy = (cut || zero_dy) ? 0.0f : add_up(n - 1);
#ifdef XS_PROFILE
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#endif
    XS_BTICK(0);
    // ---- the gradient of the step for the lane's element
    float delta[4] = {0.0f, 0.0f, 0.0f, 0.0f};
    if (there) {
      const float dyt = dht + bwd_recurrent_dy(dy, p.clip, n == 0);
      const float dct = dc + dyt * c9[0];
      const float dnt = dn - dyt * c9[1];
      delta[0] = c9[2] * dct + c9[3] * dnt;
      delta[1] = c9[4] * dct + c9[5] * dnt;
      delta[2] = c9[6] * dct;
      delta[3] = c9[7] * dyt;
      dc = restart ? 0.0f : c9[8] * dct;  // (a row that starts a document at t took nothing from the step before)
      dn = restart ? 0.0f : c9[8] * dnt;
    }
    zero_dy = restart;
    if (!cut) {
      // ---- publish (rows outside the batch: zeros), re-arm the words of two steps ago.  These waves do not poll, so they wait here until
      //      the L2 has what they re-armed a step ago: a peer that sees this publication may ask for those words next.  (Stores a step
      //      old; ms a training call at 4 heads of 256 before there was a wait / with it: B 16 x T 1024 1.694 / 1.687, B 8 x T 512 0.816 / 0.825.)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      // (the pattern stays unique: a half of all ones, which only a NaN can give, becomes 0xFFFE, a NaN as well)
      const u16x2_t lo = __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, pack_bf16x2(delta[0], delta[1])), u16x2_t{0xFFFE, 0xFFFE});
      const u16x2_t hi = __builtin_elementwise_min(__builtin_bit_cast(u16x2_t, pack_bf16x2(delta[2], delta[3])), u16x2_t{0xFFFE, 0xFFFE});
      // (plain stores: as stores of device scope, which the forward's kernels use, they measured 0.1 to 0.5 ms slower here)
      *reinterpret_cast<uint2 *>(ring + (n % kBwdRing) * ring_stride + pub_off) = uint2{__builtin_bit_cast(uint32_t, lo), __builtin_bit_cast(uint32_t, hi)};
      *reinterpret_cast<uint2 *>(ring + ((n + kBwdRing - 2) % kBwdRing) * ring_stride + pub_off) = uint2{0xFFFFFFFFu, 0xFFFFFFFFu};
    }
    XS_BTICK(1);
    // ---- while the deltas are on their way: their copies for d_wx, the next step's inputs
    wx_t *const copy = stash + (((n & 1) * 4 + prow) * UW + pu) * 4;
    if constexpr (DWX16) *reinterpret_cast<uint2 *>(copy) = uint2{pack_bf16x2(delta[0], delta[1]), pack_bf16x2(delta[2], delta[3])};
    else *reinterpret_cast<f32x4 *>(copy) = f32x4{delta[0], delta[1], delta[2], delta[3]};
    if (n + 1 < p.T) read_inputs(n + 1);
    XS_BTICK(4);
    lds_barrier();  // A(n)
    XS_BTICK(5);
  }
  // ---- gradient w.r.t. the initial state (the stabiliser's part is zero by the rule; NaN all over when a wait ran out)
  const bool mixed = bwd_placement_mixed(p, group, M);
  dy = (cut || zero_dy) ? 0.0f : add_up(p.T - 1);
  if (there) {
    const bool poisoned = mixed || __hip_atomic_load(p.abort_word, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) != 0u;
    const long long o = (long long)row * H + ecol;
    p.d_s0[o] = poisoned ? kPoison : dy;
    p.d_s0[BH + o] = poisoned ? kPoison : dc;
    p.d_s0[2 * BH + o] = poisoned ? kPoison : dn;
    p.d_s0[3 * BH + o] = 0.0f;
  }
#ifdef XS_PROFILE
  __syncthreads();
  if (group == 0 && member == 0 && lane == 0 && wave == NMW && p.B >= 4) {
    long long *out = reinterpret_cast<long long *>(p.d_s0 + 3 * BH);
    for (int i = 0; i < 8; ++i) out[i] = bprof[i];
  }
#endif
}

}  // namespace
