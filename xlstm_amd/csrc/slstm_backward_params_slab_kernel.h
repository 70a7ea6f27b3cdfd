// Gradients of the recurrent matrix and the bias from gate deltas in bf16 (what training in bf16 leaves): the product that
// slstm_backward_params_kernel.h describes, d R = delta^T . y_{t-1} per head.  Included by slstm_hip.hip only, behind that header.
//
// The kernel there takes 128 rows of the result per workgroup, brings its operands through registers and gathers MFMA
// fragments with 16-bit LDS reads.  Its time went on waiting: two chunks of 24 KiB in flight per compute unit, each for 0.26 us of
// MFMA, every one through registers (transposing reads alone, in the same structure: no change, 0.76 ms at head dim 1024).
// Here a workgroup (eight waves) owns 256 rows m x NT columns n, which halves what is read per product, and
//   - chunks of 32 k go straight from memory to a ring of LDS stages (buffer_load .. lds, 16 bytes a lane; three of 32
//     KiB in flight at NT 256, five below), one barrier per chunk, waits counted by hand: every wave issues the same number of loads
//     for every chunk, those past the slice's end with an empty descriptor (zeros, no traffic);
//   - a lane gets its 8 k of a fragment by two transposing reads (ds_read_b64_tr_b16: 4 k x 16 columns per lane group).
//     A load fills LDS in lane order, so instead of padding the 32-byte pieces of a row are permuted by its number: lane i asks
//     memory for the piece that belongs at its place, and the four rows that 16 lanes read at once hit different banks;
//   - rows that start a document (the forward's operand was zero) are masked out of the y fragments, by flags that travel
//     with the chunk; the bias sums are two more MFMAs per wave against a fragment of ones.
//
// Bound: at NT 256 a chunk is 1,024 cycles of MFMA per SIMD, about as many of LDS (128 KiB read, 32 written), and 32 KiB from the L2 per compute unit.
// Measured against the kernel it replaces: B 16 x T 512 x 4 heads of 1024 762 -> 357 us (0.77 PFLOP/s), B 16 x T 2048 x 4
// heads of 256 229 -> 137 us (335 MB of operands, 0.50 PFLOP/s); with chunks stepped by additions instead of 90 scalar instructions of products,
// and asked for behind the MFMAs (alone, in a loop): 371 -> 355, 131 -> 125 us.  Of the 355 the requests with the barriers alone take 220, MFMAs and LDS
// reads without memory 309: the eight waves of a compute unit do both in step, so the two add up where they should overlap.
#pragma once

namespace {

constexpr int kSlabMT = 256;
constexpr int param_slab_stages(int nt) { return nt == 256 ? 4 : 6; }
constexpr int param_slab_stage_bytes(int nt) { return kParamKC * (kSlabMT + nt) * 2 + kParamKC * 4; }
constexpr int param_slab_lds_bytes(int nt) { return param_slab_stages(nt) * param_slab_stage_bytes(nt); }

typedef short s16x4_t __attribute__((ext_vector_type(4)));
// ds_read_b64_tr_b16: lane l of a group of 16 asks for 4 elements of row l / 4 and gets the 4 rows' elements of column l
__device__ __forceinline__ uint2 lds_read_tr_b16(const unsigned char *src) {
  typedef __attribute__((address_space(3))) s16x4_t *lds_ptr;
  return __builtin_bit_cast(uint2, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_ptr)(const_cast<unsigned char *>(src))));
}

template <int NT>  // columns of the result per workgroup: 64, 128 or 256; dhp is a multiple of it
__global__ __launch_bounds__(512) void slstm_bwd_param_slab_kernel(BwdParamParams p) {
  constexpr int KC = kParamKC, S = param_slab_stages(NT), STAGE = param_slab_stage_bytes(NT);
  constexpr int WN = NT / 64, WM = 8 / WN, MTILES = kSlabMT / WM / 16;
  constexpr int ROWA = kSlabMT * 2, ROWB = NT * 2, BOFF = KC * ROWA, FOFF = BOFF + KC * ROWB;
  constexpr int NB = NT == 256 ? 2 : 1;    // loads of y per thread and chunk (NT 64: by half of each wave's lanes)
  constexpr int BLANES = NT == 64 ? 32 : 64, BPIECES = NT / 8;
  constexpr int LOADS = 2 + NB + 1;        // ... of a wave: deltas, y, flags
  extern __shared__ __attribute__((aligned(1024))) unsigned char slab_lds[];

  const int dh = p.dh, dhp = p.dhp, H = p.NH * dh;
  const int tiles_m = 4 * dhp / kSlabMT, tiles_n = dhp / NT, tiles = tiles_m * tiles_n;
  const int xcd = blockIdx.x & 7, slot = blockIdx.x >> 3;  // (a (head, K slice) group on one XCD: see slstm_bwd_param_kernel)
  const int group = (slot / tiles) * 8 + xcd, tile = slot % tiles;
  if (group >= p.NH * p.ksplit) return;
  const int head = group / p.ksplit, ks = group % p.ksplit;
  const int m0 = (tile / tiles_n) * kSlabMT, n0 = (tile % tiles_n) * NT;
  const int tid = threadIdx.x, lane = tid & 63, wave = (int)uniform((uint32_t)(tid >> 6)), q = lane >> 4, r16 = lane & 15;
  const int wm = wave / WN, wn = wave % WN;
  const long long BH = (long long)p.B * H;
  const long long nchunks = (long long)p.B * p.tchunks;
  const int c_lo = (int)(nchunks * ks / p.ksplit), c_hi = (int)(nchunks * (ks + 1) / p.ksplit);

  // the permutation of a row's 32-byte pieces (rows of 128 bytes: every other row starts at the same bank, and there are four pieces)
  auto swap_a = [](int k) { return (k & 3) | (((k >> 3) & 1) << 2); };
  auto swap_b = [](int k) { return NT == 64 ? ((k >> 1) & 1) | (((k >> 3) & 1) << 1) : (k & 3) | (((k >> 3) & 1) << 2); };
  // ---- what this thread brings of a chunk: 16-byte pieces, at place `tid` (+ 512) of the chunk's rows
  constexpr uint32_t kNone = 0x80000000u;  // past the end of every descriptor: zeros
  uint32_t a_off[2], b_off[NB];
  int a_row[2], b_row[NB];                 // the chunk's step
  long long a_col[2];                      // (element offsets, or -1: a unit that is not there)
  int b_col[NB];
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const int idx = tid + 512 * i, k = idx >> 5, dcol = m0 + ((idx & 31) ^ (swap_a(k) << 1)) * 8;
    a_row[i] = k;
    a_col[i] = dcol % dhp < dh ? (long long)(dcol / dhp) * H + (long long)head * dh + dcol % dhp : -1;
    a_off[i] = a_col[i] >= 0 ? (uint32_t)((k * p.d_wx_st + a_col[i]) * 2) : kNone;
  }
#pragma unroll
  for (int i = 0; i < NB; ++i) {
    const int idx = (NT == 64 ? wave * 32 + (lane & 31) : tid) + 512 * i, k = idx / BPIECES, yn = ((idx % BPIECES) ^ (swap_b(k) << 1)) * 8;
    b_row[i] = k;
    b_col[i] = n0 + yn < dh ? yn : -1;
    b_off[i] = b_col[i] >= 0 ? (uint32_t)((k * BH + yn) * 2) : kNone;
  }
  const uint32_t lds0 = (uint32_t)(unsigned long long)((__attribute__((address_space(3))) unsigned char *)slab_lds);
  // the next chunk to ask for: its place and what its descriptors cover, stepped with additions (nearly all chunks follow the last one in
  // their batch row)
  int f_left = c_hi - c_lo, f_b = c_lo / p.tchunks, f_t = c_lo % p.tchunks;
  uint32_t f_dst = lds0;
  const int tail = p.T - (p.tchunks - 1) * KC, bwidth = NT < dh - n0 ? NT : dh - n0;
  const uint32_t a_step = (uint32_t)(KC * p.d_wx_st * 2), b_step = (uint32_t)(KC * BH * 2);
  const uint32_t a_full = (uint32_t)(((KC - 1) * p.d_wx_st + 4ll * H) * 2), a_tail = (uint32_t)(((tail - 1) * p.d_wx_st + 4ll * H) * 2);
  const uint32_t b_full = (uint32_t)(((KC - 1) * BH + bwidth) * 2), b_tail = (uint32_t)(((tail - 1) * BH + bwidth) * 2);
  unsigned long long a_at = 0, b_at = 0, r_at = 0;
  auto row_start = [&](int t) {
    a_at = reinterpret_cast<unsigned long long>(p.d_wx) + ((long long)f_b * p.d_wx_sb + (long long)t * KC * p.d_wx_st) * 2;
    b_at = reinterpret_cast<unsigned long long>(p.h_out) + (((long long)t * KC - 1) * BH + (long long)f_b * H + (long long)head * dh + n0) * 2;
    r_at = p.reset ? reinterpret_cast<unsigned long long>(p.reset) + (long long)f_b * p.reset_sb + (long long)t * KC : 0;
  };
  if (f_left > 0) row_start(f_t);
  auto descriptor = [&](unsigned long long v, uint32_t bytes) { return u32x4_t{uniform((uint32_t)v), uniform((uint32_t)(v >> 32) & 0xFFFFu), uniform(bytes), 0x00020000u}; };
  auto request = [&]() {
    const bool there = f_left > 0, last = f_t == p.tchunks - 1;
    const u32x4_t ars = descriptor(a_at, there ? (last ? a_tail : a_full) : 0u);
#pragma unroll
    for (int i = 0; i < 2; ++i) bwd_fetch_to_lds_b128(ars, uniform(f_dst + (uint32_t)(wave * 1024 + 8192 * i)), a_off[i]);
    // y_{t-1}: step t's operand is row t - 1 of the outputs (in front of step 0: nothing, see below)
    const u32x4_t brs = descriptor(b_at, there ? (last ? b_tail : b_full) : 0u);
#pragma unroll
    for (int i = 0; i < NB; ++i)
      if (lane < BLANES)
        bwd_fetch_to_lds_b128(brs, uniform(f_dst + BOFF + (uint32_t)(wave * BLANES * 16 + 8192 * i)), f_t == 0 && b_row[i] == 0 ? kNone : b_off[i]);
    const u32x4_t frs = descriptor(r_at, p.reset && there ? (uint32_t)(last ? tail : KC) : 0u);
    if (lane < 4) bwd_fetch_to_lds_u8(frs, uniform(f_dst + FOFF + (uint32_t)(wave * 16)), (uint32_t)(4 * wave + lane));
    --f_left;
    a_at += a_step; b_at += b_step; r_at += KC;
    if (++f_t == p.tchunks) {
      f_t = 0; ++f_b;
      row_start(0);
    }
    f_dst = f_dst == lds0 + (S - 1) * STAGE ? lds0 : f_dst + STAGE;
  };

  // ---- fragments: lane (q, r16) takes k = 8 q .. 8 q + 7 of column r16 of a 16 x 16 tile
  const int kr = 8 * q + (r16 >> 2), c8 = (r16 & 3) * 8;
  int a_frag[MTILES], b_frag[4];
#pragma unroll
  for (int i = 0; i < MTILES; ++i) a_frag[i] = kr * ROWA + (((wm * MTILES + i) ^ swap_a(kr)) * 32) + c8;
#pragma unroll
  for (int j = 0; j < 4; ++j) b_frag[j] = BOFF + kr * ROWB + (((wn * 4 + j) ^ swap_b(kr)) * 32) + c8;
  const bool counts = n0 == 0;  // the bias sums: the first column tile's workgroups, two row tiles a wave
  int s_frag[2];
#pragma unroll
  for (int j = 0; j < 2; ++j) s_frag[j] = kr * ROWA + (((wm * MTILES + wn * 2 + j) ^ swap_a(kr)) * 32) + c8;
  f32x4 acc[MTILES][4], sums[2];
#pragma unroll
  for (int i = 0; i < MTILES; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  sums[0] = sums[1] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  auto gather = [&](const unsigned char *src, int row) {
    const uint2 lo = lds_read_tr_b16(src), hi = lds_read_tr_b16(src + 4 * row);
    return uint4{lo.x, lo.y, hi.x, hi.y};
  };
  auto compute = [&](int stage, bool flags, bool bias) {
    const unsigned char *const st = slab_lds + stage * STAGE;
    uint4 bf[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) bf[j] = gather(st + b_frag[j], ROWB);
    if (flags) {  // (a row that starts a document: the forward's operand was zero)
      const uint4 f0 = *reinterpret_cast<const uint4 *>(st + FOFF + q * 32), f1 = *reinterpret_cast<const uint4 *>(st + FOFF + q * 32 + 16);
      auto keep = [](uint32_t lo, uint32_t hi) { return ((lo & 0xFFu) ? 0u : 0xFFFFu) | ((hi & 0xFFu) ? 0u : 0xFFFF0000u); };
      const uint4 m{keep(f0.x, f0.y), keep(f0.z, f0.w), keep(f1.x, f1.y), keep(f1.z, f1.w)};
#pragma unroll
      for (int j = 0; j < 4; ++j) bf[j] = uint4{bf[j].x & m.x, bf[j].y & m.y, bf[j].z & m.z, bf[j].w & m.w};
    }
#pragma unroll
    for (int i = 0; i < MTILES; ++i) {
      const uint4 af = gather(st + a_frag[i], ROWA);
#pragma unroll
      for (int j = 0; j < 4; ++j)
        acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, af), __builtin_bit_cast(bf16x8, bf[j]), acc[i][j], 0, 0, 0);
    }
    if (bias) {
      const uint4 ones{0x3F803F80u, 0x3F803F80u, 0x3F803F80u, 0x3F803F80u};
#pragma unroll
      for (int j = 0; j < 2; ++j)
        sums[j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, gather(st + s_frag[j], ROWA)), __builtin_bit_cast(bf16x8, ones), sums[j], 0, 0, 0);
    }
  };

  const bool flags = p.reset != nullptr;
#pragma unroll
  for (int i = 0; i < S - 1; ++i) request();
  int stage = 0;
  for (int c = c_lo; c < c_hi; ++c) {
    asm volatile("s_waitcnt vmcnt(%0)" :: "n"((S - 2) * LOADS) : "memory");  // (this wave's part of chunk c has landed)
    lds_barrier();  // ... and everybody's; the stage of chunk c - 1 has been read
    compute(stage, flags, counts);
    request();      // chunk c + S - 1, into that stage, while the last MFMAs run (in front of them: 359 us where 355 now)
    if (++stage == S) stage = 0;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if (ks == 0 && p.s0) {  // what the initial state contributes: k = 32 batch rows, step 0's deltas against the y of s0
    for (int b0 = 0; b0 < p.B; b0 += KC) {
      lds_barrier();
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int b = b0 + a_row[i];
        uint4 v{0u, 0u, 0u, 0u};
        if (b < p.B && a_col[i] >= 0)
          v = *reinterpret_cast<const uint4 *>(reinterpret_cast<const uint16_t *>(reinterpret_cast<const void *>(p.d_wx)) + (long long)b * p.d_wx_sb + a_col[i]);
        *reinterpret_cast<uint4 *>(slab_lds + (tid + 512 * i) * 16) = v;
      }
#pragma unroll
      for (int i = 0; i < NB; ++i) {
        if (lane >= BLANES) continue;
        const int b = b0 + b_row[i];
        uint4 v{0u, 0u, 0u, 0u};
        if (b < p.B && b_col[i] >= 0 && !(p.reset && p.reset[(long long)b * p.reset_sb])) {
          const float *src = p.s0 + (long long)b * H + (long long)head * dh + n0 + b_col[i];
          const float4 lo = *reinterpret_cast<const float4 *>(src), hi = *reinterpret_cast<const float4 *>(src + 4);
          v = uint4{pack_bf16x2(lo.x, lo.y), pack_bf16x2(lo.z, lo.w), pack_bf16x2(hi.x, hi.y), pack_bf16x2(hi.z, hi.w)};
        }
        *reinterpret_cast<uint4 *>(slab_lds + BOFF + ((NT == 64 ? wave * 32 + lane : tid) + 512 * i) * 16) = v;
      }
      lds_barrier();
      compute(0, false, false);
    }
  }

  // ---- the slice's share: lane (q, r16) holds rows 4 q .. 4 q + 3, column r16 of every 16 x 16 tile
#pragma unroll
  for (int i = 0; i < MTILES; ++i)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int row = m0 + (wm * MTILES + i) * 16 + 4 * q + e;
      if (row % dhp >= dh) continue;
      float *const dst = p.d_r + ((long long)head * 4 * dh + (row / dhp) * dh + row % dhp) * dh + n0 + wn * 64 + r16;
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (n0 + wn * 64 + 16 * j + r16 < dh) atomicAdd(dst + 16 * j, acc[i][j][e]);
    }
  if (counts && r16 == 0) {
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int row = m0 + (wm * MTILES + wn * 2 + j) * 16 + 4 * q + e;
        if (row % dhp < dh) atomicAdd(p.d_bias + (long long)head * 4 * dh + (row / dhp) * dh + row % dhp, sums[j][e]);
      }
  }
}

}  // namespace
