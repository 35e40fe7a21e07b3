// gemm_dd.h -- bf16 products whose two operands both move by LDS-DMA
// (included by gemm_fast.hip inside its namespace, after the loaders).
//
// Every wave issues its share of both operands' DMA and computes a wave tile.
// A ring of NS TR-deep stages: stage s + NS is loaded into the slot of stage s
// once every wave has read it.
//
// A wave issues in order, so a burst of LDS reads or DMA instructions ahead of
// the MFMAs idles the matrix core while the burst issues.  A stage is two half
// stages of 32; a half runs its MFMAs from fragments read during the half
// before, and every LDS read of the next half's fragments and every DMA
// instruction of a later stage has a fixed place between two MFMAs.  With
// bursts a 192 x 128 stage took 0.72 us, spread out 0.385 us; its MFMAs alone
// take 0.38 us.
//
// For the same reason a DMA instruction in the loop is the load and little
// else: lane offsets that hold the operand's edges are set up once, one select
// cuts the reduction's partial stage, and stages past the last one load with
// num_records 0.

// f(0), f(1), ... f(N - 1) with compile-time arguments
template <class F, int... I>
CONCORD_DEV void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>()), ...);
}
template <int N, class F>
CONCORD_DEV void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>());
}
#define CONCORD_INLINE_LAMBDA __attribute__((always_inline))

// LDS byte address -> pointer
CONCORD_DEV const lds_char* lds_at(uint32_t a) { return (const lds_char*)(uintptr_t)0 + a; }

// an LDS read address with a constant part: the instruction's 16-bit offset
// holds constants below 64 KB, a second register serves the rest
struct FarBase {
  uint32_t lo, hi;
  CONCORD_DEV void init(uint32_t a) {
    lo = a;
    hi = a + 65536u;
    pin(lo);
    pin(hi);
  }
  CONCORD_DEV const lds_char* at(uint32_t o) const { return lds_at(o >= 65536u ? hi : lo) + (o & 65535u); }
};

// dma16 to LDS address base + OFF (the s_nop: M0's wait state, as there)
template <int OFF>
CONCORD_DEV void dma16_at(i32x4 rsrc, uint32_t voff, uint32_t soff, uint32_t base) {
  asm volatile("s_add_u32 m0, %3, %4\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, %2 offen lds"
               :
               : "v"(voff), "s"(rsrc), "s"(soff), "s"(base), "n"(OFF)
               : "memory", "m0", "scc");
}

// operand [rows][r], r contiguous (x, dy, a row-major weight): RowsDma's tile
// of swizzled 128-byte rows, one ds_read_b128 per fragment
template <int ROWS, int WT, int NW>
struct DdRows {
  static constexpr int TILE = ROWS * 128, NF = WT / 16, PER = ROWS / 8 / NW;
  static_assert(PER * 8 * NW == ROWS, "rows split evenly over the waves");
  uint32_t voff[PER];   // lane offset of instruction q; kOOB past the last row
  i32x4 rs;
  uint32_t ring, dst;
  FarBase base[2];      // half kk
  int32_t kc[2];        // reduction offset of the lane's chunk, q even / odd
  // src: the operand at the tile's first row; woff: the wave's first row
  CONCORD_DEV void init(const uint16_t* src, int64_t ld, int64_t left, int64_t R, int wave, int lane, int woff,
                        uint32_t ring_) {
    ring = ring_;
    dst = uni(ring + (uint32_t)(wave * PER * 1024));
    const uint64_t a = (uint64_t)(uintptr_t)src;
    rs = i32x4{(int32_t)(uint32_t)a, (int32_t)(uint32_t)((a >> 32) & 0xFFFF), (int32_t)nrec(((left - 1) * ld + R) * 2),
               0x00020000};
    for (int e = 0; e < 4; ++e) rs[e] = __builtin_amdgcn_readfirstlane(rs[e]);
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int r = (wave * PER + q) * 8 + lane / 8;
      const int c = (lane % 8) ^ ((r >> 1) & 7);
      kc[q & 1] = c * 8;
      voff[q] = r < left ? (uint32_t)((r * ld + c * 8) * 2) : kOOB;
    }
    if (PER == 1) kc[1] = kc[0];
#pragma unroll
    for (int kk = 0; kk < 2; ++kk)
      base[kk].init(ring + (uint32_t)((woff + (lane & 15)) * 128 + (((kk * 4 + (lane >> 4)) ^ ((lane & 14) >> 1)) * 16)));
  }
  CONCORD_DEV uint32_t soff(int64_t r0) const { return (uint32_t)(r0 * 2); }
  // instruction Q of a stage with rem columns, into slot SLOT
  template <int Q, int SLOT> CONCORD_DEV void issue(uint32_t so, i32x4 r, int rem) const {
    dma16_at<SLOT * TILE + Q * 1024>(r, kc[Q & 1] < rem ? voff[Q] : kOOB, so, dst);
  }
  CONCORD_DEV bf16x8 frag(int slot, int x, int kk) const {
    const lds_char* q = base[kk].at((uint32_t)(slot * TILE + x * 2048));
    return __builtin_bit_cast(bf16x8, *(const __attribute__((address_space(3))) i32x4*)q);
  }
};

// operand [r][cols] (a weight read by its reduction): TrDma's row-major tile,
// two transpose reads per fragment
template <int COLS, int WT, int NW>
struct DdCols {
  static constexpr int ROWB = COLS * 2, RPI = 1024 / ROWB;   // rows per wave instruction
  static constexpr int TILE = TR * ROWB, NF = WT / 16, PER = TR / RPI / NW;
  static_assert(PER * RPI * NW == TR, "rows split evenly over the waves");
  uint32_t voff[PER];   // lane offset of instruction q; kOOB past the last column
  i32x4 rs;
  uint32_t ring, dst, ld2;
  int32_t row;   // the lane's row of instruction 0
  FarBase fb[NF];
  // src: the operand at the tile's first column; woff: the wave's first column
  CONCORD_DEV void init(const uint16_t* src, int64_t ld, int64_t left, int64_t R, int wave, int lane, int woff,
                        uint32_t ring_) {
    ring = ring_;
    dst = uni(ring + (uint32_t)(wave * PER * 1024));
    row = wave * PER * RPI + lane / (ROWB / 16);
    ld2 = (uint32_t)(ld * 2);
    const uint64_t a = (uint64_t)(uintptr_t)src;
    // (left is a multiple of 8, or the operand is padded to one)
    const int64_t bytes = ((R - 1) * ld + (left < COLS ? (left + 7) / 8 * 8 : COLS)) * 2;
    rs = i32x4{(int32_t)(uint32_t)a, (int32_t)(uint32_t)((a >> 32) & 0xFFFF), (int32_t)nrec(bytes), 0x00020000};
    for (int e = 0; e < 4; ++e) rs[e] = __builtin_amdgcn_readfirstlane(rs[e]);
#pragma unroll
    for (int q = 0; q < PER; ++q) {
      const int r = row + q * RPI, c = (lane % (ROWB / 16)) ^ (trf(r) << 1);
      voff[q] = c * 8 < left ? (uint32_t)((r * ld + c * 8) * 2) : kOOB;
    }
    const int p = lane & 15, gq = lane >> 4;
    const uint32_t fsw = (uint32_t)(((p >> 2) | ((gq & 1) << 2)) * 32);
    const uint32_t lbase = (uint32_t)((8 * gq + (p >> 2)) * ROWB + 8 * (p & 3));
#pragma unroll
    for (int x = 0; x < NF; ++x) fb[x].init(ring + lbase + ((uint32_t)(((woff >> 4) + x) * 32) ^ fsw));
  }
  CONCORD_DEV uint32_t soff(int64_t r0) const { return (uint32_t)(r0 * ld2); }
  // instruction Q of a stage with rem rows, into slot SLOT
  template <int Q, int SLOT> CONCORD_DEV void issue(uint32_t so, i32x4 r, int rem) const {
    dma16_at<SLOT * TILE + Q * 1024>(r, row < rem - Q * RPI ? voff[Q] : kOOB, so, dst);
  }
  CONCORD_DEV bf16x8 frag(int slot, int x, int kk) const {
    const uint32_t o = (uint32_t)(slot * TILE + kk * 32 * ROWB);
    const v4i16 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)fb[x].at(o));
    const v4i16 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_v4i16*)fb[x].at(o + 4 * ROWB));
    return __builtin_bit_cast(bf16x8, __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7));
  }
};

// places of one half stage's reads between its NI x NJ MFMAs (row x outer).
// The B fragments of both halves live at once; so do the A fragments where
// the accumulators leave room (256 VGPRs), else the first NI - 1 are refilled
// in place, each after the last MFMA of its row.
template <int NI, int NJ>
struct DdPlan {
  static constexpr int NM = NI * NJ, NR = NI + NJ;
  static constexpr bool FULL = NM * 4 + 8 * NR <= 208;
  static constexpr int NIP = FULL ? 0 : NI - 1;
  static constexpr int aset(int h, int x) { return x < NIP ? 0 : h; }
  static constexpr int pos_b(int y) { return FULL ? (y * NM * 3) / (NR * 4) : 2 * y; }
  static constexpr int pos_a(int x) {
    if (FULL) return ((NJ + x) * NM * 3) / (NR * 4);
    return x < NIP ? (x + 1) * NJ + 2 : 2 * NJ + 1;
  }
};

// half H of a stage: its MFMAs; the next half's fragments from slot SN, half
// kk = H ^ 1; the ND DMA instructions dma(0), ... dma(ND - 1)
template <int H, int SN, int ND, int NI, int NJ, class SA, class SB, class RD>
CONCORD_DEV void dd_half(f32x4 (&acc)[NI][NJ], bf16x8 (&fa)[2][NI], bf16x8 (&fb)[2][NJ], const SA& a, const SB& b,
                         RD&& dma) {
  typedef DdPlan<NI, NJ> P;
  static_for<P::NM>([&](auto mc) CONCORD_INLINE_LAMBDA {
    constexpr int m = decltype(mc)::value, x = m / NJ, y = m % NJ;
    static_for<NI>([&](auto xc) CONCORD_INLINE_LAMBDA {
      constexpr int r = decltype(xc)::value;
      if constexpr (P::pos_a(r) == m) fa[P::aset(H ^ 1, r)][r] = a.frag(SN, r, H ^ 1);
    });
    static_for<NJ>([&](auto yc) CONCORD_INLINE_LAMBDA {
      constexpr int r = decltype(yc)::value;
      if constexpr (P::pos_b(r) == m) fb[H ^ 1][r] = b.frag(SN, r, H ^ 1);
    });
    constexpr int d0 = (m * ND) / P::NM, d1 = ((m + 1) * ND) / P::NM;
    static_for<d1 - d0>([&](auto dc) CONCORD_INLINE_LAMBDA { dma(std::integral_constant<int, d0 + decltype(dc)::value>()); });
    // D^T: MFMA rows = j (B tile), columns = i (A tile)
    acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[H][y], fa[P::aset(H, x)][x], acc[x][y], 0, 0, 0);
    __builtin_amdgcn_sched_barrier(0);
  });
}

// the main loop over the reduction range [r_begin, r_end)
template <int NS, int NI, int NJ, class SA, class SB>
CONCORD_DEV void dd_loop(f32x4 (&acc)[NI][NJ], const SA& sa, const SB& sb, int64_t r_begin, int64_t r_end) {
  constexpr int PERT = SA::PER + SB::PER;
  typedef DdPlan<NI, NJ> P;
  const int nst = r_end > r_begin ? (int)((r_end - r_begin + TR - 1) / TR) : 0;
  const int last = nst > 0 ? (int)(r_end - r_begin - (int64_t)(nst - 1) * TR) : 0;
  struct Stage {
    i32x4 ra, rb;
    uint32_t ao, bo;
    int rem;
  };
  auto at = [&](int s) CONCORD_INLINE_LAMBDA {
    Stage t{sa.rs, sb.rs, 0u, 0u, s == nst - 1 ? last : TR};
    const bool live = s < nst;
    const int64_t r0 = r_begin + (int64_t)(live ? s : 0) * TR;
    t.ra[2] = live ? t.ra[2] : 0;
    t.rb[2] = live ? t.rb[2] : 0;
    t.ao = sa.soff(r0);
    t.bo = sb.soff(r0);
    return t;
  };
  auto issue = [&](const Stage& t, auto slc, auto dc) CONCORD_INLINE_LAMBDA {
    constexpr int d = decltype(dc)::value, SL = decltype(slc)::value;
    if constexpr (d < SA::PER) sa.template issue<d, SL>(t.ao, t.ra, t.rem);
    else sb.template issue<d - SA::PER, SL>(t.bo, t.rb, t.rem);
  };
  static_for<NS>([&](auto sc) CONCORD_INLINE_LAMBDA {
    const Stage t = at(decltype(sc)::value);
    static_for<PERT>([&](auto dc) CONCORD_INLINE_LAMBDA { issue(t, sc, dc); });
  });
#pragma unroll
  for (int x = 0; x < NI; ++x)
#pragma unroll
    for (int y = 0; y < NJ; ++y) acc[x][y] = f32x4{0.f, 0.f, 0.f, 0.f};
  __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 1) * PERT));   // own stage-0 DMA landed
  lds_barrier();
  bf16x8 fa[2][NI], fb[2][NJ];
  static_for<NI>([&](auto xc) CONCORD_INLINE_LAMBDA { fa[0][decltype(xc)::value] = sa.frag(0, decltype(xc)::value, 0); });
  static_for<NJ>([&](auto yc) CONCORD_INLINE_LAMBDA { fb[0][decltype(yc)::value] = sb.frag(0, decltype(yc)::value, 0); });
  // the barrier of stage s stands between its halves: its slot has been read
  // (every fragment of its second half is in registers) and stage s + 1 has
  // landed.  After the last stage the reads take a slot no MFMA uses.
  auto stage = [&](int s, auto slc) CONCORD_INLINE_LAMBDA {
    constexpr int SL = decltype(slc)::value;
    dd_half<0, SL, 0, NI, NJ>(acc, fa, fb, sa, sb, [](auto) {});
    __builtin_amdgcn_s_waitcnt(vmcnt_imm((NS - 2) * PERT));   // own stage s + 1 DMA landed
    lds_barrier();
    const Stage t = at(s + NS);
    dd_half<1, (SL + 1) % NS, PERT, NI, NJ>(acc, fa, fb, sa, sb,
                                            [&](auto dc) CONCORD_INLINE_LAMBDA { issue(t, slc, dc); });
  };
  int s = 0;
  for (; s + NS <= nst; s += NS)
    static_for<NS>([&](auto sc) CONCORD_INLINE_LAMBDA { stage(s + decltype(sc)::value, sc); });
  static_for<NS - 1>([&](auto sc) CONCORD_INLINE_LAMBDA {
    if (s + decltype(sc)::value < nst) stage(s + decltype(sc)::value, sc);
  });
  // no DMA may still be writing LDS when the ring is reused or the block ends
  __builtin_amdgcn_s_waitcnt(vmcnt_imm(0));
}

// FWD_BF16 (b rows) and DGRAD_BF16 (b columns).  Bound by the MFMAs and, with
// every CU busy, by the clock they leave (a 256 x 256 stage takes 1.17 us on 20
// CUs, 1.3 us on 256), then by a block's 5 - 8 us outside the loop.  Against
// kernels whose producer waves copied operands through registers or read the
// weight tile 8 bytes at a time: dgrad 4096 x 1280 x 10240 128.7 -> 101.7 us,
// 8192 x 640 x 5120 67.5 -> 51.3, 4096 x 1280 x 1280 21.8 -> 18.0; forward
// 4096 x 10240 x 1280 113.6 -> 109.1, 4096 x 1280 x 1280 22.0 -> 18.5,
// 2048 x 1280 x 5120 40.4 -> 35.0.
//
// CARRY (8 waves): workgroups from dg_blocks on run the v-hat reduction of the
// split WGRAD rw issued just before on the stream, on the CUs the tiles leave
// idle, two reduction blocks at a time.
template <int MODE, int BI, int BJ, int WI, int WJ, int NS, bool CARRY = false>
__global__ __launch_bounds__(64 * WI * WJ, 1) void gemm_dd_kernel(GemmArgs g, GemmArgs rw, int dg_blocks) {
  constexpr int NW = WI * WJ, WTI = BI / WI, WTJ = BJ / WJ, NI = WTI / 16, NJ = WTJ / 16;
  constexpr bool FWD = MODE == MODE_FWD_BF16;
  typedef DdRows<BI, WTI, NW> SA;
  typedef typename std::conditional<FWD, DdRows<BJ, WTJ, NW>, DdCols<BJ, WTJ, NW>>::type SB;
  constexpr int RING = NS * (SA::TILE + SB::TILE), OUT = BI * (BJ + 8) * 2;
  __shared__ __attribute__((aligned(1024))) char lds[RING > OUT ? RING : OUT];
  if constexpr (CARRY) {
    if ((int)blockIdx.x >= dg_blocks) {
      ReduceVh<256, 128, 4, 2>::run_pairs(rw, (int)blockIdx.x - dg_blocks, (int)gridDim.x - dg_blocks,
                                          reinterpret_cast<float*>(lds));
      return;
    }
  }
  const int t = threadIdx.x, lane = t & 63, wave = __builtin_amdgcn_readfirstlane(t >> 6);
  int split, bi, bj, slot;
  gemm_tile_of<BI, BJ>(g, blockIdx.x, split, bi, bj, slot);
  const int64_t i0 = (int64_t)bi * BI, j0 = (int64_t)bj * BJ;
  const int64_t r_begin = (int64_t)split * g.r_split, r_end = min(g.R, r_begin + g.r_split);
  const int wi = wave / WJ, wj = wave % WJ;
  const uint16_t* gb = reinterpret_cast<const uint16_t*>(g.b);
  SA sa;
  SB sb;
  const uint32_t ring = lds_addr(lds);
  sa.init(g.a + i0 * g.lda, g.lda, g.I - i0, g.R, wave, lane, wi * WTI, ring);
  sb.init(FWD ? gb + j0 * g.ldb : gb + j0, g.ldb, g.J - j0, g.R, wave, lane, wj * WTJ, ring + NS * SA::TILE);
  f32x4 acc[NI][NJ];
  dd_loop<NS, NI, NJ>(acc, sa, sb, r_begin, r_end);
  epilogue<MODE, NI, NJ, BI, BJ, NW>(g, acc, i0, j0, wi * WTI, wj * WTJ, split, slot, wave, t, 64 * NW,
                                     reinterpret_cast<uint16_t*>(lds));
}
