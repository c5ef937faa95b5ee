// Small-tile NT GEMM for gfx950: C[M,N] = A[M,K] . B[N,K]^T on output tiles
// from 16x16 to 256x128, for grids that 256x256 tiles cannot fill the chip
// with (decoding batches, short prompts, experts with few tokens).
//
// Every output element is accumulated by the 256x256 kernels' MFMA sequence
// (16x16 fragments, the same K order, the B fragment as the MFMA's first
// operand), so the results are bit-identical to theirs.
//
// K is walked in the same stages of 128 bytes per row.  A stage's TM + TN rows
// land in one slot of an LDS ring of NS slots by LDS-DMA, in units of 8 rows
// (1 KiB, one DMA of one wave), with the 16-byte chunks swizzled as in the
// 256x256 kernels (chunk c of row r at c ^ ((r >> 1) & 7)).  Iteration s of
// the loop
//   s_waitcnt vmcnt(DMAs of stages s+2 .. s+NS-1) lgkmcnt(0); s_barrier
//       -- stage s+1 landed for every wave; every wave has read stage s
//   DMA of stage s+NS into the slot of stage s
//   LDS reads of stage s+1 into the second register set
//   MFMAs of stage s
// so NS - 1 stages are in flight, one barrier per stage, and the reads run
// beside the MFMAs.  Stages past the end are issued with a dead offset (they
// write zeros), which keeps the DMA counts constant.
//
// What bounds them: tiles up to 64x64 the operands from HBM (decoding), the
// others LDS, whose 128 bytes per cycle carry (FM + FN) fragment reads per
// wave and the DMA writes: 384 cycles of a 64x64 tile's stage against 128 of
// MFMAs, 768 against 512 for 128x128 (a direct load of the A fragments into
// registers takes the A half off LDS but measured 1.6x slower: 16 rows of 64
// bytes per load).  Measured per call, one MI355X, 256x256 tiles before ->
// now: BF16 16 x 4096 x 8192 121 -> 14.4 us (67 MB of weights, 4.7 TB/s), BF16
// 1000 x 3000 x 2056 42.8 -> 22.6 us, BF8 1024 x 4096 x 7168 57.9 -> 28.5 us,
// MXFP4 64 x 8192 x 8192 37.8 -> 10.3 us.
//
// MXFP4 adds E8M0 scale chunks (4 stages of every tile row's scales) in a
// ring of their own, requested with their first stage and read whole into
// registers with its operands.
#pragma once

#include "g9_gemm.hpp"

namespace g9 {

// Geometry of a small tile: TM x TN outputs, NW waves of which WM x WN
// compute (the others only load), NS ring slots.
template <Op OP_, int TM_, int TN_, int NW_, int WM_, int WN_, int NS_>
struct Tile {
  static constexpr Op OP = OP_;
  static constexpr int TM = TM_, TN = TN_, NW = NW_, WM = WM_, WN = WN_, NS = NS_;
  static_assert(TM % (16 * WM) == 0 && TN % (16 * WN) == 0 && WM * WN <= NW, "16x16 fragments");
  static constexpr int FM = TM / 16 / WM, FN = TN / 16 / WN;  // fragments per computing wave
  static constexpr int kThreads = 64 * NW;
  static constexpr int kUnits = (TM + TN) / 8;  // 1 KiB DMA units per stage
  static constexpr int U = kUnits / NW;         // per wave
  static_assert(kUnits % NW == 0, "DMA units divide among the waves");
  // Every unit of a wave belongs to one operand.
  static constexpr bool kOneOperand = (TM / 8) % U == 0;
  static constexpr int kSlot = (TM + TN) * kRowBytes;
  static constexpr bool kScaled = OpInfo<OP>::kScaled;
  // Scale chunks: per operand, 32-byte rows rounded up to whole 1 KiB units
  // (K-major: 32 group rows of T bytes, likewise).
  static constexpr int kScUnitsA = kScaled ? (TM + 31) / 32 : 0, kScUnitsB = kScaled ? (TN + 31) / 32 : 0;
  static constexpr int kScUnits = kScUnitsA + kScUnitsB;
  static constexpr int USC = (kScUnits + NW - 1) / NW;  // scale DMAs per wave and chunk
  static constexpr int kScSlot = kScUnits * 1024;
  static constexpr int NSC = kScaled ? (NS + 3) / 4 : 0;  // scale ring slots
  static constexpr int kScBase = NS * kSlot;
  static constexpr int kStagePitch = TN * 2 + 16;  // epilogue staging row pitch
  static constexpr int kRing = kScBase + NSC * kScSlot;
  static constexpr int kLds = kRing > TM * kStagePitch ? kRing : TM * kStagePitch;
  static_assert(kLds <= 160 * 1024, "LDS");
  // Workgroups that fit a CU's LDS and registers, and with it the waves per
  // SIMD (512 registers a lane and SIMD: accumulators, operand sets, scales
  // and ~64 addresses and temporaries).
  static constexpr int kRegs = 4 * FM * FN + 16 * (FM + FN) + (kScaled ? 4 * (FM + FN) : 0) + 64;
  static constexpr int kOccLds = 160 * 1024 / kLds, kOccRegs = 512 / kRegs * 4 / NW;
  static constexpr int kOcc = kOccRegs < 1 || kOccLds < 1 ? 1 : kOccLds < kOccRegs ? kOccLds : kOccRegs;
  static constexpr int kWavesPerSimd = kOcc * NW >= 4 ? (kOcc * NW + 3) / 4 : 1;
  // DMAs of stages first .. last (each stage's U operand DMAs; a stage that
  // is a multiple of 4 also requests its scale chunk).
  static constexpr int dmas(int first, int last) {
    int n = 0;
    for (int t = first; t <= last; ++t) n += U + (kScaled && t % 4 == 0 ? USC : 0);
    return n;
  }
  // vmcnt that leaves the requests of stages first .. last in flight (at most
  // 63, the counter's range: a lower count waits for more).
  static constexpr int keep(int first, int last) { return dmas(first, last) < 63 ? dmas(first, last) : 63; }
  static constexpr int NM = FM * FN * (OP == Op::BF8 ? 1 : 2);  // MFMAs per wave and stage
  static constexpr int NR = 2 * (FM + FN);                      // 16-byte LDS reads per wave and stage
  static constexpr bool kInterleave = NM >= 4 && WM * WN == NW;
  static constexpr int kReadSlots = NM * 3 / 4 > 0 ? NM * 3 / 4 : 1;  // MFMA slots the reads spread over
};

template <class T>
struct TileFrags {
  u32x4 a[T::FM][2], b[T::FN][2];
};
// A lane's scale bytes of one chunk per fragment: byte 2 (st & 1) + e of word
// st >> 1 is stage st, MFMA step e.
template <class T>
struct TileScales {
  u32x2 a[T::kScaled ? T::FM : 1], b[T::kScaled ? T::FN : 1];
};

template <class T>
struct TilePipe {
  static constexpr Op OP = T::OP;
  static constexpr int U = T::U, NR = T::kOneOperand ? 1 : U;
  rsrc_t r[NR];
  u32 v[U];
  rsrc_t rs[T::USC ? T::USC : 1];
  u32 vs[T::USC ? T::USC : 1], cstep[T::USC ? T::USC : 1];
  u32 ba[2], bb[2];  // LDS read bases of chunks 0, 1 of the lane's A / B row
  u32 sa, sb;        // LDS read bases of its scales
  u32 lds0, dst, sdst[T::USC ? T::USC : 1];
  int lane, wave, ns;
  u32 kshift;
  u32 psel;  // FP4: v_perm selector of the lane group's byte

  // Rows valid in the tile: `rows` of the operand from tile row t * TILE on.
  G9_DEV static u32 valid(int rows, int t, int tile) {
    return (u32)__builtin_amdgcn_readfirstlane(min(max(rows - t * tile, 0), tile));
  }

  G9_DEV void init(const GemmParams& p, char* smem, int tm, int tn) {
    lds0 = (u32)(uintptr_t)to_lds(smem);
    lane = threadIdx.x & 63;
    wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    ns = p.ns;
    kshift = p.kshift;
    const u32 va = valid(p.M, tm, T::TM), vb = valid(p.N, tn, T::TN);
    // The K tail's shift of every stage, as in the 256x256 kernels.
    const char* pa = p.a + (size_t)(tm * T::TM) * p.lda - kshift;
    const char* pb = p.b + (size_t)(tn * T::TN) * p.ldb - kshift;
    dst = lds0 + (u32)wave * (U * 1024);
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int g = wave * U + u;
      const bool isa = g < T::TM / 8;
      if (u < NR) r[u] = make_rsrc(isa ? pa : pb, isa ? va * p.lda + kshift : vb * p.ldb + kshift);
      const int row = 8 * g - (isa ? 0 : T::TM) + (lane >> 3);
      const int ch = (lane & 7) ^ ((row >> 1) & 7);
      v[u] = (u32)row * (isa ? p.lda : p.ldb) + 16u * ch;
    }
    const int wm = wave / T::WN, wn = wave % T::WN;
    const int gi = lane >> 4, rr = lane & 15, sw = (rr >> 1) & 7;
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const u32 slot = (u32)((4 * c + gi) ^ sw) * 16;
      ba[c] = lds0 + (u32)(wm * T::FM * 16 + rr) * kRowBytes + slot;
      bb[c] = lds0 + (u32)(T::TM + wn * T::FN * 16 + rr) * kRowBytes + slot;
    }
    if constexpr (T::kScaled) {
#pragma unroll
      for (int k = 0; k < T::USC; ++k) {
        // Unit q of the chunk; the waves past the last unit repeat it.
        const int q = min(wave * T::USC + k, T::kScUnits - 1);
        const bool isa = q < T::kScUnitsA;
        const int unit = isa ? q : q - T::kScUnitsA;
        const unsigned char* base = isa ? p.a_sc : p.b_sc;
        const u32 ld = isa ? p.ldsa : p.ldsb;
        const int row0 = isa ? tm * T::TM : tn * T::TN;
        const u32 rows = isa ? va : vb;
        sdst[k] = lds0 + T::kScBase + (u32)q * 1024;
        if constexpr (OpInfo<OP>::kPreshuffled) {
          // Chunk c of row m: 32 bytes at c * ld + 32 m.
          const u32 nch = (u32)(p.ns + kScChunk - 1) / kScChunk;
          rs[k] = make_rsrc(base, (nch - 1) * ld + (u32)(isa ? p.M : p.N) * kScRowBytes);
          vs[k] = (u32)(row0 + 32 * unit) * kScRowBytes + 16u * lane;
          cstep[k] = ld;
        } else if constexpr (OpInfo<OP>::kKMajor) {
          // Group G of the chunk: T bytes (one per row) at G * ld; the chunk
          // lands as 32 group rows of T bytes.  The range ends on a whole
          // dword, as in the 256x256 kernels.
          const int per = isa ? T::TM / 16 : T::TN / 16;  // 16-row pieces per group row
          const int piece = 64 * unit + lane;
          const int grp = piece / per, part = piece % per;
          rs[k] = make_rsrc(base + row0, ((u32)p.K / 32 - 1) * ld + ((rows + 3) & ~3u));
          vs[k] = grp < 32 ? (u32)grp * ld + 16u * part : kDeadOff;
          cstep[k] = 32u * ld;
        } else {
          // Row m of the chunk: 32 bytes at m * ld + 32 c, up to the last
          // row's last byte and kept scalar, as in the 256x256 kernels.
          const u32 end = rows ? (rows - 1) * ld + 8u * (u32)p.ns : 0u;
          rs[k] = make_rsrc(base + (size_t)row0 * ld, (u32)__builtin_amdgcn_readfirstlane((int)end));
          vs[k] = (u32)(32 * unit + (lane >> 1)) * ld + 16u * (lane & 1);
          cstep[k] = kScRowBytes;
        }
      }
      const u32 a0 = lds0 + T::kScBase, b0 = a0 + T::kScUnitsA * 1024;
      const int ra = wm * T::FM * 16 + rr, rb = wn * T::FN * 16 + rr;
      if constexpr (OpInfo<OP>::kPreshuffled) {
        const u32 unit = 8u * (u32)(gi ^ ((rr >> 2) & 3));
        sa = a0 + ra * 32 + unit;
        sb = b0 + rb * 32 + unit;
      } else if constexpr (OpInfo<OP>::kKMajor) {
        sa = a0 + gi * T::TM + ra;
        sb = b0 + gi * T::TN + rb;
      } else {
        sa = a0 + ra * 32;
        sb = b0 + rb * 32;
        // Byte gi of two words, as bytes 0 and 1 (the low word is v_perm's
        // second source).
        psel = (u32)gi | ((u32)(4 + gi) << 8) | 0x0c0c0000u;
      }
    }
  }

  // Requests stage t into the slot at byte offset `slot`, and (when t opens a
  // chunk) its scale chunk into the scale slot at `scslot`.
  template <bool SC>
  G9_DEV void issue(int t, u32 slot, u32 scslot) const {
    if constexpr (SC) issue_chunk(t, scslot);
    const u32 soff = stage_off(t);
    static_for<U>([&](auto UC) { issue_unit<decltype(UC)::value>(soff, slot); });
  }
  G9_DEV u32 stage_off(int t) const { return t < ns ? (u32)t * kRowBytes : kDeadOff; }
  template <int u>
  G9_DEV void issue_unit(u32 soff, u32 slot) const {
    dma16(r[u < NR ? u : 0], lds_ptr(dst + slot + u * 1024), v[u], soff);
  }
  G9_DEV void issue_chunk(int t, u32 scslot) const {
#pragma unroll
    for (int k = 0; k < T::USC; ++k)
      dma16(rs[k], lds_ptr(sdst[k] + scslot), vs[k], t < ns ? (u32)(t / 4) * cstep[k] : kDeadOff);
  }
  // Stage 0 with a K tail: chunks before k = 0 load zeros.
  G9_DEV void issue_first() const {
    if constexpr (T::kScaled) {
      issue<true>(0, 0, 0);
    } else {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int row = 8 * (wave * U + u) + (lane >> 3);  // the swizzle repeats every 16 rows
        const u32 ch = (u32)((lane & 7) ^ ((row >> 1) & 7));
        dma16(r[u < NR ? u : 0], lds_ptr(dst + u * 1024), ch * 16 < kshift ? kDeadOff : v[u], 0u);
      }
    }
  }

  G9_DEV static G9_LDS void* lds_ptr(u32 a) { return (G9_LDS void*)(uintptr_t)a; }
  G9_DEV static u32x4 lds16(u32 a) { return *(const G9_LDS u32x4*)(uintptr_t)a; }
  G9_DEV void read(TileFrags<T>& f, u32 slot) const {
#pragma unroll
    for (int c = 0; c < 2; ++c) {
      const u32 xa = ba[c] + slot, xb = bb[c] + slot;
#pragma unroll
      for (int i = 0; i < T::FM; ++i) f.a[i][c] = lds16(xa + i * 16 * kRowBytes);
#pragma unroll
      for (int j = 0; j < T::FN; ++j) f.b[j][c] = lds16(xb + j * 16 * kRowBytes);
    }
  }
  // Read number R of read(): fragment order, both chunks of a fragment together.
  // x: the slot's read bases (A chunks 0, 1, then B), opaque so the fragment
  // offsets stay in the instructions.
  template <int R>
  G9_DEV void read_one(TileFrags<T>& f, const u32 (&x)[4]) const {
    constexpr int c = R & 1, i = R >> 1;
    if constexpr (i < T::FM)
      f.a[i][c] = lds16(x[c] + i * 16 * kRowBytes);
    else
      f.b[i - T::FM][c] = lds16(x[2 + c] + (i - T::FM) * 16 * kRowBytes);
  }
  // The lane's 8 scale bytes of fragment `f` of an operand with T rows per
  // group row, read at `base`.
  template <int TR>
  G9_DEV u32x2 scale_bytes(u32 base, int f) const {
    if constexpr (OpInfo<OP>::kPreshuffled) {
      return *(const G9_LDS u32x2*)(uintptr_t)(base + f * 16 * kScRowBytes);
    } else if constexpr (OpInfo<OP>::kKMajor) {
      // Groups gi, 4 + gi, ..., 28 + gi of the row.
      u32 w[2];
#pragma unroll
      for (int h = 0; h < 2; ++h) {
        u32 x = 0;
#pragma unroll
        for (int k = 0; k < 4; ++k)
          x |= (u32) * (const G9_LDS unsigned char*)(uintptr_t)(base + f * 16 + (4 * h + k) * 4 * TR) << (8 * k);
        w[h] = x;
      }
      return u32x2{w[0], w[1]};
    } else {
      // Words 2 st + e of the row's 32 bytes hold groups 8 st + 4 e + 0..3:
      // byte gi of each.
      const u32x4 lo = lds16(base + f * 16 * kScRowBytes), hi = lds16(base + f * 16 * kScRowBytes + 16);
      const u32 l0 = __builtin_amdgcn_perm(lo.y, lo.x, psel), l1 = __builtin_amdgcn_perm(lo.w, lo.z, psel);
      const u32 h0 = __builtin_amdgcn_perm(hi.y, hi.x, psel), h1 = __builtin_amdgcn_perm(hi.w, hi.z, psel);
      return u32x2{l0 | (l1 << 16), h0 | (h1 << 16)};
    }
  }
  G9_DEV void read_scales(TileScales<T>& s, u32 scslot) const {
    if constexpr (T::kScaled) {
#pragma unroll
      for (int i = 0; i < T::FM; ++i) s.a[i] = scale_bytes<T::TM>(sa + scslot, i);
#pragma unroll
      for (int j = 0; j < T::FN; ++j) s.b[j] = scale_bytes<T::TN>(sb + scslot, j);
    }
  }
};

template <class T>
using TileAcc = f32x4[T::FM][T::FN];

// MFMA step e of a stage (ST: its place in its scale chunk) on fragments b, a
// with scales sb, sa.  Inline assembly with the accumulator tied in place, as
// in the 256x256 kernels (see mma() there for the hazards this leaves to the
// caller).
template <Op OP, int ST, int e>
G9_DEV void tile_mma(f32x4& acc, const u32x4 (&b)[2], const u32x4 (&a)[2], const u32x2& sb, const u32x2& sa) {
  if constexpr (OP == Op::F16) {
    asm("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(acc) : "v"(b[e]), "v"(a[e]));
  } else if constexpr (OP == Op::BF16) {
    asm("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(acc) : "v"(b[e]), "v"(a[e]));
  } else if constexpr (OP == Op::BF8) {
    const i32x8 x = __builtin_bit_cast(i32x8, __builtin_shufflevector(b[0], b[1], 0, 1, 2, 3, 4, 5, 6, 7));
    const i32x8 y = __builtin_bit_cast(i32x8, __builtin_shufflevector(a[0], a[1], 0, 1, 2, 3, 4, 5, 6, 7));
    asm("v_mfma_f32_16x16x128_f8f6f4 %0, %1, %2, %0 cbsz:1 blgp:1" : "+a"(acc) : "v"(x), "v"(y));
  } else {
    mfma_scaled<2 * (ST & 1) + e>(acc, b[e], a[e], ST >> 1 ? sb.y : sb.x, ST >> 1 ? sa.y : sa.x);
  }
}
// MFMA number K of a stage: step-major, then A fragments, B fragments in
// snake order (consecutive MFMAs share an operand).
template <class T, int ST, int K>
G9_DEV void tile_mfma(TileAcc<T>& acc, const TileFrags<T>& f, const TileScales<T>& s) {
  constexpr int e = K / (T::FM * T::FN), i = (K / T::FN) % T::FM, j0 = K % T::FN;
  constexpr int j = (i % 2) ? T::FN - 1 - j0 : j0;
  tile_mma<T::OP, ST, e>(acc[i][j], f.b[j], f.a[i], s.b[T::kScaled ? j : 0], s.a[T::kScaled ? i : 0]);
}

// Ends every path out of an MFMA sequence (see settle_acc).
template <class T>
G9_DEV void settle_tile(TileAcc<T>& acc) {
  mfma_drain();
#pragma unroll
  for (int i = 0; i < T::FM; ++i)
#pragma unroll
    for (int j = 0; j < T::FN; ++j) asm volatile("" : "+a"(acc[i][j]));
}

// One output tile (tm, tn) of C.
template <class T>
G9_DEV void tile_gemm(const GemmParams& p, char* smem, int tm, int tn, int out, float scale) {
  TilePipe<T> P;
  P.init(p, smem, tm, tn);
  TileAcc<T> acc;
#pragma unroll
  for (int i = 0; i < T::FM; ++i)
#pragma unroll
    for (int j = 0; j < T::FN; ++j) {
      acc[i][j] = f32x4{};
      asm volatile("" : "+a"(acc[i][j]));
    }
  const bool computes = T::WM * T::WN == T::NW || P.wave < T::WM * T::WN;
  TileFrags<T> f[2];
  TileScales<T> sc, scn;
  P.issue_first();
  static_for<T::NS - 1>([&](auto S) {
    constexpr int t = decltype(S)::value + 1;
    P.template issue<T::kScaled && t % 4 == 0>(t, t * T::kSlot, (t / 4) * T::kScSlot);
  });
  waitcnt<T::keep(1, T::NS - 1), 0>();
  barrier();
  if (computes) {
    P.read(f[0], 0);
    P.read_scales(sc, 0);
  }
  // Byte offsets of stage s's slot, and of the scale slots of the chunks read
  // and requested next.
  u32 slot = 0, scr = T::NSC > 1 ? T::kScSlot : 0, scw = ((T::NS + 3) / 4 % (T::NSC ? T::NSC : 1)) * T::kScSlot;
  auto step = [&](auto QC, int s) {
    constexpr int Q = decltype(QC)::value;  // s % 4
    constexpr int kWait = T::keep(Q + 2, Q + T::NS - 1);
    waitcnt<kWait, 0>();
    barrier();
    constexpr bool kChunkW = T::kScaled && (Q + T::NS) % 4 == 0;
    if constexpr (kChunkW) {
      P.issue_chunk(s + T::NS, scw);
      scw = scw + T::kScSlot == T::NSC * T::kScSlot ? 0 : scw + T::kScSlot;
    }
    const u32 soff = P.stage_off(s + T::NS);
    const u32 wr = slot;
    slot = slot + T::kSlot == T::NS * T::kSlot ? 0 : slot + T::kSlot;
    if constexpr (T::kInterleave) {
      // MFMAs with the stage's reads and DMAs spread between them (a wave
      // issues in order: bunched, they hold its MFMAs up).
      const u32 x[4] = {opaque(P.ba[0] + slot), opaque(P.ba[1] + slot), opaque(P.bb[0] + slot), opaque(P.bb[1] + slot)};
      static_for<T::NM>([&](auto KC) {
        constexpr int K = decltype(KC)::value;
        tile_mfma<T, Q, K>(acc, f[Q & 1], sc);
        static_for<T::NR>([&](auto R) {
          if constexpr (decltype(R)::value * T::kReadSlots / T::NR == K)
            P.template read_one<decltype(R)::value>(f[(Q + 1) & 1], x);
        });
        static_for<T::U>([&](auto D) {
          if constexpr (decltype(D)::value * T::NM / T::U == K) P.template issue_unit<decltype(D)::value>(soff, wr);
        });
        if constexpr (T::kScaled && Q == 3 && K == T::kReadSlots - 1) P.read_scales(scn, scr);
        __builtin_amdgcn_sched_barrier(0);
      });
    } else {
      static_for<T::U>([&](auto D) { P.template issue_unit<decltype(D)::value>(soff, wr); });
      if (computes) {
        P.read(f[(Q + 1) & 1], slot);
        if constexpr (T::kScaled && Q == 3) P.read_scales(scn, scr);
        static_for<T::NM>([&](auto K) { tile_mfma<T, Q, decltype(K)::value>(acc, f[Q & 1], sc); });
      }
    }
    if constexpr (T::kScaled && Q == 3) {
      scr = scr + T::kScSlot == T::NSC * T::kScSlot ? 0 : scr + T::kScSlot;
      sc = scn;
    }
  };
  int s = 0;
  for (; s + 4 <= p.ns; s += 4) static_for<4>([&](auto Q) { step(Q, s + decltype(Q)::value); });
  settle_tile<T>(acc);
  static_for<3>([&](auto Q) {
    if (s + decltype(Q)::value < p.ns) step(Q, s + decltype(Q)::value);
  });
  settle_tile<T>(acc);
  waitcnt<0, 0>();
  barrier();
  // Epilogue: 16-bit rows staged in LDS, out in 16-byte row chunks.
  const int tid = threadIdx.x;
  if (computes) {
    const int wm = P.wave / T::WN, wn = P.wave % T::WN, rr = P.lane & 15, gi = P.lane >> 4;
#pragma unroll
    for (int i = 0; i < T::FM; ++i)
#pragma unroll
      for (int j = 0; j < T::FN; ++j) {
        const f32x4 q = acc[i][j] * scale;
        const u32x2 h = out == OUT_BF16 ? pack4_bf16(q) : pack4_f16(q);
        lds_write8(smem + ((wm * T::FM + i) * 16 + rr) * T::kStagePitch + ((wn * T::FN + j) * 16 + 4 * gi) * 2, h);
      }
  }
  waitcnt<63, 0>();
  barrier();
  constexpr int kChunks = T::TN / 8;
#pragma unroll
  for (int c = 0; c < T::TM * kChunks; c += T::kThreads) {
    const int q = c + tid;
    if (T::TM * kChunks % T::kThreads != 0 && q >= T::TM * kChunks) break;
    const int row = q / kChunks, ch = q % kChunks;
    put_c16(p, tm * T::TM + row, tn * T::TN + ch * 8, lds_read16(smem + row * T::kStagePitch + ch * 16));
  }
}

}  // namespace g9
