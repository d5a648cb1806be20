// fp32 GEMM on the CDNA4 fp32 matrix cores: C = A * op(B) (+ bias).
//
// Counterpart of gemm_fp32_ga100_kernel (src/cuda/fp32_matmul.cu:31-184):
// same contract (row-major, any M/N/K, fully bounds-checked loads and stores),
// but the products run on the matrix cores with fp32 accumulation (on the bf16
// instruction, each float as three bf16 planes, or on v_mfma_f32_16x16x4_f32)
// instead of the reference's separate __fmul_rn/__fadd_rn SIMT loop, which exists
// only to dodge a GA100 FMA limit (fp32_matmul.cu:20-26).
//
// Any alignment is accepted: global memory is read by 4-byte LDS-DMA
// (buffer_load_dword ... lds, 256 contiguous LDS bytes per instruction), with
// an out-of-range offset (hardware zero-fill) for every element past M, N or
// K, so ragged shapes such as 4097 x 3001 x 2049 need no special casing.
// Operands whose rows are 16-byte aligned with K (and N for B given as [K,N])
// a multiple of 4 use 16-byte LDS-DMA instead (DMA16: buffer_load_dwordx4 ...
// lds, 1 KiB per instruction): a quarter of the load instructions and their
// address work.  The DMA fills a ring of four stages of BK = 16 k, two at a time
// while the two before are multiplied; one wait and barrier per pair certifies that the
// next pair has landed and that every wave is done with the slots about to be refilled.
// Products of one stage (K <= 16) have a kernel of their own with one slot.
//
// LDS layouts (per stage):
//   A, and B given as [N,K]: rows of 16 floats (64 bytes) in groups of 16 rows
//     (1 KiB); the 16-byte chunk c (k = 4c..4c+3) of row r sits at slot
//     f32_slot(r % 16, c) of its group, a layout measured free of LDS bank
//     conflicts for the fragment read (16 consecutive rows at one chunk per 16
//     lanes, ds_read_b128).  A DMA instruction writes a quarter of a group
//     (4-byte DMA) or a whole group (16-byte DMA), each lane fetching the
//     element f32_slot_src names for its slot.
//   B given as [K,N]: [k][n], rows of BN floats, 16-float segment s of row k
//     stored at segment s ^ ((k/4)%4): the fragment read of MFMA step s
//     (rows s, 4+s, 8+s, 12+s at 16 columns, ds_read_b32) hits 64 distinct
//     banks, and one DMA instruction writes 64 consecutive floats of a row.
// Lane group g holds k = 4g .. 4g+3 of a stage (one ds_read_b128 of A): the eight k of a
// bf16 instruction's lane come from a pair of stages, four fp32 instructions use one each.
#pragma once

#include "device_common.h"

namespace cmpext3 {

// NS: ring slots, four (two stages loaded and two multiplied at a time) or one (K <= BK).
template <int BM, int BN, int NS>
struct F32Shape {
  static constexpr int BK = 16;
  static constexpr int NT = 256;  // 2 x 2 waves
  static constexpr int WTM = BM / 2, WTN = BN / 2;
  static constexpr int FM = WTM / 16, FN = WTN / 16;
  static constexpr int A_BYTES = BM * BK * 4;
  static constexpr int B_BYTES = BN * BK * 4;
  static constexpr int STAGE = A_BYTES + B_BYTES;
  static constexpr int A_DMA = A_BYTES / 256 / 4;  // 256-byte DMA instructions per wave per stage
  static constexpr int B_DMA = B_BYTES / 256 / 4;
  // DMA16: 1 KiB instructions t = 4i + wave, i < A16 (B16), skipping t >= A_BYTES / 1024
  static constexpr int A16 = (A_BYTES / 1024 + 3) / 4;
  static constexpr int B16 = (B_BYTES / 1024 + 3) / 4;
  static_assert(BN % 64 == 0 && BM % 32 == 0, "whole DMA instructions per wave, 64-float B rows");
  static_assert(NS * STAGE <= 160 * 1024, "LDS");
};

// 16-byte slot (0..63) of chunk c (0..3) of row r (0..15) in its 1 KiB group of 16 rows:
// with bits r0..r3 of r and c0, c1 of c, slot bits are r1^c0^c1, r0^r1^r3, r0^r3, r0,
// r2, r2^c1.  Found by sweeping GF(2)-linear layouts of the group on MI355X with the LDS
// bank-conflict counter (SQ_LDS_BANK_CONFLICT): for the fragment read (lane l reads chunk
// l / 16 of row l % 16, ds_read_b128) this one measured zero conflict cycles at every
// LDS base offset tried, where the earlier chunk ^ (r / 4) % 4 swizzle (four rows per 256
// bytes) took one extra cycle per read, as did a third of the layouts swept.
__device__ __forceinline__ int f32_slot(int r, int c) {
  const int r0 = r & 1, r1 = (r >> 1) & 1, r2 = (r >> 2) & 1, r3 = (r >> 3) & 1, c0 = c & 1, c1 = (c >> 1) & 1;
  return (r1 ^ c0 ^ c1) | ((r0 ^ r1 ^ r3) << 1) | ((r0 ^ r3) << 2) | (r0 << 3) | (r2 << 4) | ((r2 ^ c1) << 5);
}
// The row (0..15) and chunk whose data slot s of a group holds (the inverse of f32_slot).
__device__ __forceinline__ void f32_slot_src(int s, int& r, int& c) {
  const int s0 = s & 1, s1 = (s >> 1) & 1, s2 = (s >> 2) & 1, s3 = (s >> 3) & 1, s4 = (s >> 4) & 1, s5 = (s >> 5) & 1;
  const int r0 = s3, r1 = s1 ^ s2, r2 = s4, r3 = s2 ^ s3, c1 = s4 ^ s5, c0 = s0 ^ r1 ^ c1;
  r = r0 | (r1 << 1) | (r2 << 2) | (r3 << 3);
  c = c0 | (c1 << 1);
}
// Byte offset of 16-byte chunk `chunk` (0..3) of row `row` in a block of rows of 16 floats.
__device__ __forceinline__ uint32_t f32_off(int row, int chunk) {
  return (uint32_t)((row >> 4) * 1024 + 16 * f32_slot(row & 15, chunk));
}

// ---- fp32 products on the bf16 matrix cores ----
// A float x, taken as 2^16 x, is the exact sum of three bf16 values: h, 2^16 x rounded
// to 8 significant bits, m, the top 8 bits of the signed rest, and l, what is left
// (scaled, every bit of every float, subnormal ones too, is above bf16's smallest,
// 2^-133).  Of the nine products of two such sums, six are summed in fp32 by
// v_mfma_f32_16x16x32_bf16: h h in one accumulator, the five small ones (h m, m h, m m,
// h l, l h, in sum about 2^-7 of h h) in another, so that they are rounded at their own
// size, and the two are added at the end.  (In one accumulator the instruction cut the
// small products off below the sum's last bits, always the same way: sums of 8192
// positive products were off by 1.6e-5, the fp32 instruction's by 1.2e-6.)  m l, l m
// and l l are left out, together at most 2^-23 of the product, and m's sign is
// independent of x's, so that they do not add up.  A chain rounds once per 32 k where
// the fp32 instruction's (16x16x4) rounds 8 times.  Relative Frobenius error against
// float64 on MI355X, fp32 instruction -> this: 512 x 512 x 8192 normal 1.62e-6 ->
// 0.57e-6, positive (uniform in [0, 1)) 1.19e-6 -> 0.42e-6, x 2048 8.1e-7 -> 2.7e-7 and
// 6.0e-7 -> 2.2e-7, x 128 2.0e-7 -> 0.67e-7, x 32 1.0e-7 -> 0.41e-7, x 16 7.4e-8 ->
// 3.6e-8, x 4 // Infinities, NaN, floats of 2^96 and more and sums of 2^96 and more (their scaled values
// overflow) are seen in the sums, and the tile is then computed again on the fp32
// instruction: such a tile takes about 2.4 times as long as one that has none.
// Splitting an element takes 6.5 vector instructions in each wave that reads it, as many
// cycles as its products where a wave's block is small: that bounds the 96 x 64 and 64 x
// 64 tiles (rounding by bf16 conversions took longer, 12 cycles each; one wave per K
// stage, which splits less, left too few waves; sums of 32 k in registers of their own,
// added to the total on the vector units, took 5 % longer than the two accumulators).
// MI355X, fp32 instruction -> this: 4096^3 (128 x 128) 946 -> 732 us, 4097 x 3001 x 2049
// (96 x 64, 4-byte DMA) 394 -> 362, 4100 x 3000 x 2048 (96 x 64) 369 -> 333, 3000 x 2000 x
// 1000 (64 x 64) 101 -> 97.
constexpr float kF32Scale = 65536.f;                      // of a split float
constexpr float kF32Unscale = 1.f / (65536.f * 65536.f);  // of a sum of products
template <typename V>
struct F32Planes {
  V h, m, l;  // u32x4: 8 k, two 16-k stages of 4; u32x2: one stage's 4
};
// Words i, i+1 of the planes of four floats.
template <typename V>
__device__ __forceinline__ void f32_split4(F32Planes<V>& p, int i, f32x4 x) {
#pragma unroll
  for (int w = 0; w < 2; ++w) {
    uint32_t h[2], m[2], l[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const float a = x[2 * w + e];
      // t = 2^32 a + 2^16 a to 24 bits, so t - 2^32 a is 2^16 a to 8 bits, exactly, and so is the rest
      const float t = a * (kF32Scale * 65536.f + kF32Scale);
      const float hi = __builtin_fmaf(a, -kF32Scale * 65536.f, t);
      const float rest = __builtin_fmaf(a, kF32Scale, -hi);
      h[e] = __float_as_uint(hi);
      m[e] = __float_as_uint(rest);
      l[e] = __float_as_uint(rest - __uint_as_float(m[e] & 0xFFFF0000u));
    }
    p.h[i + w] = pack_hi16(h[0], h[1]);
    p.m[i + w] = pack_hi16(m[0], m[1]);
    p.l[i + w] = pack_hi16(l[0], l[1]);
  }
}
__device__ __forceinline__ f32x4 f32_mma(u32x4 b, u32x4 a, f32x4 c) { return Mfma<__bf16>::mma(b, a, c); }
__device__ __forceinline__ f32x4 f32_mma(u32x2 b, u32x2 a, f32x4 c) {
  typedef short s16x4 __attribute__((ext_vector_type(4)));
  return __builtin_amdgcn_mfma_f32_16x16x16bf16_1k(__builtin_bit_cast(s16x4, b), __builtin_bit_cast(s16x4, a), c, 0,
                                                   0, 0);
}

// SPLITK: grid.z = batch * p.splits; this workgroup sums its split's K range and
// stores the sums into p.partials (bias added by the reduction).
// EXACT: on the fp32 instruction.  Otherwise returns true, with nothing written, when the
// tile needs that (see above).  NS: ring slots; one for K <= 16 (EXACT).
template <bool KN, int BM, int BN, bool SPLITK, bool DMA16, bool EXACT, int NS = 4>
__device__ __forceinline__ bool f32_tile(const GemmParams& p, unsigned char* smem) {
  using S = F32Shape<BM, BN, NS>;
  constexpr int FM = S::FM, FN = S::FN;
  static_assert(NS == 4 || (NS == 1 && EXACT && !SPLITK), "a ring of four stages, or one stage");

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;

  int tm, tn;
  int bzi;
  tile_coords(blockIdx.x, blockIdx.z, gridDim.z, p.tiles_m, p.tiles_n, p.group_m, tm, tn, bzi);
  const int m0 = tm * BM, n0 = tn * BN;
  const int M = p.M, N = p.N;
  const int64_t lda = p.lda, ldb = p.ldb;
  // split-K: entry bzi of the grid's z range is split bzi % splits of batch entry bzi / splits
  const int ks = SPLITK ? bzi % p.splits : 0;
  const int64_t bz = SPLITK ? bzi / p.splits : bzi;
  const int kbeg = SPLITK ? ks * p.ksplit : 0;
  const int K = SPLITK ? min(p.K - kbeg, p.ksplit) : p.K;  // this workgroup's K range
  const float* Abase = (const float*)p.A + bz * p.stride_a + (int64_t)m0 * lda + kbeg;
  const float* Bbase = KN ? (const float*)p.B + bz * p.stride_b + (int64_t)kbeg * ldb + n0
                          : (const float*)p.B + bz * p.stride_b + (int64_t)n0 * ldb + kbeg;

  // ---- DMA sources: the inverse of the LDS layouts, relative to the stage's k0 ----
  // Row blocks: 4-byte instruction t writes slots 16 (t % 4) .. +15 of group t / 4, lane l
  // element l % 4 of slot 16 (t % 4) + l / 4.
  uint32_t a_off[S::A_DMA];
#pragma unroll
  for (int i = 0; i < S::A_DMA; ++i) {
    const int t = wave * S::A_DMA + i;
    int r, c;
    f32_slot_src(16 * (t & 3) + (lane >> 2), r, c);
    const int row = 16 * (t >> 2) + r;
    const int k = 4 * c + (lane & 3);
    a_off[i] = (m0 + row < M) ? (uint32_t)(row * lda + k) * 4u : kBufOOB;
  }
  // B: [K,N] -> instruction t writes row k = t / (BN/64), floats 64*(t%(BN/64)) ..
  //    +63; lane l lands in segment slot 4*(t%(BN/64)) + l/16, which holds data
  //    segment slot ^ ((k/4)%4).  [N,K] -> as A.
  uint32_t b_off[S::B_DMA];
#pragma unroll
  for (int i = 0; i < S::B_DMA; ++i) {
    const int t = wave * S::B_DMA + i;
    if (KN) {
      constexpr int PER_ROW = BN / 64;
      const int k = t / PER_ROW;
      const int seg = (4 * (t % PER_ROW) + (lane >> 4)) ^ ((k >> 2) & 3);
      const int n = 16 * seg + (lane & 15);
      b_off[i] = (n0 + n < N) ? (uint32_t)(k * ldb + n) * 4u : kBufOOB;
    } else {
      int r, c;
      f32_slot_src(16 * (t & 3) + (lane >> 2), r, c);
      const int row = 16 * (t >> 2) + r;
      const int k = 4 * c + (lane & 3);
      b_off[i] = (n0 + row < N) ? (uint32_t)(row * ldb + k) * 4u : kBufOOB;
    }
  }
  // DMA16 sources: A (and B as [N,K]) instruction t writes group t (rows 16t .. 16t+15),
  // lane l slot l; B as [K,N]: instruction t writes floats 256t + 4l .. +3 of the stage's
  // [16][BN] block.
  uint32_t va_off[S::A16], vb_off[S::B16];
  int va_k[S::A16], vb_k[S::B16];
  if constexpr (DMA16) {
#pragma unroll
    for (int i = 0; i < S::A16; ++i) {
      int r, c;
      f32_slot_src(lane, r, c);
      const int row = 16 * (4 * i + wave) + r;
      const int k = 4 * c;
      va_off[i] = (m0 + row < M) ? (uint32_t)(row * lda + k) * 4u : kBufOOB;
      va_k[i] = k;
    }
#pragma unroll
    for (int i = 0; i < S::B16; ++i) {
      if (KN) {
        const int f = 256 * (4 * i + wave) + 4 * lane;
        const int k = f / BN;
        const int n = 16 * (((f % BN) >> 4) ^ ((k >> 2) & 3)) + (f & 15);
        vb_off[i] = (n0 + n < N) ? (uint32_t)(k * ldb + n) * 4u : kBufOOB;
        vb_k[i] = k;
      } else {
        int r, c;
        f32_slot_src(lane, r, c);
        const int row = 16 * (4 * i + wave) + r;
        const int k = 4 * c;
        vb_off[i] = (n0 + row < N) ? (uint32_t)(row * ldb + k) * 4u : kBufOOB;
        vb_k[i] = k;
      }
    }
  }
  // Stage st's loads.  A stage wholly inside K loads every piece unchecked; only the stage
  // that holds K's end (and those past it, all zeros) compares each piece's k with K (the
  // per-piece compare and select on every stage cost 7 %: cfg5 419.5 -> 391.7 us).
  auto load_stage = [&](int st) {
    const int k0 = st * S::BK;
    const int krem = K - k0;
    const uint32_t dst = lds_addr(smem) + (uint32_t)((st % NS) * S::STAGE);
    const i32x4 ra = make_rsrc_sgpr(Abase + k0);
    const i32x4 rb = make_rsrc_sgpr(KN ? Bbase + (int64_t)k0 * ldb : Bbase + k0);
    const bool whole = krem >= S::BK;  // wave-uniform
    if constexpr (DMA16) {
      if (whole) {
#pragma unroll
        for (int i = 0; i < S::A16; ++i)
          if (4 * i + wave < S::A_BYTES / 1024) dma_load16(ra, va_off[i], dst + (4 * i + wave) * 1024);
#pragma unroll
        for (int i = 0; i < S::B16; ++i)
          if (4 * i + wave < S::B_BYTES / 1024) dma_load16(rb, vb_off[i], dst + S::A_BYTES + (4 * i + wave) * 1024);
        return;
      }
#pragma unroll
      for (int i = 0; i < S::A16; ++i)
        if (4 * i + wave < S::A_BYTES / 1024)
          dma_load16(ra, va_k[i] < krem ? va_off[i] : kBufOOB, dst + (4 * i + wave) * 1024);
#pragma unroll
      for (int i = 0; i < S::B16; ++i)
        if (4 * i + wave < S::B_BYTES / 1024)
          dma_load16(rb, vb_k[i] < krem ? vb_off[i] : kBufOOB, dst + S::A_BYTES + (4 * i + wave) * 1024);
    } else {
      if (whole) {
#pragma unroll
        for (int i = 0; i < S::A_DMA; ++i) dma_load4(ra, a_off[i], dst + (wave * S::A_DMA + i) * 256);
#pragma unroll
        for (int i = 0; i < S::B_DMA; ++i) dma_load4(rb, b_off[i], dst + S::A_BYTES + (wave * S::B_DMA + i) * 256);
        return;
      }
      // each piece's k is found again here from an opaque copy of the lane: kept in registers
      // over the loop, the ten of a 96 x 64 tile's were spilled (4097 x 3001 x 2049 370 -> 364 us)
      int ln = lane;
      asm volatile("" : "+v"(ln));
      auto row_k = [&](int t) {
        int r, c;
        f32_slot_src(16 * (t & 3) + (ln >> 2), r, c);
        return 4 * c + (ln & 3);
      };
#pragma unroll
      for (int i = 0; i < S::A_DMA; ++i) {
        const int t = wave * S::A_DMA + i;
        dma_load4(ra, row_k(t) < krem ? a_off[i] : kBufOOB, dst + t * 256);
      }
#pragma unroll
      for (int i = 0; i < S::B_DMA; ++i) {
        const int t = wave * S::B_DMA + i;
        dma_load4(rb, (KN ? t / (BN / 64) : row_k(t)) < krem ? b_off[i] : kBufOOB, dst + S::A_BYTES + t * 256);
      }
    }
  };

  // ---- fragments: lane (r16 = l%16, g = l/16) ----
  const int r16 = lane & 15, g = lane >> 4;
  const uint32_t fa = f32_off(wm * S::WTM + r16, g);  // + 1024 per 16 rows
  const uint32_t fb_nk = S::A_BYTES + f32_off(wn * S::WTN + r16, g);
  // [K,N] B, MFMA step s, fragment j: row 4g + s, segment (wn*FN + j) ^ g, column r16.
  const uint32_t fb_kn = S::A_BYTES + (uint32_t)(4 * g * BN * 4 + 4 * r16);

  f32x4 acc[FM][FN];
  f32x4 small[FM][FN];  // the sums of the small products (not EXACT)
  // This wave's fragments of a stage (4 k per lane: k = 4g .. 4g+3)
  auto read_a = [&](int slot, int i) { return *(const f32x4*)(smem + slot * S::STAGE + fa + i * 1024); };
  auto read_b = [&](int slot, int j) {
    const unsigned char* stage = smem + slot * S::STAGE;
    if (!KN) return *(const f32x4*)(stage + fb_nk + j * 1024);
    f32x4 x;
#pragma unroll
    for (int s = 0; s < 4; ++s) x[s] = *(const float*)(stage + fb_kn + s * BN * 4 + (((wn * FN + j) ^ g) << 6));
    return x;
  };

  // The stages in ring slots slot and slot + 1 (V = u32x4: 32 k), or the one in slot (u32x2:
  // 16 k), on the bf16 instruction: B's next block is read and split among the current
  // one's products.  The fences between blocks bound the registers.  128 x 128 tiles of B as
  // [N,K] take products and vector instructions in a fixed pattern: x[512, 4096] W[4096,
  // 4096]^T 110 -> 107 us, x[100, 4096] 36.1 -> 34.6; as [K,N] it was slower (4096^3 730 ->
  // 746), on the small tiles no faster.
  auto split_stages = [&](int slot, auto v) {
    using V = decltype(v);
    using P = F32Planes<V>;
    constexpr bool PAIR = sizeof(V) == sizeof(u32x4);
    P pa[FM], pb[FN];
    auto split_a = [&](int i) {
      f32_split4(pa[i], 0, read_a(slot, i));
      if constexpr (PAIR) f32_split4(pa[i], 2, read_a(slot + 1, i));
    };
    auto split_b = [&](int j) {
      f32_split4(pb[j], 0, read_b(slot, j));
      if constexpr (PAIR) f32_split4(pb[j], 2, read_b(slot + 1, j));
    };
#pragma unroll
    for (int i = 0; i < FM; ++i) split_a(i);
    split_b(0);
    static_for<FN>([&](auto jc) {
      constexpr int j = decltype(jc)::value;
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (j + 1 < FN) split_b(j + 1);
      auto product = [&](f32x4(&sum)[FM][FN], V P::*b, V P::*a) {
#pragma unroll
        for (int i = 0; i < FM; ++i) sum[i][j] = f32_mma(pb[j].*b, pa[i].*a, sum[i][j]);
      };
      product(small, &P::l, &P::h);
      product(small, &P::h, &P::l);
      product(small, &P::m, &P::m);
      product(small, &P::m, &P::h);
      product(small, &P::h, &P::m);
      product(acc, &P::h, &P::h);
      if constexpr (PAIR && !KN && BM == 128 && j + 1 < FN) {
        static_for<6 * FM>([&](auto) {
          __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);  // one product,
          __builtin_amdgcn_sched_group_barrier(0x002, 2, 0);  // its share of the splitting (52 instructions)
        });
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  auto exact_stage = [&](int slot) {  // on the fp32 instruction
    f32x4 x[FM];
#pragma unroll
    for (int i = 0; i < FM; ++i) x[i] = read_a(slot, i);
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const f32x4 y = read_b(slot, j);
#pragma unroll
      for (int s = 0; s < 4; ++s)
#pragma unroll
        for (int i = 0; i < FM; ++i) acc[i][j] = mma_f32(y[s], x[i][s], acc[i][j]);
    }
  };
  // every load has landed and every wave's reads are done
  auto certify = [&]() { asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" : : : "memory"); };

#pragma unroll
  for (int i = 0; i < FM; ++i)
#pragma unroll
    for (int j = 0; j < FN; ++j) acc[i][j] = small[i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
  if constexpr (NS == 1) {
    load_stage(0);
    certify();
    exact_stage(0);
  } else {
    // Two stages at a time: stages st+2 and st+3 load into the slots that the iteration
    // before read while st and st+1 are multiplied.  Nothing is loaded past K, and an odd
    // stage is multiplied alone, by 16x16x16 products (a stage of zeros beside it took as
    // long as a full one: 20000 x 256 x 40 12.7 -> 11.5 us, 4096 x 4096 x 40 26.1 -> 24.3,
    // 1000 x 1001 x 24 7.5 -> 7.1).
    const int nst = (K + S::BK - 1) / S::BK;
    auto load_pair = [&](int st) {
      if (st < nst) load_stage(st);
      if (st + 1 < nst) load_stage(st + 1);
    };
    load_pair(0);
    certify();
    for (int st = 0; st + 1 < nst; st += 2) {
      const int slot = st & 2;
      load_pair(st + 2);
      if constexpr (EXACT) {
        exact_stage(slot);
        exact_stage(slot + 1);
      } else {
        split_stages(slot, u32x4{});
      }
      certify();
    }
    if (nst > 0 && (nst & 1)) {  // the last stage alone (a split past K's end has none)
      const int slot = (nst - 1) & 2;
      if constexpr (EXACT)
        exact_stage(slot);
      else
        split_stages(slot, u32x2{});
      certify();
    }
  }
  if constexpr (!EXACT) {
    bool again = false;
#pragma unroll
    for (int i = 0; i < FM; ++i)
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        acc[i][j] += small[i][j];
#pragma unroll
        for (int e = 0; e < 4; ++e) again |= !(__builtin_fabsf(acc[i][j][e]) <= 3.402823466e+38f);
        acc[i][j] *= kF32Unscale;
      }
    // (through the ring, which is free: __syncthreads_or's own LDS would cost the 96 x 64 tile
    // its fourth workgroup per CU)
    uint32_t* any = (uint32_t*)smem;
    const uint64_t lanes = __ballot(again);
    if (lane == 0) any[wave] = lanes != 0;
    __syncthreads();
    const uint32_t redo = any[0] | any[1] | any[2] | any[3];
    __syncthreads();
    if (redo) return true;
  }

  if constexpr (SPLITK) {  // fp32 partial sums, four consecutive columns per store (N % 4 == 0)
    const int batch = (int)gridDim.z / p.splits;
    float* part = p.partials + ((int64_t)ks * batch + bz) * M * N;
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int m = m0 + wm * S::WTM + i * 16 + r16;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int n = n0 + wn * S::WTN + j * 16 + 4 * g;
        if (m < M && n < N) *(f32x4*)(part + (int64_t)m * N + n) = acc[i][j];
      }
    }
    return false;
  }
  // acc[i][j][e] = C[m0 + wm*WTM + 16i + r16][n0 + wn*WTN + 16j + 4g + e]; elements
  // outside C get an out-of-range offset and are dropped by the store.
  const __amdgpu_buffer_rsrc_t crs = make_rsrc((float*)p.C + bz * p.stride_c + (int64_t)m0 * p.ldc + n0);
  const float* bias = p.bias_row ? nullptr : (const float*)p.bias;    // per column
  const float* rbias = p.bias_row ? (const float*)p.bias : nullptr;   // per row
  float bv[FN][4];
#pragma unroll
  for (int j = 0; j < FN; ++j)
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const int n = n0 + wn * S::WTN + j * 16 + 4 * g + e;
      bv[j][e] = (bias != nullptr && n < N) ? bias[n] : 0.f;
    }
  // C rows 16-byte aligned and N % 4 == 0: one 16-byte store per lane and block (the four
  // columns are all inside C or all outside), measured 8.3 -> 1.9 us per workgroup epilogue
  // on MI355X with every workgroup of a 256-CU launch storing at once.
  if (((p.ldc | N) & 3) == 0 && ((uintptr_t)((const float*)p.C + bz * p.stride_c) & 15) == 0) {
#pragma unroll
    for (int i = 0; i < FM; ++i) {
      const int row = wm * S::WTM + i * 16 + r16;
      const bool row_ok = m0 + row < M;
      const float bm = (rbias != nullptr && row_ok) ? rbias[m0 + row] : 0.f;
#pragma unroll
      for (int j = 0; j < FN; ++j) {
        const int col = wn * S::WTN + j * 16 + 4 * g;
        f32x4 v = acc[i][j];
        if (bias != nullptr) v += f32x4{bv[j][0], bv[j][1], bv[j][2], bv[j][3]};
        if (rbias != nullptr) v += bm;
        buf_store16(crs, row_ok && n0 + col < N ? (uint32_t)(row * p.ldc + col) * 4u : kBufOOB, v);
      }
    }
    return false;
  }
#pragma unroll
  for (int i = 0; i < FM; ++i) {
    const int row = wm * S::WTM + i * 16 + r16;
    const bool row_ok = m0 + row < M;
    const float bm = (rbias != nullptr && row_ok) ? rbias[m0 + row] : 0.f;
#pragma unroll
    for (int j = 0; j < FN; ++j) {
      const int col = wn * S::WTN + j * 16 + 4 * g;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const bool ok = row_ok && n0 + col + e < N;
        const float x = bias != nullptr ? acc[i][j][e] + bv[j][e]
                        : rbias != nullptr ? acc[i][j][e] + bm : acc[i][j][e];
        buf_store4(crs, ok ? (uint32_t)(row * p.ldc + col + e) * 4u : kBufOOB, x);
      }
    }
  }
  return false;
}

// WAVES: waves per SIMD the kernel is compiled for (caps its registers at 512 / WAVES).
template <bool KN, int BM, int BN, int WAVES, bool SPLITK = false, bool DMA16 = false>
__global__ void __launch_bounds__(256, WAVES) gemm_f32_kernel(const GemmParams p) {
  using S = F32Shape<BM, BN, 4>;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[4 * S::STAGE];
  if (p.K <= kF32ShortK || f32_tile<KN, BM, BN, SPLITK, DMA16, false>(p, smem))
    f32_tile<KN, BM, BN, SPLITK, DMA16, true>(p, smem);
}

// K <= kF32ShortK: products of one stage are bound by writing C, and each sum has too few
// terms for the planes to round it less often than the fp32 instruction does.  One load and
// no ring, so that eight workgroups share a CU and some write their tiles while others wait
// for their operands.  MI355X, 64 x 64 tiles, the ring kernel on planes -> this: 4096 x 4096
// x 16 22.4 -> 15.9 us (4.2 TB/s written), 8192 x 1024 x 8 13.7 -> 10.3, 3000 x 2001 x 1 (rows
// not 16-byte aligned) 20.4 -> 18.0, 1000 x 1001 x 16 6.8 -> 5.7.
template <bool KN, int BM, int BN, int WAVES, bool DMA16>
__global__ void __launch_bounds__(256, WAVES) gemm_f32_short_kernel(const GemmParams p) {
  using S = F32Shape<BM, BN, 1>;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[S::STAGE];
  f32_tile<KN, BM, BN, false, DMA16, true, 1>(p, smem);
}

}  // namespace cmpext3
