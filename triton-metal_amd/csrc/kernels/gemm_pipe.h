// Pipelined MFMA matrix product for gfx950 (16-bit and FP8 inputs, fp32
// accumulation): one workgroup of 4 waves (2 x 2) per (64 RT) x (64 CT) tile of
//
//   C[b, m, n] = sum_k A[b, m, k] B[b, k, n]  (+ Z[b, m, n] | Z[b, m, 0] | Z[b, 0, n])
//
// with either operand k-contiguous or row-contiguous, any M, N, K and alignment.
// Semantics: make_matmul_kernel, make_fused_linear_kernel and the strided dot
// template (_msl_templates.py:447-585, 4013-4135; _lowerer_templates.py:
// 1116-1540).
//
// K runs in stages of 128 bytes per row through a ring of NS stages in LDS.
// Both operands go global -> LDS through bounds-checked buffer descriptors (rows
// and k past the operand deposit zeros), the copies of a stage spread over two
// of the four k steps, one barrier per stage; the operands of the next k step are
// read while the current one multiplies.  The 256 x 256 tile gives a wave 128 x
// 128 outputs (accumulators in AGPRs, one wave per SIMD): 192 KB of LDS reads per
// stage fall to 128.
//
// What bounds it (256 x 256 tiles on every CU, bf16, us per stage): MFMA on
// constant data 1.11, with random data and the LDS reads 1.28 (the clock under
// the power limit), copies alone 0.88, all of it 1.49; the rest is 13 us per round
// of tiles (first copies, C).  us, kernels it replaced -> this: fp16 2000 x 11008
// x 4096 260 -> 196, e4m3 2048 x 4096 x 4096 178 -> 59, transposed A with add-
// matrix 4096 x 4096 x 2000 204 -> 86.  (Aligned products whose 256-tiles fill the
// chip keep gemm_t256: 4096^3 on one set of buffers 118, here 123.)
#pragma once
#include "common.h"

// Kernel arguments (ops_mm.cpp holds the same struct).
struct MmParams {
  const void* A;
  const void* B;
  void* C;
  const void* Z;
  long long sa_b, sb_b, sc_b, sz_b;  // batch strides (elements)
  long long sc_m, sc_n, sz_m, sz_n;  // C and Z strides (elements)
  int M, N, K;
  int lda, ldb;      // row stride (k-contiguous) or k stride (row-contiguous), elements
  int tiles_m, tiles_n;
  int epi;           // 0: Z unused; else + Z (add-rows / -cols: sz_n / sz_m 0)
  int out_dt, z_dt;  // TM_DT_F32 / F16 / BF16
  int vec_z;         // Z's columns contiguous (sz_n 1)
  int fix;           // pieces that no copy may take whole (FIX_*)
};

namespace mm {

enum { F16 = 0, BF16 = 1, E4M3 = 2, E5M2 = 3 };

// MmParams::fix: a k-contiguous operand whose K is no whole number of 16-byte
// pieces; a row-contiguous one whose rows do not start on 16 bytes (a piece
// across the end of its last k row could reach into another page).  Those
// pieces are filled by element loads.
enum { FIX_AK = 1, FIX_BK = 2, FIX_AR = 4, FIX_BR = 8 };

typedef short s4v_t __attribute__((ext_vector_type(4)));
typedef int i2v_t __attribute__((ext_vector_type(2)));
typedef int i8v_t __attribute__((ext_vector_type(8)));
typedef __attribute__((address_space(3))) s4v_t lds_s4_t;
typedef __attribute__((address_space(3))) i2v_t lds_i2_t;
typedef __attribute__((address_space(3))) u4_t lds_u4_t;
typedef __attribute__((address_space(3))) f4_t lds_f4_t;
typedef __attribute__((address_space(3))) float lds_f_t;

// voffset of a copy whose source is past the operand: beyond every buffer's
// extent (the host keeps them below 2 GiB), so the load deposits zeros.
constexpr uint32_t kOob = 0x80000000u;

// Global -> LDS copy through a buffer descriptor: lane l deposits 16 bytes at
// lds + 16 l (the source at any alignment of its elements), zeros where a dword
// is past the buffer.  Issued in asm for the
// reasons dma16 is (common.h); waited for with wait_vm.
TM_DEV void buf16(u4_t rsrc, uint32_t voff, uint32_t lds) {
  asm volatile("s_mov_b32 m0, %2\n\ts_nop 0\n\tbuffer_load_dwordx4 %0, %1, 0 offen lds" ::"v"(voff),
               "s"(rsrc), "s"(lds)
               : "memory", "m0");
}

TM_DEV u4_t buf_rsrc(const void* base, uint32_t bytes) {
  const uint64_t a = (uint64_t)base;
  u4_t r;
  r.x = __builtin_amdgcn_readfirstlane((uint32_t)a);
  r.y = __builtin_amdgcn_readfirstlane((uint32_t)(a >> 32) & 0xffffu);
  r.z = __builtin_amdgcn_readfirstlane(bytes);
  r.w = 0x00020000u;
  return r;
}

// One operand's tile: 64 R rows x 128 bytes of k, either [row][k] (RC false:
// rows of 128 bytes, piece p of row r at p ^ ((r >> 1) & 7), so that the 16
// rows of a read phase fall in 16 different 16-byte bank groups) or [k][row]
// (RC true: rows of 64 R elements, piece p of row k at p ^ sw(k), so that the
// four k rows of a transposing read fall in different 64-byte bank groups).
template <int KIND, bool RC, int R> struct Tile {
  static constexpr int ES = KIND >= E4M3 ? 1 : 2;
  static constexpr int BK = 128 / ES;
  static constexpr int ROWS = 64 * R;
  static constexpr int BYTES = ROWS * 128;
  static constexpr int NCP = 2 * R;      // copies per wave per step (4 waves)
  static constexpr int RB = ROWS * ES;   // bytes of a [k] row (RC)
  static constexpr int PPR = RB / 16;    // pieces of a [k] row (RC)

  // 16-byte piece swizzle of k row kr (RC); 16-bit: 4 k rows x 64 bytes per
  // read phase, 8-bit: 8 k rows x 32 bytes
  static TM_DEV int sw_rc(int kr) {
    if constexpr (ES == 2) {
      if constexpr (PPR >= 16) return 4 * (kr & 3);
      else return 4 * ((kr >> 1) & 1);
    } else {
      if constexpr (PPR >= 16) return 2 * (kr & 7);
      else if constexpr (PPR >= 8) return 2 * ((kr >> 1) & 3);
      else return 2 * ((kr >> 2) & 1);
    }
  }
  // voffset of copy i of this wave (relative to the tile's first row / column
  // and k = 0), kOob for rows past `rows`
  static TM_DEV uint32_t voff(int wave, int lane, int i, int ld, int rows) {
    const int blk = NCP * wave + i;
    if constexpr (!RC) {
      const int r = 8 * blk + (lane >> 3), p = (lane & 7) ^ ((r >> 1) & 7);
      return r < rows ? (uint32_t)r * (uint32_t)ld * ES + 16u * p : kOob;
    } else {
      const int s = 64 * blk + lane, kr = s / PPR, p = (s % PPR) ^ sw_rc(kr);
      return p * (16 / ES) < rows ? (uint32_t)kr * (uint32_t)ld * ES + 16u * p : kOob;
    }
  }
  // whether copy i's piece lies before k = left of the step
  static TM_DEV bool in_k(int wave, int lane, int i, int left) {
    const int blk = NCP * wave + i;
    if constexpr (!RC) {
      const int r = 8 * blk + (lane >> 3), p = (lane & 7) ^ ((r >> 1) & 7);
      return (p + 1) * (16 / ES) <= left;
    } else {
      return (64 * blk + lane) / PPR < left;
    }
  }
  // One piece of the stage at LDS `st` from n elements at src, zeros after
  static TM_DEV void piece(uint32_t dst, const uint8_t* src, int n) {
    u4_t v = {0u, 0u, 0u, 0u};
    for (int e = 0; e < n; ++e) {
      const uint32_t x = ES == 2 ? ((const uint16_t*)src)[e] : src[e];
      const int at = e * ES;
#pragma unroll
      for (int d = 0; d < 4; ++d)
        if ((at >> 2) == d) v[d] |= x << (8 * (at & 3));
    }
    *(lds_u4_t*)(dst) = v;
  }
  // The pieces of the last step that the copies left out: base = the tile's
  // first row (column) at the step's k, kl = k left (1 .. BK), rows as voff
  static TM_DEV void fill(uint32_t st, const uint8_t* base, int ld, int kl, int rows, int tid) {
    constexpr int EP = 16 / ES;
    if constexpr (!RC) {
      const int pc = kl / EP;
      for (int r = tid; r < ROWS; r += 256)
        piece(st + 128 * r + 16 * (pc ^ ((r >> 1) & 7)),
              base + ((size_t)r * ld + pc * EP) * ES, r < rows ? kl - pc * EP : 0);
    } else if (rows % EP && tid == 0) {
      const int pc = rows / EP, kr = kl - 1;
      piece(st + RB * kr + 16 * (pc ^ sw_rc(kr)), base + ((size_t)kr * ld + pc * EP) * ES,
            rows - pc * EP);
    }
  }
};

// FP8 operands are staged as bytes and become fp16 between the LDS read and the
// MFMA (every e4m3 / e5m2 value is exactly an fp16 value).  The FP8 MFMAs run
// at up to twice the rate but do not keep the product sums to fp32: 1.3e-5
// relative error against 4e-8 on the same inputs.
template <int KIND> TM_DEV u4_t from_bytes(uint32_t lo, uint32_t hi) {
  if constexpr (KIND == E5M2) {  // fp16 with the mantissa's low byte zero
    return u4_t{perm_b32(0, lo, 0x010c000cu), perm_b32(0, lo, 0x030c020cu),
                perm_b32(0, hi, 0x010c000cu), perm_b32(0, hi, 0x030c020cu)};
  } else {
    return u4_t{h2_bits(__builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, false))),
                h2_bits(__builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 1.0f, true))),
                h2_bits(__builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, false))),
                h2_bits(__builtin_bit_cast(h2_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 1.0f, true)))};
  }
}

// Reader of one operand's tile.  The per-lane LDS addresses are computed once;
// k step and (k-contiguous) row block are immediate offsets of the reads.  A
// read of k step kk (four to a stage) gives lane l row l % 32 of a 32-row
// block with, in either layout, the same k in its 16 bytes: 16-bit
// k = 16 kk + 8 (l / 32) + e, 8-bit k = 32 kk + 16 (l / 32) + e.
template <int KIND, bool RC, int R, int RT> struct Reader {
  using T = Tile<KIND, RC, R>;
  // k-contiguous: one address per piece pair (pieces 2 q + lane / 32);
  // row-contiguous: one per 32-row block (the swizzle crosses blocks)
  static constexpr int NAD = RC ? RT : 4;
  uint32_t ad[NAD];

  TM_DEV Reader(uint32_t base, int row0, int lane) {
    if constexpr (!RC) {
      const int r = row0 + (lane & 31), sw = (r >> 1) & 7;
#pragma unroll
      for (int q = 0; q < 4; ++q) ad[q] = base + 128u * r + 16u * ((2 * q + (lane >> 5)) ^ sw);
    } else {
      // 16-lane group g of the wave, lane j of it: the lanes of a transposing
      // read address 8 bytes of 4 (8) k rows x 16 tile rows
      const int g = lane >> 4, j = lane & 15, h = g >> 1;
      const int c = row0 + 16 * (g & 1) + (T::ES == 2 ? 4 * (j & 3) : 8 * (j & 1));
      const int k = T::ES == 2 ? 8 * h + (j >> 2) : 16 * h + (j >> 1);
      constexpr int EP = 16 / T::ES;
#pragma unroll
      for (int rb = 0; rb < RT; ++rb)
        ad[rb] = base + (uint32_t)(k * T::RB + 16 * (((c + 32 * rb) / EP) ^ T::sw_rc(k)) +
                                   (c % EP) * T::ES);
    }
  }

  TM_DEV u4_t read(int rb, int kk) const {
    if constexpr (!RC) {
      return *(lds_u4_t*)(ad[kk] + rb * 4096);
    } else if constexpr (T::ES == 2) {
      const uint32_t a = ad[rb] + 16 * kk * T::RB;
      const u2_t lo =
          __builtin_bit_cast(u2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t*)(a)));
      const u2_t hi = __builtin_bit_cast(
          u2_t, __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_s4_t*)(a + 4 * T::RB)));
      return u4_t{lo.x, lo.y, hi.x, hi.y};
    } else {
      const uint32_t a = ad[rb] + 32 * kk * T::RB;
      const i2v_t lo = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i2_t*)(a));
      const i2v_t hi = __builtin_amdgcn_ds_read_tr8_b64_v2i32((lds_i2_t*)(a + 8 * T::RB));
      return u4_t{(uint32_t)lo.x, (uint32_t)lo.y, (uint32_t)hi.x, (uint32_t)hi.y};
    }
  }
};

template <int DT> TM_DEV u4_t pack8(f4_t x, f4_t y) {
  if constexpr (DT == TM_DT_BF16)
    return u4_t{pack_bf16x2(x[0], x[1]), pack_bf16x2(x[2], x[3]), pack_bf16x2(y[0], y[1]),
                pack_bf16x2(y[2], y[3])};
  else
    return u4_t{pack_f16x2(x[0], x[1]), pack_f16x2(x[2], x[3]), pack_f16x2(y[0], y[1]),
                pack_f16x2(y[2], y[3])};
}

// 16 bytes at an element's own alignment (one dwordx4 access: global memory
// takes any alignment), for rows that do not start on 16 bytes
typedef u4_t u4e_t __attribute__((aligned(2)));
typedef f4_t f4e_t __attribute__((aligned(4)));

// x, y += the 8 consecutive elements at Z + i
TM_DEV void add8(const void* Z, long long i, int dt, f4_t* x, f4_t* y) {
  if (dt == TM_DT_F32) {
    *x += *(const f4e_t*)((const float*)Z + i);
    *y += *(const f4e_t*)((const float*)Z + i + 4);
  } else {
    const u4_t z = *(const u4e_t*)((const uint16_t*)Z + i);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      const uint16_t b = (uint16_t)(z[e >> 1] >> (16 * (e & 1)));
      const float f = dt == TM_DT_BF16 ? bf16_bits_to_f32(b) : f16_bits_to_f32(b);
      if (e < 4) (*x)[e] += f;
      else (*y)[e - 4] += f;
    }
  }
}

// tile index of this workgroup: the 8 XCDs take workgroups in turn, so each
// gets a contiguous run of the tile order, which walks 8 tile rows column by
// column (the tiles in flight on an XCD share A and B panels in its L2)
TM_DEV void tile_of(int id, int tiles_m, int tiles_n, int* tm, int* tn) {
  const int total = tiles_m * tiles_n;
  const int q = total >> 3, r = total & 7, x = id & 7, i = id >> 3;
  const int t = x * q + (x < r ? x : r) + i;
  const int per = 8 * tiles_n;
  const int grp = t / per, in = t - grp * per;
  const int first = grp * 8, gm = tiles_m - first < 8 ? tiles_m - first : 8;
  *tn = in / gm;
  *tm = first + (in - *tn * gm);
}

}  // namespace mm

template <int KIND, bool ARC, bool BRC, int RT, int CT, int NS>
__device__ __forceinline__ void mm_body(const MmParams& p) {
  using namespace mm;
  using TA = Tile<KIND, ARC, RT>;
  using TB = Tile<KIND, BRC, CT>;
  constexpr int ES = TA::ES, BK = TA::BK, BM = 64 * RT, BN = 64 * CT;
  constexpr int NKK = 4;  // k steps per stage (two MFMAs each for 8-bit operands)
  constexpr bool FP8 = ES == 1;
  // [NS A stages | NS B stages]
  constexpr int STA = TA::BYTES, STB = TB::BYTES, LDSB = NS * STA;
  __shared__ __align__(1024) uint8_t smem[NS * (STA + STB)];
  const uint32_t lds0 = lds_off(smem);

  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN, K = p.K;
  const int mr = p.M - m0, nr = p.N - n0;  // rows / columns left (may exceed the tile)
  const long long b = blockIdx.y;

  // ---- copies.  The buffers start at the step's k, so their offsets stay
  // within one tile's rows (k-contiguous) or one step's k rows (row-contiguous)
  const uint8_t* abase = (const uint8_t*)p.A +
      (size_t)(b * p.sa_b + (ARC ? (long long)m0 : (long long)m0 * p.lda)) * ES;
  const uint8_t* bbase = (const uint8_t*)p.B +
      (size_t)(b * p.sb_b + (BRC ? (long long)n0 : (long long)n0 * p.ldb)) * ES;
  const int ar = mr < BM ? mr : BM, br = nr < BN ? nr : BN;
  // row-contiguous buffers end with the last aligned piece that holds an
  // element (the bounds check drops whole dwords)
  constexpr int EP = 16 / ES;
  const int arp = (ar + EP - 1) / EP * EP, brp = (br + EP - 1) / EP * EP;
  const int arl = (p.fix & FIX_AR) ? ar : arp, brl = (p.fix & FIX_BR) ? br : brp;  // last step
  const size_t astep = ARC ? (size_t)p.lda * BK * ES : 128u;
  const size_t bstep = BRC ? (size_t)p.ldb * BK * ES : 128u;
  uint32_t av[TA::NCP], bv[TB::NCP];
#pragma unroll
  for (int i = 0; i < TA::NCP; ++i) av[i] = TA::voff(wave, lane, i, p.lda, ar);
#pragma unroll
  for (int i = 0; i < TB::NCP; ++i) bv[i] = TB::voff(wave, lane, i, p.ldb, br);
  const int nk = (K + BK - 1) / BK;
  const uint32_t la = lds0 + 1024u * TA::NCP * wave, lb = lds0 + LDSB + 1024u * TB::NCP * wave;

  // copy i of step kt (A's first, then B's) into stage s; pieces at or past
  // k = K, and whole steps past the last one, deposit zeros
  auto copy = [&](auto ic, int s, int kt) {
    constexpr int i = decltype(ic)::value;
    const int left = K - kt * BK, ks = kt < nk ? kt : nk - 1;
    const int kl = K - ks * BK;  // k left from the buffer's start, > 0
    if constexpr (i < TA::NCP) {
      const uint32_t v = TA::in_k(wave, lane, i, left) ? av[i] : kOob;
      const u4_t r = buf_rsrc(abase + ks * astep,
                              ARC ? ((uint32_t)((kl < BK ? kl : BK) - 1) * p.lda + (ks + 1 < nk ? arp : arl)) * ES
                                  : ((uint32_t)(ar - 1) * p.lda + kl) * ES);
      buf16(r, v, la + s * STA + 1024 * i);
    } else {
      constexpr int j = i - TA::NCP;
      const uint32_t v = TB::in_k(wave, lane, j, left) ? bv[j] : kOob;
      const u4_t r = buf_rsrc(bbase + ks * bstep,
                              BRC ? ((uint32_t)((kl < BK ? kl : BK) - 1) * p.ldb + (ks + 1 < nk ? brp : brl)) * ES
                                  : ((uint32_t)(br - 1) * p.ldb + kl) * ES);
      buf16(r, v, lb + s * STB + 1024 * j);
    }
  };
  // copies per wave and step: the first NC1 are issued behind the step's
  // barrier, the rest one substep later (spread over two substeps they disturb
  // the MFMAs least: 4096 x 4096 x 8192 bf16 205 us, all behind the barrier 213,
  // over all four substeps 224)
  constexpr int NC = TA::NCP + TB::NCP, NC1 = NC / 2, NM = RT * CT * (FP8 ? 2 : 1);
  auto copies = [&](int s, int kt) {
    static_for<0, NC>([&](auto i) { copy(i, s, kt); });
  };

  Reader<KIND, ARC, RT, RT> rda(lds0, 32 * RT * wm, lane);
  Reader<KIND, BRC, CT, CT> rdb(lds0 + LDSB, 32 * CT * wn, lane);

  f16_t acc[RT][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = f16_t{};

  // operands of two k steps; 8-bit ones also as read, before they become fp16
  constexpr int NV = FP8 ? 2 : 1;
  u4_t ao[2][RT][NV], bo[2][CT][NV], raw[FP8 ? RT + CT : 1];
  auto rd = [&](auto Sc, auto yc, int kk) {
    constexpr int S = decltype(Sc)::value, y = decltype(yc)::value;
    u4_t v;
    if constexpr (y < CT) v = rdb.read(y, kk);
    else v = rda.read(y - CT, kk);
    if constexpr (FP8) raw[y] = v;
    else if constexpr (y < CT) bo[S][y][0] = v;
    else ao[S][y - CT][0] = v;
  };
  auto widen = [&](auto Sc, auto yc) {
    constexpr int S = decltype(Sc)::value, y = decltype(yc)::value;
    if constexpr (FP8) {
      u4_t* o = y < CT ? bo[S][y] : ao[S][y - CT];
      o[0] = from_bytes<KIND>(raw[y].x, raw[y].y);
      o[1] = from_bytes<KIND>(raw[y].z, raw[y].w);
    }
  };
  static_for<0, NS - 1>([&](auto kt) { copies(kt, kt); });
  static_for<0, NC1>([&](auto i) { copy(i, NS - 1, NS - 1); });
  wait_vm<(NS - 2) * NC + NC1>();
  asm volatile("s_barrier" ::: "memory");
  // the last step's pieces that the copies left out, once the step has landed
  auto fill = [&](int s) {
    const int kl = K - (nk - 1) * BK;
    if (p.fix & (ARC ? FIX_AR : FIX_AK))
      TA::fill(lds0 + s * STA, abase + (nk - 1) * astep, p.lda, kl, ar, tid);
    if (p.fix & (BRC ? FIX_BR : FIX_BK))
      TB::fill(lds0 + LDSB + s * STB, bbase + (nk - 1) * bstep, p.ldb, kl, br, tid);
    lds_barrier();
  };
  if (p.fix && nk == 1) fill(0);
  {
    std::integral_constant<int, 0> z;
    static_for<0, RT + CT>([&](auto y) { rd(z, y, 0); });
    static_for<0, RT + CT>([&](auto y) { widen(z, y); });
  }

  // MFMAs of one k step on operand set S, with the reads of k step kk into the
  // other set spread between them
  auto substep = [&](auto Sc, int kk, auto&& after) {
    constexpr int S = decltype(Sc)::value;
    constexpr std::integral_constant<int, 1 - S> other;
    static_for<0, NM>([&](auto xc) {
      constexpr int x = decltype(xc)::value, v = x / (RT * CT), i = x % (RT * CT) / CT, j = x % CT;
      if constexpr (x < CT + RT) rd(other, xc, kk);
      if constexpr (x == NM - 1) static_for<NM, CT + RT>([&](auto y) { rd(other, y, kk); });
      // operands swapped: the result holds 4 consecutive columns n per lane
      acc[i][j] = mfma32<KIND == BF16>(bo[S][j][v], ao[S][i][v], acc[i][j]);
      after(xc);
      if constexpr (FP8)  // the second half's slots widen what the first half's read
        static_for<0, CT + RT>([&](auto y) {
          if constexpr (NM / 2 + decltype(y)::value * (NM / 2) / (CT + RT) == x) widen(other, y);
        });
      __builtin_amdgcn_sched_barrier(0);
    });
  };
  // One step per stage.  Its last substep starts with the barrier after which
  // every wave has read this stage and every wave's copies of the next step
  // have landed; the copies of step kt + NS then go into this stage.  (After
  // the last step the reads fetch another stage's old data, unused.)
  int st = 0;  // stage of step kt
  for (int kt = 0; kt < nk; ++kt) {
    const int prev = st == 0 ? NS - 1 : st - 1, up = st == NS - 1 ? 1 - NS : 1;
    static_for<0, NKK - 1>([&](auto kc) {
      constexpr int kk = decltype(kc)::value;
      substep(std::integral_constant<int, kk & 1>{}, kk + 1, [&](auto xc) {
        constexpr int x = decltype(xc)::value;
        if constexpr (kk == 0)
          static_for<NC1 + x * (NC - NC1) / NM, NC1 + (x + 1) * (NC - NC1) / NM>(
              [&](auto i) { copy(i, prev, kt + NS - 1); });
      });
    });
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * NC) : "memory");
    if (p.fix && kt + 2 == nk) fill(st + up);
#pragma unroll
    for (int q = 0; q < decltype(rda)::NAD; ++q) rda.ad[q] += up * STA;
#pragma unroll
    for (int q = 0; q < decltype(rdb)::NAD; ++q) rdb.ad[q] += up * STB;
    substep(std::integral_constant<int, (NKK - 1) & 1>{}, 0, [&](auto xc) {
      constexpr int x = decltype(xc)::value;
      static_for<x * NC1 / NM, (x + 1) * NC1 / NM>([&](auto i) { copy(i, st, kt + NS); });
    });
    st += up;
  }

  // ---- epilogue.  acc[i][j] of lane l: row m = 32 i + l % 32 of the wave's
  // rows, columns n = 32 j + 8 (e / 4) + 4 (l / 32) + e % 4.
  const int mw = m0 + 32 * RT * wm, nw = n0 + 32 * CT * wn;
  const int l32 = lane & 31, h = lane >> 5;
  // through LDS in blocks of 32 rows x 32 CT columns of fp32 per wave, so that
  // C (and an add-matrix Z) move in row-contiguous 16-byte pieces
  constexpr int LDW = 32 * CT + 4;  // floats per staged row
  static_assert(4 * 32 * LDW * 4 <= NS * (STA + STB), "epilogue staging");
  wait_vm<0>();
  __syncthreads();  // the stages are free
  const uint32_t eb = lds0 + (uint32_t)wave * 32 * LDW * 4;
  const long long cb = b * p.sc_b, zb = b * p.sz_b;
  const bool full = mw + 32 * RT <= p.M && nw + 32 * CT <= p.N;
  static_for<0, RT>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int q = 0; q < 4; ++q)
        *(lds_f4_t*)(eb + 4u * (l32 * LDW + 32 * j + 8 * q + 4 * h)) =
            f4_t{acc[i][j][4 * q], acc[i][j][4 * q + 1], acc[i][j][4 * q + 2],
                 acc[i][j][4 * q + 3]};
    {
      // out in pieces of 8 columns, 4 CT lanes to a row; ragged tiles skip the
      // pieces outside (and write the one across N's end by elements below)
      constexpr int LPR = 4 * CT, NP = 2 * CT;
      const int c = 8 * (lane % LPR), n = nw + c;
      const auto row = [&](int t) { return t * (64 / LPR) + lane / LPR; };
      f4_t x[NP], y[NP];
#pragma unroll
      for (int t = 0; t < NP; ++t) {
        x[t] = *(lds_f4_t*)(eb + 4u * (row(t) * LDW + c));
        y[t] = *(lds_f4_t*)(eb + 4u * (row(t) * LDW + c + 4));
      }
#pragma unroll
      for (int t = 0; t < NP; ++t) {
        const int m = mw + 32 * i + row(t);
        if (!full && (m >= p.M || n + 8 > p.N)) continue;
        if (p.epi) {
          const long long zi = zb + (long long)m * p.sz_m + n * p.sz_n;
          if (p.vec_z) {
            add8(p.Z, zi, p.z_dt, &x[t], &y[t]);
          } else if (p.sz_n == 0) {
            const float z = load_as_f32_rt(p.Z, zi, p.z_dt);
            x[t] += z;
            y[t] += z;
          } else {
#pragma unroll
            for (int e = 0; e < 4; ++e) {
              x[t][e] += load_as_f32_rt(p.Z, zi + e * p.sz_n, p.z_dt);
              y[t][e] += load_as_f32_rt(p.Z, zi + (e + 4) * p.sz_n, p.z_dt);
            }
          }
        }
        const long long ci = cb + (long long)m * p.sc_m + n;
        if (p.out_dt == TM_DT_F32) {
          *(f4e_t*)((float*)p.C + ci) = x[t];
          *(f4e_t*)((float*)p.C + ci + 4) = y[t];
        } else if (p.out_dt == TM_DT_BF16) {
          *(u4e_t*)((uint16_t*)p.C + ci) = pack8<TM_DT_BF16>(x[t], y[t]);
        } else {
          *(u4e_t*)((uint16_t*)p.C + ci) = pack8<TM_DT_F16>(x[t], y[t]);
        }
      }
    }
    // the columns past the last whole piece, element by element, a lane per row
    const int nf = p.N & ~7;
    if (nf < p.N && nf >= nw && nf < nw + 32 * CT) {
      const int m = mw + 32 * i + l32;
      if (m < p.M && h == 0)
        for (int n = nf; n < p.N; ++n) {
          float v = *(lds_f_t*)(eb + 4u * (l32 * LDW + n - nw));
          if (p.epi)
            v += load_as_f32_rt(p.Z, zb + (long long)m * p.sz_m + n * p.sz_n, p.z_dt);
          store_as_f32_rt(p.C, cb + (long long)m * p.sc_m + n, p.out_dt, v);
        }
    }
  });
}
