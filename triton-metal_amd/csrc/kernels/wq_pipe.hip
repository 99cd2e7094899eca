// Weight-only matmul on pipelined MFMA tiles, for the sizes the streaming and
// wide kernels do not take (K a multiple of 128 only, any M and N % 16 == 0) and for
// products large enough to fill the chip with 128 x 128 tiles:
//
//   Y[m, n] = sum_k X[m, k] (q(n, k) - z(n, g)) s(n, g)   (+ bias[n])
//
// int4 with groups of 128 (any zero-points) and int8 with one scale per
// channel and no zero-points; fp16 or bf16 activations; arithmetic of
// make_int4_matmul_kernel / make_int8_matmul_kernel (_msl_templates.py:
// 2652-2745) with fp32 sums.
//
// A workgroup of 4 waves (2 x 2) owns 64 RT rows x 128 columns; K runs in
// stages of 64 k through a three-stage LDS ring filled by bounds-checked
// global -> LDS copies (rows past M or N deposit zeros).  The weights stay
// packed in LDS and become exact 16-bit operands in registers, so nothing is
// rounded before the fp32 sums.  int8: q.  int4, per group
//   y += s (sum x (q - c) - (z - c) sum x)
// with c the centre of the operands and the group's sum x from wq_pipe_prep,
// which also writes X in the order the int4 operands come out in (n0 n4 n1 n5 n2
// n6 n3 n7 of each 8).  fp16: c = z without zero-points or with uint8 ones (one
// packed subtraction per pair of operands and no second term), -64 with fp16 ones;
// bf16: c = -128.  (c = -1024, the cheapest fp16 operand, left ten bits less to the
// fp32 sums: relative error of the fp16 result at K = 7040 2.079e-4 against 2.076e-4
// in exact sums, 2.084e-4 against 2.066e-4 for activations of mean 1.  bf16's sums
// are 1.5e-6 off, a thousandth of the result's rounding.)
// A lane holds one column per 32-column block (its scale is one register) and
// 16 rows.  With a k slice per grid row the fp32 sums go to P[slice][M][N].
// Two workgroups share a CU: the VALU work of one (per MFMA 4 operations of the
// group updates and 1.3 of the int4 operand builds) overlaps the MFMAs of the
// other.  us, start -> here: int4 M = 1000 K = 4096 N = 28672 bf16 593 -> 277 (850
// TFLOP/s), K = 11008 N = 4096 fp16 239 -> 128, M = 228 K = 7040 N = 2816 bf16 1367
// -> 30; int8 M = 700 K = 4096 N = 22016 fp16 167 -> 153.
#include "wq_common.h"
#include "gemm_pipe.h"

struct WqPipeParams {
  const void* X;       // [M, K], int4: as wq_pipe_prep writes it
  const uint16_t* X0;  // [M, K] as the caller has it
  const uint8_t* W;
  const void* S;
  const void* Z;
  const float* SX;     // int4: [K / 128][M rounded up to 4] sums of each group
  void* Y;             // [M, N], or null: P
  float* P;            // [slices][M][N]
  const uint16_t* bias;
  int M, N, K, kslice; // kslice: k per grid row, a multiple of 128
  int tiles_m, tiles_n, sxld;
};

// X in operand order and the sums of its groups: a thread per 8 k, 16 threads
// per group; grid (M, ceil(K / 2048)): any number of rows (y holds 65535).
template <bool BF16> TM_DEV void wq_pipe_prep_body(const uint16_t* X, uint16_t* XP, float* SX,
                                                   int K, int sxld) {
  const int m = blockIdx.x, k = 2048 * blockIdx.y + 8 * threadIdx.x;
  if (k >= K) return;  // K % 128 == 0: whole groups of 16 lanes leave
  const u4_t x = ldg128(X + (size_t)m * K + k);
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const uint16_t lo = x[i] & 0xffff, hi = x[i] >> 16;
    s += BF16 ? bf16_bits_to_f32(lo) + bf16_bits_to_f32(hi)
              : f16_bits_to_f32(lo) + f16_bits_to_f32(hi);
  }
  s = row16_sum(s);
  *(u4_t*)(XP + (size_t)m * K + k) = perm_x8(x);
  if ((threadIdx.x & 15) == 0) SX[(size_t)(k >> 7) * sxld + m] = s;
}
extern "C" __global__ __launch_bounds__(256) void wq_pipe_prep_f16(const uint16_t* X, uint16_t* XP,
                                                                   float* SX, int K, int sxld) {
  wq_pipe_prep_body<false>(X, XP, SX, K, sxld);
}
extern "C" __global__ __launch_bounds__(256) void wq_pipe_prep_bf16(const uint16_t* X,
                                                                    uint16_t* XP, float* SX,
                                                                    int K, int sxld) {
  wq_pipe_prep_body<true>(X, XP, SX, K, sxld);
}

template <int QB, bool BF16, int ZDT, int RT>
__device__ __forceinline__ void wq_pipe_body(const WqPipeParams& p) {
  using namespace mm;
  constexpr int CT = 2, NS = 3, BM = 64 * RT, BN = 64 * CT;
  constexpr int WB = QB == 4 ? 32 : 64;            // weight bytes of a row per stage
  // int4 operands: q - z (fp16 with uint8 or no z); 64 + q (fp16), 128 + q (bf16),
  // with a term left for the group's sums of x
  constexpr bool LESS = QB == 4 && !BF16 && ZDT != TM_DT_F16, SUMX = QB == 4 && !LESS;
  constexpr int STX = BM * 128, STW = BN * WB, STS = SUMX ? 1024 : 0;
  constexpr int ST = STX + STW + STS;
  constexpr int NCX = 2 * RT, NCW = STW / 4096;    // copies per wave
  constexpr int NC = NCX + NCW + (SUMX ? 1 : 0);
  constexpr int PW = WB / 16;                      // pieces of a weight row
  constexpr int LDW = 32 * CT + 4;
  constexpr int EPI = 4 * 32 * LDW * 4;
  __shared__ __align__(1024) uint8_t smem[NS * ST > EPI ? NS * ST : EPI];
  const uint32_t lds0 = lds_off(smem);
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave >> 1, wn = wave & 1, l32 = lane & 31, h = lane >> 5;
  int tm, tn;
  tile_of(blockIdx.x, p.tiles_m, p.tiles_n, &tm, &tn);
  const int m0 = tm * BM, n0 = tn * BN, K = p.K;
  const int k0 = blockIdx.y * p.kslice, k1 = min(K, k0 + p.kslice);
  const int nk = (k1 - k0) / 64, ng = K / 128;
  const int ar = min(p.M - m0, BM), br = min(p.N - n0, BN);

  // ---- copies
  const int wrow = QB == 4 ? K / 2 : K;            // bytes of a weight row
  const uint8_t* xb = (const uint8_t*)p.X + ((size_t)m0 * K + k0) * 2;
  const uint8_t* wb = p.W + (size_t)n0 * wrow + (QB == 4 ? k0 / 2 : k0);
  uint32_t xv[NCX], wv[NCW];
#pragma unroll
  for (int i = 0; i < NCX; ++i) xv[i] = Tile<F16, false, RT>::voff(wave, lane, i, K, ar);
  // weight rows: piece q of row r at q ^ (r >> 3) & 1 (32-byte rows) or
  // q ^ (r >> 2) & 3 (64-byte rows): the 16 rows of a read phase in 16
  // different 16-byte bank groups
  const auto wsw = [](int r) { return QB == 4 ? (r >> 3) & 1 : (r >> 2) & 3; };
#pragma unroll
  for (int i = 0; i < NCW; ++i) {
    const int s = 64 * (NCW * wave + i) + lane, r = s / PW, q = (s % PW) ^ wsw(r);
    wv[i] = r < br ? (uint32_t)r * (uint32_t)wrow + 16u * q : kOob;
  }
  // stage kt into ring slot s (whole steps past the slice deposit zeros)
  auto copies = [&](int s, int kt) {
    const int ks = kt < nk ? kt : nk - 1;
    const uint32_t base = lds0 + s * ST;
    const u4_t rx = buf_rsrc(xb + (size_t)ks * 128,
                             ((uint32_t)(ar - 1) * K + (uint32_t)(K - k0 - 64 * ks)) * 2);
    const u4_t rw = buf_rsrc(wb + (size_t)ks * WB,
                             (uint32_t)br * (uint32_t)wrow - (uint32_t)(QB == 4 ? k0 / 2 : k0) -
                                 (uint32_t)(ks * WB));
#pragma unroll
    for (int i = 0; i < NCX; ++i)
      buf16(rx, kt < nk ? xv[i] : kOob, base + 1024 * (NCX * wave + i));
#pragma unroll
    for (int i = 0; i < NCW; ++i)
      buf16(rw, kt < nk ? wv[i] : kOob, base + STX + 1024 * (NCW * wave + i));
    if constexpr (SUMX) {
      // the group's sums of x for this tile's rows (each wave copies the same
      // bytes to the same place)
      const int g = (k0 + 64 * ks) >> 7;
      const u4_t rs = buf_rsrc(p.SX + (size_t)g * p.sxld, (uint32_t)p.sxld * 4);
      buf16(rs, 16 * lane < BM * 4 ? (uint32_t)(m0 * 4 + 16 * lane) : kOob, base + STX + STW);
    }
  };

  // ---- readers
  // X piece of step t (row 32 RT wm + l32, rows of 128 bytes): half h takes
  // k = 32 h + 8 t .. (int4) or 16 (2 (t / 2) + h) + 8 (t % 2) .. (int8)
  uint32_t xa[4];
  {
    const int r = 32 * RT * wm + l32, sw = (r >> 1) & 7;
#pragma unroll
    for (int t = 0; t < 4; ++t)
      xa[t] = lds0 + 128u * r +
              16u * ((QB == 4 ? 4 * h + t : 4 * (t >> 1) + 2 * h + (t & 1)) ^ sw);
  }
  const int wr = 32 * CT * wn + l32;  // weight row of column block 0 (block j: + 32 j)
  uint32_t wa[2];
#pragma unroll
  for (int s = 0; s < 2; ++s)
    wa[s] = lds0 + STX + (uint32_t)wr * WB + 16u * ((QB == 4 ? h : 2 * s + h) ^ wsw(wr));
  const uint32_t sa = lds0 + STX + STW + 4u * (32 * RT * wm + 4 * h);

  constexpr int NY = QB == 4 ? RT : 1;
  f16_t acc[RT][CT], y[NY][CT];
#pragma unroll
  for (int i = 0; i < RT; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) acc[i][j] = f16_t{};
#pragma unroll
  for (int i = 0; i < NY; ++i)
#pragma unroll
    for (int j = 0; j < CT; ++j) y[i][j] = f16_t{};

  // scales and zero-points of the lane's columns, one group ahead
  constexpr int SDT = BF16 ? TM_DT_BF16 : TM_DT_F16;
  int col[CT];
#pragma unroll
  for (int j = 0; j < CT; ++j) col[j] = min(n0 + 32 * CT * wn + 32 * j + l32, p.N - 1);
  typename Raw<SDT>::T sraw[CT];
  typename Raw<ZDT>::T zraw[CT];
  float sc[CT], zc[CT];  // scale and z - c
  h2_t c2[CT];           // 1024 + z (LESS)
  auto load_sz = [&](int g) {
    if constexpr (QB == 4) {
      g = min(g, ng - 1);
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        sraw[j] = ld_raw<SDT>(p.S, (size_t)col[j] * ng + g);
        zraw[j] = ld_raw<ZDT>(p.Z, (size_t)col[j] * ng + g);
      }
    }
  };
  auto take_sz = [&]() {
    if constexpr (QB == 4) {
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        sc[j] = raw_to_f32<SDT>(sraw[j]);
        zc[j] = (LESS ? 1024.0f : BF16 ? 128.0f : 64.0f) + raw_to_f32<ZDT>(zraw[j]);
        if constexpr (LESS) c2[j] = h2_t{(half_t)zc[j], (half_t)zc[j]};
      }
    }
  };

  load_sz(k0 >> 7);
#pragma unroll
  for (int s = 0; s < NS - 1; ++s) copies(s, s);
  const uint32_t mask = vgpr_const(SUMX && !BF16 ? kMask64 : 0x000F000Fu);
  const uint32_t magic = vgpr_const(SUMX && !BF16 ? kMagic64 : w4_magic<BF16>());
  int st = 0, kt = 0;
  // one stage: wait for it, refill the slot read last, multiply
  auto stage = [&](bool first) {
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"((NS - 2) * NC) : "memory");
    const int off = st * ST;
    if (first) {
      take_sz();
      load_sz(((k0 + 64 * kt) >> 7) + 1);
    }
    copies(st == 0 ? NS - 1 : st - 1, kt + NS - 1);
    u4_t w[2][CT];
#pragma unroll
    for (int s = 0; s < (QB == 4 ? 1 : 2); ++s)
#pragma unroll
      for (int j = 0; j < CT; ++j) w[s][j] = *(lds_u4_t*)(wa[s] + off + 32 * WB * j);
    u4_t x[4][RT];
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < RT; ++i) x[t][i] = *(lds_u4_t*)(xa[t] + off + 4096 * i);
    if (LESS && first) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = f16_t{};
    }
    f4_t sx[RT][4];
    if (SUMX && first) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int q = 0; q < 4; ++q) sx[i][q] = *(lds_f4_t*)(sa + off + 4 * (32 * i + 8 * q));
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) acc[i][j][e] = -zc[j] * sx[i][e >> 2][e & 3];
    }
#pragma unroll
    for (int t = 0; t < 4; ++t) {
      u4_t o[CT];
#pragma unroll
      for (int j = 0; j < CT; ++j) {
        if constexpr (LESS) o[j] = w4_less(w4_operand(w[0][j][t], mask, magic), c2[j]);
        else if constexpr (QB == 4 && BF16) o[j] = w4_operand(w[0][j][t], mask, magic);
        else if constexpr (QB == 4) o[j] = w4_operand64(w[0][j][t], mask, magic, 4, 8);
        else o[j] = w8_operand<BF16>(w[t >> 1][j][2 * (t & 1)], w[t >> 1][j][2 * (t & 1) + 1]);
      }
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j) acc[i][j] = mfma32<BF16>(x[t][i], o[j], acc[i][j]);
    }
    st = st == NS - 1 ? 0 : st + 1;
    ++kt;
  };
  while (kt < nk) {
    stage(true);
    stage(false);
    if constexpr (QB == 4) {
#pragma unroll
      for (int i = 0; i < RT; ++i)
#pragma unroll
        for (int j = 0; j < CT; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) y[i][j][e] = fmaf(sc[j], acc[i][j][e], y[i][j][e]);
    }
  }

  // ---- epilogue: lane l holds column 32 j + l % 32, rows 8 (e / 4) + 4 h + e % 4
  wait_vm<0>();
  __syncthreads();
  if constexpr (QB == 8) {
#pragma unroll
    for (int j = 0; j < CT; ++j) sc[j] = load_as_f32<SDT>(p.S, col[j]);
  }
  const uint32_t eb = lds0 + (uint32_t)wave * 32 * LDW * 4;
  const int mw = m0 + 32 * RT * wm, nw = n0 + 32 * CT * wn;
  float* P = p.P ? p.P + (size_t)blockIdx.y * p.M * p.N : nullptr;
  constexpr int LPR = 4 * CT, NP = 2 * CT;  // lanes of a row, pieces of 8 columns per lane
  f4_t size = {0.f, 0.f, 0.f, 0.f};         // infinite or NaN: so is one of the outputs
  static_for<0, RT>([&](auto ic) {
    constexpr int i = decltype(ic)::value;
#pragma unroll
    for (int j = 0; j < CT; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        float v;
        if constexpr (QB == 4) v = y[i][j][e];
        else v = sc[j] * acc[i][j][e];
        *(lds_f_t*)(eb + 4u * ((8 * (e >> 2) + 4 * h + (e & 3)) * LDW + 32 * j + l32)) = v;
      }
    const int c = 8 * (lane % LPR), n = nw + c;  // N % 16 == 0: whole pieces
#pragma unroll
    for (int t = 0; t < NP; ++t) {
      const int r = t * (64 / LPR) + lane / LPR, m = mw + 32 * i + r;
      f4_t a = *(lds_f4_t*)(eb + 4u * (r * LDW + c));
      f4_t b = *(lds_f4_t*)(eb + 4u * (r * LDW + c + 4));
      const bool in = m < p.M && n < p.N;
      if constexpr (!LESS) {
#pragma unroll
        for (int e = 0; e < 4; ++e) size[e] += __builtin_fabsf(a[e]) + __builtin_fabsf(b[e]);
      }
      if (!in) continue;
      const size_t o = (size_t)m * p.N + n;
      if (P) {
        *(f4_t*)(P + o) = a;
        *(f4_t*)(P + o + 4) = b;
      } else {
        if (p.bias) add8(p.bias, n, SDT, &a, &b);
        *(u4e_t*)((uint16_t*)p.Y + o) = pack8<SDT>(a, b);
      }
    }
  });
  if constexpr (!LESS) {
    // outputs that came out infinite or NaN again, as wq_general sums them
    // (wq_direct), piece by piece by the whole wave; the lane that holds the piece
    // reads back what it stored.  One sum of sizes finds them, and the code stands
    // in one place: a test of each output cost every call 0.4 us.
    for (uint64_t todo = __ballot(not_finite((size[0] + size[1]) + (size[2] + size[3]))); todo;
         todo &= todo - 1) {
      const int l = __builtin_ctzll(todo), n = nw + 8 * (l % LPR);
      if (n >= p.N) continue;
#pragma unroll 1
      for (int x = 0; x < RT * NP * 8; ++x) {
        const int e = x & 7, t = x >> 3;
        const int m = mw + 32 * (t / NP) + (t % NP) * (64 / LPR) + l / LPR;
        if (m >= p.M) break;  // (rows rise with t)
        const size_t o = (size_t)m * p.N + n + e;
        bool bad = false;
        if (lane == l) bad = not_finite(P ? P[o] : load_as_f32<SDT>(p.Y, o));
        if (!__ballot(bad)) continue;
        const float d = wq_direct<QB, BF16, ZDT>(
            p.X0 + (size_t)m * K, p.W + (size_t)(n + e) * wrow, p.S, p.Z,
            (size_t)(n + e) * (QB == 4 ? ng : 1), k0, k1, lane);
        if (lane != l) continue;
        if (P) P[o] = d;
        else store_as_f32_rt(p.Y, o, SDT, d + (p.bias ? load_as_f32<SDT>(p.bias, n + e) : 0.0f));
      }
    }
  }
}

// wq_pipe_q<bits>_<act>_z<zeros>_r<RT>
#define TM_WQ_PIPE(QB, AN, BF, ZN, ZDT, RT)                                                    \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(2, 2)))      \
      void wq_pipe_q##QB##_##AN##_z##ZN##_r##RT(WqPipeParams p) {                               \
    wq_pipe_body<QB, BF, ZDT, RT>(p);                                                          \
  }
#define TM_WQ_PIPE_RT(QB, AN, BF, ZN, ZDT) \
  TM_WQ_PIPE(QB, AN, BF, ZN, ZDT, 1)       \
  TM_WQ_PIPE(QB, AN, BF, ZN, ZDT, 2)
TM_WQ_PIPE_RT(4, f16, false, n, -1)
TM_WQ_PIPE_RT(4, f16, false, s, TM_DT_F16)
TM_WQ_PIPE_RT(4, f16, false, u, 3)
TM_WQ_PIPE_RT(4, bf16, true, n, -1)
TM_WQ_PIPE_RT(4, bf16, true, s, TM_DT_BF16)
TM_WQ_PIPE_RT(4, bf16, true, u, 3)
TM_WQ_PIPE_RT(8, f16, false, n, -1)
TM_WQ_PIPE_RT(8, bf16, true, n, -1)
