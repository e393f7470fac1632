// gemm_split.hip — fp32 GEMM on the bf16 matrix cores of CDNA4, every operand
// split into three bf16 pieces (v_mfma_f32_32x32x16_bf16).
//
// x = h + m + l with h, m, l the successive bf16 roundings: 3 x 8 significant
// bits hold all 24 bits of an fp32 value, once the operands are scaled by 2^24:
// the last bit of the smallest subnormal, 2^-149, is then a normal bf16 value. A
// scaled value past the bf16 range or a sum past the fp32 range (operands from
// 2^104, results from 2^80) comes out non-finite and is recomputed on the fp32
// MFMAs. A product keeps the six terms down
// to 2^-16 of the largest (h.h, h.m, m.h, h.l, m.m, l.h; the dropped ones lie
// below 2^-26), accumulated in fp32, smallest first. Against float64 the sums
// are closer than the fp32 MFMA's, because 16 products enter the accumulator
// per rounding instead of four: relative error 1.6e-7 vs 2.0e-7 at K = 128,
// 3.4e-7 vs 4.0e-7 at K = 512, 1.01e-6 vs 1.15e-6 at K = 4096 (N(0,1)
// operands, one wavefront's 32 x 32 tile).
//
// What bounds it: six MFMAs at the bf16 rate (1.7 PFLOP/s from registers, the
// part's power limit) against one at the fp32 rate (0.15), so 1.9x the fp32
// ceiling. To stay near it, each wavefront owns 32 rows x 128 columns: its A
// rows are private, so they go global -> registers -> pieces with no LDS and
// no repeated conversion; only the B tile, shared by the block's wavefronts,
// is staged in LDS, already split and in fragment order (one conflict-free
// ds_read_b128 per piece and fragment).
#pragma once
#include "common.hip"
#include "gemm_mfma.hip"  // block_tile_of, batch_tile

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef float floatx2 __attribute__((ext_vector_type(2)));
typedef float floatx16 __attribute__((ext_vector_type(16)));
typedef unsigned uintx4 __attribute__((ext_vector_type(4)));

namespace zk {

// Barrier for LDS only: global loads and stores stay in flight across it.
__device__ __forceinline__ void lds_only_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

struct Pieces {
  bf16x8 h, m, l;
};
// Two values at a time: v_cvt_pk_bf16_f32 rounds a pair into one register.
__device__ __forceinline__ unsigned pack_bf16(float a, float b) {
  const floatx2 v = {a, b};
  return __builtin_bit_cast(unsigned, __builtin_convertvector(v, bf16x2));
}
__device__ __forceinline__ Pieces split_pieces(const float (&x)[8]) {
  uintx4 h, m, l;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    const float x0 = x[2 * c], x1 = x[2 * c + 1];
    h[c] = pack_bf16(x0, x1);
    const float r0 = x0 - __builtin_bit_cast(float, h[c] << 16);
    const float r1 = x1 - __builtin_bit_cast(float, h[c] & 0xffff0000u);
    m[c] = pack_bf16(r0, r1);
    const float q0 = r0 - __builtin_bit_cast(float, m[c] << 16);
    const float q1 = r1 - __builtin_bit_cast(float, m[c] & 0xffff0000u);
    l[c] = pack_bf16(q0, q1);
  }
  Pieces p;
  p.h = __builtin_bit_cast(bf16x8, h);
  p.m = __builtin_bit_cast(bf16x8, m);
  p.l = __builtin_bit_cast(bf16x8, l);
  return p;
}

constexpr int kSplitBK = 32;  // k-tile: two 16-wide MFMA steps
// Of either operand before it is split: one multiplication per value, 0-4 %
// of a case's time (returns of 98,304 rows 392 -> 410 us, two layers of 24,576
// rows forward and backward 250 -> 253); sums in the ordinary range keep their bits.
constexpr float kSplitScale = 0x1p24f;

// LDS of one block in bytes: the B tile's pieces, double buffered.
template <int CT>  // 32-wide column tiles of the block
constexpr int split_smem_bytes() {
  return 2 * CT * 2 * 3 * 1024;
}

// Reduction index of element c (0..7) of lane group g in step s of a k-tile:
// quads 4 s + g and 4 s + 2 + g of the tile's eight, so that a lane reads its
// share of a K-contiguous row as four float4s and the two lane groups of a
// row read adjacent 16 bytes. Any bijection gives the same product as long
// as A and B agree.
__device__ __forceinline__ constexpr int split_k(int s, int g, int c) {
  return 16 * s + 8 * (c / 4) + 4 * g + c % 4;
}

// C[M x N] tile (mt, nt) with the epilogues of gemm_body, k-tiles
// [split * kt_per_split, ...). WM x WN wavefronts of TR x TN 32 x 32 tiles each. A: K-contiguous rows (AK; optionally
// gathered) or [K x M]; B: K-contiguous rows (BKC) or [K x N] (optionally
// gathered). VEC: K-contiguous operands have float4-aligned rows. EXACT: the
// slice's k-tiles lie inside K. Rows past M and columns past N repeat the last
// one, operands, sums and all, so that edge tiles need no masks: their stores
// write the last row's or column's own value again. GATHER: permB may be set. ACC2: the five small
// terms in accumulators of their own, added at the end: the large ones then
// round once per 16 products (relative error 1.3e-7 instead of 3.4e-7 at K =
// 512) for 64 more registers, two instead of three wavefronts per SIMD.
template <bool AK, bool BKC, int WM, int WN, int TR, int TN, bool VEC, bool EXACT, bool GATHER,
          bool DG, bool ACC2>
__device__ __forceinline__ void split_body(char* __restrict__ smem, const GemmArgs& p, int split, int mt,
                                           int nt) {
  constexpr int CT = WN * TN;  // column tiles of the block
  constexpr int NT = 64 * WM * WN, BM = 32 * TR * WM, BN = 32 * CT, BK = kSplitBK;
  constexpr int FR = CT * 128 / NT;  // B fragments (8 reduction indices of one column) per thread
  static_assert(FR >= 1 && FR * NT == CT * 128, "whole fragments per thread");
  static_assert(BKC || BN % 64 == 0, "N-contiguous B: a wavefront loads one reduction index at a time");
  if (p.guard && *p.guard == 0) return;
  const int m0 = mt * BM, n0 = nt * BN;
  if (m0 >= p.M || n0 >= p.N || split >= p.nsplit) return;  // uniform
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;
  const int li = lane & 31, lg = lane >> 5;
  const int K = p.K;
  const int KT = (K + BK - 1) / BK;
  const int kt0 = split * p.kt_per_split;
  const int kt1 = min(KT, kt0 + p.kt_per_split);

  // ---- A: this lane's rows (or columns of [K x M]), one per row tile.
  const int mw = m0 + 32 * TR * wm, nw = n0 + 32 * TN * wn;  // the wavefront's first row and column
  int mc[TR];
  const float* arow[TR];
#pragma unroll
  for (int i = 0; i < TR; ++i) {
    const int m = mw + 32 * i + li;
    mc[i] = min(m, p.M - 1);
    arow[i] = nullptr;
    if (AK) arow[i] = p.A + (long long)(p.permA ? p.permA[mc[i]] : mc[i]) * p.lda;
  }
  float araw[2][TR][8];
  // Loads of a k-tile that lies inside K (all of them in an exact fit) need
  // no clamps; the last one of a ragged K reads clamped, valid addresses and
  // its elements past K are zeroed before they are split.
  auto load_a = [&](int k0, int s) {
    auto go = [&](auto inside) {
      constexpr bool IN = decltype(inside)::value;
#pragma unroll
      for (int i = 0; i < TR; ++i) {
        float* d = araw[s][i];
        if constexpr (AK && VEC) {
#pragma unroll
          for (int h = 0; h < 2; ++h) {
            int k = k0 + 4 * (4 * s + 2 * h + lg);
            if (!IN) k = min(k, ((K + 3) & ~3) - 4);
            const float4 v = *reinterpret_cast<const float4*>(arow[i] + k);
            d[4 * h] = v.x, d[4 * h + 1] = v.y, d[4 * h + 2] = v.z, d[4 * h + 3] = v.w;
          }
        } else {
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            if constexpr (AK) {
              const int k = k0 + split_k(s, lg, c);
              d[c] = arow[i][IN ? k : min(k, K - 1)];
            } else if constexpr (IN) {
              const float* row = p.A + (long long)(k0 + split_k(s, 0, c)) * p.lda;  // uniform
              d[c] = row[(unsigned)(4 * lg * p.lda + mc[i])];
            } else {
              d[c] = p.A[(long long)min(k0 + split_k(s, lg, c), K - 1) * p.lda + mc[i]];
            }
          }
        }
      }
    };
    if (EXACT || k0 + BK <= K)
      go(std::true_type{});
    else
      go(std::false_type{});
  };

  // ---- B: this thread's fragments. K-contiguous: lane group tid % 2 and SB
  // of the two steps of BP columns. N-contiguous: column nbc, units u0 ..
  // u0 + FR - 1 of the four (step, lane group) pairs (uniform over the
  // wavefront).
  constexpr int SB = FR >= 2 ? 2 : 1;   // steps per thread and column
  constexpr int BP = BKC ? FR / SB : 1;  // columns per thread
  constexpr int TPC = 4 / SB;            // threads per column
  const float* brow[BP];
  const int gb = tid & 1;
  const int sb0 = SB == 2 ? 0 : (tid >> 1) & 1;
  const int nbc = BKC ? 0 : tid % BN;
  const int u0 = BKC ? 0 : __builtin_amdgcn_readfirstlane(tid / BN) * FR;
  const int ncl = min(n0 + nbc, p.N - 1);
  if constexpr (BKC) {
#pragma unroll
    for (int b = 0; b < BP; ++b) {
      const int n = n0 + tid / TPC + b * (NT / TPC);
      brow[b] = p.B + (long long)min(n, p.N - 1) * p.ldb;
    }
  }
  float braw[FR][8];
  int bperm[!BKC && GATHER ? FR : 1][8];
  auto fetch_b = [&](int k0) {  // gathered rows of the k-tile at k0
    if constexpr (!BKC && GATHER) {
      if (!p.permB) return;
#pragma unroll
      for (int f = 0; f < FR; ++f)
#pragma unroll
        for (int c = 0; c < 8; ++c) bperm[f][c] = p.permB[min(k0 + split_k((u0 + f) / 2, (u0 + f) % 2, c), K - 1)];
    }
  };
  auto load_b = [&](int k0) {
    auto go = [&](auto inside) {
      constexpr bool IN = decltype(inside)::value;
      if constexpr (BKC) {
#pragma unroll
        for (int b = 0; b < BP; ++b)
#pragma unroll
          for (int sx = 0; sx < SB; ++sx) {
            const int s = sb0 + sx;
            float* d = braw[SB * b + sx];
            if constexpr (VEC) {
#pragma unroll
              for (int h = 0; h < 2; ++h) {
                int k = k0 + 4 * (4 * s + 2 * h + gb);
                if (!IN) k = min(k, ((K + 3) & ~3) - 4);
                const float4 v = *reinterpret_cast<const float4*>(brow[b] + k);
                d[4 * h] = v.x, d[4 * h + 1] = v.y, d[4 * h + 2] = v.z, d[4 * h + 3] = v.w;
              }
            } else {
#pragma unroll
              for (int c = 0; c < 8; ++c) {
                const int k = k0 + split_k(s, gb, c);
                d[c] = brow[b][IN ? k : min(k, K - 1)];
              }
            }
          }
      } else {
#pragma unroll
        for (int f = 0; f < FR; ++f)
#pragma unroll
          for (int c = 0; c < 8; ++c) {
            const int kk = k0 + split_k((u0 + f) / 2, (u0 + f) % 2, c);
            int r = IN ? kk : min(kk, K - 1);
            if constexpr (GATHER) r = p.permB ? bperm[f][c] : r;
            const float* row = p.B + (long long)r * p.ldb;  // uniform
            braw[f][c] = row[(unsigned)ncl];
          }
      }
    };
    if (EXACT || k0 + BK <= K)
      go(std::true_type{});
    else
      go(std::false_type{});
  };
  // LDS: piece q of fragment (column tile j, step s) is 64 x 16 bytes at
  // ((j * 2 + s) * 3 + q) * 1024; lane (i, g) of the fragment sits in slot
  // 32 g + (i ^ 12 g), which keeps the two lane groups of a row in different
  // banks when a thread pair stores them.
  auto slot = [](int i, int g) { return 32 * g + (i ^ (12 * g)); };
  auto store_b = [&](int buf, int k0) {
    char* base = smem + buf * (CT * 2 * 3 * 1024);
#pragma unroll
    for (int f = 0; f < FR; ++f) {
      const int s = BKC ? sb0 + f % SB : (u0 + f) / 2;
      const int g = BKC ? gb : (u0 + f) % 2;
      const int n = BKC ? tid / TPC + (f / SB) * (NT / TPC) : nbc;
      if (!EXACT && k0 + BK > K) {
#pragma unroll
        for (int c = 0; c < 8; ++c)
          if (k0 + split_k(s, g, c) >= K) braw[f][c] = 0.f;
      }
#pragma unroll
      for (int c = 0; c < 8; ++c) braw[f][c] *= kSplitScale;
      const Pieces q = split_pieces(braw[f]);
      char* d = base + ((n / 32) * 2 + s) * 3 * 1024 + slot(n & 31, g) * 16;
      *reinterpret_cast<bf16x8*>(d) = q.h;
      *reinterpret_cast<bf16x8*>(d + 1024) = q.m;
      *reinterpret_cast<bf16x8*>(d + 2048) = q.l;
    }
  };

  // The matrix core truncates a small product towards minus infinity when it
  // meets a large accumulator: 1e-8 to 3e-8 of |C| on average, far below the
  // rounding of one element but visible in a sum over a whole batch. So every
  // other strip (in rows, column blocks and split-K slices) accumulates -C.
  // (With ACC2 the small products never meet the large accumulator.)
  const bool neg = !ACC2 && (mt * WM + wm + nt + split) % 2;
  const float scale = neg ? -kSplitScale : kSplitScale;
  float unscale = (neg ? -1.f : 1.f) / (kSplitScale * kSplitScale);
  constexpr int U = TN % 2 == 0 ? 2 : 1;  // column tiles whose MFMAs alternate
  floatx16 acc[TR][TN], lo[ACC2 ? TR : 1][ACC2 ? TN : 1];
#pragma unroll
  for (int i = 0; i < TR; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        acc[i][j][r] = 0.f;
        if constexpr (ACC2) lo[i][j][r] = 0.f;
      }
  const bool rowsum = !AK && p.rowsumA != nullptr && nt == 0 && wn == 0;
  float rs[TR] = {};

  // Pipeline: while the MFMAs of k-tile t run from LDS buffer t & 1, the B
  // tile of t + 1 is split into the other buffer (read by every wavefront
  // before the last barrier) and the loads of A t + 1 (each step's registers
  // are reloaded as soon as they are split) and B t + 2 are in flight. One
  // LDS barrier per k-tile.
  if (kt0 < kt1) {
    fetch_b(kt0 * BK);
    load_b(kt0 * BK);
    load_a(kt0 * BK, 0);
    load_a(kt0 * BK, 1);
    store_b(0, kt0 * BK);
    if (kt0 + 1 < kt1) {
      fetch_b((kt0 + 1) * BK);
      load_b((kt0 + 1) * BK);
      if (kt0 + 2 < kt1) fetch_b((kt0 + 2) * BK);
    }
  }
  lds_only_barrier();
  const int rslot = slot(li, lg) * 16 + wn * TN * 2 * 3 * 1024;
  auto iteration = [&](int kt) {
    const int cur = (kt - kt0) & 1;
    const char* base = smem + cur * (CT * 2 * 3 * 1024) + rslot;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      if (!EXACT && (kt + 1) * BK > K) {
#pragma unroll
        for (int i = 0; i < TR; ++i)
#pragma unroll
          for (int c = 0; c < 8; ++c)
            if (kt * BK + split_k(s, lg, c) >= K) araw[s][i][c] = 0.f;
      }
      bf16x8 ah[TR], am[TR], al[TR];
#pragma unroll
      for (int i = 0; i < TR; ++i) {
        if (rowsum) {
#pragma unroll
          for (int c = 0; c < 8; ++c) rs[i] += araw[s][i][c];
        }
#pragma unroll
        for (int c = 0; c < 8; ++c) araw[s][i][c] *= scale;
        const Pieces q = split_pieces(araw[s][i]);
        ah[i] = q.h, am[i] = q.m, al[i] = q.l;
      }
      if (kt + 1 < kt1) {
        load_a((kt + 1) * BK, s);
        if (s == 0) {
          store_b(cur ^ 1, (kt + 1) * BK);
          if (kt + 2 < kt1) {
            load_b((kt + 2) * BK);
            if (kt + 3 < kt1) fetch_b((kt + 3) * BK);
          }
        }
      }
      // Two column tiles at a time, so that consecutive MFMAs do not depend on
      // each other; the terms of one accumulator smallest first.
#pragma unroll
      for (int j = 0; j < TN; j += U) {
        bf16x8 bh[U], bm[U], bl[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
          const char* d = base + ((j + u) * 2 + s) * 3 * 1024;
          bh[u] = *reinterpret_cast<const bf16x8*>(d);
          bm[u] = *reinterpret_cast<const bf16x8*>(d + 1024);
          bl[u] = *reinterpret_cast<const bf16x8*>(d + 2048);
        }
        auto term = [&](const bf16x8 (&x)[TR], const bf16x8 (&y)[U], auto small) {
#pragma unroll
          for (int i = 0; i < TR; ++i)
#pragma unroll
            for (int u = 0; u < U; ++u) {
              constexpr bool LO = ACC2 && decltype(small)::value;
              floatx16& c = LO ? lo[LO ? i : 0][LO ? j + u : 0] : acc[i][j + u];
              c = __builtin_amdgcn_mfma_f32_32x32x16_bf16(x[i], y[u], c, 0, 0, 0);
            }
        };
        term(al, bh, std::true_type{});
        term(am, bm, std::true_type{});
        term(ah, bl, std::true_type{});
        term(am, bh, std::true_type{});
        term(ah, bm, std::true_type{});
        term(ah, bh, std::false_type{});
      }
    }
    lds_only_barrier();
  };
  // Staged epilogue (DG: exact-fit data gradients, kEpiEluGrad only): half of the strip's columns
  // at a time goes through this wavefront's own LDS, so that the ELU' operand
  // is read and dL/dz written as float4 row segments.
  static_assert(!DG || EXACT, "whole tiles");
  constexpr int SCOLS = 64, SPITCH = SCOLS + 4, SROWS = 4;  // rows per pass of 64 lanes
  constexpr int SHALF = TN * 32 / SCOLS, SPASS = 32 / SROWS;
  static_assert(!DG || 32 * SPITCH * 4 * WM * WN <= split_smem_bytes<CT>(), "a half strip per wavefront");
  float4 yq[DG ? SPASS : 1];
  const int sr = lane / 16, sc = (lane % 16) * 4;
  auto load_y = [&](int i, int h) {
    if constexpr (DG) {
#pragma unroll
      for (int ps = 0; ps < SPASS; ++ps)
        yq[ps] = *reinterpret_cast<const float4*>(p.Y + (long long)min(mw + 32 * i + SROWS * ps + sr, p.M - 1) * p.ldy + nw +
                                                  SCOLS * h + sc);
    }
  };
  for (int kt = kt0; kt < kt1; ++kt) iteration(kt);
  if constexpr (ACC2) {
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] += lo[i][j][r];
  }
  load_y(0, 0);

  // Where the pieces do not hold the operands -- infinities (inf - inf), values
  // that round to a bf16 infinity -- or a scaled sum overflows, the sums come
  // out non-finite. Such a wavefront recomputes its strip with fp32 MFMAs
  // straight from memory.
  {
    float nan = 0.f;
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) nan = nan + acc[i][j][r] * 0.f;  // 0, or NaN once a sum is not finite
    if (__any(nan != 0.f)) {
      unscale = 1.f;
#pragma unroll
      for (int i = 0; i < TR; ++i)
#pragma unroll
        for (int j = 0; j < TN; ++j)
#pragma unroll
          for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.f;
      const int kend = min(K, kt1 * BK);
      for (int kb = kt0 * BK; kb < kend; kb += 2) {
        const int k = kb + lg, kc = min(k, kend - 1);
        const bool in = k < kend;
        float av[TR];
#pragma unroll
        for (int i = 0; i < TR; ++i) av[i] = AK ? arow[i][kc] : p.A[(long long)kc * p.lda + mc[i]];
#pragma unroll
        for (int j = 0; j < TN; ++j) {
          const int n = min(nw + 32 * j + li, p.N - 1);
          const long long r = !BKC && GATHER && p.permB ? p.permB[kc] : kc;
          const float bv = BKC ? p.B[(long long)n * p.ldb + kc] : p.B[r * p.ldb + n];
#pragma unroll
          for (int i = 0; i < TR; ++i)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(in ? av[i] : 0.f, in ? bv : 0.f, acc[i][j], 0, 0, 0);
        }
      }
    }
  }

  if (rowsum) {
#pragma unroll
    for (int i = 0; i < TR; ++i) {
      rs[i] += __shfl_xor(rs[i], 32, 64);
      if (lg == 0 && mw < p.M) p.rowsumA[(long long)split * p.M + mc[i]] = rs[i];
    }
  }

  // Epilogue: register r of acc[i][j] is row 8 (r / 4) + 4 lg + r % 4 of row
  // tile i, column 32 j + li.
  float* C = p.C + (long long)split * p.split_stride;
  static_assert(TR == 1, "one row tile per wavefront: a strip past M is skipped whole");
  if (mw >= p.M || nw >= p.N) return;  // (no barrier follows)
  auto emit = [&](auto f) {
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) {
        const int n = min(nw + 32 * j + li, p.N - 1);
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const int mm = min(mw + 32 * i + 4 * lg + 8 * (r / 4) + r % 4, p.M - 1);
          C[(long long)mm * p.ldc + n] = f(acc[i][j][r] * unscale, j, mm, n);
        }
      }
  };
  if constexpr (DG) {
    float* st = reinterpret_cast<float*>(smem) + wave * 32 * SPITCH;
#pragma unroll
    for (int i = 0; i < TR; ++i)
#pragma unroll
      for (int h = 0; h < SHALF; ++h) {
        if (i + h > 0) load_y(i, h);
#pragma unroll
        for (int jj = 0; jj < SCOLS / 32; ++jj)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            st[(4 * lg + 8 * (r / 4) + r % 4) * SPITCH + 32 * jj + li] =
                  acc[i][SCOLS / 32 * h + jj][r] * unscale;
#pragma unroll
        for (int ps = 0; ps < SPASS; ++ps) {
          const int row = SROWS * ps + sr;
          float4 v = *reinterpret_cast<const float4*>(st + row * SPITCH + sc);
          v.x *= elu_grad_from_act(yq[ps].x);
          v.y *= elu_grad_from_act(yq[ps].y);
          v.z *= elu_grad_from_act(yq[ps].z);
          v.w *= elu_grad_from_act(yq[ps].w);
          *reinterpret_cast<float4*>(C + (long long)min(mw + 32 * i + row, p.M - 1) * p.ldc + nw + SCOLS * h + sc) = v;
        }
      }
    return;
  }
  if (p.epi == kEpiBiasN) {
    float b[TN];
#pragma unroll
    for (int j = 0; j < TN; ++j) b[j] = p.bias[min(nw + 32 * j + li, p.N - 1)];
    if (p.act)
      emit([&](float v, int j, int, int) { return elu(v + b[j]); });
    else
      emit([&](float v, int j, int, int) { return v + b[j]; });
  } else if (p.epi == kEpiBiasM) {
    if (p.act)
      emit([&](float v, int, int mm, int) { return elu(v + p.bias[(long long)mm * p.bias_stride]); });
    else
      emit([&](float v, int, int mm, int) { return v + p.bias[(long long)mm * p.bias_stride]; });
  } else if (p.epi == kEpiEluGrad) {
    emit([&](float v, int, int mm, int n) { return v * elu_grad_from_act(p.Y[(long long)mm * p.ldy + n]); });
  } else {
    emit([&](float v, int, int, int) { return v; });
  }
}

// Tile (mt, nt) of slice `split`: slices inside K run the form without clamps
// and masks in the k-loop. DG additionally needs whole column tiles and
// float4-aligned rows of C and Y (p.vecB, set by the host).
template <bool AK, bool BKC, int WM, int WN, int TR, int TN, bool VEC, bool DG, bool ACC2>
__device__ __forceinline__ void split_tile(char* __restrict__ smem, const GemmArgs& p, const BlockTile& bt) {
  const int kt1 = min((p.K + kSplitBK - 1) / kSplitBK, (bt.z + 1) * p.kt_per_split);
  constexpr bool GATHER = !AK && !BKC;  // the input layer's weight gradient of a shuffled minibatch
  const bool whole = kt1 * kSplitBK <= p.K && (!DG || (p.vecB && (bt.nt + 1) * 32 * TN * WN <= p.N));
  if (whole && !(GATHER && p.permB))
    split_body<AK, BKC, WM, WN, TR, TN, VEC, true, false, DG, ACC2>(smem, p, bt.z, bt.mt, bt.nt);
  else if (GATHER && whole)
    split_body<AK, BKC, WM, WN, TR, TN, VEC, true, true, false, ACC2>(smem, p, bt.z, bt.mt, bt.nt);
  else
    split_body<AK, BKC, WM, WN, TR, TN, VEC, false, GATHER, false, ACC2>(smem, p, bt.z, bt.mt, bt.nt);
}

}  // namespace zk

#define ZK_SPLIT(NAME, AK, BKC, VEC, DG, ACC2)                                                 \
  extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(ACC2 ? 2 : 3))) \
  void NAME(zk::GemmBatch b) {                                                                 \
    __shared__ __align__(16) char smem[zk::split_smem_bytes<4>()];                             \
    int prob;                                                                                  \
    const zk::BlockTile bt = zk::batch_tile(b, (int)blockIdx.x, prob);                         \
    zk::split_tile<AK, BKC, 4, 1, 1, 4, VEC, DG, ACC2>(smem, b.g[prob], bt);                         \
  }
// Naming: a{k,m} = A K- or M-contiguous, b{k,n} = B K- or N-contiguous, _s
// element loads of K-contiguous rows that are not 16-byte aligned, _dg the
// data gradients (ELU' epilogue), _acc2 the forwards with K > 128, whose errors
// pass through every later layer.
ZK_SPLIT(zk_split_ak_bk, true, true, true, false, false)
ZK_SPLIT(zk_split_ak_bk_acc2, true, true, true, false, true)
ZK_SPLIT(zk_split_ak_bk_s, true, true, false, false, false)
ZK_SPLIT(zk_split_ak_bn, true, false, true, false, false)
ZK_SPLIT(zk_split_ak_bn_s, true, false, false, false, false)
ZK_SPLIT(zk_split_ak_bn_dg, true, false, true, true, false)
ZK_SPLIT(zk_split_am_bn, false, false, true, false, false)

// One layer's backward as one launch (GemmPair): the split-K weight-gradient
// blocks of both nets, then their data-gradient blocks with the ELU' epilogue
// (disjoint outputs, one LDS allocation). The data gradients' epilogues, which
// move 2.5x the bytes of their k-loops, overlap the weight gradients' MFMAs.
extern "C" __global__ __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(3)))
void zk_split_bwd(zk::GemmPair b) {
  __shared__ __align__(16) char smem[zk::split_smem_bytes<4>()];
  const int g = (int)blockIdx.x;
  int prob;
  if (g < b.nw) {
    const zk::BlockTile bt = zk::batch_tile(b.w, g, prob);
    zk::split_tile<false, false, 4, 1, 1, 4, true, false, false>(smem, b.w.g[prob], bt);
  } else {
    const zk::BlockTile bt = zk::batch_tile(b.d, g - b.nw, prob);
    zk::split_tile<true, false, 4, 1, 1, 4, true, true, false>(smem, b.d.g[prob], bt);
  }
}
