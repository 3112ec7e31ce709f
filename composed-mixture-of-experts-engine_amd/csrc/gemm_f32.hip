// Grouped SwiGLU expert GEMMs in float32 (the reference module's default dtype) for gfx950.
//
// The same six products as the bf16 kernels (gemm.hip) -- C[m, n] = sum_k A[m, k] B[n, k] per expert segment,
// with the SwiGLU forward / backward fused into the epilogues -- on v_mfma_f32_32x32x2_f32: float32 products and
// float32 sums, as the reference's float32 F.linear computes them (pkg/distributed/moe_layer.py L:166-198,
// L:326-337).  The fp32 MFMA peak is 1/16 of the bf16 one, so a block is small enough that two share a CU:
// 128x128 tiles, eight waves of 32x64, 32-wide k slices double-buffered in LDS and refilled through registers one
// slice ahead.  Eight waves and not four of 64x64: an MFMA takes 64 cycles and a slice ends in a barrier, so it is
// waves that hide it (E = 8, H = 1024, F = 4096, 512 rows an expert, all six products: 2810 -> 2690 us; a 16-wide
// slice 2750; one block a CU, 32 or 64 wide, 2900).
//
// An MFMA may take its two k values from any positions as long as A and B agree: in MFMA s of a group of 8 k, lane l
// supplies k = 8 grp + 4 (l / 32) + s for its row (A) or column (B), so the four MFMAs of a group cover its 8 k once
// each.  LDS holds an operand tile in its own order, so neither is transposed on the way in:
//   operand mode 0 ("rows"): element (i, k) at P[i*ld + k]: [i][k] with a pitch of 36 floats; a lane reads the four k
//                            of a group with one 16-byte read
//   operand mode 1 ("cols"): element (i, k) at P[k*ld + i]: [k][i] with a pitch of 136 floats; a lane reads its k's
//                            one by one (4 bytes; the half waves are 4 rows = 32 banks apart, so no two lanes meet)
//   GROUP 0: rows of one expert segment (tile prefix from k_gemm_tiles with bm = 128); GROUP 1: the reduction
//   runs over the expert's rows (weight gradients; experts without rows get zeros).
//   EPI 0 store C; EPI 1 SwiGLU forward (the B tile interleaves 32 gate and 32 up rows, so a lane holds g and u
//   of the same (row, f) in its two n blocks): act = silu(g) u and hgu = [g | u]; EPI 2 SwiGLU backward from
//   C = dA and hgu: dh = [dA u silu'(g) | dA silu(g)].
#include <algorithm>
#include <type_traits>

#include "common.h"

namespace moe {

struct GemmF32Args {
  const float* A;
  int64_t lda;
  const float* B;
  const float* B2;     // second B source: k >= b_split (cols mode) / up rows (EPI 1)
  int64_t ldb;
  int64_t b_estride;   // per-expert stride of B / B2 (row-grouped)
  int b_split;
  float* C;
  float* C2;           // EPI 1: hgu; k-grouped: rows >= c_split
  int64_t ldc;
  int64_t c_estride;   // per-expert stride of C / C2 (k-grouped)
  int c_split;
  const float* X;      // EPI 2: hgu
  int F;
  const int* offsets;  // [E+1]
  const int* tile_off; // [E+1] m-tile prefix with bm = 128 (row-grouped)
  int E;
  int M, N, K;         // k-grouped: M, N; row-grouped: N, K
  float* part;         // row-grouped: partial tiles of the split last round (null: no split)
  int npart;           // ... and how many of them an XCD has room for
};

constexpr int FBM = 128, FBN = 128, FBK = 32;
constexpr int FNT = 512;                 // threads: eight waves, two on each SIMD
constexpr int FNJ = FBM * FBK / (4 * FNT);  // 16-byte units of an operand slice a thread moves
constexpr int FCH = FBK / 4;           // ... and of one row of it
constexpr int FKP = FBK + 4;    // rows mode: LDS row pitch (floats): 144 bytes, keeps 16-byte reads aligned
constexpr int FIP = FBM + 8;    // cols mode: pitch of a k row (floats); 4 pitches are 32 banks mod 64
constexpr int fop(int mode) { return mode ? FBK * FIP : FBM * FKP; }  // floats of an operand tile

__device__ __forceinline__ f32x16 mfma32x32x2_f32(float a, float b, const f32x16& c) {
  return __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, c, 0, 0, 0);
}

// silu and its derivative in float32 with the library exponential (the reference's torch silu, x / (1 + e^-x))
__device__ __forceinline__ float sig32(float g) { return 1.f / (1.f + expf(-g)); }

// The last round of a row-grouped product, split over k as gemm.hip's.  A round of an XCD is 64 blocks, two on each of
// its 32 CUs; when a CU's pair ends its two places are filled at once, so what is left after the whole rounds runs in
// pairs beside idle CUs (only the first 32 blocks of a launch are spread one to a CU).  The last n % 64 tiles become S
// parts each, summed by k_gemm_reduce_f32; S has the least estimated time in slices of one tile (two tiles on a CU
// take twice that), with about 4 slices for writing and reading back a 64 KB partial tile and 3 for the reduction's
// launch.  E = 8, H = 1024, F = 4096, 4096 rows in ragged segments: fwd2 and dxp have about 300 tiles for 256 CUs.
constexpr int kSplitMaxF32 = 192;
__device__ __forceinline__ int split_of_f32(int n, int nk, int npart) {
  const int r = n & 63;
  int best = 1, cost = n <= 32 ? nk : 2 * nk;
  for (int S = 2; S <= 16; ++S) {
    if (r * S > npart || S > nk) break;
    const int c = (n <= 32 && r * S <= 32 ? 1 : 2 * ((r * S + 63) >> 6)) * ((nk + S - 1) / S + 4) + 3;
    if (c < cost) {
      cost = c;
      best = S;
    }
  }
  return r ? best : 1;
}

// The row-grouped tiles of an XCD, n of them.  Column tiles [nt0, nt0 + tn) of every expert, so that each XCD has the
// same share of each segment's full and partly filled row tiles; with few column tiles that 8 XCDs cannot share
// evenly, a contiguous range of all tiles from `first`.  Either way the row tiles of one weight panel run on one XCD.
struct F32Range {
  int n, first, nt0, tn;
};
__device__ __forceinline__ F32Range f32_range(const GemmF32Args& g, int xcd, int Tn) {
  if ((Tn & 7) == 0 || Tn >= 64) {
    const int lo = Tn * xcd >> 3, hi = Tn * (xcd + 1) >> 3;
    return {g.tile_off[g.E] * (hi - lo), 0, lo, hi - lo};
  }
  const int total = g.tile_off[g.E] * Tn, chunk = (total + 7) >> 3;
  return {max(0, min(chunk, total - xcd * chunk)), xcd * chunk, 0, Tn};
}

struct F32Tile {
  int e, mbase, mlen, nt;
};
// Tile i of the range: m fastest within an expert's column tile.
__device__ __forceinline__ F32Tile f32_tile(const GemmF32Args& g, const F32Range& x, int i) {
  const int L = x.first + i;
  int lo = 0, hi = g.E - 1;  // largest e with tile_off[e] * tn <= L
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (g.tile_off[mid] * x.tn <= L) lo = mid;
    else hi = mid - 1;
  }
  F32Tile t;
  t.e = lo;
  const int cnt = g.tile_off[lo + 1] - g.tile_off[lo];
  const int local = L - g.tile_off[lo] * x.tn, col = local / cnt;
  t.nt = x.nt0 + col;
  t.mbase = g.offsets[lo] + (local - col * cnt) * FBM;
  t.mlen = min(FBM, g.offsets[lo + 1] - t.mbase);
  return t;
}

template <int AMODE, int BMODE, int GROUP, int EPI>
__global__ __launch_bounds__(FNT, 2) void k_gemm_f32(GemmF32Args g) {
  __shared__ __attribute__((aligned(16))) float sa[2][fop(AMODE)];
  __shared__ __attribute__((aligned(16))) float sb[2][fop(BMODE)];
  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wv = tid >> 6;

  // ---- tile decode (the grid is sized for the most tiles any routing can produce; surplus blocks exit).  XCD
  // blockIdx mod 8 ----
  constexpr bool SPLIT = GROUP == 0;
  const int xcd = (int)(blockIdx.x & 7);
  int slot = (int)(blockIdx.x >> 3);
  int e, mbase, mlen, kbase = 0, klen, nt;
  float* part_out = nullptr;  // where a part of a split tile goes
  if constexpr (GROUP == 0) {
    const int Tn = (EPI == 1) ? (2 * g.F + FBN - 1) / FBN : (g.N + FBN - 1) / FBN;
    const F32Range x = f32_range(g, xcd, Tn);
    klen = g.K;
    if (g.part != nullptr) {
      const int full = x.n & ~63, nkt = (g.K + FBK - 1) / FBK;
      const int S = split_of_f32(x.n, nkt, g.npart);
      if (slot >= full && S > 1) {
        const int j = slot - full, t = j / S, p = j - t * S;
        if (t >= x.n - full) return;
        slot = full + t;
        kbase = nkt * p / S * FBK;
        klen = min(g.K, nkt * (p + 1) / S * FBK) - kbase;
        part_out = g.part + (int64_t)(xcd * g.npart + j) * (FBM * FBN);
      }
    }
    if (slot >= x.n) return;
    const F32Tile t = f32_tile(g, x, slot);
    e = t.e;
    mbase = t.mbase;
    mlen = t.mlen;
    nt = t.nt;
  } else {
    const int Tm = (g.M + FBM - 1) / FBM, Tn = (g.N + FBN - 1) / FBN;
    const int total = g.E * Tm * Tn, chunk = (total + 7) >> 3;
    const int L = xcd * chunk + slot;
    if (slot >= chunk || L >= total) return;
    e = L / (Tm * Tn);
    const int r = L - e * Tm * Tn;
    const int mt = r / Tn;
    nt = r - mt * Tn;
    mbase = mt * FBM;
    mlen = min(FBM, g.M - mbase);
    kbase = g.offsets[e];
    klen = g.offsets[e + 1] - kbase;
  }
  const int n0 = nt * FBN;
  const int nlen = (EPI == 1) ? min(FBN, 2 * (g.F - nt * (FBN / 2))) : min(FBN, g.N - n0);
  const int nk = (klen + FBK - 1) / FBK;

  // ---- operand sources, FNJ 16-byte units q = tid + FNT j a thread.  Rows mode: row q / FCH, k chunk (q % FCH) * 4 of
  // the slice; cols mode: k-row q / 32, i chunk (q % 32) * 4.  Rows / columns past the tile are clamped to valid ones
  // (their results are never stored); k past the reduction reads zeros. ----
  const float* arow[FNJ];
  const float* brow[FNJ];
#pragma unroll
  for (int j = 0; j < FNJ; ++j) {
    const int q = tid + FNT * j;
    if constexpr (AMODE == 0) {
      const int i = min(q / FCH, mlen - 1);
      arow[j] = g.A + (int64_t)(mbase + i) * g.lda + kbase + (q % FCH) * 4;
    } else {
      const int ic = (q & 31) * 4;
      arow[j] = g.A + (int64_t)kbase * g.lda + mbase + (ic < mlen ? ic : 0);
    }
    if constexpr (BMODE == 0) {
      const int i = min(q / FCH, nlen - 1);
      if constexpr (EPI == 1) {
        const int f = nt * (FBN / 2) + (i >> 6) * 32 + (i & 31);
        brow[j] = (((i >> 5) & 1) ? g.B2 : g.B) + (int64_t)e * g.b_estride + (int64_t)f * g.ldb + kbase + (q % FCH) * 4;
      } else {
        brow[j] = g.B + (int64_t)e * g.b_estride + (int64_t)(n0 + i) * g.ldb + (SPLIT ? kbase : 0) + (q % FCH) * 4;
      }
    } else {
      const int ic = (q & 31) * 4;
      const int off = n0 + (ic < nlen ? ic : 0);
      if constexpr (GROUP == 0) brow[j] = g.B + (int64_t)e * g.b_estride + (int64_t)(SPLIT ? kbase : 0) * g.ldb + off;
      else brow[j] = g.B + (int64_t)kbase * g.ldb + off;
    }
  }
  const float* b2row0 = nullptr;  // cols-mode B with a split (dxp): the second source's column base
  const int bsplit = g.b_split - (SPLIT ? kbase : 0);  // in this block's k (not positive: all from the second source)
  if constexpr (BMODE == 1 && GROUP == 0) {
    const int ic = (tid & 31) * 4;
    b2row0 = g.b_split > 0 ? g.B2 + (int64_t)e * g.b_estride + n0 + (ic < nlen ? ic : 0) : nullptr;
  }

  f32x4 ra[FNJ], rb[FNJ];
  auto load = [&](int kt) {
    const int k0 = kt * FBK;
#pragma unroll
    for (int j = 0; j < FNJ; ++j) {
      const int q = tid + FNT * j;
      if constexpr (AMODE == 0) {
        const int k = k0 + (q % FCH) * 4;
        ra[j] = k < klen ? *reinterpret_cast<const f32x4*>(arow[j] + k0) : f32x4{0.f, 0.f, 0.f, 0.f};
      } else {
        const int k = k0 + (q >> 5);
        ra[j] = k < klen ? *reinterpret_cast<const f32x4*>(arow[j] + (int64_t)k * g.lda) : f32x4{0.f, 0.f, 0.f, 0.f};
      }
      if constexpr (BMODE == 0) {
        const int k = k0 + (q % FCH) * 4;
        rb[j] = k < klen ? *reinterpret_cast<const f32x4*>(brow[j] + k0) : f32x4{0.f, 0.f, 0.f, 0.f};
      } else {
        const int k = k0 + (q >> 5);
        const float* src;
        if constexpr (GROUP == 0) {
          // all units of a thread share its column (FNT is a multiple of 32), so the second source's column base
          // b2row0 serves them all
          if (g.b_split > 0 && k >= bsplit) src = b2row0 + (int64_t)(k - bsplit) * g.ldb;
          else src = brow[j] + (int64_t)k * g.ldb;
        } else {
          src = brow[j] + (int64_t)k * g.ldb;
        }
        rb[j] = k < klen ? *reinterpret_cast<const f32x4*>(src) : f32x4{0.f, 0.f, 0.f, 0.f};
      }
    }
  };
  auto store = [&](int buf) {
#pragma unroll
    for (int j = 0; j < FNJ; ++j) {
      const int q = tid + FNT * j;
      if constexpr (AMODE == 0) {
        *reinterpret_cast<f32x4*>(&sa[buf][(q / FCH) * FKP + (q % FCH) * 4]) = ra[j];
      } else {
        *reinterpret_cast<f32x4*>(&sa[buf][(q >> 5) * FIP + (q & 31) * 4]) = ra[j];
      }
      if constexpr (BMODE == 0) {
        *reinterpret_cast<f32x4*>(&sb[buf][(q / FCH) * FKP + (q % FCH) * 4]) = rb[j];
      } else {
        *reinterpret_cast<f32x4*>(&sb[buf][(q >> 5) * FIP + (q & 31) * 4]) = rb[j];
      }
    }
  };

  // fragment of a 32-wide block at `base`, group grp of the slice: the lane's four k
  auto frag = [&](const float* t, auto mode, int base, int grp) -> f32x4 {
    const int i = base + (lane & 31), k = grp * 8 + (lane >> 5) * 4;
    if constexpr (decltype(mode)::value == 0) return *reinterpret_cast<const f32x4*>(&t[i * FKP + k]);
    else return f32x4{t[k * FIP + i], t[(k + 1) * FIP + i], t[(k + 2) * FIP + i], t[(k + 3) * FIP + i]};
  };
  using AM = std::integral_constant<int, AMODE>;
  using BM = std::integral_constant<int, BMODE>;

  // Wave w: rows [32 (w / 2), ...+32) and columns [64 (w % 2), ...+64) of the tile.  Waves w and w + 4 share a SIMD,
  // so where a segment's last rows fill at most half a tile, the waves without rows leave every SIMD half its MFMAs.
  const int wm0 = (wv >> 1) * 32, wn0 = (wv & 1) * 64;
  const bool rows = wm0 < mlen;
  f32x16 acc[2];
#pragma unroll
  for (int ni = 0; ni < 2; ++ni)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[ni][r] = 0.f;

  if (nk > 0) {
    load(0);
    store(0);
    __syncthreads();
    for (int kt = 0; kt < nk; ++kt) {
      const int buf = kt & 1;
      if (kt + 1 < nk) load(kt + 1);  // in flight during this slice's MFMAs
      if (rows) {
#pragma unroll
        for (int grp = 0; grp < FBK / 8; ++grp) {
          const f32x4 fa = frag(sa[buf], AM{}, wm0, grp);
          const f32x4 fb0 = frag(sb[buf], BM{}, wn0, grp), fb1 = frag(sb[buf], BM{}, wn0 + 32, grp);
#pragma unroll
          for (int s = 0; s < 4; ++s) {
            acc[0] = mfma32x32x2_f32(fa[s], fb0[s], acc[0]);
            acc[1] = mfma32x32x2_f32(fa[s], fb1[s], acc[1]);
          }
        }
      }
      if (kt + 1 < nk) {
        store(buf ^ 1);  // the other buffer was last read in slice kt-1, before the barrier that ended it
        __syncthreads();
      }
    }
  }

  // ---- epilogue straight from the accumulators: acc[ni][r] = C[wm0 + 8 (r/4) + 4 (lane/32) + r%4]
  // [wn0 + ni*32 + lane%32]; 32 lanes of a row write 128 consecutive bytes ----
  const int jl = lane & 31;
  if constexpr (SPLIT) {
    if (part_out != nullptr) {  // a part of a split tile: fp32, [128][128]
#pragma unroll
      for (int r = 0; r < 16; ++r) {
        const int ri = wm0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
        if (ri >= mlen) continue;
        part_out[ri * FBN + wn0 + jl] = acc[0][r];
        part_out[ri * FBN + wn0 + 32 + jl] = acc[1][r];
      }
      return;
    }
  }
#pragma unroll
  for (int r = 0; r < 16; ++r) {
    const int ri = wm0 + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3);
    if (ri >= mlen) continue;
    const int64_t row = mbase + ri;
    if constexpr (EPI == 1) {
      // the wave's two n blocks: gate (ni = 0) and up (ni = 1) of the same 32 f
      const int f = nt * (FBN / 2) + (wn0 >> 6) * 32 + jl;
      if (f >= g.F) continue;
      const float gv = acc[0][r], uv = acc[1][r];
      g.C[row * g.ldc + f] = gv * sig32(gv) * uv;
      if (g.C2 != nullptr) {
        g.C2[row * 2 * (int64_t)g.F + f] = gv;
        g.C2[row * 2 * (int64_t)g.F + g.F + f] = uv;
      }
    } else {
#pragma unroll
      for (int ni = 0; ni < 2; ++ni) {
        const int c = n0 + wn0 + ni * 32 + jl;
        if (c >= g.N) continue;
        const float v = acc[ni][r];
        if constexpr (EPI == 2) {
          const float gv = g.X[row * 2 * (int64_t)g.F + c], uv = g.X[row * 2 * (int64_t)g.F + g.F + c];
          const float sg = sig32(gv);
          g.C[row * g.ldc + c] = v * uv * sg * (1.f + gv * (1.f - sg));
          g.C[row * g.ldc + g.F + c] = v * gv * sg;
        } else if constexpr (GROUP == 0) {
          g.C[row * g.ldc + c] = v;
        } else {
          const bool second = g.c_split > 0 && row >= g.c_split;
          float* base = (second ? g.C2 : g.C) + (int64_t)e * g.c_estride;
          base[(second ? row - g.c_split : row) * g.ldc + c] = v;
        }
      }
    }
  }
}

// Sums the parts of the split tiles (k_gemm_f32, split_of_f32) in split order and forms the product's epilogue: block
// (t, y) takes 16 rows of the t-th split tile of XCD t / 64.
template <int EPI>
__global__ __launch_bounds__(256) void k_gemm_reduce_f32(GemmF32Args g) {
  const int xcd = (int)(blockIdx.x >> 6), t = (int)(blockIdx.x & 63);
  const int Tn = (EPI == 1) ? (2 * g.F + FBN - 1) / FBN : (g.N + FBN - 1) / FBN;
  const F32Range x = f32_range(g, xcd, Tn);
  if (t >= (x.n & 63)) return;
  const int S = split_of_f32(x.n, (g.K + FBK - 1) / FBK, g.npart);
  if (S == 1) return;
  const F32Tile d = f32_tile(g, x, (x.n & ~63) + t);
  const float* const src = g.part + (int64_t)(xcd * g.npart + t * S) * (FBM * FBN);
  auto sum = [&](int at) {
    f32x4 s = *reinterpret_cast<const f32x4*>(src + at);
    for (int p = 1; p < S; ++p) s += *reinterpret_cast<const f32x4*>(src + (int64_t)p * (FBM * FBN) + at);
    return s;
  };
  for (int u = threadIdx.x; u < 16 * FBN / 4; u += 256) {
    const int r = (int)blockIdx.y * 16 + u / (FBN / 4), c = (u % (FBN / 4)) * 4;
    if (r >= d.mlen) continue;
    const int64_t row = d.mbase + r;
    if constexpr (EPI == 1) {
      // tile column c: pair c / 64 of 32 gate columns and the 32 up columns of the same f
      const int f = d.nt * (FBN / 2) + (c >> 6) * 32 + (c & 31);
      if ((c & 32) || f >= g.F) continue;
      const f32x4 gv = sum(r * FBN + c), uv = sum(r * FBN + c + 32);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        g.C[row * g.ldc + f + j] = gv[j] * sig32(gv[j]) * uv[j];
        if (g.C2 != nullptr) {
          g.C2[row * 2 * (int64_t)g.F + f + j] = gv[j];
          g.C2[row * 2 * (int64_t)g.F + g.F + f + j] = uv[j];
        }
      }
    } else {
      const int n0 = d.nt * FBN + c;
      if (n0 >= g.N) continue;  // N % 4 == 0
      const f32x4 v = sum(r * FBN + c);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        if constexpr (EPI == 2) {
          const float gv = g.X[row * 2 * (int64_t)g.F + n0 + j], uv = g.X[row * 2 * (int64_t)g.F + g.F + n0 + j];
          const float sg = sig32(gv);
          g.C[row * g.ldc + n0 + j] = v[j] * uv * sg * (1.f + gv * (1.f - sg));
          g.C[row * g.ldc + g.F + n0 + j] = v[j] * gv * sg;
        } else {
          g.C[row * g.ldc + n0 + j] = v[j];
        }
      }
    }
  }
}

__global__ __launch_bounds__(1024) void k_gemm_tiles_f32(const int* __restrict__ offsets, int E,
                                                         int* __restrict__ tile_off) {
  // tile_off[e+1] = sum_{e' <= e} ceil(rows_e' / 128) (one block, E <= 1024)
  __shared__ int part[1024];
  const int tid = threadIdx.x;
  part[tid] = tid < E ? (offsets[tid + 1] - offsets[tid] + FBM - 1) / FBM : 0;
  __syncthreads();
  for (int o = 1; o < E; o <<= 1) {
    const int v = tid >= o ? part[tid - o] : 0;
    __syncthreads();
    part[tid] += v;
    __syncthreads();
  }
  if (tid == 0) tile_off[0] = 0;
  if (tid < E) tile_off[tid + 1] = part[tid];
}

namespace {
bool a16f(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15u) == 0; }

template <int AM, int BMD, int GR, int EP>
int launch_f32(const char* name, hipStream_t s, const GemmF32Args& a, int64_t R) {
  int64_t blocks, Tn = 0;
  if constexpr (GR == 0) {
    Tn = EP == 1 ? (2 * (int64_t)a.F + FBN - 1) / FBN : ((int64_t)a.N + FBN - 1) / FBN;
    blocks = ((R + FBM - 1) / FBM + a.E) * Tn;
  } else {
    blocks = (int64_t)a.E * ((a.M + FBM - 1) / FBM) * ((a.N + FBN - 1) / FBN);
  }
  if (blocks <= 0) return 0;
  // an XCD's share is the largest eighth of the column tiles (f32_range), or of all tiles
  if constexpr (GR == 0) blocks = 8 * std::max((blocks + 7) / 8, ((R + FBM - 1) / FBM + a.E) * ((Tn + 7) / 8));
  else blocks = (blocks + 7) / 8 * 8;
  if (GR == 0 && a.part != nullptr) blocks += 8 * a.npart;  // the parts of each XCD's split tiles
  MOE_LAUNCH(name, (k_gemm_f32<AM, BMD, GR, EP>), dim3((unsigned)blocks), dim3(FNT), 0, s, a);
  if constexpr (GR == 0) {
    if (a.part != nullptr)
      MOE_LAUNCH("k_gemm_reduce_f32", k_gemm_reduce_f32<EP>, dim3(8 * 64, FBM / 16), dim3(256), 0, s, a);
  }
  return check_launch(name);
}

// Partial tiles: 16 a tile, at most kSplitMaxF32 an XCD; none for a product of 16 rounds or more, or where the caller's
// workspace has no room for them.  cols: columns of the product's tiles (2F for the gate/up product).
int split_parts_f32(int64_t R, int64_t E, int64_t cols) {
  const int64_t tiles = ((R + FBM - 1) / FBM + E) * ((cols + FBN - 1) / FBN);
  return (int)std::min<int64_t>(kSplitMaxF32, 16 * ((tiles + 7) / 8));
}
size_t split_bytes_f32(int64_t R, int64_t E, int64_t cols) {
  if (R <= 0 || E <= 0 || R / FBM * ((cols + FBN - 1) / FBN) >= 16 * 512) return 0;
  return (size_t)8 * split_parts_f32(R, E, cols) * FBM * FBN * sizeof(float);
}
void take_split_f32(GemmF32Args& a, int64_t R, int64_t cols, void* ws, size_t ws_bytes) {
  const size_t used = moe_swiglu_f32_workspace(a.E), need = split_bytes_f32(R, a.E, cols);
  if (need == 0 || ws_bytes < used + need) return;
  a.part = reinterpret_cast<float*>(static_cast<char*>(ws) + used);
  a.npart = split_parts_f32(R, a.E, cols);
}

int check_f32(const char* what, int64_t R, int64_t H, int64_t F, int64_t E) {
  if (R < 0 || H < 4 || F < 32 || E < 1 || E > 1024 || H % 4 || F % 32)
    return fail_arg("%s: bad shape R=%lld H=%lld F=%lld E=%lld (need H%%4==0, F%%32==0, E<=1024)", what,
                    (long long)R, (long long)H, (long long)F, (long long)E);
  return 0;
}
}  // namespace
}  // namespace moe

using namespace moe;

extern "C" size_t moe_swiglu_f32_workspace(int64_t E) { return (size_t)((E + 1) * 4 + 255) & ~(size_t)255; }

extern "C" size_t moe_swiglu_f32_split_workspace(int64_t R, int64_t H, int64_t F, int64_t E) {
  // the most that one of the products takes: 2F (gate/up), F (dact) or H columns (the others), each by its own size
  return std::max({split_bytes_f32(R, E, 2 * F), split_bytes_f32(R, E, F), split_bytes_f32(R, E, H)});
}

extern "C" size_t moe_swiglu_fwd_f32_split_workspace(int64_t R, int64_t H, int64_t F, int64_t E) {
  if (swiglu_small_takes(R, H, F, E, 4)) return 0;
  return std::max(split_bytes_f32(R, E, 2 * F), split_bytes_f32(R, E, H));
}

extern "C" int moe_swiglu_fwd_f32(const float* xp, const float* w_gate, const float* w_up, const float* w_down,
                                  const int32_t* offsets, int64_t R, int64_t H, int64_t F, int64_t E, float* act,
                                  float* hgu, float* y, void* workspace, size_t ws_bytes, void* stream) {
  if (int rc = check_f32("moe_swiglu_fwd_f32", R, H, F, E)) return rc;
  if (R == 0) return 0;
  if (!xp || !w_gate || !w_up || !w_down || !offsets || !act || !y || !a16f(xp) || !a16f(w_gate) || !a16f(w_up) ||
      !a16f(w_down))
    return fail_arg("moe_swiglu_fwd_f32: null or misaligned pointer");
  if (!workspace || ws_bytes < moe_swiglu_f32_workspace(E))
    return set_error("moe_swiglu_fwd_f32: workspace"), MOE_EWORKSPACE;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  if (a16f(act) && a16f(y) && (!hgu || a16f(hgu)) && swiglu_small_takes(R, H, F, E, 4))
    return swiglu_small_fwd(true, xp, w_gate, w_up, w_down, offsets, R, H, F, E, act, hgu, y, s);
  int* tile_off = static_cast<int*>(workspace);
  MOE_LAUNCH("k_gemm_tiles_f32", k_gemm_tiles_f32, dim3(1), dim3(1024), 0, s, offsets, (int)E, tile_off);
  GemmF32Args a{};
  a.offsets = offsets;
  a.tile_off = tile_off;
  a.E = (int)E;
  a.F = (int)F;
  // fwd1: [act | hgu] = xp . [Wg ; Wu]^T
  a.A = xp;
  a.lda = H;
  a.B = w_gate;
  a.B2 = w_up;
  a.ldb = H;
  a.b_estride = F * H;
  a.C = act;
  a.C2 = hgu;
  a.ldc = F;
  a.N = (int)(2 * F);
  a.K = (int)H;
  take_split_f32(a, R, 2 * F, workspace, ws_bytes);
  if (int rc = launch_f32<0, 0, 0, 1>("k_gemm_swiglu_fwd1_f32", s, a, R)) return rc;
  // fwd2: y = act . Wd^T
  GemmF32Args b{};
  b.offsets = offsets;
  b.tile_off = tile_off;
  b.E = (int)E;
  b.F = (int)F;
  b.A = act;
  b.lda = F;
  b.B = w_down;
  b.ldb = F;
  b.b_estride = H * F;
  b.C = y;
  b.ldc = H;
  b.N = (int)H;
  b.K = (int)F;
  take_split_f32(b, R, H, workspace, ws_bytes);
  return launch_f32<0, 0, 0, 0>("k_gemm_swiglu_fwd2_f32", s, b, R);
}

extern "C" int moe_swiglu_bwd_f32(const float* dy, const float* xp, const float* act, const float* hgu,
                                  const float* w_gate, const float* w_up, const float* w_down, const int32_t* offsets,
                                  int64_t R, int64_t H, int64_t F, int64_t E, float* dh, float* dxp, float* dw_gate,
                                  float* dw_up, float* dw_down, void* workspace, size_t ws_bytes, void* stream) {
  if (int rc = check_f32("moe_swiglu_bwd_f32", R, H, F, E)) return rc;
  if (!dy || !xp || !act || !hgu || !w_gate || !w_up || !w_down || !offsets || !dh || !dxp || !dw_gate || !dw_up ||
      !dw_down)
    return fail_arg("moe_swiglu_bwd_f32: null pointer argument");
  if (!a16f(dy) || !a16f(xp) || !a16f(act) || !a16f(dh) || !a16f(w_gate) || !a16f(w_up) || !a16f(w_down))
    return fail_arg("moe_swiglu_bwd_f32: operands must be 16-byte aligned");
  if (!workspace || ws_bytes < moe_swiglu_f32_workspace(E))
    return set_error("moe_swiglu_bwd_f32: workspace"), MOE_EWORKSPACE;
  hipStream_t s = reinterpret_cast<hipStream_t>(stream);
  int* tile_off = static_cast<int*>(workspace);
  MOE_LAUNCH("k_gemm_tiles_f32", k_gemm_tiles_f32, dim3(1), dim3(1024), 0, s, offsets, (int)E, tile_off);
  if (R > 0) {
    // dA: dh = epilogue(dy . Wd)   (B[n = f][k = h] = Wd[h][f])
    GemmF32Args a{};
    a.offsets = offsets;
    a.tile_off = tile_off;
    a.E = (int)E;
    a.F = (int)F;
    a.A = dy;
    a.lda = H;
    a.B = w_down;
    a.ldb = F;
    a.b_estride = H * F;
    a.C = dh;
    a.ldc = 2 * F;
    a.X = hgu;
    a.N = (int)F;
    a.K = (int)H;
    take_split_f32(a, R, F, workspace, ws_bytes);
    if (int rc = launch_f32<0, 1, 0, 2>("k_gemm_swiglu_dact_f32", s, a, R)) return rc;
    // dxp = dh . [Wg ; Wu]   (B[n = h][k = j] = W1[j][h])
    GemmF32Args b{};
    b.offsets = offsets;
    b.tile_off = tile_off;
    b.E = (int)E;
    b.F = (int)F;
    b.A = dh;
    b.lda = 2 * F;
    b.B = w_gate;
    b.B2 = w_up;
    b.b_split = (int)F;
    b.ldb = H;
    b.b_estride = F * H;
    b.C = dxp;
    b.ldc = H;
    b.N = (int)H;
    b.K = (int)(2 * F);
    take_split_f32(b, R, H, workspace, ws_bytes);
    if (int rc = launch_f32<0, 1, 0, 0>("k_gemm_swiglu_dxp_f32", s, b, R)) return rc;
  }
  // dWd_e = dy_e^T . act_e   (M = H, N = F, K = rows of e)
  GemmF32Args c{};
  c.offsets = offsets;
  c.E = (int)E;
  c.A = dy;
  c.lda = H;
  c.B = act;
  c.ldb = F;
  c.C = dw_down;
  c.ldc = F;
  c.c_estride = H * F;
  c.M = (int)H;
  c.N = (int)F;
  if (int rc = launch_f32<1, 1, 1, 0>("k_gemm_swiglu_dwd_f32", s, c, R)) return rc;
  // [dWg_e ; dWu_e] = dh_e^T . xp_e   (M = 2F, N = H, K = rows of e)
  GemmF32Args d{};
  d.offsets = offsets;
  d.E = (int)E;
  d.A = dh;
  d.lda = 2 * F;
  d.B = xp;
  d.ldb = H;
  d.C = dw_gate;
  d.C2 = dw_up;
  d.c_split = (int)F;
  d.ldc = H;
  d.c_estride = F * H;
  d.M = (int)(2 * F);
  d.N = (int)H;
  return launch_f32<1, 1, 1, 0>("k_gemm_swiglu_dw1_f32", s, d, R);
}
