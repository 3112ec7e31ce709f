// Grouped SwiGLU expert products for few rows per expert (decode batches, small prompts), bf16 and fp32.
//
// With r rows an expert costs 6 r F H flops over 3 F H weights: below about a hundred rows the weights' stream
// bounds both forward products, and the 256-row (bf16) and 128-row (fp32) tiles of gemm.hip / gemm_f32.hip leave
// most of the memory system idle: one block a CU, two k slices in flight, and as few tiles as the output is wide.
// Here a block owns 16 NF weight rows of one expert (gate/up product: 8 NF gate and the matching 8 NF up rows) and
// streams them once, its NW waves each taking every NW-th 128-byte column chunk, straight from HBM into MFMA
// fragments: v_mfma_f32_16x16x32_bf16 / v_mfma_f32_16x16x4_f32 with 16 weight rows as the M operand and 16 token
// rows as the N operand, so a lane's 16-byte load is its fragment: lane 16 q + r reads bytes [16 q, 16 q + 16) of a
// 64-byte half chunk of row r, and the four lanes of a row make one 64-byte request.  The k slot a value lands in
// is free as long as both operands agree.  Each wave keeps one whole chunk of weights in flight beyond the one it
// multiplies.  The tokens' fragments come from L2 (re-read by every block).  The waves' partial sums meet in LDS
// in wave order (fp32), where the SwiGLU is formed with the large kernels' own roundings.  Every 64 rows of an
// expert (fp32: 32) are a pass of their own blocks over its weights, so a skewed routing's passes run beside each other.
// No tile table: a block finds its rows from `offsets`.
//
// Blocks start their chunks at different columns (a hash of the expert and its column tile, wrapping around the row):
// rows lie a power of two apart, and blocks that walk them in step ask the same few memory channels.  The start decides
// the order of a row's sums, so it depends on nothing else: a row has the same bits whatever other experts' rows, and its
// own expert's, are beside it.  (The passes of a tile over the same weights walk them together.)  Measured at E = 8,
// H = 4096, F = 14336, one row an expert: 591 us for both products in step, 487 us started apart (5.8 TB/s of weights);
// 718 / 558 us with non-temporal loads (each 128-byte line is asked for in two halves, which a cached load fetches once).
//
// Against the 256-row tiles (split last rounds included), bf16, both products, us, tiles -> here; "routed" is the top-K
// of random logits, "skewed" the same with a Zipf(1.1) bias on the experts:
//   rows an expert, mean    1 each       16 routed   16 skewed   24 routed   24 skewed   28 routed   32 each    64 each
//   E 8,   H 4096, F 14336  643 -> 485   630 -> 563  635 -> 595  637 -> 602  641 -> 696  638 -> 654  636 -> 634  651 -> 806
//   E 128, H 2048, F 768    303 -> 210   308 -> 263  211 -> 212  308 -> 288  244 -> 256  310 -> 307  313 -> 297  343 -> 393
//   E 32,  H 2048, F 4096   404 -> 269   404 -> 323  384 -> 353  402 -> 360  375 -> 375  404 -> 383  409 -> 368  409 -> 461
// With passes of 32 rows an expert's further rows cost as many more streams of its weights: 24 skewed 777, 288 and 426.
// Routings that put nearly all rows on a few of many experts are what is left to the tiles' favour (E 128, Zipf(2), 16
// rows: 118 -> 148).  fp32, E = 8, H = 1024, F = 4096, one row each, against its 128-row tiles: 463 -> 77 us; its sums
// are slow enough that rows and not weights bound a pass, and it keeps 32 of them.
#include <algorithm>

#include "common.h"

namespace moe {

struct SmallArgs {
  const uint8_t* A;    // rows [R][K]
  const uint8_t* B;    // weights [E][N][K] (gate for the gate/up product)
  const uint8_t* B2;   // up weights
  void* C;             // act [R][F] / y [R][N]
  void* C2;            // hgu [R][2F] (gate/up product; null for inference)
  const int* offsets;  // [E+1]
  int64_t b_ebytes;    // bytes of one expert's matrix
  uint32_t kbytes;     // bytes of a row of A and B
  int N;               // output columns: F (gate/up) or H
  int Tn;              // column tiles
  int E;
};

namespace {


__device__ __forceinline__ float sig_bf(float g) { return __builtin_amdgcn_rcpf(1.f + __expf(-g)); }
__device__ __forceinline__ float sig_f32(float g) { return 1.f / (1.f + expf(-g)); }

template <bool F32>
__device__ __forceinline__ f32x4 mma16(const u32x4& w, const u32x4& a, f32x4 c) {
  if constexpr (F32) {
#pragma unroll
    for (int s = 0; s < 4; ++s)
      c = __builtin_amdgcn_mfma_f32_16x16x4f32(__uint_as_float(w[s]), __uint_as_float(a[s]), c, 0, 0, 0);
    return c;
  } else {
    return mfma16x16x32(__builtin_bit_cast(bf16x8, w), __builtin_bit_cast(bf16x8, a), c);
  }
}

// One pass: rows [row0, row0 + min(rows, 16 MT)) of the segment against the block's 16 NF weight rows.
template <bool F32, bool GU, int NF, int NW, int MT>
__device__ __forceinline__ void small_pass(const SmallArgs& g, const uint8_t* base0, const uint8_t* base1, int64_t row0,
                                           int rows, int n0, uint32_t tile, float* red) {
  const int tid = threadIdx.x, lane = tid & 63, wv = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int r = lane & 15, q = lane >> 4;
  const uint32_t kb = g.kbytes;
  constexpr int RP = NF * 16 + 4;  // floats a row of the partial sums
  // fragment f of the 16 NF weight rows: GU: the first NF / 2 gate rows, the others up rows; rows past N repeat the last
  uint32_t wo[NF], ao[MT];
#pragma unroll
  for (int f = 0; f < NF; ++f) {
    const int n = GU ? n0 + (f % (NF / 2)) * 16 + r : min(n0 + f * 16 + r, g.N - 1);
    wo[f] = (uint32_t)n * kb + q * 16;
  }
#pragma unroll
  for (int m = 0; m < MT; ++m) ao[m] = (uint32_t)min(m * 16 + r, rows - 1) * kb + q * 16;
  const uint8_t* const arow = g.A + row0 * kb;

  // the tokens' fragments of the chunk being multiplied are loaded just before it (MT >= 2: an L2 round trip hidden
  // by the other waves) or with its weights (MT == 1, where there are registers for both)
  constexpr int AB = MT == 1 ? 2 : 1;
  u32x4 wb[2][NF][2], ab[AB][MT][2];
  auto load_a = [&](int b, int c) {
    const uint32_t k0 = (uint32_t)c * 128;
#pragma unroll
    for (int s = 0; s < 2; ++s) {
      const bool in = k0 + s * 64 + q * 16 < kb;
      const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
      for (int m = 0; m < MT; ++m) {
        const u32x4 v = *reinterpret_cast<const u32x4*>(arow + (ao[m] + (in ? k0 + s * 64 : 0u)));
        ab[b][m][s] = in ? v : z;
      }
    }
  };
  auto load = [&](int b, int c) {
    if constexpr (AB == 2) load_a(b, c);
    const uint32_t k0 = (uint32_t)c * 128;
    if (k0 + 128 <= kb) {
#pragma unroll
      for (int s = 0; s < 2; ++s) {
#pragma unroll
        for (int f = 0; f < NF; ++f)
          wb[b][f][s] = *reinterpret_cast<const u32x4*>((GU && f >= NF / 2 ? base1 : base0) + (wo[f] + (k0 + s * 64)));
      }
    } else {  // the row's last, partial chunk: 16-byte units past its end are zeros on both sides
#pragma unroll
      for (int s = 0; s < 2; ++s) {
        const bool in = k0 + s * 64 + q * 16 < kb;
        const uint32_t k = in ? k0 + s * 64 : 0u;
        const u32x4 z = {0u, 0u, 0u, 0u};
#pragma unroll
        for (int f = 0; f < NF; ++f) {
          const u32x4 v = *reinterpret_cast<const u32x4*>((GU && f >= NF / 2 ? base1 : base0) + (wo[f] + k));
          wb[b][f][s] = in ? v : z;
        }
      }
    }
  };
  f32x4 acc[NF][MT];
#pragma unroll
  for (int f = 0; f < NF; ++f)
#pragma unroll
    for (int m = 0; m < MT; ++m) acc[f][m] = f32x4{0.f, 0.f, 0.f, 0.f};
  auto mma = [&](int b, int c) {
    if constexpr (AB == 1) load_a(0, c);
#pragma unroll
    for (int s = 0; s < 2; ++s)
#pragma unroll
      for (int f = 0; f < NF; ++f)
#pragma unroll
        for (int m = 0; m < MT; ++m) acc[f][m] = mma16<F32>(wb[b][f][s], ab[AB == 2 ? b : 0][m][s], acc[f][m]);
  };
  const int nc = (int)((kb + 127) / 128);
  const int start = (int)__umulhi(tile * 0x9E3779B1u, (uint32_t)nc);
  auto at = [&](int i) {
    const int c = i + start;
    return c < nc ? c : c - nc;
  };
  int c = wv;
  if (c < nc) {
    load(0, at(c));
    for (;;) {
      if (c + NW < nc) load(1, at(c + NW));
      mma(0, at(c));
      c += NW;
      if (c >= nc) break;
      if (c + NW < nc) load(0, at(c + NW));
      mma(1, at(c));
      c += NW;
      if (c >= nc) break;
    }
  }

  // acc[f][m][j] of lane 16 q + r: weight row 16 f + 4 q + j, token row 16 m + r
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    if (m * 16 >= rows) break;
    if (m > 0) __syncthreads();
#pragma unroll
    for (int f = 0; f < NF; ++f)
      *reinterpret_cast<f32x4*>(&red[(wv * 16 + r) * RP + f * 16 + q * 4]) = acc[f][m];
    __syncthreads();
    constexpr int PAIRS = GU ? NF * 4 : NF * 8;  // column pairs a row
    for (int u = tid; u < 16 * PAIRS; u += NW * 64) {
      const int mr = u / PAIRS, p = (u % PAIRS) * 2;
      if (m * 16 + mr >= rows) continue;
      const int64_t row = row0 + m * 16 + mr;
      float v[2] = {0.f, 0.f}, w[2] = {0.f, 0.f};
#pragma unroll
      for (int x = 0; x < NW; ++x) {
        const float2 s = *reinterpret_cast<const float2*>(&red[(x * 16 + mr) * RP + p]);
        v[0] += s.x;
        v[1] += s.y;
        if constexpr (GU) {
          const float2 t = *reinterpret_cast<const float2*>(&red[(x * 16 + mr) * RP + NF * 8 + p]);
          w[0] += t.x;
          w[1] += t.y;
        }
      }
      const int n = n0 + p;
      if constexpr (F32) {
        float* C = static_cast<float*>(g.C);
        if constexpr (GU) {
          *reinterpret_cast<float2*>(C + row * g.N + n) =
              float2{v[0] * sig_f32(v[0]) * w[0], v[1] * sig_f32(v[1]) * w[1]};
          if (g.C2 != nullptr) {
            float* h = static_cast<float*>(g.C2) + row * 2 * (int64_t)g.N + n;
            *reinterpret_cast<float2*>(h) = float2{v[0], v[1]};
            *reinterpret_cast<float2*>(h + g.N) = float2{w[0], w[1]};
          }
        } else if (n < g.N) {
          *reinterpret_cast<float2*>(C + row * g.N + n) = float2{v[0], v[1]};
        }
      } else {
        uint16_t* C = static_cast<uint16_t*>(g.C);
        const uint32_t vb = pack2bf(v[0], v[1]);
        if constexpr (GU) {
          // gate and up rounded to bf16, then act, as the 256-row tiles' epilogue
          const uint32_t ub = pack2bf(w[0], w[1]);
          const float g0 = __uint_as_float(vb << 16), g1 = __uint_as_float(vb & 0xffff0000u);
          *reinterpret_cast<uint32_t*>(C + row * g.N + n) =
              pack2bf(g0 * sig_bf(g0) * __uint_as_float(ub << 16), g1 * sig_bf(g1) * __uint_as_float(ub & 0xffff0000u));
          if (g.C2 != nullptr) {
            uint16_t* h = static_cast<uint16_t*>(g.C2) + row * 2 * (int64_t)g.N + n;
            *reinterpret_cast<uint32_t*>(h) = vb;
            *reinterpret_cast<uint32_t*>(h + g.N) = ub;
          }
        } else if (n < g.N) {
          *reinterpret_cast<uint32_t*>(C + row * g.N + n) = vb;
        }
      }
    }
  }
}

// Rows of a pass: 64 take 250 registers of the 256 that two waves a SIMD have (NF = 4).
template <bool F32>
constexpr int pass_rows() {
  return F32 ? 32 : 64;
}

template <bool F32, bool GU, int NF, int NW>
__global__ __launch_bounds__(NW * 64, 8 / NW) void k_gemm_small(SmallArgs g) {
  __shared__ __attribute__((aligned(16))) float red[NW * 16 * (NF * 16 + 4)];
  constexpr int PR = pass_rows<F32>();
  const int slot = (int)(blockIdx.x / g.Tn), nt = (int)(blockIdx.x % g.Tn);
  int e = slot, pass = 0;
  if (slot >= g.E) {  // the (slot - E)-th of the passes past the experts' first ones
    const int lane = threadIdx.x & 63;
    int x = slot - g.E;
    for (int e0 = 0;; e0 += 64) {
      if (e0 >= g.E) return;
      const int i = e0 + lane;
      const int c = i < g.E ? max((g.offsets[i + 1] - g.offsets[i] + PR - 1) / PR - 1, 0) : 0;
      int upto = c;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const int v = __shfl_up(upto, o);
        upto += lane >= o ? v : 0;
      }
      const unsigned long long past = __ballot(x < upto);
      if (past) {
        const int l = __builtin_ctzll(past);
        e = e0 + l;
        pass = x - (__shfl(upto, l) - __shfl(c, l)) + 1;
        break;
      }
      x -= __shfl(upto, 63);
    }
    e = __builtin_amdgcn_readfirstlane(e);
    pass = __builtin_amdgcn_readfirstlane(pass);
  }
  const int m0 = g.offsets[e] + pass * PR, hi = g.offsets[e + 1];
  if (m0 >= hi) return;
  const int n0 = nt * NF * (GU ? 8 : 16);
  const uint8_t* const b0 = g.B + (int64_t)e * g.b_ebytes;
  const uint8_t* const b1 = GU ? g.B2 + (int64_t)e * g.b_ebytes : nullptr;
  const uint32_t tile = (uint32_t)(e * g.Tn + nt);
  if (PR > 32 && hi - m0 > 32) small_pass<F32, GU, NF, NW, PR / 16>(g, b0, b1, m0, min(PR, hi - m0), n0, tile, red);
  else if (hi - m0 > 16) small_pass<F32, GU, NF, NW, 2>(g, b0, b1, m0, min(32, hi - m0), n0, tile, red);
  else small_pass<F32, GU, NF, NW, 1>(g, b0, b1, m0, hi - m0, n0, tile, red);
}

// 64 weight rows and four waves a block; where that leaves fewer than 512 blocks (two a CU), 32 rows and eight
// waves: fp32 E = 8, H = 1024, F = 4096 (128 blocks of the down projection) 104 -> 77 us.
template <bool F32, bool GU>
int launch_small(const char* name, hipStream_t s, SmallArgs a, int64_t E, int64_t R) {
  a.E = (int)E;
  const int64_t slots = E + R / pass_rows<F32>();  // every expert's first pass, and as many more as R rows can need
  if (cdiv(a.N, GU ? 32 : 64) * E >= 512) {
    a.Tn = cdiv(a.N, GU ? 32 : 64);
    MOE_LAUNCH(name, (k_gemm_small<F32, GU, 4, 4>), dim3((unsigned)(a.Tn * slots)), dim3(256), 0, s, a);
  } else {
    a.Tn = cdiv(a.N, GU ? 16 : 32);
    MOE_LAUNCH(name, (k_gemm_small<F32, GU, 2, 8>), dim3((unsigned)(a.Tn * slots)), dim3(512), 0, s, a);
  }
  return check_launch(name);
}
}  // namespace

// Up to 24 rows an expert on average (fp32: 32): routed rows gain 6-16% there on every layer measured and nothing at 28;
// skewed ones gain up to 16 and give back at most 9% at 24 (figures at the top).  The host does not know the rows of each
// expert.  A weight slice and a pass's rows are addressed by 32-bit byte offsets.
bool swiglu_small_takes(int64_t R, int64_t H, int64_t F, int64_t E, int elem) {
  const int64_t lim = (int64_t)1 << 32;
  return R <= (elem == 4 ? 32 : 24) * E && H * F * elem < lim && 64 * std::max(H, F) * elem < lim &&
         (E + R / 32) * std::max((F + 15) / 16, (H + 31) / 32) < ((int64_t)1 << 31);
}

int swiglu_small_fwd(bool f32, const void* xp, const void* w_gate, const void* w_up, const void* w_down,
                     const int* offsets, int64_t R, int64_t H, int64_t F, int64_t E, void* act, void* hgu, void* y,
                     hipStream_t s) {
  const int elem = f32 ? 4 : 2;
  SmallArgs a{};
  a.offsets = offsets;
  a.b_ebytes = H * F * elem;
  a.A = static_cast<const uint8_t*>(xp);
  a.B = static_cast<const uint8_t*>(w_gate);
  a.B2 = static_cast<const uint8_t*>(w_up);
  a.C = act;
  a.C2 = hgu;
  a.kbytes = (uint32_t)(H * elem);
  a.N = (int)F;
  const int rc = f32 ? launch_small<true, true>("k_gemm_small_fwd1_f32", s, a, E, R)
                     : launch_small<false, true>("k_gemm_small_fwd1", s, a, E, R);
  if (rc) return rc;
  SmallArgs b{};
  b.offsets = offsets;
  b.b_ebytes = H * F * elem;
  b.A = static_cast<const uint8_t*>(act);
  b.B = static_cast<const uint8_t*>(w_down);
  b.C = y;
  b.kbytes = (uint32_t)(F * elem);
  b.N = (int)H;
  return f32 ? launch_small<true, false>("k_gemm_small_fwd2_f32", s, b, E, R)
             : launch_small<false, false>("k_gemm_small_fwd2", s, b, E, R);
}

}  // namespace moe
