// gfx950 prompt products for few tokens (and for matrices too small to fill the chip with large tiles).
//
// The tiled products of prefill.hip give a workgroup 128 or 256 weight rows and walk K block by block: with 4096 rows
// that is 32 workgroups on 256 CUs, and a 14336-column product takes the 112 blocks' latency whatever the token count.
// Here a workgroup owns 16 or 32 weight rows and its eight waves share K: in one round wave w multiplies block 8 r + w,
// so every matrix has rows / 16 workgroups and the weights of a round, 1 KiB of every row, are in flight at once.
#include <math.h>
#include <stdlib.h>

#include <algorithm>

#include "act.hpp"
#include "launch.hpp"

namespace qph {

typedef int v4i __attribute__((ext_vector_type(4)));

__device__ __forceinline__ float sk_silu_mul(float g, float u) { return g / (1.f + exp_poly(0.f - g)) * u; }   // kernels_x86.cpp:427-431

// LDS written by this wave is visible, every wave is here; global loads stay in flight (__syncthreads would wait for them)
__device__ __forceinline__ void lds_barrier() {
  asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory");
}

// ------------------------------------------------------------------ q8, K split over the waves
// Tile: 16 RT weight rows x 16 NTT tokens per workgroup, 8 waves.  Round r: wave w forms the exact int32 block sums of
// block 8 r + w for the whole tile on v_mfma_i32_16x16x64_i8 - weights straight from HBM into registers, activations in the order the quantiser leaves for it (PfQuantArgs::tiled: a fragment is
// 1 KiB of consecutive bytes) - T = hi plane, T = 256 T + 128 sum(W), then the lo plane on top (sum(W) from the same fragments against a constant
// plane), and leaves (float)T in LDS.  After one barrier every thread carries its four rows' fp32 chain over the round's eight blocks in order,
// acc = fma(bs, (float)isum, acc): rows_q8's order (kernels_x86.cpp:55-71), bit-identical to the tiled products.  The sums
// of two rounds have their own LDS, so a round costs one barrier.
// The weights of the next DA rounds and the activations of the next DB - 1 are in flight over the barriers; workgroups
// are persistent, and the stream of rounds runs through their row tiles without a gap.
// Token tiles of one row tile go to workgroups 8 apart - the same XCD - so their weights come from its L2.
// Measured (MI355X, weights from HBM, us; before: the 128-row tiles): 4096 x 14336 at 16 / 40 / 77 / 128 tokens
// 126 / 128 / 146 / 156 -> 20 / 32 / 37 / 42; 4096 x 4096 39 / 39 / 40 / 41 -> 8 / 11 / 14 / 16; 896 x 4864
// 44 / 45 / 47 / 47 -> 8 / 8 / 10 / 10.  At 16 tokens the weights alone take 17 of the 20 us (58.7 MB at ~5 TB/s and
// ~5 us from the launch to the first data); at more tokens the activations' L2 reads and the issue of ~250 instructions
// per wave and round bound it (without any loads 40 tokens take 20 of 37 us).
// Depth: 2 rounds of each; 4 of the weights, or of both, were slower (4096 x 14336, 16 tokens 20.2 / 21.0 / 21.9 us).
constexpr int kSkWaves = 8, kSkDepth = 2;
template <int RT, int NTT, int DA, int DB>
__global__ __launch_bounds__(kSkWaves * 64) void k_skinny_q8(GemmArgs a, int nrt, int ntk) {
  constexpr int RW = 16 * RT, NT = 16 * NTT, P = RW + 4;   // rows, tokens, floats between two tokens' rows in LDS
  extern __shared__ __align__(16) float sums[];            // [2 rounds][8 blocks][NT][P]
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  const int nb = a.cols / kQB, rounds = (nb + kSkWaves - 1) / kSkWaves;
  const bool paired = a.w2 != nullptr;   // rows 0-15 of the tile from the gate matrix, 16-31 the same rows of the up matrix
  // the workgroup's token tile tk and its row tiles rt0, rt0 + rts, ...
  const int rts = gridDim.x / ntk, rt0 = ((int)blockIdx.x >> 3) / ntk * 8 + (blockIdx.x & 7), tk = ((int)blockIdx.x >> 3) % ntk;
  const int mine = rt0 < nrt ? (nrt - rt0 + rts - 1) / rts : 0;
  if (!mine) return;

  struct Tile { const int8_t *w, *w2; const float *scale, *scale2, *bias; float *y; int rows, ldy, r0; };
  auto tile_of = [&](int rt) {
    Tile t{a.w, a.w2, a.scale, a.scale2, a.bias, a.y, a.rows, a.ldy, rt * (paired ? 16 : RW)};
    if (a.nseg > 1) {
      int base = 0;
      bool found = false;
#pragma unroll
      for (int s = 0; s < kGemmMaxSeg; s++)
        if (!found && s < a.nseg) {
          const GemmSeg &g = a.seg[s];
          const int n = (g.rows + RW - 1) / RW;
          if (rt < base + n || s == a.nseg - 1) {
            t = Tile{g.w, nullptr, g.scale, nullptr, g.bias, g.y, g.rows, g.ldy, (rt - base) * RW};
            found = true;
          }
          base += n;
        }
    }
    return t;
  };

  // the load streams.  Every step loads, past the last round the last one again (from the caches): a load under a
  // condition would make the compiler's waits assume it was not issued and drain the newer ones
  int atile = 0, around = 0, bround = 0, sround = 0;
  // weights: an instruction takes 8 rows x 128 bytes, whole lines.  Lane l of load h holds row 8 h + l % 8, 16-byte piece
  // l / 8; to_frag turns the two into the fragments of the block's two 64-deep steps: row l % 16, piece 2 (l / 16) + step
  const int8_t *wrow[RT][2];
  auto a_tile = [&]() {
    const Tile t = tile_of(rt0 + atile * rts);
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int h = 0; h < 2; h++)
        wrow[i][h] = (paired && i == 1 ? t.w2 : t.w) + 16 * (lane >> 3) +
                     (size_t)min(t.r0 + (paired ? 0 : 16 * i) + 8 * h + (lane & 7), t.rows - 1) * a.cols;
  };
  auto load_a = [&](v4i (&A)[RT][2]) {
    const int b = min(around * kSkWaves + wave, nb - 1);
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int h = 0; h < 2; h++) A[i][h] = *(const v4i *)(wrow[i][h] + (size_t)b * kQB);
    if (around + 1 < rounds) around++;
    else if (atile + 1 < mine) { around = 0; atile++; a_tile(); }
  };
  auto to_frag = [&](const v4i (&R)[2], v4i (&F)[2]) {
#pragma unroll
    for (int k = 0; k < 4; k++) {
      const int x = R[0][k], y = R[1][k];
      F[0][k] = __builtin_amdgcn_update_dpp(x, y, kDppRowRor8, 0xf, 0xc, false);   // lanes 8-15 of each row: load 1, lane - 8
      F[1][k] = __builtin_amdgcn_update_dpp(y, x, kDppRowRor8, 0xf, 0x3, false);   // lanes 0-7: load 0, lane + 8
    }
  };
  // activations: the same rounds for every row tile
  const int nt16 = (a.ntok + 15) / 16;
  uint32_t boff[NTT];   // the planes of a chunk of tokens stay below 4 GiB
#pragma unroll
  for (int n = 0; n < NTT; n++) boff[n] = (uint32_t)min(tk * NTT + n, nt16 - 1) * 16 * a.ldq + 16 * lane;
  auto load_b = [&](v4i (&H)[NTT][2], v4i (&L)[NTT][2]) {
    const size_t o = (size_t)min(bround * kSkWaves + wave, nb - 1) * 2048;
    const int8_t *hb = a.th + o, *lb = a.tl + o;
#pragma unroll
    for (int n = 0; n < NTT; n++)
#pragma unroll
      for (int ks = 0; ks < 2; ks++) {
        H[n][ks] = *(const v4i *)(hb + boff[n] + 1024 * ks);
        L[n][ks] = *(const v4i *)(lb + boff[n] + 1024 * ks);
      }
    bround = bround + 1 < rounds ? bround + 1 : 0;
  };

  // the chain's thread: token ct of the tile, rows 4 cq .. 4 cq + 3
  const bool chain = tid < NT * RW / 4;
  const int ct = tid / (RW / 4), cq = tid % (RW / 4), ctok = tk * NT + ct;
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  const float *bsp = a.xb + (size_t)min(ctok, a.ntok - 1) * a.ldb;
  auto load_s = [&](float4 &s0, float4 &s1) {   // ldb covers whole rounds
    s0 = *(const float4 *)(bsp + sround * kSkWaves); s1 = *(const float4 *)(bsp + sround * kSkWaves + 4);
    sround = sround + 1 < rounds ? sround + 1 : 0;
  };
  // the tile's row scales and its bias or residual values arrive under its rounds (loaded in the first one)
  Tile tl = tile_of(rt0);
  int ctile = 0, cround = 0;
  float4 sc4, ex4;
  auto load_c = [&]() {
    const int row = min(tl.r0 + (paired ? 4 * (cq & 3) : 4 * cq), tl.rows - 1), n4 = min(3, tl.rows - 1 - row);
    const float *sc = (paired && cq >= 4 ? tl.scale2 : tl.scale) + row;
    sc4 = make_float4(sc[0], sc[min(1, n4)], sc[min(2, n4)], sc[n4]);
    if (!paired && (a.resid || tl.bias)) {
      const float *ex = a.resid ? tl.y + (size_t)min(ctok, a.ntok - 1) * tl.ldy + row : tl.bias + row;
      ex4 = make_float4(ex[0], ex[min(1, n4)], ex[min(2, n4)], ex[n4]);
    }
  };

  v4i A[DA][RT][2], H[DB][NTT][2], L[DB][NTT][2];
  float4 bs[2][2];
  const v4i c64 = {0x40404040, 0x40404040, 0x40404040, 0x40404040};
  a_tile();
  load_s(bs[0][0], bs[0][1]);
#pragma unroll
  for (int i = 0; i < DA; i++) {   // in the order the steps issue them: activations of step i + DB - 1, weights of i + DA
    if (i < DB - 1) load_b(H[i], L[i]);
    load_a(A[i]);
  }

  auto step = [&](v4i (&A)[RT][2], v4i (&H)[NTT][2], v4i (&L)[NTT][2], v4i (&Hn)[NTT][2], v4i (&Ln)[NTT][2], int par) {
    const int b0 = cround * kSkWaves;
    if (cround == 0 && chain) load_c();
    load_s(bs[par ^ 1][0], bs[par ^ 1][1]);
    load_b(Hn, Ln);
    float *sb = sums + par * (kSkWaves * NT * P);
    if (b0 + wave < nb) {
      float *sw = sb + wave * (NT * P);
#pragma unroll
      for (int i = 0; i < RT; i++) {
        v4i F[2];
        to_frag(A[i], F);
        v4i S = {0, 0, 0, 0};   // 64 sum(W) of the lane's four rows
        S = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[0], c64, S, 0, 0, 0);
        S = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[1], c64, S, 0, 0, 0);
        S = S * 2;
#pragma unroll
        for (int n = 0; n < NTT; n++) {
          v4i T = {0, 0, 0, 0};
          T = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[0], H[n][0], T, 0, 0, 0);
          T = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[1], H[n][1], T, 0, 0, 0);
          T = T * 256 + S;
          T = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[0], L[n][0], T, 0, 0, 0);
          T = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[1], L[n][1], T, 0, 0, 0);
          const int t0 = T[0], t1 = T[1], t2 = T[2], t3 = T[3];
          *(float4 *)(sw + (16 * n + lr) * P + 16 * i + 4 * lg) = make_float4((float)t0, (float)t1, (float)t2, (float)t3);
        }
      }
    }
    load_a(A);
    lds_barrier();
    if (chain) {
      const float *sp = sb + ct * P + 4 * cq;
      const float4 w0 = bs[par][0], w1 = bs[par][1];
      const float wv[kSkWaves] = {w0.x, w0.y, w0.z, w0.w, w1.x, w1.y, w1.z, w1.w};
      auto fold = [&](float w, const float4 &s) {
        acc.x = __builtin_fmaf(w, s.x, acc.x); acc.y = __builtin_fmaf(w, s.y, acc.y);
        acc.z = __builtin_fmaf(w, s.z, acc.z); acc.w = __builtin_fmaf(w, s.w, acc.w);
      };
      if (b0 + kSkWaves <= nb) {
        float4 s[kSkWaves];
#pragma unroll
        for (int j = 0; j < kSkWaves; j++) s[j] = *(const float4 *)(sp + j * (NT * P));
#pragma unroll
        for (int j = 0; j < kSkWaves; j++) fold(wv[j], s[j]);
      } else {
#pragma unroll
        for (int j = 0; j < kSkWaves - 1; j++)
          if (b0 + j < nb) fold(wv[j], *(const float4 *)(sp + j * (NT * P)));
      }
    }
    if (++cround < rounds) return;
    cround = 0;
    if (chain) {
      float v[4] = {acc.x * sc4.x, acc.y * sc4.y, acc.z * sc4.z, acc.w * sc4.w};
      float *yt = tl.y + (size_t)ctok * tl.ldy;
      if (paired) {
        // gate rows in quads 0-3, the same rows of up in quads 4-7 of the token's eight lanes: a gate lane finishes its
        // first two rows, the up lane four lanes on the other two
        const float u0 = dpp_f<kDppRowShl4>(v[0]), u1 = dpp_f<kDppRowShl4>(v[1]);
        const float g2 = dpp_f<kDppRowShr4>(v[2]), g3 = dpp_f<kDppRowShr4>(v[3]);
        const bool lo = cq < 4;
        const int row = tl.r0 + 4 * (cq & 3) + (lo ? 0 : 2);
        const float h0 = sk_silu_mul(lo ? v[0] : g2, lo ? u0 : v[2]), h1 = sk_silu_mul(lo ? v[1] : g3, lo ? u1 : v[3]);
        if (ctok < a.ntok) {
          if (row < tl.rows) yt[row] = h0;
          if (row + 1 < tl.rows) yt[row + 1] = h1;
        }
      } else if (ctok < a.ntok) {
        const int row = tl.r0 + 4 * cq;
        if (a.resid || tl.bias) {   // rounded products, then added: no contraction
          asm volatile("" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]));
          v[0] += ex4.x; v[1] += ex4.y; v[2] += ex4.z; v[3] += ex4.w;
        }
        if (row + 3 < tl.rows && (tl.ldy & 3) == 0) *(float4 *)(yt + row) = make_float4(v[0], v[1], v[2], v[3]);
        else
#pragma unroll
          for (int i = 0; i < 4; i++) if (row + i < tl.rows) yt[row + i] = v[i];
      }
      acc = make_float4(0.f, 0.f, 0.f, 0.f);
    }
    if (++ctile < mine) tl = tile_of(rt0 + ctile * rts);
  };
  const int steps = mine * rounds;
  static_assert(DA % DB == 0 && DB % 2 == 0, "ring slots repeat every DA steps");
  for (int i = 0; i < steps; i += DA) {
#pragma unroll
    for (int k = 0; k < DA; k++)
      if (i + k < steps) step(A[k], H[k % DB], L[k % DB], H[(k + DB - 1) % DB], L[(k + DB - 1) % DB], k & 1);
  }
}

// row tiles one workgroup walks
static int sk_tiles_per_wg(int nrt, int ntk, int cus) {
  const int most = std::max(1, cus / (8 * ntk));
  return ((nrt + 7) / 8 + most - 1) / most;
}
static int sk_row_tiles(const GemmArgs &a, int rt) {
  const int rw = a.w2 ? 16 : 16 * rt;
  if (a.nseg < 2) return (a.rows + rw - 1) / rw;
  int n = 0;
  for (int s = 0; s < a.nseg; s++) n += (a.seg[s].rows + rw - 1) / rw;
  return n;
}
template <int RT, int NTT, int DA, int DB>
static hipError_t launch_skinny_t(const GemmArgs &a, int nrt, int cus, hipStream_t st) {
  const int nt16 = (a.ntok + 15) / 16, ntk = (nt16 + NTT - 1) / NTT;
  // 8 ntk g workgroups: per XCD g row tiles at a time by every token tile; one to a CU, with equal shares of the row tiles
  const int per = sk_tiles_per_wg(nrt, ntk, cus), g = ((nrt + 7) / 8 + per - 1) / per;
  const size_t lds = 2ull * kSkWaves * 16 * NTT * (16 * RT + 4) * 4;
  hipLaunchKernelGGL((k_skinny_q8<RT, NTT, DA, DB>), dim3((unsigned)(8 * ntk * g)), dim3(kSkWaves * 64), lds, st, a, nrt, ntk);
  return hipGetLastError();
}
// The tile shape and the time it is expected to take: a start of ~5 us, then per row tile of a workgroup its rounds and
// ~0.8 us for its end (round times from the shapes above and 14336 x 4096 pairs, with every CU busy)
double skinny_cost(const GemmArgs &a, int cus, int *rt, int *ntt) {
  static const double round_us[2][4] = {{1.05, 1.3, 1.9, 1.9}, {1.5, 1.9, 2.3, 2.6}};
  const int rounds = (a.cols / kQB + kSkWaves - 1) / kSkWaves, nt16 = (a.ntok + 15) / 16;
  double best = 1e30;
  for (int r = a.w2 ? 2 : 1; r <= 2; r++)
    for (int n = 1; n <= 4; n++) {
      const int ntk = (nt16 + n - 1) / n, per = sk_tiles_per_wg(sk_row_tiles(a, r), ntk, cus);
      const int waves = (8 * ntk + cus - 1) / cus;   // more token tiles than CUs / 8: several workgroups to a CU
      const double c = 5 + waves * per * (rounds * round_us[r - 1][n - 1] + 0.8);
      if (c < best) { best = c; *rt = r; *ntt = n; }
    }
  return best;
}
hipError_t launch_skinny(const GemmArgs &a, int rt, int ntt, int cus, hipStream_t st) {
  if (a.kind != MK_Q8 || a.ldb % 8 || a.ldb < round_up(a.cols / kQB, 8) || (a.w2 && rt != 2)) return hipErrorInvalidValue;
  const int nrt = sk_row_tiles(a, rt);
#define QPH_SK(R, N) if (rt == R && ntt == N) return launch_skinny_t<R, N, kSkDepth, kSkDepth>(a, nrt, cus, st);
  QPH_SK(1, 1) QPH_SK(1, 2) QPH_SK(1, 3) QPH_SK(1, 4) QPH_SK(2, 1) QPH_SK(2, 2) QPH_SK(2, 3) QPH_SK(2, 4)
#undef QPH_SK
  return hipErrorInvalidValue;
}

}  // namespace qph
