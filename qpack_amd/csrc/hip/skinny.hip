// gfx950 prompt products for few tokens (and for matrices too small to fill the chip with large tiles).
//
// The tiled products of prefill.hip give a workgroup 128 or 256 weight rows and walk K block by block: with 4096 rows
// that is 32 workgroups on 256 CUs, and a 14336-column product takes the 112 blocks' latency whatever the token count.
// Here a workgroup owns 16 or 32 weight rows and its eight waves share K: in one round wave w multiplies block 8 r + w,
// so every matrix has rows / 16 workgroups and the weights of a round, 1 KiB of every row, are in flight at once.
#include <math.h>
#include <stdlib.h>

#include <algorithm>
#include <type_traits>

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
// block 8 r + w for the whole tile on v_mfma_i32_16x16x64_i8 - weights straight from HBM into registers, activations in the order the quantiser leaves for it (PfQuantArgs::th: a fragment is
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
// ORD: the fp32 order of a row's block sums.  0: one chain; 1: the decode matvec's split chain - shares of the blocks
// chained each from zero, then summed pairwise; the share sums wait in LDS; 2: k_attn_wo's - a chain per kv group times the
// row scale, the groups summed in order.  1 and 2 give a token's row the bits its decode step gives it.
template <int RT, int NTT, int DA, int DB, int ORD>
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
  float *shares = sums + 2 * kSkWaves * NT * P + tid;   // ORD 1: [4 rows][8 shares][chain threads]
  constexpr int CT = NT * RW / 4;
  int share_len[4], left[4], nshare[4];                      // ORD 1: blocks per share, left in it, shares stored
  float4 ysum = make_float4(0.f, 0.f, 0.f, 0.f);             // ORD 2
  int gleft = a.group_blocks;
  auto load_c = [&]() {
    if constexpr (ORD == 1) {
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const int r = tl.r0 + (paired ? 4 * (cq & 3) : 4 * cq) + i, gw = (paired ? r : r / a.deal.ns) % a.deal.waves;
        const int n = (a.deal.units - gw + a.deal.waves - 1) / a.deal.waves * a.deal.ns;   // rows of the wave that has this one
        const int lanes = n <= 8 ? 8 : n <= 16 ? 4 : n <= 32 ? 2 : 1;
        share_len[i] = left[i] = (nb + 4 * lanes - 1) / (4 * lanes) * 4; nshare[i] = 0;
      }
    }
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
      auto fold = [&](int j, const float4 &s) {
        acc.x = __builtin_fmaf(wv[j], s.x, acc.x); acc.y = __builtin_fmaf(wv[j], s.y, acc.y);
        acc.z = __builtin_fmaf(wv[j], s.z, acc.z); acc.w = __builtin_fmaf(wv[j], s.w, acc.w);
        if constexpr (ORD == 1) {
          if ((j & 3) == 3 || b0 + j == nb - 1) {   // shares are whole multiples of four blocks, the last may end early
            float *ap[4] = {&acc.x, &acc.y, &acc.z, &acc.w};
#pragma unroll
            for (int i = 0; i < 4; i++) {
              left[i] -= 4;
              if (left[i] == 0 || b0 + j == nb - 1) { shares[(8 * i + nshare[i]++) * CT] = *ap[i]; *ap[i] = 0.f; left[i] = share_len[i]; }
            }
          }
        }
        if constexpr (ORD == 2) {
          if (--gleft == 0) {
            float4 p = make_float4(acc.x * sc4.x, acc.y * sc4.y, acc.z * sc4.z, acc.w * sc4.w);
            asm volatile("" : "+v"(p.x), "+v"(p.y), "+v"(p.z), "+v"(p.w));   // rounded parts, then added
            ysum.x += p.x; ysum.y += p.y; ysum.z += p.z; ysum.w += p.w;
            acc = make_float4(0.f, 0.f, 0.f, 0.f); gleft = a.group_blocks;
          }
        }
      };
      if (b0 + kSkWaves <= nb) {
        float4 s[kSkWaves];
#pragma unroll
        for (int j = 0; j < kSkWaves; j++) s[j] = *(const float4 *)(sp + j * (NT * P));
#pragma unroll
        for (int j = 0; j < kSkWaves; j++) fold(j, s[j]);
      } else {
#pragma unroll
        for (int j = 0; j < kSkWaves - 1; j++)
          if (b0 + j < nb) fold(j, *(const float4 *)(sp + j * (NT * P)));
      }
    }
    if (++cround < rounds) return;
    cround = 0;
    if (chain) {
      if constexpr (ORD == 1) {   // ((c0 + c1) + (c2 + c3)) + ((c4 + c5) + (c6 + c7)), absent shares zero
        float *ap[4] = {&acc.x, &acc.y, &acc.z, &acc.w};
#pragma unroll
        for (int i = 0; i < 4; i++) {
          float c[8];
#pragma unroll
          for (int k = 0; k < 8; k++) c[k] = k < nshare[i] ? shares[(8 * i + k) * CT] : 0.f;
          *ap[i] = ((c[0] + c[1]) + (c[2] + c[3])) + ((c[4] + c[5]) + (c[6] + c[7]));
        }
      }
      float v[4] = {acc.x * sc4.x, acc.y * sc4.y, acc.z * sc4.z, acc.w * sc4.w};
      if constexpr (ORD == 2) { v[0] = ysum.x; v[1] = ysum.y; v[2] = ysum.z; v[3] = ysum.w; ysum = make_float4(0.f, 0.f, 0.f, 0.f); }
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
template <int RT, int NTT, int ORD>
static hipError_t launch_skinny_t(const GemmArgs &a, int nrt, int cus, hipStream_t st) {
  const int nt16 = (a.ntok + 15) / 16, ntk = (nt16 + NTT - 1) / NTT;
  // 8 ntk g workgroups: per XCD g row tiles at a time by every token tile; one to a CU, with equal shares of the row tiles
  const int per = sk_tiles_per_wg(nrt, ntk, cus), g = ((nrt + 7) / 8 + per - 1) / per;
  const size_t lds = 2ull * kSkWaves * 16 * NTT * (16 * RT + 4) * 4 + (ORD == 1 ? 16 * NTT * 16 * RT * 8 * 4 : 0);
  hipLaunchKernelGGL((k_skinny_q8<RT, NTT, kSkDepth, kSkDepth, ORD>), dim3((unsigned)(8 * ntk * g)), dim3(kSkWaves * 64), lds, st, a, nrt, ntk);
  return hipGetLastError();
}
// The tile shape and the time it is expected to take: a start of ~5 us, then per row tile of a workgroup its rounds and
// ~0.8 us for its end (round times from the shapes above and 14336 x 4096 pairs, with every CU busy).  Every XCD reads the
// tokens' planes once per row tile: beyond its 4 MiB of L2 they come from the shared cache, all XCDs together at ~7 TB/s,
// and a row tile takes no less than that (896 x 4864 at 1152 / 1536 / 2048 tokens, expected by the rounds alone 54 / 54 / 60
// us: 57 / 72 / 97, with this 59 / 76 / 99; 4096 x 14336 at 2048 600: 1057, with this 1089)
double skinny_cost(const GemmArgs &a, int cus, int *rt, int *ntt) {
  static const double round_us[2][4] = {{1.05, 1.3, 1.9, 1.9}, {1.5, 1.9, 2.3, 2.6}};
  const int rounds = (a.cols / kQB + kSkWaves - 1) / kSkWaves, nt16 = (a.ntok + 15) / 16;
  const double planes = 32.0 * nt16 * a.cols, planes_us = planes > 4e6 ? planes * 8 / 7e6 : 0;
  double best = 1e30;
  for (int r = a.w2 ? 2 : 1; r <= 2; r++)
    for (int n = 1; n <= 4; n++) {
      const int ntk = (nt16 + n - 1) / n, per = sk_tiles_per_wg(sk_row_tiles(a, r), ntk, cus);
      const int waves = (8 * ntk + cus - 1) / cus;   // more token tiles than CUs / 8: several workgroups to a CU
      const double c = 5 + per * (std::max(waves * rounds * round_us[r - 1][n - 1], planes_us) + waves * 0.8);
      if (c < best) { best = c; *rt = r; *ntt = n; }
    }
  return best;
}
hipError_t launch_skinny(const GemmArgs &a, int rt, int ntt, int cus, hipStream_t st) {
  if (a.kind != MK_Q8 || a.ldb % 8 || a.ldb < round_up(a.cols / kQB, 8) || (a.w2 && rt != 2) ||
      (size_t)round_up(a.ntok, 16) * a.ldq >> 32)   // the kernel's offsets into a plane are 32 bits
    return hipErrorInvalidValue;
  const int nrt = sk_row_tiles(a, rt);
  if (a.deal.waves > 0 || a.group_blocks > 0) {   // the decode step's orders: one tile of at most 16 tokens
    if (a.ntok > 16 || a.nseg > 1 || (a.deal.waves > 0 && (a.group_blocks > 0 || a.deal.ns < 1)) || (a.group_blocks > 0 && a.w2))
      return hipErrorInvalidValue;
    if (a.group_blocks > 0) return rt == 1 ? launch_skinny_t<1, 1, 2>(a, nrt, cus, st) : launch_skinny_t<2, 1, 2>(a, sk_row_tiles(a, 2), cus, st);
    return rt == 1 ? launch_skinny_t<1, 1, 1>(a, nrt, cus, st) : launch_skinny_t<2, 1, 1>(a, sk_row_tiles(a, 2), cus, st);
  }
#define QPH_SK(R, N) if (rt == R && ntt == N) return launch_skinny_t<R, N, 0>(a, nrt, cus, st);
  QPH_SK(1, 1) QPH_SK(1, 2) QPH_SK(1, 3) QPH_SK(1, 4) QPH_SK(2, 1) QPH_SK(2, 2) QPH_SK(2, 3) QPH_SK(2, 4)
#undef QPH_SK
  return hipErrorInvalidValue;
}

// ------------------------------------------------------------------ q4 and q1 weights
// q4 on the f16 matrix cores: a group (32 columns) is a dot product of 4-bit integers with 16-bit ones, at most 8 x 32 x
// 32767 < 2^23 in size, so v_mfma_f32_16x16x32_f16 gives it exactly, as a float: the weights n = nibble - 8 are exact
// halves, the activation goes in as two halves q = hi + lo (hi = 256 (q >> 8), lo = q & 255), every product and partial sum
// is an integer below 2^24.  What is left for the vector ALU is one fma per output and group, with the group's fp16 scale;
// on the int8 cores it is a shift-add, a conversion and an fma, and the offset corrections.
//   blk = sum over the block's groups of scale * sum, acc = fma(bs[token][block], blk, acc)
// q1 on the int8 matrix cores, which do twice the columns in the time: a group is a whole block (128 columns, two steps),
// so the integer work after it is a fourth of q4's.  A bit becomes the byte +-64 (0x40 or 0xc0: a shift, a mask and an
// or for four; a set bit, weight +1, is -64); with T = 32 sum(W) + the hi plane, 256 T + the plane lo - 128 = 64 times the
// group's sum, exact in int32 and as a float (the sum is below 2^22), and -1 / 64 goes into the scale.  64 sum(W) is one more
// product, with a constant plane.
// Tile: 16 RT rows x 16 NTT tokens per workgroup; its 8 waves take every eighth block each, add no barrier until the tile's
// end, and their fp32 partials are summed there through LDS, 32 tokens at a time: pairwise, so that the error is below one
// chain's at every block count above 8 (in rounding variances of one block's size, 9 blocks: chain 45, in wave order 52,
// pairwise 37; 38: 741, 282, 224).  Up to 8 blocks a wave has one at most and any such sum would round each block once more than
// the chain acc = fma(bs, blk, acc) does; the waves then leave blk itself and the chain runs at the end.
// Operands: weights from HBM to registers as stored.  q4: lane l loads the 16 bytes of group l / 16 of row l % 16; a 4 x 4
// transpose of dwords over the four 16-lane rows (permlane swaps) gives every lane dword l / 16 of each group, and a dword
// becomes four half pairs with a mask, 0x6400 (1024 + nibble) and one packed subtraction.  q1: dword l / 16 of the block.
// Activations in the order these fragments have (PfQuantArgs::fp: 1 KiB of consecutive bytes each), straight from L2 to
// registers, one block ahead (q4 with 64 rows by 48 tokens, or 32 by 64, spills: 2 to 4 times slower).  The rows' scales of
// a block (one load) are handed to the lanes through LDS, the tokens' block scales stay in LDS from the start.
// Measured (MI355X, weights from HBM, us; before: 128 x 128 tiles on the int8 cores): q4 3584 x 18944 at 150 tokens 780 ->
// 99, 18944 x 3584 255 -> 71, 896 x 4864 at 512 tokens 164 -> 20.  37888 x 3584 at 512 tokens take 244 us: with the two
// planes 1.14 POP/s, what a large bf16 matrix product reaches here (1.12 PFLOP/s).  Without any loads 150 tokens of 18944 x
// 3584 take 9 % less, without the unpacking and the scaling 5 %, with one plane 15 %: no single resource is left to relieve.
// q1 at 300 tokens (before: on the f16 cores like q4) 28672 x 4096 200 -> 119, 4096 x 14336 116 -> 72.
typedef _Float16 h2v __attribute__((ext_vector_type(2)));
typedef _Float16 h4v __attribute__((ext_vector_type(4)));
typedef _Float16 h8v __attribute__((ext_vector_type(8)));
typedef float f4v __attribute__((ext_vector_type(4)));

// lane l of dword j: group l / 16's dword j -> dword l / 16 of group j
__device__ __forceinline__ void transpose4(uint32_t &a, uint32_t &b, uint32_t &c, uint32_t &d) {
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3\n\ts_nop 1\n\t"
               "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1"
               : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
}
// halves (b0.lo, b2.lo, b0.hi, b2.hi, b1.lo, b3.lo, b1.hi, b3.hi) of the dword's four bytes, each nibble - 8.  A nibble in
// mantissa bits 0-3 under the exponent of 1024 is 1024 + n, in bits 4-7 under that of 64 it is 64 + n: exact halves, so is
// the difference.  c1 / c2 (0x64006400 / 0x54005400) come in registers: v_and_or_b32 takes one constant besides
__device__ __forceinline__ h8v q4_half8(uint32_t w, uint32_t c1, uint32_t c2) {
  const uint32_t v = w >> 8;
  const h2v o1 = {(_Float16)1032, (_Float16)1032}, o2 = {(_Float16)72, (_Float16)72};
  auto bits = [](h2v x) { return __builtin_bit_cast(uint32_t, x); };
  const uint32_t p0 = bits(__builtin_bit_cast(h2v, (w & 0x000f000fu) | c1) - o1);
  const uint32_t p1 = bits(__builtin_bit_cast(h2v, (w & 0x00f000f0u) | c2) - o2);
  const uint32_t p2 = bits(__builtin_bit_cast(h2v, (v & 0x000f000fu) | c1) - o1);
  const uint32_t p3 = bits(__builtin_bit_cast(h2v, (v & 0x00f000f0u) | c2) - o2);
  return __builtin_bit_cast(h8v, make_uint4(p0, p1, p2, p3));
}
// step s of a q1 dword: bytes (bits 4 s + j of its four bytes), j = 0..3, as -64 (set) or +64: they differ in the sign bit only
__device__ __forceinline__ v4i q1_bytes16(uint32_t w, int s, uint32_t c) {
  uint32_t p[4];
#pragma unroll
  for (int j = 0; j < 4; j++) p[j] = ((w << (7 - 4 * s - j)) & 0x80808080u) | c;
  return __builtin_bit_cast(v4i, make_uint4(p[0], p[1], p[2], p[3]));
}

template <int KIND, int RT, int NTT, bool ORD>
__global__ __launch_bounds__(kSkWaves * 64) void k_lowbit(GemmArgs a, int nrt, int ntk, int tg, int rg) {
  constexpr bool Q4 = KIND == MK_Q4;
  constexpr int RW = 16 * RT, NT = 16 * NTT, P = RW + 4, SB = Q4 ? 8 : 2;   // SB: scale bytes per row and block
  constexpr int NS = Q4 ? 4 : 2, BB = NS * 2048;                            // MFMA steps and activation bytes per block
  typedef typename std::conditional<Q4, h8v, v4i>::type frag_t;
  extern __shared__ __align__(16) char hsm[];
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6), lr = lane & 15, lg = lane >> 4;
  const int nb = a.cols / kQB;
  constexpr int RN = NTT < 2 ? NTT : 2, RT16 = 16 * RN;       // token tiles whose partials are summed at a time
  float *red = (float *)hsm;                                  // [8 waves][16 RN][P] partials
  char *scl = hsm + (size_t)kSkWaves * RT16 * P * 4 + wave * (RW * SB);   // this wave's block scales [RW][SB]
  float *bsl = (float *)(hsm + (size_t)kSkWaves * (RT16 * P * 4 + RW * SB));   // [nb][NT]
  const bool paired = a.w2 != nullptr;   // the tile's first RW / 2 rows from the gate matrix, the others the same rows of up
  // token tile tk and row tiles rt0, rt0 + rts, ...: the XCD's workgroups are dealt in sets of tg token tiles x rg row tiles
  const int q = (int)blockIdx.x >> 3, in_set = q % (tg * rg);
  const int rts = 8 * rg, rt0 = in_set / tg * 8 + (blockIdx.x & 7), tk = q / (tg * rg) * tg + in_set % tg;
  const int mine = rt0 < nrt && tk < ntk ? (nrt - rt0 + rts - 1) / rts : 0;
  if (!mine) return;
  const int rowb = Q4 ? a.cols / 2 : a.cols / 8, blkb = Q4 ? 64 : 16;   // bytes per row, per row and block

  struct Tile { const uint8_t *w, *w2; const uint16_t *st, *st2; const float *bias; float *y; int rows, ldy, r0; };
  auto tile_of = [&](int rt) {
    Tile t{(const uint8_t *)a.w, (const uint8_t *)a.w2, a.st, a.st2, a.bias, a.y, a.rows, a.ldy, rt * (paired ? RW / 2 : RW)};
    if (a.nseg > 1) {
      int base = 0;
      bool found = false;
#pragma unroll
      for (int s = 0; s < kGemmMaxSeg; s++)
        if (!found && s < a.nseg) {
          const GemmSeg &g = a.seg[s];
          const int n = (g.rows + RW - 1) / RW;
          if (rt < base + n || s == a.nseg - 1) {
            t = Tile{(const uint8_t *)g.w, nullptr, g.st, nullptr, g.bias, g.y, g.rows, g.ldy, (rt - base) * RW};
            found = true;
          }
          base += n;
        }
    }
    return t;
  };

  // the tokens' block scales
  for (int i = tid; i < nb * NT; i += kSkWaves * 64) {
    const int b = i / NT, t = tk * NT + i % NT;
    bsl[i] = a.xb[(size_t)min(t, a.ntok - 1) * a.ldb + b];
  }

  // this wave's stream: blocks wave, wave + 8, ... of each of its row tiles
  const int nj = wave < nb ? (nb - wave + kSkWaves - 1) / kSkWaves : 0;
  int ltile = 0, lj = 0;   // the next weights to load
  const uint8_t *wrow[RT];
  const char *srow;
  size_t sstep = 0;
  auto w_tile = [&]() {
    const Tile t = tile_of(rt0 + ltile * rts);
#pragma unroll
    for (int i = 0; i < RT; i++) {
      const bool up = paired && i >= RT / 2;
      const int row = min(t.r0 + 16 * (up ? i - RT / 2 : i) + lr, t.rows - 1);
      wrow[i] = (up ? t.w2 : t.w) + (size_t)row * rowb + (Q4 ? 16 : 4) * lg;
    }
    const int l = lane & (RW - 1);
    const bool up = paired && l >= RW / 2;
    srow = (const char *)(up ? t.st2 : t.st) + (size_t)min(t.r0 + (up ? l - RW / 2 : l), t.rows - 1) * SB;
    sstep = (size_t)t.rows * SB;
  };
  typedef typename std::conditional<Q4, uint4, uint32_t>::type raw_t;
  typedef typename std::conditional<Q4, uint2, uint16_t>::type scr_t;
  auto load_w = [&](raw_t (&A)[RT], scr_t &S) {
    const int b = min(wave + kSkWaves * lj, nb - 1);
#pragma unroll
    for (int i = 0; i < RT; i++) A[i] = *(const raw_t *)(wrow[i] + (size_t)b * blkb);
    S = *(const scr_t *)(srow + (size_t)b * sstep);
    if (lj + 1 < nj) lj++;
    else if (ltile + 1 < mine) { lj = 0; ltile++; w_tile(); }
  };
  const int nt16 = (a.ntok + 15) / 16;
  const char *fb[NTT];
#pragma unroll
  for (int n = 0; n < NTT; n++) fb[n] = (const char *)a.fp + (size_t)min(tk * NTT + n, nt16 - 1) * nb * BB + 16 * lane;
  int bj = 0;
  frag_t B[NS][NTT][2];
  auto load_b = [&](int s, int n) {
    const char *p = fb[n] + (size_t)min(wave + kSkWaves * bj, nb - 1) * BB + 2048 * s;
#pragma unroll
    for (int pl = 0; pl < 2; pl++) B[s][n][pl] = *(const frag_t *)(p + 1024 * pl);
  };

  f4v acc[RT][NTT];
  auto zero = [&]() {
#pragma unroll
    for (int i = 0; i < RT; i++)
#pragma unroll
      for (int n = 0; n < NTT; n++) acc[i][n] = (f4v){0.f, 0.f, 0.f, 0.f};
  };
  zero();
  raw_t A[RT];
  scr_t S;
  uint32_t c1 = Q4 ? 0x64006400u : 0x40404040u, c2 = 0x54005400u;
  asm volatile("" : "+v"(c1), "+v"(c2));
  w_tile();
  load_w(A, S);
#pragma unroll
  for (int s = 0; s < NS; s++)
#pragma unroll
    for (int n = 0; n < NTT; n++) load_b(s, n);
  bj = nj > 1 ? 1 : 0;
  __syncthreads();   // the block scales

  auto block = [&](int b) {
    // this block's row scales to the lanes that hold the rows (LDS operations of a wave complete in order)
    if (RW == 64 || lane < RW) *(scr_t *)(scl + (lane & (RW - 1)) * SB) = S;
    uint32_t q[RT][4];
#pragma unroll
    for (int i = 0; i < RT; i++) {
      if constexpr (Q4) {
        q[i][0] = A[i].x; q[i][1] = A[i].y; q[i][2] = A[i].z; q[i][3] = A[i].w;
        transpose4(q[i][0], q[i][1], q[i][2], q[i][3]);
      } else {
        q[i][0] = A[i];
      }
    }
    load_w(A, S);   // the next block's
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
    h4v sc[RT][4];   // q4: row i's four groups; q1: [0] the four rows
#pragma unroll
    for (int i = 0; i < RT; i++) {
      if (Q4) {
#pragma unroll
        for (int k = 0; k < 2; k++) {
          const h8v v = *(const h8v *)(scl + (16 * i + 4 * lg + 2 * k) * SB);
          sc[i][2 * k] = __builtin_shufflevector(v, v, 0, 1, 2, 3);
          sc[i][2 * k + 1] = __builtin_shufflevector(v, v, 4, 5, 6, 7);
        }
      } else {
        sc[i][0] = *(const h4v *)(scl + (16 * i + 4 * lg) * SB);
      }
    }
    float bs[NTT];
#pragma unroll
    for (int n = 0; n < NTT; n++) bs[n] = bsl[b * NT + 16 * n + lr];
    if constexpr (Q4) {
      f4v blk[RT][NTT];
#pragma unroll
      for (int s = 0; s < 4; s++) {
        h8v F[RT];
#pragma unroll
        for (int i = 0; i < RT; i++) F[i] = q4_half8(q[i][s], c1, c2);
#pragma unroll
        for (int n = 0; n < NTT; n++)
#pragma unroll
          for (int i = 0; i < RT; i++) {
            f4v T = (f4v){0.f, 0.f, 0.f, 0.f};
            T = __builtin_amdgcn_mfma_f32_16x16x32_f16(F[i], B[s][n][0], T, 0, 0, 0);
            T = __builtin_amdgcn_mfma_f32_16x16x32_f16(F[i], B[s][n][1], T, 0, 0, 0);
#pragma unroll
            for (int r = 0; r < 4; r++) {
              const float w = (float)sc[i][r][s];
              blk[i][n][r] = s == 0 ? w * T[r] : __builtin_fmaf(w, T[r], blk[i][n][r]);
            }
          }
#pragma unroll
        for (int n = 0; n < NTT; n++) load_b(s, n);
      }
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int n = 0; n < NTT; n++)
#pragma unroll
          for (int r = 0; r < 4; r++) acc[i][n][r] = ORD ? blk[i][n][r] : __builtin_fmaf(bs[n], blk[i][n][r], acc[i][n][r]);
    } else {
      v4i F[2][RT], R[RT];
      const v4i ones = (v4i){0x01010101, 0x01010101, 0x01010101, 0x01010101};
#pragma unroll
      for (int i = 0; i < RT; i++) {
        R[i] = (v4i){0, 0, 0, 0};
#pragma unroll
        for (int s = 0; s < 2; s++) {
          F[s][i] = q1_bytes16(q[i][0], s, c1);
          R[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[s][i], ones, R[i], 0, 0, 0);
        }
      }
      float w[RT][4];
#pragma unroll
      for (int i = 0; i < RT; i++)
#pragma unroll
        for (int r = 0; r < 4; r++) { R[i][r] >>= 1; w[i][r] = -0.015625f * (float)sc[i][0][r]; }
#pragma unroll
      for (int n = 0; n < NTT; n++) {
        v4i T[RT];
#pragma unroll
        for (int i = 0; i < RT; i++) {
          T[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[0][i], B[0][n][0], R[i], 0, 0, 0);
          T[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[1][i], B[1][n][0], T[i], 0, 0, 0);
        }
#pragma unroll
        for (int i = 0; i < RT; i++) {
#pragma unroll
          for (int r = 0; r < 4; r++) T[i][r] = (int)((uint32_t)T[i][r] << 8);
          T[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[0][i], B[0][n][1], T[i], 0, 0, 0);
          T[i] = __builtin_amdgcn_mfma_i32_16x16x64_i8(F[1][i], B[1][n][1], T[i], 0, 0, 0);
        }
#pragma unroll
        for (int s = 0; s < 2; s++) load_b(s, n);
#pragma unroll
        for (int i = 0; i < RT; i++)
#pragma unroll
          for (int r = 0; r < 4; r++) {
            const float blk = w[i][r] * (float)T[i][r];
            acc[i][n][r] = ORD ? blk : __builtin_fmaf(bs[n], blk, acc[i][n][r]);
          }
      }
    }
    bj = bj + 1 < nj ? bj + 1 : 0;
  };

  for (int tile = 0; tile < mine; tile++) {
    for (int j = 0; j < nj; j++) block(wave + kSkWaves * j);
    const Tile t = tile_of(rt0 + tile * rts);
#pragma unroll
    for (int n0 = 0; n0 < NTT; n0 += RN) {
#pragma unroll
      for (int n = n0; n < n0 + RN && n < NTT; n++)
#pragma unroll
        for (int i = 0; i < RT; i++)
          *(f4v *)(red + (wave * RT16 + 16 * (n - n0) + lr) * P + 16 * i + 4 * lg) = acc[i][n];
      lds_barrier();
      auto part = [&](int w, int tok, int row) { return *(const f4v *)(red + (w * RT16 + tok) * P + row); };
      auto sum = [&](int tok, int row) {
        if constexpr (ORD) {   // no loop up to nb: its reads would wait for one another (pairs of 4864 x 896, 1024 tokens: 83 us, this 77)
          f4v v = (f4v){0.f, 0.f, 0.f, 0.f}, p[kSkWaves];   // a wave without a block left zeros
          float bs[kSkWaves];
#pragma unroll
          for (int w = 0; w < kSkWaves; w++) {
            p[w] = part(w, tok, row);
            const float b = bsl[min(w, nb - 1) * NT + 16 * n0 + tok];
            bs[w] = w < nb ? b : 0.f;
          }
#pragma unroll
          for (int w = 0; w < kSkWaves; w++)
#pragma unroll
            for (int r = 0; r < 4; r++) v[r] = __builtin_fmaf(bs[w], p[w][r], v[r]);
          return v;
        } else {
          return ((part(0, tok, row) + part(1, tok, row)) + (part(2, tok, row) + part(3, tok, row))) +
                 ((part(4, tok, row) + part(5, tok, row)) + (part(6, tok, row) + part(7, tok, row)));
        }
      };
      const int quads = paired ? RW / 8 : RW / 4, ntoks = NTT - n0 < RN ? 16 * (NTT - n0) : RT16;
      for (int e = tid; e < ntoks * quads; e += kSkWaves * 64) {
        const int tok = e / quads, cq = e % quads, gt = tk * NT + 16 * n0 + tok, row = t.r0 + 4 * cq;
        if (gt >= a.ntok) continue;
        f4v v = sum(tok, 4 * cq);
        float *yt = t.y + (size_t)gt * t.ldy;
        if (paired) {
          const f4v u = sum(tok, RW / 2 + 4 * cq);
#pragma unroll
          for (int r = 0; r < 4; r++) v[r] = sk_silu_mul(v[r], u[r]);
        }
        if (row + 3 < t.rows && (t.ldy & 3) == 0) {
          if (a.resid) v += *(const f4v *)(yt + row);
          else if (t.bias) v += *(const f4v *)(t.bias + row);
          *(f4v *)(yt + row) = v;
        } else {
#pragma unroll
          for (int r = 0; r < 4; r++)
            if (row + r < t.rows) yt[row + r] = a.resid ? yt[row + r] + v[r] : t.bias ? v[r] + t.bias[row + r] : v[r];
        }
      }
      lds_barrier();
    }
    zero();
  }
}

// scales of a q4 / q1 matrix [rows][G] -> block-major: out[block][row][4] (q4) or out[block][row] (q1)
__global__ __launch_bounds__(256) void k_scale_blocks(const uint16_t *sc, int rows, int G, int per, uint16_t *out) {
  const int64_t i = (int64_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (int64_t)rows * G) return;
  const int r = (int)(i / G), g = (int)(i % G);
  out[((size_t)(g / per) * rows + r) * per + g % per] = sc[i];
}
hipError_t launch_scale_blocks(int kind, const uint16_t *sc, int rows, int cols, uint16_t *out, hipStream_t st) {
  if (cols % kQB || rows <= 0 || (kind != MK_Q4 && kind != MK_Q1)) return hipErrorInvalidValue;
  const int per = kind == MK_Q4 ? 4 : 1, G = cols / kQB * per;
  const int64_t n = (int64_t)rows * G;
  hipLaunchKernelGGL(k_scale_blocks, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, sc, rows, G, per, out);
  return hipGetLastError();
}

// token tiles in sets of tg: the workgroups on the chip at a time share a set's activations, which then stay in the XCDs'
// L2 while the weights stream past (18944 x 3584, 2048 tokens: one set of 64 tiles 1194 us, sets of 16 / 8 / 4 / 2
// 919 / 865 / 861 / 910; up to 16 tiles one set is as fast)
static void lowbit_sets(int ntk, int *sets, int *tg) {
  const int cap = ntk <= 16 ? 16 : 8;
  *sets = (ntk + cap - 1) / cap; *tg = (ntk + *sets - 1) / *sets;
}
static size_t lowbit_lds(int kind, int rt, int ntt, int nb) {
  return (size_t)kSkWaves * (16 * std::min(ntt, 2) * (16 * rt + 4) * 4 + 16 * rt * (kind == MK_Q4 ? 8 : 2)) + (size_t)nb * 16 * ntt * 4;
}
static int lowbit_row_tiles(const GemmArgs &a, int rt) {
  const int rw = a.w2 ? 8 * rt : 16 * rt;
  if (a.nseg < 2) return (a.rows + rw - 1) / rw;
  int n = 0;
  for (int s = 0; s < a.nseg; s++) n += (a.seg[s].rows + rw - 1) / rw;
  return n;
}
template <int KIND, int RT, int NTT, bool ORD>
static hipError_t launch_lowbit_o(const GemmArgs &a, int cus, hipStream_t st) {
  const int nrt = lowbit_row_tiles(a, RT), nt16 = (a.ntok + 15) / 16, ntk = (nt16 + NTT - 1) / NTT;
  int sets, tg;
  lowbit_sets(ntk, &sets, &tg);
  const int per = sk_tiles_per_wg(nrt, tg, cus), rg = ((nrt + 7) / 8 + per - 1) / per;
  const size_t lds = lowbit_lds(KIND, RT, NTT, a.cols / kQB);
  if (lds > 160 * 1024) return hipErrorInvalidValue;
  hipLaunchKernelGGL((k_lowbit<KIND, RT, NTT, ORD>), dim3((unsigned)(8 * sets * tg * rg)), dim3(kSkWaves * 64), lds, st, a, nrt, ntk, tg, rg);
  return hipGetLastError();
}
template <int KIND, int RT, int NTT>
static hipError_t launch_lowbit_t(const GemmArgs &a, int cus, hipStream_t st) {
  return a.cols / kQB <= kSkWaves ? launch_lowbit_o<KIND, RT, NTT, true>(a, cus, st) : launch_lowbit_o<KIND, RT, NTT, false>(a, cus, st);
}
// The tile shape for a launch: a start of ~5 us, then per row tile of a workgroup every wave's blocks and ~1 us for each
// pass of its end (block times with every CU busy, fitted to the shapes above, within 10 % of what they take).  32-row
// tiles where 64-row ones leave CUs idle; 64 tokens for q1 where there are enough tiles (28672 x 4096 at 512 tokens: 32
// tokens a tile 219 us, 64 178; 4096 x 14336 at 50 tokens: 64 x 64 37 us, 32 x 32 20.5).
static void lowbit_tile(const GemmArgs &a, int cus, int *rt, int *ntt) {
  static const int shape[5][2] = {{2, 1}, {2, 2}, {4, 1}, {4, 2}, {4, 4}};
  static const double block_us[2][5] = {{1.55, 2.0, 2.1, 2.45, 0}, {0.65, 1.1, 1.1, 1.63, 2.6}};   // q4, q1
  const bool q1 = a.kind == MK_Q1;
  const int rounds = (a.cols / kQB + kSkWaves - 1) / kSkWaves, nt16 = (a.ntok + 15) / 16;
  double best = 1e30;
  for (int i = 0; i < (q1 ? 5 : 4); i++) {
    const int ntk = (nt16 + shape[i][1] - 1) / shape[i][1];
    int sets, tg;
    lowbit_sets(ntk, &sets, &tg);
    const double c = sets * sk_tiles_per_wg(lowbit_row_tiles(a, shape[i][0]), tg, cus) * (rounds * block_us[q1][i] + (shape[i][1] + 1) / 2);
    if (c < best) { best = c; *rt = shape[i][0]; *ntt = shape[i][1]; }
  }
}
hipError_t launch_lowbit(const GemmArgs &a, int cus, hipStream_t st) {
  if ((a.kind != MK_Q4 && a.kind != MK_Q1) || !a.fp || a.ldb < a.cols / kQB || (a.w2 && !a.st2)) return hipErrorInvalidValue;
  int rt, ntt;
  lowbit_tile(a, cus, &rt, &ntt);
  if (const char *e = getenv("QPH_SKINNY")) {   // test hook: the tile (two digits, rows / 16 and tokens / 16)
    rt = atoi(e) / 10 >= 4 ? 4 : 2; ntt = std::max(1, std::min(2, atoi(e) % 10));
    if (a.kind == MK_Q1 && atoi(e) == 44) ntt = 4;
  }
#define QPH_HF(R, N)                                                      \
  if (rt == R && ntt == N)                                                \
    return a.kind == MK_Q4 ? launch_lowbit_t<MK_Q4, R, N>(a, cus, st) : launch_lowbit_t<MK_Q1, R, N>(a, cus, st);
  QPH_HF(2, 1) QPH_HF(2, 2) QPH_HF(4, 1) QPH_HF(4, 2)
  if (a.kind == MK_Q1 && rt == 4 && ntt == 4) return launch_lowbit_t<MK_Q1, 4, 4>(a, cus, st);
#undef QPH_HF
  return hipErrorInvalidValue;
}

}  // namespace qph
