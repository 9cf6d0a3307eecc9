// Daylight-coefficient x sky-matrix product (dctimestep / rmtxop multiply,
// util/cmatrix.c:421-474, util/rmatrix.c:806-836):
//   C[m][n][c] = sum_k A[m][k][c] * B[k][n][c]   for c = R, G, B.
//
// mode 1 (default): BF16 MFMA with split operands.  Each FP32 value x is
// carried as hi = bf16(x), lo = bf16(x - hi); the product is accumulated in
// FP32 as hi*hi + hi*lo + lo*hi, which leaves a relative error near 2^-16
// per term instead of bf16's 2^-8.  gfx950's double-rate bf16 MFMAs do the
// products; both operands are first re-laid out K-contiguous per channel, in
// the tiles the product kernels load whole.
// mode 0: plain FP32 FMA, tiled through LDS (accuracy baseline).
#include <hip/hip_runtime.h>
#include <mutex>
#include <type_traits>
#include "rg_render.hpp"

namespace rg {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef unsigned short u16x8 __attribute__((ext_vector_type(8)));

__device__ __forceinline__ unsigned short f2bf(float f) {   // round to nearest even
  uint32_t u = __float_as_uint(f);
  u += 0x7fffu + ((u >> 16) & 1u);
  return (unsigned short)(u >> 16);
}
__device__ __forceinline__ float bf2f(unsigned short h) { return __uint_as_float((uint32_t)h << 16); }

// Both operands to hi/lo planes in one launch: blocks [0, nba) split
// A[M][K][3] into [3][M][Kp] (one element per thread), the others take a
// 32 (k) x 32 (n) tile of B[K][N][3] with its three channels (96 contiguous
// floats per k row) through LDS into [3][N][Kp] (K-contiguous per channel).
// K is zero-padded to Kp.
__global__ void __launch_bounds__(256) k_split(const float* A, const float* B, int M, int K, int N, int Kp,
                                               unsigned nba, unsigned short* Ah, unsigned short* Al,
                                               unsigned short* Bh, unsigned short* Bl) {
  __shared__ float tile[3][32][33];
  if (blockIdx.x < nba) {
    const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
    if (i >= (size_t)3 * M * Kp) return;
    const int k = (int)(i % Kp);
    const size_t r = i / Kp;
    const int m = (int)(r % M), c = (int)(r / M);
    const float x = k < K ? A[((size_t)m * K + k) * 3 + c] : 0.0f;
    const unsigned short h = f2bf(x);
    Ah[i] = h;
    Al[i] = f2bf(x - bf2f(h));
    return;
  }
  const unsigned bt = blockIdx.x - nba;
  const int ntn = (N + 31) / 32;
  const int n0 = (int)(bt % ntn) * 32, k0 = (int)(bt / ntn) * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;   // 32 x 8
  for (int j = ty; j < 32; j += 8) {
    const int k = k0 + j;
#pragma unroll
    for (int e = tx; e < 96; e += 32) {
      const int n = n0 + e / 3;
      tile[e % 3][j][e / 3] = (k < K && n < N) ? B[((size_t)k * N + n) * 3 + e % 3] : 0.0f;
    }
  }
  __syncthreads();
  for (int j = ty; j < 96; j += 8) {
    const int c = j / 32, n = n0 + j % 32, k = k0 + tx;
    if (n < N && k < Kp) {
      const float x = tile[c][tx][j % 32];
      const unsigned short h = f2bf(x);
      const size_t o = ((size_t)c * N + n) * Kp + k;
      Bh[o] = h;
      Bl[o] = f2bf(x - bf2f(h));
    }
  }
}

// Between writes of a wavefront's own LDS and reads of it by its other lanes:
// a wavefront's LDS instructions complete in order, so only the compiler has
// to keep them so (no instruction).
__device__ __forceinline__ void wave_lds_order() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

constexpr int DB = 256;        // 4 wavefronts, 2 (m) x 2 (n)
#ifndef RG_DCSKY_WB
#define RG_DCSKY_WB 4          // 16-column tiles per wavefront along n
#endif
constexpr int WA = 2;          // 16-row tiles per wavefront along m
constexpr int WB = RG_DCSKY_WB;
constexpr int BM = 32 * WA, BN = 32 * WB;   // block tile
constexpr int GROUP_M = 8;     // m tiles walked together (L2 reuse of B)

__device__ __forceinline__ bf16x8 ld8(const unsigned short* p) {
  u16x8 v = *(const u16x8*)p;
  return __builtin_bit_cast(bf16x8, v);
}

// Block -> tile.  Workgroups are dispatched round-robin over the 8 XCDs, so
// block b runs on XCD b % 8; each XCD is given a contiguous range of tiles,
// walked in groups of GROUP_M row tiles, so the operand rows it re-reads stay
// in its own L2.
__device__ __forceinline__ bool tile_of(int Mt, int Nt, int& tm, int& tn) {
  const int T = Mt * Nt;
  const int per = (T + 7) / 8;
  const int b = blockIdx.x;
  const int slot = b >> 3;
  const int tile = (b & 7) * per + slot;
  if (slot >= per || tile >= T) return false;
  const int group = tile / (GROUP_M * Nt);
  const int first = group * GROUP_M;
  const int gsz = min(Mt - first, GROUP_M);
  const int in = tile - group * GROUP_M * Nt;
  tm = first + in % gsz;
  tn = in / gsz;
  return true;
}

// The MFMA computes D = X * Y with X the B fragment (rows = sky columns n)
// and Y the A fragment (columns = sensors m), so each lane ends up holding 4
// consecutive n of one m: with the three channels that is 12 consecutive
// floats of C, written as three 16-byte stores.
__global__ void __launch_bounds__(DB) k_dcsky_mfma(const unsigned short* Ah, const unsigned short* Al,
                                                   const unsigned short* Bh, const unsigned short* Bl, float* C,
                                                   int M, int N, int Kp, int Mt, int Nt) {
  int tm, tn;
  if (!tile_of(Mt, Nt, tm, tn)) return;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int wm = wave >> 1, wn = wave & 1;
  const int m0 = tm * BM + wm * 16 * WA, n0 = tn * BN + wn * 16 * WB;
  const int r16 = lane & 15, kq = (lane >> 4) * 8;
  f32x4 acc[3][WA][WB];
  for (int c = 0; c < 3; ++c)
    for (int a = 0; a < WA; ++a)
      for (int b = 0; b < WB; ++b) acc[c][a][b] = f32x4{0.f, 0.f, 0.f, 0.f};
  // clamp rows/cols so loads stay in bounds; their results are not stored
  size_t ao[WA], bo[WB];
  for (int a = 0; a < WA; ++a) ao[a] = (size_t)min(m0 + 16 * a + r16, M - 1) * Kp + kq;
  for (int b = 0; b < WB; ++b) bo[b] = (size_t)min(n0 + 16 * b + r16, N - 1) * Kp + kq;
  for (int c = 0; c < 3; ++c) {
    const unsigned short* ah = Ah + (size_t)c * M * Kp;
    const unsigned short* al = Al + (size_t)c * M * Kp;
    const unsigned short* bh = Bh + (size_t)c * N * Kp;
    const unsigned short* bl = Bl + (size_t)c * N * Kp;
    bf16x8 fah[WA], fal[WA], fbh[WB], fbl[WB];
    for (int a = 0; a < WA; ++a) { fah[a] = ld8(ah + ao[a]); fal[a] = ld8(al + ao[a]); }
    for (int b = 0; b < WB; ++b) { fbh[b] = ld8(bh + bo[b]); fbl[b] = ld8(bl + bo[b]); }
    for (int k = 0; k < Kp; k += 32) {
      // prefetch the next K step while this one is on the matrix cores
      bf16x8 nah[WA], nal[WA], nbh[WB], nbl[WB];
      const int kn = k + 32 < Kp ? k + 32 : k;
      for (int a = 0; a < WA; ++a) { nah[a] = ld8(ah + ao[a] + kn); nal[a] = ld8(al + ao[a] + kn); }
      for (int b = 0; b < WB; ++b) { nbh[b] = ld8(bh + bo[b] + kn); nbl[b] = ld8(bl + bo[b] + kn); }
      for (int a = 0; a < WA; ++a)
        for (int b = 0; b < WB; ++b) {
          acc[c][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fbh[b], fah[a], acc[c][a][b], 0, 0, 0);
          acc[c][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fbl[b], fah[a], acc[c][a][b], 0, 0, 0);
          acc[c][a][b] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fbh[b], fal[a], acc[c][a][b], 0, 0, 0);
        }
      for (int a = 0; a < WA; ++a) { fah[a] = nah[a]; fal[a] = nal[a]; }
      for (int b = 0; b < WB; ++b) { fbh[b] = nbh[b]; fbl[b] = nbl[b]; }
    }
  }
  // D layout: lane holds D[n = 4 * (lane >> 4) + i][m = lane & 15]
  const bool vec = (N & 3) == 0;
  for (int a = 0; a < WA; ++a) {
    const int m = m0 + 16 * a + r16;
    if (m >= M) continue;
    for (int b = 0; b < WB; ++b) {
      const int nb = n0 + 16 * b + (lane >> 4) * 4;
      if (nb >= N) continue;
      float* dst = C + ((size_t)m * N + nb) * 3;
      const f32x4 r = acc[0][a][b], g = acc[1][a][b], u = acc[2][a][b];
      if (vec) {   // nb + 3 < N as N is a multiple of 4; 16-byte aligned
        float4* d4 = (float4*)dst;
        d4[0] = make_float4(r[0], g[0], u[0], r[1]);
        d4[1] = make_float4(g[1], u[1], r[2], g[2]);
        d4[2] = make_float4(u[2], r[3], g[3], u[3]);
      } else {
        for (int i = 0; i < 4 && nb + i < N; ++i) {
          dst[3 * i + 0] = r[i];
          dst[3 * i + 1] = g[i];
          dst[3 * i + 2] = u[i];
        }
      }
    }
  }
}

// Ring form for long K.  A block of four wavefronts (2 x 2) computes a
// 128 x 128 tile of all three channels, each wavefront 64 x 64 of it (2 x 2
// MFMA tiles x 3 channels of accumulators: 192 registers).  The 32 x 32 x 16
// MFMA, because there is one wavefront per SIMD: alone it issues 2.2 PFLOP/s
// of them, but only 1.3 of 16 x 16 x 32 (measured, independent products).  A stage is one
// channel of one K step of 32: the A and B hi/lo tiles (128 rows x 32 K, 8 KB
// each), loaded straight into LDS by global_load_lds (no staging registers)
// into a ring of four buffers, three stages ahead of their use.  Fragments
// are read one stage ahead into a second register set, so a stage is 24 MFMAs
// with the next stage's 16 LDS reads and the fourth's 8 loads between them,
// and one barrier.
//
// The operands are laid out for it by k_split_tiled: a stage's tile of one
// plane is 8 KB in one piece, so a load instruction fetches eight whole cache
// lines.  (From row-major planes it fetched sixteen half lines, and the
// texture unit, 61 cycles per instruction, was busy 80 % of the time.)
// 20000 x 2306 x 8760: 6.5 ms (6.7 to 6.8 with the split), 1.12 PFLOP/s issued,
// where 128 x 128 tiles of 32 x 32 per wavefront staged through registers took
// 10.5 ms; matrix cores busy 54 % of the cycles, at a clock that falls to
// 1.9 GHz.  The 16-byte parts of a row sit at part ^ ((row >> 1) & 3): the eight lanes that
// read LDS together (same part, consecutive rows of 64 bytes) then cover
// eight different 16-byte columns of the banks.
constexpr int LBM = 128, LBN = 128;
constexpr int RING = 4;                       // stages in LDS
constexpr int RPLANE = 128 * 32;              // one plane of a stage (bf16)

// Operands to tiled hi/lo planes: [channel][tile of 128 rows][K step of 32]
// [row][part swizzled][8], rows and K zero-padded.  A wavefront takes 16 rows
// of one K step in all three channels: 1,536 floats, read in runs of 96 (a row
// of A) or 48 (a K row of B) consecutive ones and turned in LDS, so that each
// lane then holds eight K of one row; its six stores are 1 KB in one piece
// over the wavefront.  (Lanes reading their own 24 floats from memory touched
// 64 lines per load: 568 against 294 us for both operands of the largest
// product, 20000 x 2306 x 8760.)  Blocks [0, nba) split A[M][K][3], the others B[K][N][3].
constexpr int TROW = 97;                      // padded row in LDS (floats)
__global__ void __launch_bounds__(256) k_split_tiled(const float* A, const float* B, int M, int K, int N, int nk,
                                                     int Mt, int Nt, unsigned nba, unsigned short* Ah,
                                                     unsigned short* Al, unsigned short* Bh, unsigned short* Bl) {
  __shared__ float turn[4][16 * TROW];
  const bool isb = blockIdx.x >= nba;
  const size_t g = ((size_t)(isb ? blockIdx.x - nba : blockIdx.x) * 256 + threadIdx.x) >> 6;   // wavefront
  const int lane = threadIdx.x & 63, T = isb ? Nt : Mt, R = isb ? N : M;
  float* tl = turn[threadIdx.x >> 6];
  // wavefront -> (K step, group of 16 rows): A walks K first (a row's steps
  // follow each other in memory), B walks the rows
  const int groups = T * 8;
  if (g >= (size_t)groups * nk) return;
  const int ks = (int)(isb ? g / groups : g % nk), rg = (int)(isb ? g % groups : g / nk);
  float x[24];
#pragma unroll
  for (int j = 0; j < 24; ++j) {
    const int i = j * 64 + lane;
    int r, e;                                 // row, 3 x K + channel within the tile
    size_t at;
    if (isb) {
      const int k = i / 48, q = i % 48;
      r = q / 3;
      e = 3 * k + q % 3;
      at = ((size_t)(ks * 32 + k) * N + rg * 16) * 3 + q;
    } else {
      r = i / 96;
      e = i % 96;
      at = ((size_t)(rg * 16 + r) * K + ks * 32) * 3 + e;
    }
    x[j] = (rg * 16 + r < R && ks * 32 + e / 3 < K) ? (isb ? B : A)[at] : 0.0f;
  }
#pragma unroll
  for (int j = 0; j < 24; ++j) {
    const int i = j * 64 + lane;
    const int k = i / 48, q = i % 48;
    tl[isb ? (q / 3) * TROW + 3 * k + q % 3 : (i / 96) * TROW + i % 96] = x[j];
  }
  wave_lds_order();
  const int row = rg * 16 + (lane >> 2), part = lane & 3;
  const float* mine = tl + (lane >> 2) * TROW + part * 24;
  unsigned short* H = isb ? Bh : Ah;
  unsigned short* L = isb ? Bl : Al;
#pragma unroll
  for (int c = 0; c < 3; ++c) {
    u16x8 h, l;
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const float v = mine[3 * j + c];
      const unsigned short u = f2bf(v);
      h[j] = u;
      l[j] = f2bf(v - bf2f(u));
    }
    const size_t o = (((size_t)c * T + (row >> 7)) * nk + ks) * RPLANE + (row & 127) * 32 + (part ^ ((row >> 1) & 3)) * 8;
    *(u16x8*)(H + o) = h;
    *(u16x8*)(L + o) = l;
  }
}

// Every LDS read of this wavefront done, at most N of its loads under way,
// then the block's barrier.
template <int N>
__device__ __forceinline__ void ring_wait() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" :: "n"(N) : "memory");
}

__global__ void __launch_bounds__(256) __attribute__((amdgpu_waves_per_eu(1, 1)))
k_dcsky_ring(const unsigned short* Ah, const unsigned short* Al, const unsigned short* Bh, const unsigned short* Bl,
             float* C, int M, int N, int nkall, int Mt, int Nt) {
  __shared__ __attribute__((aligned(16))) unsigned short lds[RING][4][RPLANE];   // [buffer][Ah, Al, Bh, Bl]
  int tm, tn;
  if (!tile_of(Mt, Nt, tm, tn)) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wm = wave >> 1, wn = wave & 1;
  const int r32 = lane & 31;
  const int mb = tm * LBM, nb = tn * LBN;
  // this block's share of the K steps and, when K is split, its own partial C
  const int kb = (int)((long long)nkall * blockIdx.y / gridDim.y);
  const int nk = (int)((long long)nkall * (blockIdx.y + 1) / gridDim.y) - kb;
  C += (size_t)blockIdx.y * M * N * 3;
  // this wavefront stages plane `wave`; stage s is channel s % 3 of K step
  // s / 3.  Past the end the last stage is loaded again, so that the counts
  // of loads under way stay the same
  const int T = wave < 2 ? Mt : Nt, t = wave < 2 ? tm : tn;
  const unsigned short* src = (wave == 0 ? Ah : (wave == 1 ? Al : (wave == 2 ? Bh : Bl))) +
                              ((size_t)t * nkall + kb) * RPLANE;
  const size_t cstep = (size_t)T * nkall * RPLANE;   // next channel
  const int lo8 = lane * 8;
  int left = 3 * nk, lc = 0;
  auto load_part = [&](int buf, int j) {
    __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(src + j * 512 + lo8),
                                     (__attribute__((address_space(3))) void*)&lds[buf][wave][j * 512], 16, 0, 0);
  };
  auto next_stage = [&]() {
    if (--left <= 0) return;
    if (lc == 2) { src += RPLANE; src -= 2 * cstep; lc = 0; }
    else { src += cstep; ++lc; }
  };
  f32x16 acc[3][2][2];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int i = 0; i < 16; ++i) acc[c][0][0][i] = acc[c][0][1][i] = acc[c][1][0][i] = acc[c][1][1][i] = 0.f;
  // fragments [set][plane: Ah, Al, Bh, Bl][tile][half of the K step]
  const int ra = (wm * 64 + r32) * 32, rb = (wn * 64 + r32) * 32;
  const int part[2] = {((lane >> 5) ^ ((r32 >> 1) & 3)) * 8, ((2 + (lane >> 5)) ^ ((r32 >> 1) & 3)) * 8};
  bf16x8 fr[2][4][2][2];
  auto read_frag = [&](int buf, int f, int i) {       // i = 8 x half + 4 x tile + plane
    const int pl = i & 3, q = (i >> 2) & 1, kk = i >> 3;
    fr[f][pl][q][kk] = ld8(&lds[buf][pl][(pl < 2 ? ra : rb) + q * 1024 + part[kk]]);
  };
#pragma unroll
  for (int s = 0; s < RING; ++s) {
#pragma unroll
    for (int j = 0; j < 8; ++j) load_part(s, j);
    next_stage();
  }
  ring_wait<8 * (RING - 1)>();
#pragma unroll
  for (int i = 0; i < 16; ++i) read_frag(0, 0, i);
  // One K step (three stages).  J: its place among four, which settles each
  // stage's buffer and register set at compile time (12 stages = 3 channels x
  // 4 buffers).  The loop runs whole groups of four; leaving it in between
  // would copy all accumulators at every exit.
  auto kstep = [&](auto J) {
#pragma unroll
    for (int q = 3 * decltype(J)::value; q < 3 * decltype(J)::value + 3; ++q) {
      const int c = q % 3, buf = q % RING, f = q & 1;
      // stage s + 1 is in LDS for everyone, and everyone has read stage s
      ring_wait<8 * (RING - 2)>();
#pragma unroll
      for (int g = 0; g < 8; ++g) {
        load_part(buf, g);
        if (g < 6)
#pragma unroll
          for (int i = 0; i < 3; ++i)
            if (3 * g + i < 16) read_frag((buf + 1) % RING, f ^ 1, 3 * g + i);
#pragma unroll
        for (int i = 3 * g; i < 3 * g + 3; ++i) {
          const int kk = i / 12, p = i / 4 % 3, a = (i >> 1) & 1, b = i & 1;    // products: hi hi, lo hi, hi lo
          acc[c][a][b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fr[f][p == 1 ? 3 : 2][b][kk], fr[f][p == 2 ? 1 : 0][a][kk],
                                                                 acc[c][a][b], 0, 0, 0);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
      next_stage();
    }
  };
  for (int k = 0; k < nk / 4; ++k) {
    kstep(std::integral_constant<int, 0>());
    kstep(std::integral_constant<int, 1>());
    kstep(std::integral_constant<int, 2>());
    kstep(std::integral_constant<int, 3>());
  }
  if ((nk & 3) > 0) kstep(std::integral_constant<int, 0>());
  if ((nk & 3) > 1) kstep(std::integral_constant<int, 1>());
  if ((nk & 3) > 2) kstep(std::integral_constant<int, 2>());
  // the loads still under way write LDS: the block must not end before them
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  // D layout: lane holds D[n = 8 * (i / 4) + 4 * (lane >> 5) + i % 4][m = lane & 31]
  const bool vec = (N & 3) == 0;
#pragma unroll
  for (int a = 0; a < 2; ++a) {
    const int m = mb + wm * 64 + 32 * a + r32;
    if (m >= M) continue;
#pragma unroll
    for (int bg = 0; bg < 8; ++bg) {
      const int b = bg >> 2, i0 = (bg & 3) * 4;
      const int nq = nb + wn * 64 + 32 * b + 2 * i0 + 4 * (lane >> 5);
      if (nq >= N) continue;
      float* dst = C + ((size_t)m * N + nq) * 3;
      const f32x16 r = acc[0][a][b], g = acc[1][a][b], u = acc[2][a][b];
      if (vec) {
        float4* d4 = (float4*)dst;
        d4[0] = make_float4(r[i0], g[i0], u[i0], r[i0 + 1]);
        d4[1] = make_float4(g[i0 + 1], u[i0 + 1], r[i0 + 2], g[i0 + 2]);
        d4[2] = make_float4(u[i0 + 2], r[i0 + 3], g[i0 + 3], u[i0 + 3]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (nq + i < N) {
            dst[3 * i + 0] = r[i0 + i];
            dst[3 * i + 1] = g[i0 + i];
            dst[3 * i + 2] = u[i0 + i];
          }
      }
    }
  }
}

// Sum of the partial products of a split K, in order.
__global__ void __launch_bounds__(256) k_dcsky_sum(const float* part, float* C, size_t n, int parts) {
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= n) return;
  float v = part[i];
  for (int p = 1; p < parts; ++p) v += part[(size_t)p * n + i];
  C[i] = v;
}

// Parts the K steps of the ring form are split into: with fewer tiles than
// compute units the others would idle for the whole K (3 tiles of K = 2306:
// 133 us; in 18 parts 51 us), so K is shared by as many blocks as there
// are units for, at least four steps each.  From half as many tiles as units
// on a second round would cost what the split saves.
static int ring_parts(long long tiles, int nk) {
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  return (int)std::max<long long>(1, std::min<long long>(ncu / tiles, nk / 4));
}

// Short-K form (K <= 160, e.g. 146 Klems patches): the product is bound by
// the output write, and the operands are small enough that a wavefront keeps
// 16 rows of A (hi and lo, all K, three channels: 120 registers at K = 160)
// for the whole launch.  A block of 8 wavefronts owns a slab of 128 rows of A
// and walks a range of sky columns in chunks of 32: each chunk's B planes
// (hi/lo, three channels, all K) are loaded straight into LDS, into the buffer
// that the chunk before does not use.  No K loop over global memory, one
// barrier per chunk.
//
// Outputs go through LDS: a lane ends up with 12 consecutive floats of a row,
// and storing those as they are writes 16 bytes every 48, three times as many
// partial lines as the rows have.  Turned in LDS, a store instruction covers
// runs of 192 bytes.  2500 x 146 x 8760: 84 to 90 us (104 with 48-byte runs and the
// chunk staged through registers), 3.0 of the 6.9 TB/s that a plain fill
// reaches; what is left is the wait for the next chunk's loads, which complete
// in order behind the stores of the chunk before (the compiler does not tell
// the two buffers apart and waits for them ahead of this chunk's first LDS
// read, so they overlap nothing), and LDS reads (61 KB per wavefront and
// chunk).  Four wavefronts of 32 rows halve those and lose
// more: one wavefront per SIMD, 106 us.
// The code's own wait for those loads does not rely on that one.  With 16-byte
// stores it stands ahead of the chunk's outputs, where nothing has to be
// counted.  With 4-byte ones it would keep their addresses from being formed
// beside the MFMAs there (2500 x 146 x 8759: 164 us, 139 behind them), so it
// stands behind them and takes exactly 2 NST of them to be under way: each is
// an instruction of its own in the source, and every lane issues all of them
// in every chunk (pieces past the chunk load a valid piece again; outputs
// outside C go to `sink`).
constexpr int SW = 8;                  // wavefronts per block
constexpr int SROWS = 16 * SW;         // rows of A per block (a slab)
constexpr int SCOLS = 32;              // sky columns per staged chunk
constexpr int SHORT_KS = 5;            // K steps of 32 the short form covers (Kp <= 160)
constexpr int SINK_FLOATS = 64 * 12;   // one wavefront's worth of redirected outputs
constexpr int SOUT = 52;               // padded output row in LDS (floats): 16 columns x 3 channels

template <int KS, bool VEC>
__global__ void __launch_bounds__(64 * SW)
k_dcsky_short(const unsigned short* Ah, const unsigned short* Al, const unsigned short* Bh, const unsigned short* Bl,
              float* C, float* sink, int M, int N, int Mt, int Nt, int nrange) {
  static_assert(SROWS == LBM, "a slab is a tile of the split planes");
  constexpr int NPC = 6 * KS * 2;              // 1 KB pieces (16 rows of one K step) per chunk
  constexpr int NLD = (NPC + SW - 1) / SW;     // pieces per wavefront
  __shared__ __attribute__((aligned(16))) unsigned short lds[2][6 * KS * SCOLS * 32];   // [buffer][2 c + lo][step][row][32]
  __shared__ __attribute__((aligned(16))) float turn[SW][16 * SOUT];
  // block -> (slab, column range); blocks run on XCD b % 8, and the blocks
  // of one XCD take consecutive q: all slabs of one column range, which
  // share its B chunks in that XCD's L2
  const int per = (int)((gridDim.x + 7) / 8);
  const int q = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
  if (q >= Mt * nrange) return;
  const int slab = q % Mt, range = q / Mt;
  const int nchunk = (N + SCOLS - 1) / SCOLS;
  const int cb = (int)((long long)range * nchunk / nrange), ce = (int)((long long)(range + 1) * nchunk / nrange);
  if (cb >= ce) return;
  const int lane = threadIdx.x & 63, wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int r16 = lane & 15, part = ((lane >> 4) ^ ((r16 >> 1) & 3)) * 8;
  bf16x8 ah[3][KS], al[3][KS];
#pragma unroll
  for (int c = 0; c < 3; ++c)
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      const size_t o = (((size_t)c * Mt + slab) * KS + s) * RPLANE + (wave * 16 + r16) * 32 + part;
      ah[c][s] = ld8(Ah + o);
      al[c][s] = ld8(Al + o);
    }
  // piece p: plane p / (2 KS) (2 c + lo), K step, half of the chunk's rows
  const unsigned short* psrc[NLD];
#pragma unroll
  for (int j = 0; j < NLD; ++j) {
    const int p = min(wave + j * SW, NPC - 1);
    const int pl = p / (2 * KS), s = (p % (2 * KS)) >> 1, half = p & 1;
    psrc[j] = ((pl & 1) ? Bl : Bh) + ((size_t)(pl >> 1) * Nt * KS + s) * RPLANE + half * 512;
  }
  auto load_chunk = [&](int chunk, int buf) {
    const int n0 = chunk * SCOLS;
    const size_t at = (size_t)(n0 >> 7) * KS * RPLANE + (n0 & 127) * 32 + lane * 8;
#pragma unroll
    for (int j = 0; j < NLD; ++j)
      __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)(psrc[j] + at),
                                       (__attribute__((address_space(3))) void*)&lds[buf][min(wave + j * SW, NPC - 1) * 512],
                                       16, 0, 0);
  };
  load_chunk(cb, 0);
  // every load so far (A and the first chunk) complete here, so that no wait
  // inside the loop, where this chunk's stores are also outstanding, is
  // counted against them
  ring_wait<0>();
  float* const mysink = sink + lane * 12;
  float* const tw = turn[wave];
  constexpr int NST = VEC ? 3 : 12;      // stores per 16 columns: 16 bytes each, or 4
  for (int ch = cb; ch < ce; ++ch) {
    const int buf = (ch - cb) & 1;
    load_chunk(min(ch + 1, ce - 1), buf ^ 1);
    __builtin_amdgcn_sched_barrier(0);     // the next chunk's loads go out before the MFMAs
    f32x4 acc[2][3];
#pragma unroll
    for (int b = 0; b < 2; ++b)
#pragma unroll
      for (int c = 0; c < 3; ++c) acc[b][c] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int s = 0; s < KS; ++s) {
      // the six accumulators take turns, so that no MFMA waits for the one before it
      bf16x8 fb[2][3][2];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int c = 0; c < 3; ++c)
#pragma unroll
          for (int h = 0; h < 2; ++h)
            fb[b][c][h] = ld8(&lds[buf][((2 * c + h) * KS + s) * (SCOLS * 32) + (16 * b + r16) * 32 + part]);
#pragma unroll
      for (int p = 0; p < 3; ++p)            // hi hi, lo hi, hi lo
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int c = 0; c < 3; ++c)
            acc[b][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(fb[b][c][p == 1], p == 2 ? al[c][s] : ah[c][s],
                                                                acc[b][c], 0, 0, 0);
    }
    if (VEC) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");     // the next chunk's loads done
    // D layout: lane holds D[n = 4 * (lane >> 4) + i][m = lane & 15], 12
    // consecutive floats of row m; turned through this wavefront's own LDS
    const int m0 = slab * SROWS + wave * 16;
#pragma unroll
    for (int b = 0; b < 2; ++b) {
      const f32x4 r = acc[b][0], g = acc[b][1], u = acc[b][2];
      float4* t4 = (float4*)(tw + r16 * SOUT + (lane >> 4) * 12);
      t4[0] = make_float4(r[0], g[0], u[0], r[1]);
      t4[1] = make_float4(g[1], u[1], r[2], g[2]);
      t4[2] = make_float4(u[2], r[3], g[3], u[3]);
      wave_lds_order();
      const int f0 = (ch * SCOLS + 16 * b) * 3;
#pragma unroll
      for (int i = 0; i < NST; ++i) {
        const int l = i * 64 + lane;
        constexpr int W = VEC ? 4 : 1;         // floats per store
        const int row = l / (48 / W), f = l % (48 / W) * W;
        // N a multiple of 4 (VEC): 16-byte aligned, and a piece is inside C or outside as a whole
        const bool in = m0 + row < M && f0 + f < 3 * N;
        float* dst = in ? C + (size_t)(m0 + row) * N * 3 + f0 + f : mysink;
        if (VEC) *(float4*)dst = *(const float4*)(tw + row * SOUT + f);
        else asm volatile("global_store_dword %0, %1, off" :: "v"(dst), "v"(tw[row * SOUT + f]) : "memory");
      }
      wave_lds_order();
    }
    // every LDS read of this chunk done, and the next one's loads (issued
    // before these stores)
    ring_wait<VEC ? 63 : 2 * NST>();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// Small products in one launch, FP32 throughout: a block of 16 wavefronts
// takes 64 columns of RM rows (all three channels), each wavefront a
// sixteenth of K, and adds the parts in LDS in order.  Splitting the operands
// first takes a launch of its own, 7 us of latency whatever the size: 67 x 41
// x 5 takes 14 us here and 25 there, 100 x 578 x 100 22 and 36.  From 2^22
// multiply-adds on four rows share a column's loads (11 x 146 x 8760: 26 us,
// 44 split), which needs columns enough that a wavefront's lie in one group
// of rows (14000 x 578 x 1: 174 us with four rows, 50 with one).  The lines
// to the split forms lie where they catch up; past K = 1024 the parts' chains
// of loads are longer than the ring's split K (2000 x 2306 x 1: 125 against
// 53 us).
constexpr int TW = 16;
constexpr long long SMALL_MACS = 1ll << 23, SMALL_ROW_MACS = 1ll << 22, SMALL_WIDE_MACS = 1ll << 24;
constexpr int SMALL_K = 1024, SMALL_WIDE_N = 256;
template <int RM>
__global__ void __launch_bounds__(64 * TW) k_dcsky_small(const float* A, const float* B, float* C, int M, int K, int N) {
  __shared__ float part[TW][RM][64 * 3 + 1];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  // column `col` of the row groups laid end to end
  const size_t all = (size_t)((M + RM - 1) / RM) * N, col0 = (size_t)blockIdx.x * 64;
  const size_t col = min(col0 + lane, all - 1);
  const int m = (int)(col / N) * RM;
  const float* b = B + (col % N) * 3;
  const float* a[RM];
#pragma unroll
  for (int i = 0; i < RM; ++i) a[i] = A + (size_t)min(m + i, M - 1) * K * 3;
  const int k0 = (int)((long long)K * w / TW), k1 = (int)((long long)K * (w + 1) / TW);
  float acc[RM][3] = {};
#pragma unroll 8
  for (int k = k0; k < k1; ++k) {
    const float* bk = b + (size_t)k * N * 3;
    const float b0 = bk[0], b1 = bk[1], b2 = bk[2];
#pragma unroll
    for (int i = 0; i < RM; ++i) {
      acc[i][0] = fmaf(a[i][3 * k], b0, acc[i][0]);
      acc[i][1] = fmaf(a[i][3 * k + 1], b1, acc[i][1]);
      acc[i][2] = fmaf(a[i][3 * k + 2], b2, acc[i][2]);
    }
  }
#pragma unroll
  for (int i = 0; i < RM; ++i)
#pragma unroll
    for (int c = 0; c < 3; ++c) part[w][i][3 * lane + c] = acc[i][c];
  __syncthreads();
  for (int t = threadIdx.x; t < RM * 192; t += 64 * TW) {
    const int i = t / 192, f = t % 192;
    const size_t oc = col0 + f / 3;
    const int om = (int)(oc / N) * RM + i;
    if (oc >= all || om >= M) continue;
    float v = part[0][i][f];
#pragma unroll
    for (int k = 1; k < TW; ++k) v += part[k][i][f];
    C[((size_t)om * N + oc % N) * 3 + f % 3] = v;
  }
}

// FP32 reference path: 16x16 threads, 64x64 tile, LDS staged.
__global__ void __launch_bounds__(256) k_dcsky_f32(const float* A, const float* B, float* C, int M, int K, int N) {
  __shared__ float As[3][64][17];
  __shared__ float Bs[3][16][65];
  int tx = threadIdx.x & 15, ty = threadIdx.x >> 4;
  int m0 = blockIdx.y * 64, n0 = blockIdx.x * 64;
  float acc[3][4][4] = {};
  for (int k0 = 0; k0 < K; k0 += 16) {
    for (int t = threadIdx.x; t < 3 * 64 * 16; t += 256) {
      int c = t % 3, kk = (t / 3) % 16, mm = t / 48;
      int m = m0 + mm, k = k0 + kk;
      As[c][mm][kk] = (m < M && k < K) ? A[((size_t)m * K + k) * 3 + c] : 0.f;
    }
    for (int t = threadIdx.x; t < 3 * 64 * 16; t += 256) {
      int c = t % 3, nn = (t / 3) % 64, kk = t / 192;
      int n = n0 + nn, k = k0 + kk;
      Bs[c][kk][nn] = (n < N && k < K) ? B[((size_t)k * N + n) * 3 + c] : 0.f;
    }
    __syncthreads();
    for (int kk = 0; kk < 16; ++kk)
      for (int c = 0; c < 3; ++c)
        for (int i = 0; i < 4; ++i) {
          float a = As[c][ty * 4 + i][kk];
          for (int j = 0; j < 4; ++j) acc[c][i][j] = fmaf(a, Bs[c][kk][tx * 4 + j], acc[c][i][j]);
        }
    __syncthreads();
  }
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 4; ++j) {
      int m = m0 + ty * 4 + i, n = n0 + tx * 4 + j;
      if (m < M && n < N)
        for (int c = 0; c < 3; ++c) C[((size_t)m * N + n) * 3 + c] = acc[c][i][j];
    }
}

static void dck(hipError_t e, const char* w) {
  if (e != hipSuccess) throw std::runtime_error(std::string(w) + ": " + hipGetErrorString(e));
}

// Split planes of a call, kept per (device, stream) and grown as needed (a
// stream-ordered allocation and free per call cost about as much as the whole
// product at K = 146).  The lock is held while a call queues its kernels, so a
// buffer is only replaced after the work queued on it has finished.
struct DcScratch {
  void* p = nullptr;
  size_t bytes = 0;
};
static std::mutex g_dc_mu;
static std::map<std::pair<int, hipStream_t>, DcScratch> g_dc_scratch;

static unsigned short* dc_scratch(size_t bytes, hipStream_t st) {
  int dev = 0;
  dck(hipGetDevice(&dev), "dcsky device");
  DcScratch& s = g_dc_scratch[{dev, st}];
  if (s.bytes < bytes) {
    if (s.p) {
      dck(hipStreamSynchronize(st), "dcsky scratch sync");
      dck(hipFree(s.p), "dcsky scratch free");
      s.p = nullptr;
      s.bytes = 0;
    }
    dck(hipMalloc(&s.p, bytes), "dcsky scratch");
    s.bytes = bytes;
  }
  return (unsigned short*)s.p;
}

// Column ranges per slab for the short-K form: one block per CU at a time
// (its LDS), so the fewest ranges that keep at least 90 % of the CUs busy
// over whole rounds of blocks.
static int short_ranges(int nslab, int nchunk) {
  int dev = 0, ncu = 256;
  if (hipGetDevice(&dev) == hipSuccess) (void)hipDeviceGetAttribute(&ncu, hipDeviceAttributeMultiprocessorCount, dev);
  ncu = std::max(ncu, 1);
  int best = 1;
  double beff = 0.0;
  for (int r = 1; r <= std::min(nchunk, 64); ++r) {
    const long long G = (long long)nslab * r;
    const long long rounds = (G + ncu - 1) / ncu;
    const double eff = (double)G / (double)(rounds * ncu);
    if (eff > beff + 1e-9) { beff = eff; best = r; }
    if (eff >= 0.9) break;
  }
  return best;
}

template <int KS>
static void launch_short(const unsigned short* Ah, const unsigned short* Al, const unsigned short* Bh,
                         const unsigned short* Bl, float* C, float* sink, int M, int N, int Mt, int Nt,
                         hipStream_t st) {
  const int nrange = short_ranges(Mt, (N + SCOLS - 1) / SCOLS);
  const long long G = (long long)Mt * nrange;
  if (G > 0x7fffffffLL - 8) throw std::runtime_error("dcsky: matrix too large");
  const unsigned nblk = (unsigned)((G + 7) / 8 * 8);
  if (N % 4 == 0)
    hipLaunchKernelGGL((k_dcsky_short<KS, true>), dim3(nblk), dim3(64 * SW), 0, st, Ah, Al, Bh, Bl, C, sink, M, N,
                       Mt, Nt, nrange);
  else
    hipLaunchKernelGGL((k_dcsky_short<KS, false>), dim3(nblk), dim3(64 * SW), 0, st, Ah, Al, Bh, Bl, C, sink, M, N,
                       Mt, Nt, nrange);
}

void dcsky(const float* A, const float* B, float* C, int M, int K, int N, int mode, hipStream_t st) {
  if (mode == 0) {
    hipLaunchKernelGGL(k_dcsky_f32, dim3((N + 63) / 64, (M + 63) / 64), dim3(256), 0, st, A, B, C, M, K, N);
    return;
  }
  const bool wide = N >= SMALL_WIDE_N && M >= 4;
  const double macs = (double)M * N * K;
  if (mode == 1 && K <= SMALL_K && macs <= (double)(wide ? SMALL_WIDE_MACS : SMALL_MACS)) {
    const bool rows = wide && macs > (double)SMALL_ROW_MACS;
    const size_t cols = (size_t)(rows ? (M + 3) / 4 : M) * N;
    hipLaunchKernelGGL(rows ? k_dcsky_small<4> : k_dcsky_small<1>, dim3((unsigned)((cols + 63) / 64)), dim3(64 * TW), 0,
                       st, A, B, C, M, K, N);
    return;
  }
  // K <= 160 is bound by the output write and keeps A in registers (mode 4
  // forces that form); longer K is MFMA work and takes the ring of LDS
  // buffers (mode 3; 2500 x 146 x 8760: 155 us there).  mode 2 forces
  // per-wavefront loads, slower everywhere (2500 x 200 x 8760: 299 us where
  // the ring takes 179).
  const int k32 = (K + 31) / 32 * 32;
  if (mode == 4 && k32 > 32 * SHORT_KS) throw std::runtime_error("dcsky: mode 4 needs K <= 160");
  const bool shortk = mode == 4 || (mode == 1 && k32 <= 32 * SHORT_KS);
  const bool staged = !shortk && mode != 2;
  const bool tiled = shortk || staged;
  const int Kp = k32, nk = Kp / 32;
  const int Mt = (M + LBM - 1) / LBM, Nt = (N + LBN - 1) / LBN;      // tiles of the tiled planes
  const size_t na = (size_t)3 * (tiled ? Mt * LBM : M) * Kp, nb = (size_t)3 * (tiled ? Nt * LBN : N) * Kp;
  std::lock_guard<std::mutex> lk(g_dc_mu);
  // split planes, then (16-byte aligned) the short form's output sink or a
  // split K's partial products
  const size_t plane_bytes = (2 * (na + nb) * sizeof(unsigned short) + 255) / 256 * 256;
  const int parts = staged ? ring_parts((long long)Mt * Nt, nk) : 1;
  const size_t tail_bytes = std::max((size_t)SINK_FLOATS, parts > 1 ? (size_t)parts * M * N * 3 : 0) * sizeof(float);
  unsigned short* buf = dc_scratch(plane_bytes + tail_bytes, st);
  unsigned short *Ah = buf, *Al = buf + na, *Bh = buf + 2 * na, *Bl = buf + 2 * na + nb;
  float* sink = (float*)((char*)buf + plane_bytes);
  if (tiled) {
    const size_t nba = ((size_t)Mt * 8 * nk + 3) / 4, nbb = ((size_t)Nt * 8 * nk + 3) / 4;
    const long long tiles = (long long)Mt * Nt;
    if (nba + nbb > 0x7fffffffu || tiles > 0x7fffffffLL - 8) throw std::runtime_error("dcsky: matrix too large");
    hipLaunchKernelGGL(k_split_tiled, dim3((unsigned)(nba + nbb)), dim3(256), 0, st, A, B, M, K, N, nk, Mt, Nt,
                       (unsigned)nba, Ah, Al, Bh, Bl);
    if (shortk) {
      switch (nk) {
        case 1: launch_short<1>(Ah, Al, Bh, Bl, C, sink, M, N, Mt, Nt, st); break;
        case 2: launch_short<2>(Ah, Al, Bh, Bl, C, sink, M, N, Mt, Nt, st); break;
        case 3: launch_short<3>(Ah, Al, Bh, Bl, C, sink, M, N, Mt, Nt, st); break;
        case 4: launch_short<4>(Ah, Al, Bh, Bl, C, sink, M, N, Mt, Nt, st); break;
        default: launch_short<5>(Ah, Al, Bh, Bl, C, sink, M, N, Mt, Nt, st); break;
      }
      return;
    }
    hipLaunchKernelGGL(k_dcsky_ring, dim3((unsigned)((tiles + 7) / 8 * 8), (unsigned)parts), dim3(256), 0, st, Ah, Al,
                       Bh, Bl, parts > 1 ? sink : C, M, N, nk, Mt, Nt);
    if (parts > 1) {
      const size_t n = (size_t)M * N * 3;
      hipLaunchKernelGGL(k_dcsky_sum, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, sink, C, n, parts);
    }
    return;
  }
  const size_t nba = (na + 255) / 256, nbb = (size_t)((N + 31) / 32) * (Kp / 32);
  if (nba + nbb > 0x7fffffffu) throw std::runtime_error("dcsky: matrix too large");
  hipLaunchKernelGGL(k_split, dim3((unsigned)(nba + nbb)), dim3(256), 0, st, A, B, M, K, N, Kp, (unsigned)nba, Ah, Al,
                     Bh, Bl);
  const int Wt = (M + BM - 1) / BM, Vt = (N + BN - 1) / BN;
  const long long tiles = (long long)Wt * Vt;
  if (tiles > 0x7fffffffLL - 8) throw std::runtime_error("dcsky: matrix too large");
  hipLaunchKernelGGL(k_dcsky_mfma, dim3((unsigned)((tiles + 7) / 8 * 8)), dim3(DB), 0, st, Ah, Al, Bh, Bl, C, M, N, Kp,
                     Wt, Vt);
}

}  // namespace rg
