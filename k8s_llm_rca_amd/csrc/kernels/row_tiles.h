// A product of many rows as one workgroup's tile of 32 F rows x 256 columns, for kernels with an epilogue of their own
// (gemm_add.hip, gemm_prep.hip).
//
// One 512-thread workgroup a compute unit; F is chosen by how the tiles fill whole waves of 256
// (ops/linear.py: add_plan, prep_plan).  K comes in tiles of 64 by LDS-DMA, three of them staged (two where the rows leave no room), and is
// worked off in two phases, W's columns 0 - 127 and 128 - 255: a wave multiplies 16 F rows x 32 columns a phase and reads its rows'
// fragments once a tile.  Waves 4 - 7 run one barrier behind waves 0 - 3, so that on every SIMD one of two waves issues matrix
// instructions while the other reads fragments and asks for tiles.  In slots between barriers, u the K tile:
//   waves 0 - 3:  4u  read X0, W0    4u+1  multiply    4u+2  read W1            4u+3  multiply
//   waves 4 - 7:                     4u+1  read X1, W0  4u+2  multiply          4u+3  read W1      4u+4  multiply
// A slot's reads have ended when the next slot has (the multiplication waits for them).  So a buffer of tile u takes its next tile
// from slot 4u+2 (X0: read by waves 0 - 3 alone), 4u+3 (X1, W0) and 4u+5 (W1); each wave asks in its reading slots, W by halves of
// the waves.  A wave waits for its own share of what is read next in the reading slot before: FLY counts what it has asked for
// since.  Past the last tile the last one is asked for again, into a buffer that nobody reads, so that the counts hold.
//
#pragma once
#include <type_traits>

#include "common.h"

namespace k8s {
namespace padd {

constexpr int BN = 256, BK = 64, ROW_B = 2 * BK;          // a staged row: 128 bytes
constexpr int GM = 4;                                     // row tiles of a group that shares its columns' weights

typedef __attribute__((address_space(3))) void lds_void_t;
__device__ __forceinline__ void glds16(const uint16_t* src, unsigned char* lds_dst) {
  __builtin_amdgcn_global_load_lds(src, (lds_void_t*)lds_dst, 16, 0, 0);
}
__device__ __forceinline__ void bar() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("" ::: "memory");
}
template <int N>
__device__ __forceinline__ void vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}
__device__ __forceinline__ float last_lane(float v) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}
__device__ __forceinline__ void lds_bar() {
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
  bar();
}

// A workgroup's tile: XCD-contiguous ranges of tiles, groups of GM row tiles
__device__ __forceinline__ void tile_of(int n_mt, int n_nt, int& tm, int& tn) {
  const int T = n_mt * n_nt, b = blockIdx.x, xcd = b & 7, q = T >> 3, r = T & 7;
  const int t = (xcd < r ? xcd * (q + 1) : r * (q + 1) + (xcd - r) * q) + (b >> 3);
  const int gsz = GM * n_nt, first = t / gsz * GM, gm = min(n_mt - first, GM);
  tm = first + (t % gsz) % gm;
  tn = (t % gsz) / gm;
}

// The order of a tile's columns in which a lane has eight neighbours, 8 fhi + 4 j + v of the wave's 32
__device__ __forceinline__ int eight_columns(int h, int R) {
  const int rho = R & 31;
  return 128 * h + 32 * (R >> 5) + 8 * ((rho >> 2) & 3) + 4 * (rho >> 4) + (rho & 3);
}

// F: 16-row fragments of a wave
template <int F>
struct RowTile {
  static constexpr int BM = 32 * F, HM = 16 * F;            // rows of a tile, of a half
  static constexpr int NB = F <= 5 ? 3 : 2;                 // staged K tiles
  static constexpr int XA = (2 * F + 3) / 4;                // DMA instructions of a wave for its half of X
  static constexpr int XB = HM * ROW_B, WB = 128 * ROW_B, BUF = 2 * XB + 2 * WB;
  static constexpr int LDS = NB * BUF > HM * 1024 ? NB * BUF : HM * 1024;      // (the second: half a tile's results in fp32)
  static_assert(LDS <= 160 * 1024);

  // acc[h][i][j][v] = row m0 + HM wr + 16 i + frow of a by row col(h, 32 wc + 16 j + 4 fhi + v) of w (wave 4 wr + wc, lane 16 fhi +
  // frow).  Rows of a past M - 1 are the last again.
  template <typename Col>
  static __device__ __forceinline__ void product(const uint16_t* a, int lda, const uint16_t* w, int M, int K, int m0, unsigned char* sm,
                                                 f32x4 (&acc)[2][F][2], Col&& col) {
    const int lane = threadIdx.x & 63, wv = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int wr = wv >> 2, wc = wv & 3, nt = K / BK;
    // ---- what this wave stages: its own half of X, a part of both halves of W
    const uint16_t* xs[XA];
    uint32_t xd[XA];
#pragma unroll
    for (int i = 0; i < XA; ++i) {
      const int j = min(4 * i + wc, 2 * F - 1), R = 8 * j + (lane >> 3);      // (past the last: the last again)
      xs[i] = a + (size_t)min(m0 + HM * wr + R, M - 1) * lda + 8 * ((lane & 7) ^ ((R >> 1) & 7));
      xd[i] = wr * XB + j * 1024;
    }
    const uint16_t* wsrc[2][2];
    uint32_t wd[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int j = 8 * wr + 2 * wc + i, R = 8 * j + (lane >> 3);
#pragma unroll
      for (int h = 0; h < 2; ++h) wsrc[h][i] = w + (size_t)col(h, R) * K + 8 * ((lane & 7) ^ ((R >> 1) & 7));
      wd[i] = 2 * XB + j * 1024;
    }
    auto put_x = [&](int v, int buf) {
      const int kt = min(v, nt - 1) * BK;
#pragma unroll
      for (int i = 0; i < XA; ++i) glds16(xs[i] + kt, sm + buf * BUF + xd[i]);
    };
    auto put_w = [&](int h, int v, int buf) {
      const int kt = min(v, nt - 1) * BK;
#pragma unroll
      for (int i = 0; i < 2; ++i) glds16(wsrc[h][i] + kt, sm + buf * BUF + h * WB + wd[i]);
    };
    const int frow = lane & 15, fhi = lane >> 4;
    const int f0 = frow * ROW_B + 16 * (fhi ^ ((frow >> 1) & 7));
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[h][i][j] = f32x4{0.f, 0.f, 0.f, 0.f};
    bf16x8 xf[F][2], wf[2][2];
    auto read_x = [&](int buf) {
#pragma unroll
      for (int i = 0; i < F; ++i)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
          xf[i][ks] = *reinterpret_cast<const bf16x8*>(sm + buf * BUF + wr * XB + 16 * i * ROW_B + (f0 ^ (64 * ks)));
    };
    auto read_w = [&](int h, int buf) {
#pragma unroll
      for (int j = 0; j < 2; ++j)
#pragma unroll
        for (int ks = 0; ks < 2; ++ks)
          wf[j][ks] = *reinterpret_cast<const bf16x8*>(sm + buf * BUF + 2 * XB + h * WB + (32 * wc + 16 * j) * ROW_B + (f0 ^ (64 * ks)));
    };
    auto mul = [&](auto H) {
      constexpr int h = decltype(H)::value;
#pragma unroll
      for (int ks = 0; ks < 2; ++ks)
#pragma unroll
        for (int i = 0; i < F; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[h][i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j][ks], xf[i][ks], acc[h][i][j], 0, 0, 0);
    };
    using H0 = std::integral_constant<int, 0>;
    using H1 = std::integral_constant<int, 1>;
    auto run = [&](auto WR) {
      constexpr bool second = decltype(WR)::value;
      // DMA instructions of this wave that may be in flight behind what is read next
      constexpr int FLY = (second ? 2 : 0) + (NB == 3 ? 6 + 2 * XA : 2 + XA);
      put_x(0, 0);
      put_w(0, 0, 0);
      put_w(1, 0, 0);
      put_x(1, 1);
      if constexpr (NB == 3) {
        put_w(0, 1, 1);
        put_w(1, 1, 1);
        put_x(2, 2);
      }
      if constexpr (second) put_w(0, NB - 1, NB - 1);
      vm_wait<FLY>();
      bar();
      if constexpr (second) bar();
      int b = 0, bl = NB - 1;                                 // the buffers of tiles u and u - 1
      for (int u = 0; u < nt; ++u) {
        read_x(b);
        read_w(0, b);
        put_w(second, u - 1 + NB, bl);
        vm_wait<FLY>();
        bar();
        mul(H0{});
        bar();
        read_w(1, b);
        if constexpr (!second) put_w(1, u - 1 + NB, bl);
        put_x(u + NB, b);
        if constexpr (second) put_w(0, u + NB, b);
        vm_wait<FLY>();
        bar();
        mul(H1{});
        bar();
        bl = b;
        b = b + 1 == NB ? 0 : b + 1;
      }
      if constexpr (!second) bar();
    };
    if (wr == 0)
      run(std::false_type{});
    else
      run(std::true_type{});
    vm_wait<0>();                                             // no DMA is in flight when the buffers get another use
  }

  // Half a tile's results in the order of eight_columns, rows of 1 KB: 16-byte piece c of row r at c ^ (r & 15), no bank conflict in either direction
  static __device__ __forceinline__ void put(unsigned char* sm, const f32x4 (&acc)[2][F][2]) {
    const int lane = threadIdx.x & 63, wc = (threadIdx.x >> 6) & 3, frow = lane & 15, fhi = lane >> 4;
#pragma unroll
    for (int i = 0; i < F; ++i)
#pragma unroll
      for (int h = 0; h < 2; ++h)
#pragma unroll
        for (int j = 0; j < 2; ++j) {
          const int r = 16 * i + frow, c = (128 * h + 32 * wc + 8 * fhi + 4 * j) >> 2;
          *reinterpret_cast<f32x4*>(sm + r * 1024 + 16 * (c ^ frow)) = acc[h][i][j];
        }
  }
  static __device__ __forceinline__ f32x4 get(const unsigned char* sm, int r) {
    return *reinterpret_cast<const f32x4*>(sm + r * 1024 + 16 * ((threadIdx.x & 63) ^ (r & 15)));
  }
};

}  // namespace padd
}  // namespace k8s
