// Matrix products on the gfx950 matrix cores, for sizes from one row to the
// tens of GFLOP: D[m][n] = sum_k A[m][k] B[n][k], fp32 accumulation, an epilogue
// on four consecutive n at a time.
//
// A lane's operand fragment is 16 bytes along k: one 16x16x32 step in 16 bits,
// four 16x16x4 steps in fp32. B's rows are the MFMA's first operand, so a lane
// ends with four consecutive columns n of one row m and stores them together.
#pragma once

#include "mlc_cdna4.h"

namespace mlc {

// This workgroup's (row, column) tile of BATCHES products of MT x NT tiles,
// false past the last one. Workgroups go to the 8 XCDs in turn, so each XCD
// takes a contiguous eighth of the tiles: bands of up to 8 row tiles, columns
// outside rows, so that the tiles of one XCD at a time share few rows of A and
// few of B and find them in its L2. (With whole columns instead, 64 row tiles
// read A from memory once per column: 16384x768x3072 fp16 took 111 us, 73 now.)
template <int BATCHES, int MT, int NT>
__device__ __forceinline__ bool tile_index(int& z, int& mt, int& nt) {
  constexpr int TILES = BATCHES * MT * NT, PER = (TILES + 7) / 8, BAND = MT < 8 ? MT : 8;
  const int i = (int)(blockIdx.x / 8), t = (int)(blockIdx.x % 8) * PER + i;
  if (i >= PER || t >= TILES) return false;
  z = t / (MT * NT);
  const int u = t % (MT * NT), band = u / (BAND * NT), v = u % (BAND * NT);
  const int rows = MT - band * BAND < BAND ? MT - band * BAND : BAND;
  mt = band * BAND + v % rows;
  nt = v / rows;
  return true;
}

template <class T> struct mma_type;
template <> struct mma_type<f16> { typedef half8 frag; };
template <> struct mma_type<bf16> { typedef bf16x8 frag; };
template <> struct mma_type<float> { typedef float4v frag; };

// acc[i] += sum over the fragments' k of b[n = 4 (lane / 16) + i] a[m = lane % 16]
__device__ __forceinline__ float4v mma16(half8 b, half8 a, float4v c) { return mfma_16x16x32(b, a, c); }
__device__ __forceinline__ float4v mma16(bf16x8 b, bf16x8 a, float4v c) { return mfma_16x16x32(b, a, c); }
__device__ __forceinline__ float4v mma16(float4v b, float4v a, float4v c) {
#pragma unroll
  for (int i = 0; i < 4; ++i) c = __builtin_amdgcn_mfma_f32_16x16x4f32(b[i], a[i], c, 0, 0, 0);
  return c;
}

template <class T> __device__ __forceinline__ typename mma_type<T>::frag load_frag(const T* p) {
  return *reinterpret_cast<const typename mma_type<T>::frag*>(p);
}

// 16 bytes per lane from global memory into LDS at ``lds`` + 16 * lane.
__device__ __forceinline__ void load_to_lds(const void* g, void* lds) {
  __builtin_amdgcn_global_load_lds((const __attribute__((address_space(1))) void*)g,
                                   (__attribute__((address_space(3))) void*)lds, 16, 0, 0);
}

// Wait until at most N of this wave's vector-memory operations are in flight,
// and none of its LDS reads: the slot they read may be overwritten next.
template <int N> __device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(N) : "memory");
}

// Tiled form: unit stride along k, 16-byte aligned rows, K a multiple of
// 128 bytes per k-split. One workgroup of WM x WN x WK waves per TM x TN tile:
// WK groups of waves split k, and in a group each wave owns a TM/WM x TN/WN
// part of the tile. A group's operand rows move 128 bytes of k at a time
// straight into its ring of NST LDS stages, NST - 1 stages ahead.
//
// A fragment's 16 rows lie a row pitch apart, so loading it from global memory
// lane by lane costs a cache-line lookup per 16 bytes (15 bytes a clock per CU
// measured); through LDS eight neighbouring lanes take one 128-byte line. In
// LDS the 16-byte slot of row r is xor-ed with r / 2 (on the global side: LDS
// is written in lane order), so 16 lanes reading one slot of 16 rows hit 64
// distinct banks.
//
// Rows past M or N are read from the last row and dropped by the epilogue:
// epi(m, n, four columns of a row), or where ``transposed`` (the same for the
// whole workgroup; without a k-split) epi_t(m, n, four rows of a column).
template <class T, int M, int N, int K, int LDA, int LDB, int TM, int TN, int WM, int WN, int WK,
          int NST, class Epi, class EpiT>
__device__ __forceinline__ void gemm_tile(const T* __restrict__ a, const T* __restrict__ b,
                                          int m0, int n0, Epi epi, bool transposed, EpiT epi_t) {
  typedef typename mma_type<T>::frag frag;
  constexpr int PIECE = 128, BK = PIECE / sizeof(T);     // bytes and elements of k per stage
  constexpr int SLOTS = PIECE / 16, RPL = 64 / SLOTS;  // rows per load instruction
  constexpr int GW = WM * WN;                          // waves per k-group
  constexpr int IT = K / (BK * WK);                    // stages per k-group
  constexpr int ROWS = TM + TN, LPW = ROWS / RPL / GW;
  constexpr int RA = TM / WM / 16, RB = TN / WN / 16;
  static_assert(K % (BK * WK) == 0 && ROWS % (RPL * GW) == 0, "tile split");
  static_assert(TM % (16 * WM) == 0 && TN % (16 * WN) == 0, "wave split");
  constexpr int RING = IT < NST ? IT : NST;
  constexpr int STAGE = ROWS * PIECE;
  constexpr int PART = WK > 1 ? WK * TM * (TN + 4) * 4 : 0;
  constexpr int TW = TN / WN, RP = TW + 4, ROWBUF = 16 * RP;   // floats of a wave's row buffer
  // the column buffer of 16 rows is the larger one in fp32, and more than the
  // ring where k is one stage of a 256 x 256 tile
  constexpr int ROWBUFS = GW * ROWBUF * 4, COLBUFS = GW * TW * 20 * (int)sizeof(T);
  constexpr int EPI = WK > 1 ? PART : ROWBUFS > COLBUFS ? ROWBUFS : COLBUFS;
  constexpr int LDS = WK * RING * STAGE > EPI ? WK * RING * STAGE : EPI;
  // whether the columns of every wave's tile fit at once (16 rows always do)
  constexpr bool COLS = GW * TW * (TM / WM + 4) * (int)sizeof(T) <= LDS;
  __shared__ __attribute__((aligned(1024))) char lds[LDS];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int group = wave / GW, w = wave % GW;
  const int wm = w / WN, wn = w % WN;
  const int r = lane & 15, g = lane >> 4;
  char* const ring = lds + group * RING * STAGE;

  const char* src[LPW];
#pragma unroll
  for (int i = 0; i < LPW; ++i) {
    const int q = w + i * GW, row = q * RPL + lane / SLOTS;
    const int chunk = (lane % SLOTS) ^ (row / (16 / SLOTS) % SLOTS);
    const T* p;
    if (row < TM) {
      const int m = m0 + row;
      p = a + (int64_t)(m < M ? m : M - 1) * LDA;
    } else {
      const int n = n0 + row - TM;
      p = b + (int64_t)(n < N ? n : N - 1) * LDB;
    }
    src[i] = reinterpret_cast<const char*>(p) + group * (IT * PIECE) + chunk * 16;
  }
  auto load = [&](int it) {
    char* dst = ring + (it % RING) * STAGE + w * 1024;
#pragma unroll
    for (int i = 0; i < LPW; ++i) load_to_lds(src[i] + it * PIECE, dst + i * GW * 1024);
  };

  float4v acc[RA][RB];
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < RB; ++j) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};

  const int swz = r / (16 / SLOTS) % SLOTS;
  auto compute = [&](int it) {
    const char* st = ring + (it % RING) * STAGE;
    const char* sa = st + (wm * (TM / WM) + r) * PIECE;
    const char* sb = st + (TM + wn * (TN / WN) + r) * PIECE;
    constexpr int STEPS = PIECE / 64;
    frag fa[STEPS][RA], fb[STEPS][RB];
    auto read = [&](int s) {
      const int at = ((s * 4 + g) ^ swz) * 16;
#pragma unroll
      for (int i = 0; i < RA; ++i) fa[s][i] = *reinterpret_cast<const frag*>(sa + i * 16 * PIECE + at);
#pragma unroll
      for (int j = 0; j < RB; ++j) fb[s][j] = *reinterpret_cast<const frag*>(sb + j * 16 * PIECE + at);
    };
    read(0);
#pragma unroll
    for (int s = 0; s < STEPS; ++s) {
      if (s + 1 < STEPS) read(s + 1);  // in flight during this step's products
#pragma unroll
      for (int i = 0; i < RA; ++i)
#pragma unroll
        for (int j = 0; j < RB; ++j) acc[i][j] = mma16(fb[s][j], fa[s][i], acc[i][j]);
    }
  };
  // one group of one wave needs no barrier: its stages are its own
  auto sync = [&]() {
    if constexpr (GW > 1) __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
  };

  if constexpr (IT <= NST) {
    // the whole of k fits the ring: every load is in flight before the first product
#pragma unroll
    for (int it = 0; it < IT; ++it) load(it);
#pragma unroll
    for (int it = 0; it < IT; ++it) {
      switch (IT - 1 - it) {
        case 0: wait_vm<0>(); break;
        case 1: wait_vm<LPW>(); break;
        case 2: wait_vm<2 * LPW>(); break;
        default: wait_vm<3 * LPW>(); break;
      }
      sync();
      compute(it);
    }
  } else {
#pragma unroll
    for (int it = 0; it < NST - 1; ++it) load(it);
    int it = 0;
    for (; it < IT - (NST - 1); ++it) {
      wait_vm<(NST - 2) * LPW>();
      sync();  // everyone is past stage it - 1, whose slot the next load takes
      load(it + NST - 1);
      compute(it);
    }
#pragma unroll
    for (int t = NST - 2; t >= 0; --t, ++it) {
      switch (t) {
        case 0: wait_vm<0>(); break;
        case 1: wait_vm<LPW>(); break;
        default: wait_vm<2 * LPW>(); break;
      }
      sync();
      compute(it);
    }
  }

  if constexpr (WK == 1) {
    // Through the wave's own LDS, so that neighbouring lanes store neighbouring
    // pieces of a row (or, transposed, of a column). From the accumulators a
    // store covers 32 bytes of each of 16 rows: 16384x2304x768 fp16 took 68 us
    // so, 58 this way; 128x50257x768, whose rows are odd, 26 and 23.
    const int mw = m0 + wm * (TM / WM), nw = n0 + wn * TW;
    __syncthreads();  // the ring is read out
    if (!transposed) {
      float* rows = reinterpret_cast<float*>(lds) + w * ROWBUF;
#pragma unroll
      for (int i = 0; i < RA; ++i) {
#pragma unroll
        for (int j = 0; j < RB; ++j)
          *reinterpret_cast<float4v*>(rows + r * RP + 16 * j + 4 * g) = acc[i][j];
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q0 = 0; q0 < 4 * TW; q0 += 64) {
          const int q = q0 + lane;
          if (4 * TW % 64 != 0 && q >= 4 * TW) continue;
          const int m = q / (TW / 4), n = q % (TW / 4) * 4;
          epi(mw + 16 * i + m, nw + n, *reinterpret_cast<const float4v*>(rows + m * RP + n));
        }
        __builtin_amdgcn_wave_barrier();
      }
    } else {
      // columns of the wave's whole tile, in its storage type (what the
      // epilogue reads of a product): a store covers up to 128 bytes of each,
      // 32 with 16 rows at a time (merged q/k/v of 16384 rows 87 us so, 75 now)
      constexpr int TR = COLS ? TM / WM : 16, CP = TR + 4;
      T* cols = reinterpret_cast<T*>(lds) + w * TW * CP;
#pragma unroll
      for (int i0 = 0; i0 < RA; i0 += TR / 16) {
#pragma unroll
        for (int i = 0; i < TR / 16; ++i)
#pragma unroll
          for (int j = 0; j < RB; ++j)
#pragma unroll
            for (int e = 0; e < 4; ++e)
              st(cols + (16 * j + 4 * g + e) * CP + 16 * i + r, acc[i0 + i][j][e]);
        __builtin_amdgcn_wave_barrier();
#pragma unroll
        for (int q0 = 0; q0 < TW * TR / 4; q0 += 64) {
          const int q = q0 + lane;
          if (TW * TR / 4 % 64 != 0 && q >= TW * TR / 4) continue;
          const int m = q % (TR / 4) * 4, n = q / (TR / 4);
          float c[4];
          load_pack<4>(c, cols + n * CP + m);
          epi_t(mw + 16 * i0 + m, nw + n, float4v{c[0], c[1], c[2], c[3]});
        }
        __builtin_amdgcn_wave_barrier();
      }
    }
  } else {
    constexpr int P = TN + 4;
    float* part = reinterpret_cast<float*>(lds);
    __syncthreads();  // the ring is read out
#pragma unroll
    for (int i = 0; i < RA; ++i)
#pragma unroll
      for (int j = 0; j < RB; ++j)
        *reinterpret_cast<float4v*>(part + (group * TM + wm * (TM / WM) + 16 * i + r) * P
                                    + wn * (TN / WN) + 16 * j + 4 * g) = acc[i][j];
    __syncthreads();
    for (int q = threadIdx.x; q < TM * TN / 4; q += GW * WK * 64) {
      const int m = q / (TN / 4), n = q % (TN / 4) * 4;
      float4v s = *reinterpret_cast<const float4v*>(part + m * P + n);
#pragma unroll
      for (int k = 1; k < WK; ++k) s += *reinterpret_cast<const float4v*>(part + (k * TM + m) * P + n);
      epi(m0 + m, n0 + n, s);
    }
  }
}

// 16 bytes or 4 elements at an address aligned to one element: the hardware
// takes unaligned global accesses, one instruction instead of one an element.
template <class F, class T> __device__ __forceinline__ F load_unaligned(const T* p) {
  F f;
  __builtin_memcpy(&f, p, sizeof(F));
  return f;
}

// One operand's TR x BK tile, global to registers to LDS ([row][k], rows
// padded by 16 bytes). ROWS x K is the operand's extent. Three ways in:
//  * unit stride along k: a lane moves 16 bytes of one row;
//  * 16 bits, unit stride along the rows: a lane loads 16 bytes of eight rows
//    at two neighbouring k and writes eight pairs;
//  * otherwise a lane gathers 16 bytes along k, neighbouring lanes
//    neighbouring rows.
// Past the extent: a valid row again, zeros along k.
template <class T, int ROWS, int K, int SR, int SK, int TR, int BK, int THREADS, bool ALIGNED>
struct tile_loader {
  typedef typename mma_type<T>::frag frag;
  static constexpr int E = 16 / sizeof(T), PITCH = BK + E;
  static constexpr bool PAIRS = sizeof(T) == 2 && SK != 1 && SR == 1;
  static constexpr int LOADS = PAIRS ? 2 : 1;       // fragments a lane holds per piece
  static constexpr int PIECES = TR * (BK / E) / LOADS, PER = (PIECES + THREADS - 1) / THREADS;
  union word { frag f; T x[E]; };
  word v[PER][LOADS];
  __device__ __forceinline__ static void where(int id, int& row, int& k) {
    if constexpr (PAIRS) {
      row = id % (TR / E) * E;
      k = id / (TR / E) * 2;
    } else if constexpr (SK == 1) {
      row = id / (BK / E);
      k = id % (BK / E) * E;
    } else {
      row = id % TR;
      k = id / TR * E;
    }
  }
  __device__ __forceinline__ void load(const T* __restrict__ p, int row0, int k0) {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int id = u * THREADS + threadIdx.x;
      if (PIECES % THREADS != 0 && id >= PIECES) continue;
      int row, k;
      where(id, row, k);
      row += row0;
      k += k0;
      if constexpr (PAIRS) {
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          word w;
          w.f = frag{};
          if (K % BK == 0 || k + h < K) {
            const T* q = p + (int64_t)(k + h) * SK;
            if (ROWS % TR == 0 || row + E <= ROWS) {
              w.f = ALIGNED ? load_frag<T>(q + row) : load_unaligned<frag>(q + row);
            } else {
#pragma unroll
              for (int i = 0; i < E; ++i) w.x[i] = q[row + i < ROWS ? row + i : ROWS - 1];
            }
          }
          v[u][h] = w;
        }
      } else {
        row = row < ROWS ? row : ROWS - 1;
        const T* q = p + (int64_t)row * SR + (int64_t)k * SK;
        word w;
        w.f = frag{};
        if (SK == 1 && (K % BK == 0 || k + E <= K)) {
          w.f = ALIGNED ? load_frag<T>(q) : load_unaligned<frag>(q);
        } else {
#pragma unroll
          for (int i = 0; i < E; ++i)
            if (K % BK == 0 || k + i < K) w.x[i] = q[(int64_t)i * SK];
        }
        v[u][0] = w;
      }
    }
  }
  __device__ __forceinline__ void store(T (*lds)[PITCH]) const {
#pragma unroll
    for (int u = 0; u < PER; ++u) {
      const int id = u * THREADS + threadIdx.x;
      if (PIECES % THREADS != 0 && id >= PIECES) continue;
      int row, k;
      where(id, row, k);
      if constexpr (PAIRS) {
#pragma unroll
        for (int i = 0; i < E; ++i)
          *reinterpret_cast<pack<T, 2>*>(&lds[row + i][k]) = pack<T, 2>{{v[u][0].x[i], v[u][1].x[i]}};
      } else {
        *reinterpret_cast<frag*>(&lds[row][k]) = v[u][0].f;
      }
    }
  }
};

// Staged form: any strides, sizes and alignments. Four waves, 2 x 2 over the
// TM x TN tile; both operands pass through LDS in BK steps, the next step's
// loads in flight during this step's products.
template <class T, int M, int N, int K, int SAM, int SAK, int SBN, int SBK, int TM, int TN, int BK,
          bool ALIGN_A, bool ALIGN_B, class Epi>
__device__ __forceinline__ void gemm_staged(const T* __restrict__ a, const T* __restrict__ b,
                                            int m0, int n0, Epi epi) {
  typedef typename mma_type<T>::frag frag;
  constexpr int E = 16 / sizeof(T), S = 4 * E, P = BK + E;
  constexpr int RA = TM / 32, RB = TN / 32;
  __shared__ __attribute__((aligned(16))) T la[TM][P];
  __shared__ __attribute__((aligned(16))) T lb[TN][P];
  tile_loader<T, M, K, SAM, SAK, TM, BK, 256, ALIGN_A> ga;
  tile_loader<T, N, K, SBN, SBK, TN, BK, 256, ALIGN_B> gb;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int r = lane & 15, g = lane >> 4;
  const int wm = (wave >> 1) * (TM / 2), wn = (wave & 1) * (TN / 2);
  float4v acc[RA][RB];
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < RB; ++j) acc[i][j] = float4v{0.0f, 0.0f, 0.0f, 0.0f};
  ga.load(a, m0, 0);
  gb.load(b, n0, 0);
  for (int k0 = 0; k0 < K; k0 += BK) {
    if (k0) __syncthreads();
    ga.store(la);
    gb.store(lb);
    __syncthreads();
    if (k0 + BK < K) {
      ga.load(a, m0, k0 + BK);
      gb.load(b, n0, k0 + BK);
    }
#pragma unroll
    for (int s = 0; s < BK / S; ++s) {
      frag fa[RA], fb[RB];
#pragma unroll
      for (int i = 0; i < RA; ++i) fa[i] = *reinterpret_cast<const frag*>(&la[wm + 16 * i + r][s * S + g * E]);
#pragma unroll
      for (int j = 0; j < RB; ++j) fb[j] = *reinterpret_cast<const frag*>(&lb[wn + 16 * j + r][s * S + g * E]);
#pragma unroll
      for (int i = 0; i < RA; ++i)
#pragma unroll
        for (int j = 0; j < RB; ++j) acc[i][j] = mma16(fb[j], fa[i], acc[i][j]);
    }
  }
#pragma unroll
  for (int i = 0; i < RA; ++i)
#pragma unroll
    for (int j = 0; j < RB; ++j) epi(m0 + wm + 16 * i + r, n0 + wn + 16 * j + 4 * g, acc[i][j]);
}

// A product as its storage type T holds it, in an fp32 register.
template <class T> __device__ __forceinline__ float ld_of(float x) { return x; }
template <> __device__ __forceinline__ float ld_of<f16>(float x) { return round_f16(x); }
template <> __device__ __forceinline__ float ld_of<bf16>(float x) { return round_bf16(x); }

// Four consecutive columns of one row, dropped past M and N, in one store
// except at the end of a row.
template <class T, int M, int N, int LDC, bool ALIGNED>
__device__ __forceinline__ void store4(T* __restrict__ c, int m, int n, const float (&v)[4]) {
  if (m >= M || n >= N) return;
  T* p = c + (int64_t)m * LDC + n;
  if constexpr (ALIGNED) {
    store_pack<4>(p, v);
  } else if (n + 4 <= N) {
    const pack<T, 4> w = {{cvt<T>(v[0]), cvt<T>(v[1]), cvt<T>(v[2]), cvt<T>(v[3])}};
    __builtin_memcpy(p, &w, sizeof(w));
  } else {
#pragma unroll
    for (int i = 0; i < 4; ++i)
      if (n + i < N) st(p + i, v[i]);
  }
}

}  // namespace mlc
