// float32 GEMM on the bf16 matrix cores: C(m, n) = Σ_k A(m, k)·B(n, k), every product taken
// at float32 accuracy. Shared by the forward projections (ops_gemm.hip) and the backward
// products (ops_train.hip).
//
// Each operand value is split as x = x0 + x1 + x2 with x0 = bf16(x), x1 = bf16(x − x0),
// x2 = bf16(x − x0 − x1), all rounded to nearest: 8 + 8 + 8 significand bits and the signs
// hold the 24 bits of x exactly. (x is multiplied by kLift = 2^16 first and the sums by 2^-32 at the
// end, so that this holds for every float32: the last bit of the smallest, 2^-149, becomes bf16's
// smallest value. As they are, values below 2^-109 lose parts; at 2^-120 an output's error was
// 3.5e-5. A value from 2^112 on or an output from 2^96 on then overflows, see below. It costs
// 0.8 % of a product.) Of the nine products the six
//   x0·y0 + x0·y1 + x1·y0 + x0·y2 + x2·y0 + x1·y1
// are summed in float32 on v_mfma_f32_32x32x16_bf16; the dropped ones (x1·y2, x2·y1,
// x2·y2) are below 2^-25 of |x·y|, under the rounding of a single float32 product. A
// float32 MFMA adds k two at a time into its accumulator, this one sixteen at a time, and
// every kChunk stages the accumulators are added to a second set, so the sums see fewer
// roundings (relative error against 64 bits on unit-normal operands, the float32 MFMA's
// in brackets: K 64 7.4e-8 (1.4e-7), K 1024 2.4e-7 (5.7e-7), K 32000 2.8e-7 (3.2e-6)).
// An infinity, or a value that rounds up to one in bf16, makes an output NaN or infinite
// that float32 arithmetic may not; so every non-finite output is taken from the float32 MFMA
// over its k range instead (tile_f32).
//
// Why: the float32 MFMA peaks at 157 TFLOP/s, the bf16 one at 2.5 PFLOP/s, a sixth of which
// is 417. Measured, 4096 rows, a float32 MFMA kernel of the same tile and this one: N = K = 1024
// 94 → 53 µs (162 TFLOP/s), N 4096 317 → 222 (155), K 4096 343 → 203 (169), the 32000-row tied
// head's loss 2484 → 1636. What bounds it: the matrix unit is busy 55 % of the cycles (the head, counters), at the
// 1.5 to 1.8 GHz that the chip holds under this load; of the rest, without the split the same
// loop runs 1.3 times as fast, and the vector work (6.8 instructions an MFMA) hides under the
// MFMAs only in part. The 128 × 128 tile holds all 256 registers and spills 16 to 21.
//
// A workgroup of WM·WN·WK waves owns a TM × TN tile; a wave TM/WM × TN/WN of it and, of the
// two 16-wide k steps of a stage, one (the two partial tiles are summed through LDS at
// the end). Stages of 32 k: the values are loaded into registers two stages ahead, split
// beside the MFMAs of the stage before their own, and stored as three bf16 planes of 64-byte
// rows into the LDS buffer that is not being multiplied; one barrier a stage.
// Operands k-contiguous (KC: element (r, k) at p[r·ld + k]) or not (p[k·ld + r]).
#pragma once

#include <type_traits>

#include "gemm_big.hpp"

namespace nml {
namespace x3 {

typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));

constexpr int kK = 32;      // k per stage
constexpr int kChunk = 16;  // stages summed in one accumulator
constexpr float kLift = 0x1p16f;
// 128 × 128 tiles (one workgroup per CU) from this many of them on, 64 × 64 tiles (three
// per CU) below: N = K = 1024, 128 of the large tiles 43.2 µs against 34.9 with the small, 192
// 46.8 against 47.4, 256 51.4 against 62.9.
constexpr long long kLargeTiles = 192;

struct Operand {
  const float* p;
  long long ld;
};

// Byte offset of the 16-byte chunk c (k 8c … 8c + 7) of tile row `row` in a plane. The 16
// lanes of a fragment read (16 consecutive rows, one chunk) and of a store (the same, or 4
// rows × 4 chunks) each cover the 64 banks once.
__device__ __forceinline__ uint32_t plane_off(int row, int c) {
  return static_cast<uint32_t>(row * 64 + ((c ^ ((row >> 2) & 3)) << 4));
}

// bf16(x0) and bf16(x1) packed, low and high half (round to nearest even).
__device__ __forceinline__ uint32_t cvt_pk(float x0, float x1) {
  uint32_t h;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(h) : "v"(x0), "v"(x1));
  return h;
}

template <int TM, int TN, int WM, int WN, int WK>
struct Shape {
  static constexpr int Threads = 64 * WM * WN * WK;
  static constexpr int MI = TM / WM / 32, NJ = TN / WN / 32;
  static constexpr int Plane = (TM + TN) * 64;  // A's rows, then B's
  static constexpr int Stage = 3 * Plane;
  static constexpr size_t Flag = 2 * static_cast<size_t>(Stage);  // one int: a non-finite output
  static constexpr size_t Lds = Flag + 16;
  static_assert(MI >= 1 && NJ >= 1 && WK == 2, "tile");
  static_assert(static_cast<size_t>(TM) * (TN + 1) * 4 <= Flag, "the WK sum and tile_f32's go through LDS");
};

// The values of one operand of R rows that this thread stages. KC: 4 k of a row per task, 8
// lanes a row (whole 128-byte lines per load); else 8 k of a row, 64 lanes taking 64
// neighbouring rows at each k (256 contiguous bytes per load). NEG: the stage's second 16 k
// are stored negated. All are stored times kLift. Two stages' values are held, by the stage's
// parity.
template <bool KC, int R, int T, bool NEG>
struct Stager {
  static constexpr int V = KC ? 4 : 8;
  static constexpr int Tasks = R * (kK / V) / T;
  static constexpr int Pairs = Tasks * V / 2, Slices = 3 * Pairs;
  static_assert(Tasks >= 1 && Tasks * T == R * (kK / V) && R % 64 == 0, "whole tasks per thread");
  float v[2][Tasks][V];
  uint32_t part[3][V / 2];  // the current task's parts, packed in pairs
  const float* base;        // the tile's first row at k 0 (uniform)
  uint32_t off[Tasks];      // this task's element past it (rows past the last: the last row,
                            // whose outputs nobody stores)
  uint32_t dst;             // task 0's bytes in a plane; task i's are Step·i further
  float lift;               // ±kLift (every task's k are the same)
  static constexpr int Step = KC ? T / 8 * 64 : 0;
  static_assert(KC ? (T / 8) % 16 == 0 : Tasks == 1, "tasks differ by whole swizzle periods");

  static __device__ __forceinline__ int row_of(int i) {
    const int id = static_cast<int>(threadIdx.x) + T * i;
    return KC ? id >> 3 : id % R;
  }
  static __device__ __forceinline__ int k_of(int i) {
    const int id = static_cast<int>(threadIdx.x) + T * i;
    return KC ? (id & 7) * 4 : id / R * 8;
  }

  __device__ __forceinline__ Stager(Operand o, int r0, int rows) {
    base = o.p + (KC ? r0 * o.ld : static_cast<long long>(r0));
#pragma unroll
    for (int i = 0; i < Tasks; ++i) {
      const uint32_t r = min(row_of(i), rows - 1 - r0), k = k_of(i), ld = static_cast<uint32_t>(o.ld);
      off[i] = KC ? r * ld + k : k * ld + r;
    }
    const uint32_t k = k_of(0);
    dst = plane_off(row_of(0), k / 8) + (KC ? (k & 4) * 2 : 0);
    lift = k & 16 ? -kLift : kLift;
  }

  // a whole stage from k0
  template <int P>
  __device__ __forceinline__ void load(Operand o, int k0) {
    const float* q = base + (KC ? static_cast<long long>(k0) : k0 * o.ld);
#pragma unroll
    for (int i = 0; i < Tasks; ++i) {
      if constexpr (KC) {
        const floatx4 x = *reinterpret_cast<const floatx4*>(q + off[i]);
#pragma unroll
        for (int e = 0; e < 4; ++e) v[P][i][e] = x[e];
      } else {
#pragma unroll
        for (int e = 0; e < V; ++e) v[P][i][e] = (q + e * o.ld)[off[i]];
      }
    }
  }

  // the stage from k0 that ends at kend: zero from there on
  template <int P>
  __device__ __forceinline__ void load_tail(Operand o, int k0, int kend) {
    const float* q = base + (KC ? static_cast<long long>(k0) : k0 * o.ld);
#pragma unroll
    for (int i = 0; i < Tasks; ++i) {
      const int left = kend - k0 - k_of(i);  // values in range
#pragma unroll
      for (int e = 0; e < V; ++e) v[P][i][e] = e < left ? (KC ? q + e : q + e * o.ld)[off[i]] : 0.f;
    }
  }

  // The split of parity P's values in Slices steps: step 3·pair + p takes part p of one pair;
  // a task's last step stores its three parts at lds (this operand's rows of plane 0),
  // `plane` bytes apart.
  template <int P>
  __device__ __forceinline__ void slice(int n, char* lds, int plane) {
#pragma clang fp contract(off)
    const int i = n / 3 / (V / 2), e = n / 3 % (V / 2), p = n % 3;
    float& v0 = v[P][i][2 * e];
    float& v1 = v[P][i][2 * e + 1];
    if (p == 0) {
      v0 *= NEG ? lift : kLift;
      v1 *= NEG ? lift : kLift;
    }
    const uint32_t h = cvt_pk(v0, v1);
    part[p][e] = h;
    if (p < 2) {
      v0 -= __uint_as_float(h << 16);
      v1 -= __uint_as_float(h & 0xffff0000u);
    } else if (e == V / 2 - 1) {
#pragma unroll
      for (int q = 0; q < 3; ++q) {
        typedef uint32_t vec __attribute__((ext_vector_type(V / 2)));
        vec x;
#pragma unroll
        for (int u = 0; u < V / 2; ++u) x[u] = part[q][u];
        *reinterpret_cast<vec*>(lds + (q * plane + Step * i) + dst) = x;
      }
    }
  }
};

// The tile's products on the float32 MFMA, k two at a time, left in lds as [row][TN + 1]: the
// slow path of a tile with a non-finite output. Stages of 32 k in rows of 33 floats, the next
// one's values in registers meanwhile; each wave takes G 32 × 32 blocks. A product of
// non-finite outputs takes 2.7 times a finite one (4096 × 1024 × 1024: 142 µs against 53; with a
// lane forming each of its outputs by itself 7.6 ms), one non-finite row 2.4 times.
template <int TM, int TN, int T, bool A_KC, bool B_KC>
__device__ __forceinline__ void tile_f32(Operand a, Operand b, int M, int N, int m0, int n0, int kbeg, int kend,
                                         float* lds) {
  constexpr int BN = TN / 32, G = TM / 32 * BN / (T / 64), P = kK + 1;
  constexpr int RA = TM * kK / T, RB = TN * kK / T;  // values per thread and stage
  static_assert(G >= 1 && BN % G == 0, "a wave's blocks lie in one row of blocks");
  const int tid = threadIdx.x, lane = tid & 63;
  const int first = __builtin_amdgcn_readfirstlane(tid >> 6) * G, bm = first / BN * 32, bn = first % BN * 32;
  floatx16 acc[G];
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[g][r] = 0.f;
  float va[RA], vb[RB];
  // value i of this thread: tile row and k, neighbouring lanes along the contiguous extent
  auto row_of = [&](bool kc, int R, int i) { return kc ? (tid + T * i) / kK : (tid + T * i) % R; };
  auto k_of = [&](bool kc, int R, int i) { return kc ? (tid + T * i) % kK : (tid + T * i) / R; };
  auto fetch = [&](int k0) {
#pragma unroll
    for (int i = 0; i < RA; ++i) {
      const int m = m0 + row_of(A_KC, TM, i), k = k0 + k_of(A_KC, TM, i);
      va[i] = m < M && k < kend ? a.p[A_KC ? m * a.ld + k : k * a.ld + m] : 0.f;
    }
#pragma unroll
    for (int i = 0; i < RB; ++i) {
      const int n = n0 + row_of(B_KC, TN, i), k = k0 + k_of(B_KC, TN, i);
      vb[i] = n < N && k < kend ? b.p[B_KC ? n * b.ld + k : k * b.ld + n] : 0.f;
    }
  };
  fetch(kbeg);
  for (int k0 = kbeg; k0 < kend; k0 += kK) {
    __syncthreads();  // every wave is done with the stage before
#pragma unroll
    for (int i = 0; i < RA; ++i) lds[row_of(A_KC, TM, i) * P + k_of(A_KC, TM, i)] = va[i];
#pragma unroll
    for (int i = 0; i < RB; ++i) lds[(TM + row_of(B_KC, TN, i)) * P + k_of(B_KC, TN, i)] = vb[i];
    __syncthreads();
    if (k0 + kK < kend) fetch(k0 + kK);
#pragma unroll 4
    for (int kk = 0; kk < kK; kk += 2) {
      const int k = kk + (lane >> 5);
      const float x = lds[(bm + (lane & 31)) * P + k];
#pragma unroll
      for (int g = 0; g < G; ++g)
        acc[g] = __builtin_amdgcn_mfma_f32_32x32x2f32(x, lds[(TM + bn + 32 * g + (lane & 31)) * P + k], acc[g], 0, 0, 0);
    }
  }
  __syncthreads();
#pragma unroll
  for (int g = 0; g < G; ++g)
#pragma unroll
    for (int r = 0; r < 16; ++r)
      lds[(bm + 8 * (r >> 2) + 4 * (lane >> 5) + (r & 3)) * (TN + 1) + bn + 32 * g + (lane & 31)] = acc[g][r];
  __syncthreads();
}

// One workgroup's tile at (m0, n0) over k in [kbeg, kend); epi(m, n, value) is called for
// every element below M, N. lds: Shape::Lds bytes.
template <int TM, int TN, int WM, int WN, int WK, bool A_KC, bool B_KC, typename Epi>
__device__ __forceinline__ void tile(Operand a, Operand b, int M, int N, int m0, int n0, int kbeg, int kend,
                                     char* lds, Epi epi) {
  typedef Shape<TM, TN, WM, WN, WK> Sh;
  constexpr int MI = Sh::MI, NJ = Sh::NJ, T = Sh::Threads;
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wk = wave / (WM * WN), wm = (wave / WN) % WM, wn = wave % WN;
  floatx16 acc[MI][NJ], tot[MI][NJ];
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[i][j][r] = tot[i][j][r] = 0.f;

  typedef Stager<A_KC, TM, T, true> SA;
  typedef Stager<B_KC, TN, T, false> SB;
  SA sa(a, m0, M);
  SB sb(b, n0, N);
  int* flag = reinterpret_cast<int*>(lds + Sh::Flag);
  if (tid == 0) *flag = 0;
  constexpr int kSlices = SA::Slices + SB::Slices, kMfma = 6 * MI * NJ;
  // Multiplies the stage in buffer P (k step wk) and, with NEXT, splits parity P ^ 1's values
  // into the other buffer, a few instructions of the split behind each MFMA: the vector
  // unit works in the 32 cycles that an MFMA holds the matrix unit only on instructions
  // of the same wave (two waves, one splitting while the other multiplied, took the sum
  // of both times).
  auto stage = [&](auto par_c, auto next_c) {
    constexpr int P = decltype(par_c)::value;
    constexpr bool NEXT = decltype(next_c)::value;
    const char* buf = lds + P * Sh::Stage;
    char* out = lds + (P ^ 1) * Sh::Stage;
    const int c = 2 * wk + (lane >> 5);
    bf16x8 fa[MI][3], fb[NJ][3];
    constexpr int order[3] = {1, 0, 2}, orderb[3] = {1, 2, 0};
#pragma unroll
    for (int p = 0; p < 3; ++p) {
#pragma unroll
      for (int i = 0; i < MI; ++i)
        fa[i][order[p]] = *reinterpret_cast<const bf16x8*>(
            buf + order[p] * Sh::Plane + plane_off(wm * (TM / WM) + 32 * i + (lane & 31), c));
#pragma unroll
      for (int j = 0; j < NJ; ++j)
        fb[j][orderb[p]] = *reinterpret_cast<const bf16x8*>(
            buf + orderb[p] * Sh::Plane + TM * 64 + plane_off(wn * (TN / WN) + 32 * j + (lane & 31), c));
    }
    constexpr int pa[6] = {1, 0, 2, 1, 0, 0}, pb[6] = {1, 2, 0, 0, 1, 0};  // smallest first
    int n = 0;
#pragma unroll
    for (int q = 0; q < 6; ++q)
#pragma unroll
      for (int i = 0; i < MI; ++i)
#pragma unroll
        for (int j = 0; j < NJ; ++j) {
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fa[i][pa[q]], fb[j][pb[q]], acc[i][j], 0, 0, 0);
          if constexpr (NEXT) {
            const int upto = ((q * MI + i) * NJ + j + 1) * kSlices / kMfma;
#pragma unroll
            for (int u = 0; u < (kSlices + kMfma - 1) / kMfma; ++u)
              if (n < upto) {
                if (n < SA::Slices)
                  sa.template slice<P ^ 1>(n, out, Sh::Plane);
                else
                  sb.template slice<P ^ 1>(n - SA::Slices, out + TM * 64, Sh::Plane);
                ++n;
              }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
  };
  auto split_all = [&](auto par_c) {  // parity P's values into buffer P
    constexpr int P = decltype(par_c)::value;
#pragma unroll
    for (int n = 0; n < SA::Slices; ++n) sa.template slice<P>(n, lds + P * Sh::Stage, Sh::Plane);
#pragma unroll
    for (int n = 0; n < SB::Slices; ++n) sb.template slice<P>(n, lds + P * Sh::Stage + TM * 64, Sh::Plane);
  };
  const int S = (kend - kbeg) / kK;  // whole stages
  // stage s (past the last: the last again, no branch around the loads)
  auto load = [&](auto par_c, int s) {
    constexpr int P = decltype(par_c)::value;
    const int k0 = kbeg + min(s, S - 1) * kK;
    sa.template load<P>(a, k0);
    sb.template load<P>(b, k0);
  };
  auto flush = [&]() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          tot[i][j][r] += acc[i][j][r];
          acc[i][j][r] = 0.f;
        }
  };
  using P0 = std::integral_constant<int, 0>;
  using P1 = std::integral_constant<int, 1>;
  if (S > 0) {
    load(P0{}, 0);
    load(P1{}, 1);
    split_all(P0{});
    __syncthreads();
    int s = 0;
    for (; s + 2 < S; s += 2) {
      load(P0{}, s + 2);
      stage(P0{}, std::true_type{});
      __syncthreads();
      load(P1{}, s + 3);
      stage(P1{}, std::true_type{});
      if ((s + 2) % kChunk == 0) flush();
      __syncthreads();
    }
    if (s + 1 < S) {
      stage(P0{}, std::true_type{});
      __syncthreads();
      stage(P1{}, std::false_type{});
    } else {
      stage(P0{}, std::false_type{});
    }
    __syncthreads();
  }
  if (kbeg + S * kK < kend) {  // the last, partial stage
    sa.template load_tail<0>(a, kbeg + S * kK, kend);
    sb.template load_tail<0>(b, kbeg + S * kK, kend);
    split_all(P0{});
    __syncthreads();
    stage(P0{}, std::false_type{});
    __syncthreads();
  }
  flush();
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j) acc[i][j] = tot[i][j];

  if constexpr (WK == 2) {
    // Wave pairs (wk 0, wk 1) hold partial sums of the same tile, wk 1's of the negated
    // products (the second 16 k of A's stages are): each passes the other one half of its 16-register groups and finishes the
    // rest. (The bf16 MFMA's sums fall slightly towards −∞: mean error −2.5e-8 on 1024-term
    // sums of magnitude 0.6, the same in every row, which a column sum over 4096 rows
    // turned into 2.5e-5 of its value; with one half negated the falls cancel, 2e-6 against
    // the float32 MFMA's 4e-6.)
    float* x = reinterpret_cast<float*>(lds);
    const int pair = wave % (WM * WN);
    constexpr int G = MI * NJ;  // 32 × 32 tiles
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int r = 0; r < 8; ++r)
        x[((pair * G + g) * 16 + (wk ? r : 8 + r)) * 64 + lane] =
            wk ? acc[g / NJ][g % NJ][r] : acc[g / NJ][g % NJ][8 + r];
    __syncthreads();
#pragma unroll
    for (int g = 0; g < G; ++g)
#pragma unroll
      for (int r = 0; r < 8; ++r) {
        const float o = x[((pair * G + g) * 16 + (wk ? 8 + r : r)) * 64 + lane];
        if (wk)
          acc[g / NJ][g % NJ][8 + r] = o - acc[g / NJ][g % NJ][8 + r];
        else
          acc[g / NJ][g % NJ][r] -= o;
      }
  }
  // D layout of a 32×32 MFMA tile: lane l, register r → row 8(r/4) + 4(l/32) + r%4, col l%32.
  const int mb = m0 + wm * (TM / WM) + 4 * (lane >> 5), nb = n0 + wn * (TN / WN) + (lane & 31);
  constexpr int RN = 16 / WK;  // registers of a tile this wave finishes, from r0
  const int r0 = WK == 2 ? wk * 8 : 0;
  // This wave's outputs, and whether any is not finite: z stays 0 (a row past the last is a copy
  // of the last).
  float out[MI * NJ * RN], z = 0.f;
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < RN; ++r) {
        float v = acc[i][j][r];
        if constexpr (WK == 2) v = wk ? acc[i][j][8 + r] : v;
        v *= 1.f / kLift / kLift;
        out[(i * NJ + j) * RN + r] = v;
        z = __builtin_fmaf(v, 0.f, z);
      }
  // (asked before the stores, which the barrier would wait for)
  if (z != 0.f) *flag = 1;
  __syncthreads();
  if (*flag) {
    float* f32 = reinterpret_cast<float*>(lds);
    tile_f32<TM, TN, T, A_KC, B_KC>(a, b, M, N, m0, n0, kbeg, kend, f32);
#pragma unroll
    for (int e = 0; e < MI * NJ * RN; ++e) {
      const int t = e / RN, r = r0 + e % RN;
      const int m = mb + 32 * (t / NJ) + 8 * (r >> 2) + (r & 3) - m0, n = nb + 32 * (t % NJ) - n0;
      if (!__builtin_isfinite(out[e])) out[e] = f32[m * (TN + 1) + n];
    }
  }
#pragma unroll
  for (int e = 0; e < MI * NJ * RN; ++e) {
    const int t = e / RN, r = r0 + e % RN;
    const int m = mb + 32 * (t / NJ) + 8 * (r >> 2) + (r & 3), n = nb + 32 * (t % NJ);
    if (m < M && n < N) epi(m, n, out[e]);
  }
}

}  // namespace x3
}  // namespace nml
