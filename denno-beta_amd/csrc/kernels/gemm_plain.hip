#include "gemm_common.h"

// ---------------------------------------------------------------------------------------
// The plain product: 32-bit arithmetic for any dtype, one order of summation for every element
// whatever M is, so that logits do not depend on how a step was cut: K goes in segments of SEG; a
// segment's sum runs k ascending from zero, one fused multiply-add a step; the segments' sums are
// added in ascending order, starting from zero.  Three kernels keep to it.  Many rows (M > 64): 64 x 64
// tiles on the matrix cores, a workgroup walks all of K.  Up to 16 rows (`chain_takes`): 8 or 16 columns
// and all of K a workgroup, on the matrix cores too.  Else: a tile of 8 to 64 rows x 64 columns, and where the
// column tiles alone do not fill the chip every segment is a workgroup of its own, which asks for its
// whole share of W (64 x 128: 32 KB) at once and leaves its sum in a workspace; a second kernel adds
// the segments' sums in order and ends with the epilogue.  (Few rows used to run in the many-rows
// kernel: a hundred workgroups, each walking all of K alone.)
// ---------------------------------------------------------------------------------------
namespace plain {
constexpr int BM = 64, BN = 64, PAD = 4;
constexpr int SEG = 128;

template <typename TC>
__device__ __forceinline__ void finish(float v, int m, int n, const float* bias, TC* C, int ldc, float* resid, int ldr,
                                       int epi) {
  if (bias) v += bias[n];
  if (resid) {
    float* r = resid + static_cast<size_t>(m) * ldr + n;
    *r = *r + v;
  } else {
    C[static_cast<size_t>(m) * ldc + n] = from_float<TC>(apply_epilogue(v, epi));
  }
}

typedef float f32x16 __attribute__((ext_vector_type(16)));

// Many rows.  v_mfma_f32_32x32x2_f32 adds its two products to the sum one after the other, k ascending, each with one
// rounding, subnormals kept: the same bits as the chain of fused multiply-adds that `rows_kernel` runs, at twice the rate of
// the vector unit's single 32-bit multiply-adds (157 against 79 TFLOP/s on the card), which bounded this kernel while it used
// them: the 97 products of a GPT-2 Medium step of 2,048 rows took 242 us on average and take 142 now (62 -> 105 TFLOP/s; the
// matrix cores are busy three quarters of the largest one's time, the rest is waits for operands at the barriers).
// A workgroup's tile is 64 x 64, a wave's 32 x 32: small, because operands are cheap here (two numbers a lane for 64
// cycles of matrix work) and with four workgroups a CU a product of 1,024 columns still gives every CU two tiles.
// Slabs of 32 along K wait in registers while the slab before is multiplied, and lie in LDS with every eight k of a row in
// the order 0 2 4 6 1 3 5 7: a lane (row l % 32, k = 2 s + l / 32) then reads its four steps' numbers in one 16-byte load;
// rows 36 floats apart meet the banks evenly.  (Slabs of 16 in three buffers, the next one's operands read ahead: 149 us.)
// WHOLE: K is a multiple of 4, so four elements along K are all inside or all outside.
constexpr int LK = 32, LLD = LK + 4;

// Eight numbers along K of a row.  What lies beyond K is read from inside the row instead (a load behind a condition would be
// waited for where the paths meet, before the matrix instructions and not behind them) and zeroed by `lay8`.
template <typename TI, bool WHOLE>
__device__ __forceinline__ void load8(const TI* __restrict__ row, int k, int K, TI* v) {
  if (WHOLE) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const TI* p = row + min(k + 4 * h, K - 4);
#pragma unroll
      for (int i = 0; i < 4; ++i) v[4 * h + i] = p[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = row[min(k + i, K - 1)];
  }
}

template <typename TI>
__device__ __forceinline__ void lay8(float* at, const TI* v, int inside) {
  float f[8];
#pragma unroll
  for (int i = 0; i < 8; ++i) f[i] = i < inside ? to_float(v[i]) : 0.f;
  *reinterpret_cast<float4*>(at) = float4{f[0], f[2], f[4], f[6]};
  *reinterpret_cast<float4*>(at + 4) = float4{f[1], f[3], f[5], f[7]};
}

// SHORT: K of at most 64, a slab or two: nothing to overlap inside a workgroup, so a slab is loaded, laid down and multiplied, in half of the LDS, and eight
// workgroups a CU hide each other's waits.  (With slabs asked for that are not there, and four workgroups a CU, the long walk's kernel takes 40.3 us for 2,048 x
// 8,192 x 16 in bfloat16, 11.6 for 1 x 50,257 x 33; single multiply-adds took 32.5 and 9.0, this takes 30.9 and 9.5.)
template <typename TI, typename TC, bool WHOLE, bool SHORT>
__global__ __launch_bounds__(256, SHORT ? 8 : 4) void gemm_kernel(const TI* __restrict__ A, int lda, const TI* __restrict__ W,
                                                       const float* __restrict__ bias, TC* __restrict__ C, int ldc,
                                                       float* __restrict__ resid, int ldr, int M, int N, int K,
                                                       int epi, int mtiles, int tiles, int per_xcd) {
  __shared__ __attribute__((aligned(16))) float As[SHORT ? 1 : 2][BM * LLD];
  __shared__ __attribute__((aligned(16))) float Ws[SHORT ? 1 : 2][BN * LLD];
  // each of the 8 XCDs, among which workgroups go round, takes a run of tiles, rows first: its L2 then serves a few column
  // tiles' weights and the rows
  const int tile = static_cast<int>(blockIdx.x % 8) * per_xcd + static_cast<int>(blockIdx.x / 8);
  if (tile >= tiles) return;
  const int t = threadIdx.x, lane = t % 64, wave = t / 64;
  const int m0 = tile % mtiles * BM, n0 = tile / mtiles * BN;
  const int lrow = t / 4, lk = (t % 4) * 8;             // loader: 64 rows x 4 groups of 8 k
  // (rows beyond M and N: the last one again; what they give is not stored)
  const TI* arow = A + static_cast<size_t>(min(m0 + lrow, M - 1)) * lda;
  const TI* wrow = W + static_cast<size_t>(min(n0 + lrow, N - 1)) * K;
  const int wm = wave / 2 * 32, wn = wave % 2 * 32;
  const int fa = (wm + lane % 32) * LLD + 4 * (lane / 32), fw = (wn + lane % 32) * LLD + 4 * (lane / 32);
  f32x16 acc, tot;
#pragma unroll
  for (int r = 0; r < 16; ++r) acc[r] = tot[r] = 0.f;
  TI av[8], wv[8];
  if constexpr (SHORT) {
    for (int k0 = 0; k0 < K; k0 += LK) {
      load8<TI, WHOLE>(arow, k0 + lk, K, av);
      load8<TI, WHOLE>(wrow, k0 + lk, K, wv);
      if (k0 > 0) __syncthreads();
      lay8(&As[0][lrow * LLD + lk], av, K - k0 - lk);
      lay8(&Ws[0][lrow * LLD + lk], wv, K - k0 - lk);
      __syncthreads();
#pragma unroll
      for (int g = 0; g < LK / 8; ++g) {
        const float4 a = *reinterpret_cast<const float4*>(&As[0][fa + 8 * g]), w = *reinterpret_cast<const float4*>(&Ws[0][fw + 8 * g]);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.x, w.x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.y, w.y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.z, w.z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a.w, w.w, acc, 0, 0, 0);
      }
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) tot[r] += acc[r];
  } else {
    load8<TI, WHOLE>(arow, lk, K, av);
    load8<TI, WHOLE>(wrow, lk, K, wv);
    lay8(&As[0][lrow * LLD + lk], av, K - lk);
    lay8(&Ws[0][lrow * LLD + lk], wv, K - lk);
    load8<TI, WHOLE>(arow, LK + lk, K, av);
    load8<TI, WHOLE>(wrow, LK + lk, K, wv);
    __syncthreads();
    int buf = 0;
    for (int k0 = 0; k0 < K; k0 += LK, buf ^= 1) {
      // a slab's operands are read at once; in the middle of its matrix instructions the next slab is laid down and the one
      // after it asked for, so that only the barrier stands between two slabs' matrix instructions
      float4 a[LK / 8], w[LK / 8];
#pragma unroll
      for (int g = 0; g < LK / 8; ++g) {
        a[g] = *reinterpret_cast<const float4*>(&As[buf][fa + 8 * g]);
        w[g] = *reinterpret_cast<const float4*>(&Ws[buf][fw + 8 * g]);
      }
#pragma unroll
      for (int g = 0; g < LK / 8; ++g) {
        if (g == LK / 16) {
          __builtin_amdgcn_sched_barrier(0);
          const int inside = k0 + 2 * LK <= K ? 8 : K - (k0 + LK + lk);
          lay8(&As[buf ^ 1][lrow * LLD + lk], av, inside);      // (behind the last slab: zeros that nobody reads)
          lay8(&Ws[buf ^ 1][lrow * LLD + lk], wv, inside);
          load8<TI, WHOLE>(arow, k0 + 2 * LK + lk, K, av);
          load8<TI, WHOLE>(wrow, k0 + 2 * LK + lk, K, wv);
          __builtin_amdgcn_sched_barrier(0);
        }
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g].x, w[g].x, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g].y, w[g].y, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g].z, w[g].z, acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_32x32x2f32(a[g].w, w[g].w, acc, 0, 0, 0);
      }
      if ((k0 + LK) % SEG == 0 || k0 + LK >= K) {         // a segment ends: its sum joins the others'
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          tot[r] += acc[r];
          acc[r] = 0.f;
        }
      }
      __syncthreads();
    }
  }
  // a lane holds column lane % 32 of the rows 8 (r / 4) + 4 (lane / 32) + r % 4
  const int n = n0 + wn + lane % 32;
  if (n >= N) return;
  const float b = bias ? bias[n] : 0.f;
  const int mb = m0 + wm + 4 * (lane / 32);
  if (resid) {
    float old[16];
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = mb + 8 * (r / 4) + r % 4;
      old[r] = m < M ? resid[static_cast<size_t>(m) * ldr + n] : 0.f;
    }
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = mb + 8 * (r / 4) + r % 4;
      if (m < M) resid[static_cast<size_t>(m) * ldr + n] = old[r] + (bias ? tot[r] + b : tot[r]);
    }
  } else {
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int m = mb + 8 * (r / 4) + r % 4;
      if (m < M) C[static_cast<size_t>(m) * ldc + n] = from_float<TC>(apply_epilogue(bias ? tot[r] + b : tot[r], epi));
    }
  }
}

// four consecutive elements in one load (the few-rows kernel is launched only where they are aligned)
__device__ __forceinline__ void load4(const float* p, float* v) {
  const float4 x = *reinterpret_cast<const float4*>(p);
  v[0] = x.x, v[1] = x.y, v[2] = x.z, v[3] = x.w;
}
__device__ __forceinline__ void load4(const bf16_t* p, float* v) {
  const uint2 x = *reinterpret_cast<const uint2*>(p);
  v[0] = __uint_as_float(x.x << 16), v[1] = __uint_as_float(x.x & 0xffff0000u);
  v[2] = __uint_as_float(x.y << 16), v[3] = __uint_as_float(x.y & 0xffff0000u);
}

// Where the key and value columns of a fused projection of few rows go besides C (slot_map == null: nowhere):
// as KVScatter says it, with pools of C's own type.
template <typename TC>
struct KVRows {
  const int32_t* slot_map;
  TC* k_pool;
  TC* v_pool;
  int q_width, kv_width, dh, page_size, Hkv;
};

// such a column's value, as `finish` stored it in C, at its token's place in the cache
template <typename TC>
__device__ __forceinline__ void to_cache(float tot, int m, int n, const float* bias, int epi, const KVRows<TC>& kv) {
  if (kv.slot_map == nullptr || n < kv.q_width) return;
  const int slot = kv.slot_map[m];
  if (slot < 0) return;
  int c = n - kv.q_width;
  const bool is_value = c >= kv.kv_width;
  if (is_value) c -= kv.kv_width;
  const int page = slot / kv.page_size, off = slot % kv.page_size;
  const int hh = c / kv.dh, d = c % kv.dh;
  const size_t base = (static_cast<size_t>(page) * kv.Hkv + hh) * kv.page_size * kv.dh;
  const TC x = from_float<TC>(apply_epilogue(bias ? tot + bias[n] : tot, epi));
  if (is_value)
    kv.v_pool[base + static_cast<size_t>(d) * kv.page_size + off] = x;
  else
    kv.k_pool[base + static_cast<size_t>(off) * kv.dh + d] = x;
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// Four registers, four rows of 16 lanes: lane group g gives its register s to group s's register g (a 4 x 4 turn).  Written as assembly for
// the reason that `other_half` gives, with the idle cycles that the swaps and the matrix instruction behind them want.
__device__ __forceinline__ void turn4(float* v) {
  unsigned a = __builtin_bit_cast(unsigned, v[0]), b = __builtin_bit_cast(unsigned, v[1]), c = __builtin_bit_cast(unsigned, v[2]),
           d = __builtin_bit_cast(unsigned, v[3]);
  asm volatile(
      "s_nop 1\n\tv_permlane32_swap_b32 %0, %2\n\tv_permlane32_swap_b32 %1, %3\n\ts_nop 1\n\t"
      "v_permlane16_swap_b32 %0, %1\n\tv_permlane16_swap_b32 %2, %3\n\ts_nop 1"
      : "+v"(a), "+v"(b), "+v"(c), "+v"(d));
  v[0] = __builtin_bit_cast(float, a), v[1] = __builtin_bit_cast(float, b), v[2] = __builtin_bit_cast(float, c), v[3] = __builtin_bit_cast(float, d);
}

// Up to 16 rows: one kernel (where: chain_takes).  A workgroup owns 16 columns, or, for up to 8 rows, 8, and all of K; a wave
// takes a segment at a time, every load of it at once, straight into registers, and multiplies on the matrix cores:
// v_mfma_f32_16x16x4_f32 adds its four products to the sum one after the other, k ascending, each with one rounding: the
// bits of the chain of fused multiply-adds.  Its operands want k = 4 s + g in lane group g, and a lane's 16 bytes are
// k = 4 g + s: a 4 x 4 turn between lane groups (`turn4`).  With up to 8 rows the 16 x 16 result is two segments' 8 x 8 on its
// diagonal: lanes l % 16 < 8 bring rows and columns of one segment, the others the same rows and columns of the next (the
// blocks off the diagonal are dropped), so that twice as many workgroups ask for half as much each.  The segments' sums meet in
// LDS and are added in order.  A kernel with a workgroup a segment, whose operands go through LDS and vector
// multiply-adds, and a second one that adds the sums, against this one at 1 and 8 rows: 3,072 x 1,024 10.4 -> 6.1 and
// 10.8 -> 7.4 us, 1,024 x 1,024 7.0 -> 4.6 and 7.3 -> 5.2, 1,024 x 4,096 12.1 -> 8.7 and 12.3 -> 10.8, 1,600 x 6,400 20.0 -> 14.2
// and 20.6 -> 17.1, 50,257 x 1,024 75.5 -> 36.7 (5.6 TB/s of W) and 75.6 -> 50.5.  At one row it is bound by W's bytes and its
// chain of trips to memory; from 8 rows on what a workgroup reads of A is as much as it reads of W.
template <typename TI, typename TC, int WAVES, bool PAIR, int NB>
__global__ __launch_bounds__(WAVES * 64) void chain_kernel(const TI* __restrict__ A, int lda, const TI* __restrict__ W, const float* __restrict__ bias,
                                                            TC* __restrict__ C, int ldc, float* __restrict__ resid, int ldr, int M, int N, int K,
                                                            int epi, KVRows<TC> kv) {
  constexpr int SIDE = PAIR ? 8 : 16, EACH = PAIR ? 2 : 1;      // rows and columns of a block of the result; segments at a time
  constexpr int BLOCK = SIDE * SIDE / 4;
  extern __shared__ f32x4 sums[];                               // [segment][NB][BLOCK]: place (row / 4) * SIDE + column of a block, its four rows
  const int lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), g = lane / 16, half = PAIR ? lane % 16 / 8 : 0;
  const int n0 = blockIdx.x * (SIDE * NB), m0 = blockIdx.y * SIDE, nseg = (K + SEG - 1) / SEG;
  const TI* arow = A + static_cast<size_t>(min(m0 + lane % SIDE, M - 1)) * lda;
  const TI* wrow[NB];
#pragma unroll
  for (int b = 0; b < NB; ++b) wrow[b] = W + static_cast<size_t>(min(n0 + b * SIDE + lane % SIDE, N - 1)) * K;
  for (int s0 = wave * EACH; s0 < nseg; s0 += WAVES * EACH) {
    const int k0 = (s0 + half) * SEG + 4 * g;
    float w[NB][SEG / 16][4], a[SEG / 16][4];
    // (never a conditional load: what lies beyond K is read from the row's end and counts as zeros, the weight as well as the row)
#pragma unroll
    for (int b = 0; b < NB; ++b)
#pragma unroll
      for (int q = 0; q < SEG / 16; ++q) load4(wrow[b] + min(k0 + 16 * q, K - 4), w[b][q]);
#pragma unroll
    for (int q = 0; q < SEG / 16; ++q) load4(arow + min(k0 + 16 * q, K - 4), a[q]);
    f32x4 acc[NB];
#pragma unroll
    for (int b = 0; b < NB; ++b) acc[b] = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int q = 0; q < SEG / 16; ++q) {
      if ((s0 + EACH) * SEG > K) {      // (the same for the whole wave)
        const bool inside = k0 + 16 * q < K;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          a[q][i] = inside ? a[q][i] : 0.f;
#pragma unroll
          for (int b = 0; b < NB; ++b) w[b][q][i] = inside ? w[b][q][i] : 0.f;
        }
      }
      turn4(a[q]);
#pragma unroll
      for (int b = 0; b < NB; ++b) {
        turn4(w[b][q]);
#pragma unroll
        for (int i = 0; i < 4; ++i) acc[b] = __builtin_amdgcn_mfma_f32_16x16x4f32(a[q][i], w[b][q][i], acc[b], 0, 0, 0);
      }
    }
    // acc[b][r]: row 4 g + r, column lane % 16
#pragma unroll
    for (int b = 0; b < NB; ++b) {
      if (!PAIR)
        sums[(s0 * NB + b) * BLOCK + lane] = acc[b];
      else if (g / 2 == half && s0 + half < nseg)
        sums[((s0 + half) * NB + b) * BLOCK + g % 2 * 8 + lane % 8] = acc[b];
    }
  }
  __syncthreads();
  for (int t = threadIdx.x; t < NB * SIDE * SIDE; t += WAVES * 64) {
    const int b = t / (SIDE * SIDE), row = t / SIDE % SIDE, m = m0 + row, n = n0 + b * SIDE + t % SIDE;
    if (m >= M || n >= N) continue;
    const float* p = reinterpret_cast<const float*>(sums) + (b * BLOCK + (row / 4) * SIDE + t % SIDE) * 4 + row % 4;
    float tot = 0.f;
    int s = 0;
    for (; s + 8 <= nseg; s += 8) {
      float v[8];
#pragma unroll
      for (int i = 0; i < 8; ++i) v[i] = p[(s + i) * NB * BLOCK * 4];
#pragma unroll
      for (int i = 0; i < 8; ++i) tot += v[i];
    }
    for (; s < nseg; ++s) tot += p[s * NB * BLOCK * 4];
    finish<TC>(tot, m, n, bias, C, ldc, resid, ldr, epi);
    to_cache<TC>(tot, m, n, bias, epi, kv);
  }
}

// Few rows.  A workgroup: RM rows x 64 columns, the segments [seg0, seg0 + nseg) of K.  part == null:
// it owns all segments and ends with the epilogue; else it owns one (blockIdx.z) and writes its sum to
// part[seg][m][n].  A segment's share of W (64 rows x 128 k) and of A is asked for at once, 16 bytes a
// thread and load, eight threads to a row's 128 bytes, and goes through LDS in four slabs of 32.
template <typename TI, typename TC, int RM>
__global__ __launch_bounds__(256) void rows_kernel(const TI* __restrict__ A, int lda, const TI* __restrict__ W,
                                                    const float* __restrict__ bias, TC* __restrict__ C, int ldc,
                                                    float* __restrict__ resid, int ldr, int M, int N, int K, int epi,
                                                    float* __restrict__ part) {
  constexpr int SK = 32;                              // a slab
  constexpr int TN = RM >= 16 ? 4 : 2;                // columns per thread
  constexpr int TM = RM * BN / (256 * TN);            // rows per thread
  constexpr int CG = BN / TN;                         // threads along the columns
  static_assert(TM >= 1 && TM * TN * 256 == RM * BN, "tile");
  __shared__ float As[SK][RM + PAD];
  __shared__ float Ws[SK][BN + PAD];
  const int t = threadIdx.x;
  const int m0 = blockIdx.y * RM, n0 = blockIdx.x * BN;
  const int tx = t % CG, ty = t / CG;
  // loader: thread t takes 4 k at (t % 8) * 4 of row t / 8 (+ 32 for the second half of W's rows), in each slab
  const int lr = t / 8, lk = (t % 8) * 4;
  const int seg_first = part ? blockIdx.z : 0;
  const int seg_last = part ? blockIdx.z + 1 : (K + SEG - 1) / SEG;
  float tot[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) tot[i][j] = 0.f;

  for (int seg = seg_first; seg < seg_last; ++seg) {
    const int kseg = seg * SEG;
    // everything this segment needs, asked for at once
    float wv[SEG / SK][2][4];
    float av[SEG / SK][(RM + 31) / 32][4];
#pragma unroll
    for (int sl = 0; sl < SEG / SK; ++sl) {
      const int k = kseg + sl * SK + lk;
#pragma unroll
      for (int hf = 0; hf < 2; ++hf) {
        const int n = n0 + lr + 32 * hf;
#pragma unroll
        for (int i = 0; i < 4; ++i) wv[sl][hf][i] = 0.f;
        if (n < N && k < K) load4(W + static_cast<size_t>(n) * K + k, wv[sl][hf]);
      }
#pragma unroll
      for (int hf = 0; hf < (RM + 31) / 32; ++hf) {
        const int r = lr + 32 * hf, m = m0 + r;
#pragma unroll
        for (int i = 0; i < 4; ++i) av[sl][hf][i] = 0.f;
        if (r < RM && m < M && k < K) load4(A + static_cast<size_t>(m) * lda + k, av[sl][hf]);
      }
    }
    float acc[TM][TN];
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) acc[i][j] = 0.f;
#pragma unroll
    for (int sl = 0; sl < SEG / SK; ++sl) {
      __syncthreads();
#pragma unroll
      for (int hf = 0; hf < 2; ++hf)
#pragma unroll
        for (int i = 0; i < 4; ++i) Ws[lk + i][lr + 32 * hf] = wv[sl][hf][i];
#pragma unroll
      for (int hf = 0; hf < (RM + 31) / 32; ++hf)
        if (lr + 32 * hf < RM) {
#pragma unroll
          for (int i = 0; i < 4; ++i) As[lk + i][lr + 32 * hf] = av[sl][hf][i];
        }
      __syncthreads();
      if (kseg + sl * SK < K) {
#pragma unroll
        for (int k = 0; k < SK; ++k) {
          float a[TM], w[TN];
#pragma unroll
          for (int i = 0; i < TM; ++i) a[i] = As[k][ty * TM + i];
#pragma unroll
          for (int j = 0; j < TN; ++j) w[j] = Ws[k][tx * TN + j];
#pragma unroll
          for (int i = 0; i < TM; ++i)
#pragma unroll
            for (int j = 0; j < TN; ++j) acc[i][j] = fmaf(a[i], w[j], acc[i][j]);
        }
      }
    }
#pragma unroll
    for (int i = 0; i < TM; ++i)
#pragma unroll
      for (int j = 0; j < TN; ++j) tot[i][j] += acc[i][j];
  }
#pragma unroll
  for (int i = 0; i < TM; ++i) {
    const int m = m0 + ty * TM + i;
    if (m >= M) continue;
#pragma unroll
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + tx * TN + j;
      if (n >= N) continue;
      if (part)
        part[(static_cast<size_t>(blockIdx.z) * M + m) * N + n] = tot[i][j];
      else
        finish<TC>(tot[i][j], m, n, bias, C, ldc, resid, ldr, epi);
    }
  }
}

// the segments' sums of each element, added in ascending order from zero, then the epilogue; the keys and values
// among the columns also go to their tokens' places in the cache, so that no kernel has to copy them there
template <typename TC>
__global__ __launch_bounds__(256) void join_kernel(const float* __restrict__ part, int nseg, const float* __restrict__ bias,
                                                    TC* __restrict__ C, int ldc, float* __restrict__ resid, int ldr,
                                                    int M, int N, int epi, KVRows<TC> kv) {
  const int n = blockIdx.x * 256 + threadIdx.x, m = blockIdx.y;
  if (n >= N) return;
  float tot = 0.f;
  const float* p = part + static_cast<size_t>(m) * N + n;
  const size_t step = static_cast<size_t>(M) * N;
  int s = 0;
  for (; s + 8 <= nseg; s += 8) {       // eight loads at a time; the sum keeps its order
    float v[8];
#pragma unroll
    for (int i = 0; i < 8; ++i) v[i] = p[(s + i) * step];
#pragma unroll
    for (int i = 0; i < 8; ++i) tot += v[i];
  }
  for (; s < nseg; ++s) tot += p[s * step];
  finish<TC>(tot, m, n, bias, C, ldc, resid, ldr, epi);
  to_cache<TC>(tot, m, n, bias, epi, kv);
}

constexpr int FEW_ROWS = 64;
// Whether chain_kernel takes a product that few_rows_take takes.  Behind each size: the time of the kernel with a workgroup a
// segment and its join over chain_kernel's, 32-bit, weights from memory.
// * A workgroup's 16 waves take 32 segments a turn (16 where it has 16 rows), and one of 8 columns has all of K to itself,
//   where a workgroup a segment spreads few columns over the chip: the fewer the columns and the more rows of A are read
//   beside W's, the earlier a long K is better off there.
//     256 columns: 1 row at K = 3,072 1.13, 4,096 0.99; 8 rows at 2,048 1.12, 3,072 0.95
//     512: 4 rows at 4,096 0.99; 8 at 3,072 1.01, 4,096 0.90            768: 8 rows at 6,400 1.00, 7,680 0.88
//     1,024: 8 rows at 7,680 0.99, 12,288 0.88                          1,600: 8 rows at 16,384 1.07; 16 at 3,072 1.00, 4,096 0.95
//     3,072 (one and a half workgroups a CU): 8 rows at 7,680 0.95, 16,384 0.89; 16 at 7,680 1.03
//     8,192: 8 rows at 6,400 0.96, 8,192 1.18, 16,384 1.01
//   The sums take 256 bytes of LDS a segment (512 with two blocks of columns, 1 KB with 16 rows): 64 KB at most.
// * A workgroup costs the same however short K is, and there are eight times as many of 8 columns.
//     8,192 columns: K = 64 0.90, 128 1.14                              16,384: 128 0.75, 256 1.28
//     50,257 (whose tiles of 64 fill the chip without shares of K): 128 0.67, 256 1.08
//     with 16 rows and columns: 16,384: 32 0.85, 64 1.02                50,257: 96 0.86, 128 1.03
static bool chain_takes(int M, int N, int K) {
  if (M > 16) return false;
  const bool sixteen = M > 8 && N >= 2048;      // (workgroups of 16 rows and columns: see `run`)
  if (N > 2048 && K < (sixteen ? min(N / 256, 128) : min(N / 64, 256))) return false;
  int longest;
  if (M <= 5)
    longest = N < 512 ? 3072 : N < 768 ? 4096 : N < 1024 ? 7680 : N < 1536 ? 12288 : 16384;
  else if (M <= 8)
    longest = N < 512 ? 2048 : N < 768 ? 3072 : N < 1024 ? 6400 : N < 1536 || (N > 2048 && N < 4096) ? 7680 : 16384;
  else
    longest = N < 512 ? 3072 : N < 768 ? 4096 : N < 1024 ? 6400 : N < 1536 ? 7680 : N < 3072 ? 4096 : 7680;
  return K <= longest;
}

// floats of workspace that a product of M rows needs (0: none)
long work_floats(int M, int N, int K) {
  if (M > FEW_ROWS || chain_takes(M, N, K)) return 0;
  const int nseg = (K + SEG - 1) / SEG;
  const long tiles = (N + BN - 1) / BN;
  if (nseg < 2 || tiles >= 384) return 0;      // the column tiles alone fill the chip
  return static_cast<long>(nseg) * M * N;
}

// whether the few-rows kernel takes these operands (it loads four elements at a time: rows that do not start
// at multiples of that go the other way)
template <typename TI>
static bool few_rows_take(const void* A, int lda, const void* W, int M, int K) {
  const size_t quad = 4 * sizeof(TI);
  return M <= FEW_ROWS && reinterpret_cast<uintptr_t>(A) % quad == 0 && reinterpret_cast<uintptr_t>(W) % quad == 0 &&
         lda % 4 == 0 && K % 4 == 0;
}

// kv: a fused projection's cache write, done by chain_kernel or by the kernel that joins the segments (so only where one of
// them runs: few_rows_take and joins_of)
template <typename TI, typename TC>
static int run(const void* A, int lda, const void* W, const float* bias, void* C, int ldc, float* resid, int ldr, int M,
               int N, int K, int epi, float* work, long have, hipStream_t stream, KVRows<TC> kv = KVRows<TC>{}) {
  const TI* a = static_cast<const TI*>(A);
  const TI* w = static_cast<const TI*>(W);
  TC* c = static_cast<TC*>(C);
  if (!few_rows_take<TI>(A, lda, W, M, K)) {
    if (kv.slot_map) return DN_ERR_SHAPE;
    const int mtiles = (M + BM - 1) / BM;
    const long all = static_cast<long>(mtiles) * ((N + BN - 1) / BN);
    if (all > (1 << 30)) return DN_ERR_SHAPE;
    const int tiles = static_cast<int>(all), per_xcd = (tiles + 7) / 8;
#define DN_MANY(WHOLE, SHORT)                                                                                                    \
  hipLaunchKernelGGL((gemm_kernel<TI, TC, WHOLE, SHORT>), dim3(per_xcd * 8), dim3(256), 0, stream, a, lda, w, bias, c, ldc, resid, \
                     ldr, M, N, K, epi, mtiles, tiles, per_xcd)
    // (a short K whose tiles are two a CU at most: nobody's waits to hide, and the registers of the long walk's kernel make the shorter end:
    // 200 x 64 x 64 in bfloat16, added into the stream, 5.9 us and 6.3)
    const bool brief = K <= 2 * LK && tiles > 2 * 256;
    if (K % 4 == 0 && brief)
      DN_MANY(true, true);
    else if (K % 4 == 0)
      DN_MANY(true, false);
    else if (brief)
      DN_MANY(false, true);
    else
      DN_MANY(false, false);
#undef DN_MANY
    return 0;
  }
  if (chain_takes(M, N, K)) {
    const int nseg = (K + SEG - 1) / SEG;
    // 9 to 16 rows of few columns: two workgroups of 8 rows, since 16 columns each leave most CUs without work (1,024 x 1,024
    // at 16 rows 6.9 us and 5.3, from K = 4,096 18.4 and 11.1; 3,072 columns 7.5 and 9.3).  5 to 8 rows of very many
    // columns: two blocks of columns, since the rows are read again by every workgroup (50,257 x 1,024: 8 rows 55.0 and 50.5;
    // 1 row 36.7 and 41.8).
    const bool pair = M <= 8 || N < 2048, wide = M > 4 && M <= 8 && N >= 16384;
    const int turns = pair ? (nseg + 1) / 2 : nseg, side = pair ? 8 : 16, cols = wide ? 2 * side : side;
#define DN_CHAIN(WAVES, PAIR, NB)                                                                                                       \
  hipLaunchKernelGGL((chain_kernel<TI, TC, WAVES, PAIR, NB>), dim3((N + cols - 1) / cols, (M + side - 1) / side), dim3(WAVES * 64),     \
                     static_cast<size_t>(nseg) * NB * side * side * sizeof(float), stream, a, lda, w, bias, c, ldc, resid, ldr, M, N, K, \
                     epi, kv)
#define DN_CHAIN_W(PAIR, NB)   \
  if (turns <= 4)              \
    DN_CHAIN(4, PAIR, NB);     \
  else if (turns <= 8)         \
    DN_CHAIN(8, PAIR, NB);     \
  else                         \
    DN_CHAIN(16, PAIR, NB)
    if (pair && wide) {
      DN_CHAIN_W(true, 2);
    } else if (pair) {
      DN_CHAIN_W(true, 1);
    } else {
      DN_CHAIN_W(false, 1);
    }
#undef DN_CHAIN_W
#undef DN_CHAIN
    return 0;
  }
  const long need = work_floats(M, N, K);
  if (need > 0 && (work == nullptr || have < need)) return DN_ERR_SHAPE;     // dn_gemm_work_floats says how much
  float* part = need > 0 ? work : nullptr;
  if (kv.slot_map && !part) return DN_ERR_SHAPE;
  const int nseg = (K + SEG - 1) / SEG;
  const int rm = M <= 8 ? 8 : M <= 16 ? 16 : M <= 32 ? 32 : 64;
  dim3 grid((N + BN - 1) / BN, (M + rm - 1) / rm, part ? nseg : 1);
#define DN_ROWS(RM)                                                                                                  \
  hipLaunchKernelGGL((rows_kernel<TI, TC, RM>), grid, dim3(256), 0, stream, a, lda, w, bias, c, ldc, resid, ldr, M, N, \
                     K, epi, part)
  if (rm == 8) DN_ROWS(8);
  else if (rm == 16) DN_ROWS(16);
  else if (rm == 32) DN_ROWS(32);
  else DN_ROWS(64);
#undef DN_ROWS
  if (part)
    hipLaunchKernelGGL((join_kernel<TC>), dim3((N + 255) / 256, M), dim3(256), 0, stream, part, nseg, bias, c, ldc, resid,
                       ldr, M, N, epi, kv);
  return 0;
}

// -- what the entry points call (one function per choice of types) ---------------------------------------
// (not a product of one segment, though chain_kernel could: inner sizes of up to 128 are no model's that waits for a launch, and
// the cache's own kernel stays behind them as it stands behind more than 64 rows)
int joins_of(int M, int N, int K) { return work_floats(M, N, K) > 0 || (chain_takes(M, N, K) && K > SEG); }

int few_rows_take_of(int dtype, const void* A, int lda, const void* W, int M, int K) {
  return dtype == DN_F32 ? few_rows_take<float>(A, lda, W, M, K) : dtype == DN_BF16 ? few_rows_take<bf16_t>(A, lda, W, M, K) : 0;
}

int run_of(int in_dtype, int out_dtype, const void* A, int lda, const void* W, const float* bias, void* C, int ldc,
           float* resid, int ldr, int M, int N, int K, int epilogue, float* work, long have, hipStream_t stream) {
#define DN_LAUNCH(TI, TC) return run<TI, TC>(A, lda, W, bias, C, ldc, resid, ldr, M, N, K, epilogue, work, have, stream)
  if (in_dtype == DN_F32 && out_dtype == DN_F32) DN_LAUNCH(float, float);
  if (in_dtype == DN_F32 && out_dtype == DN_BF16) DN_LAUNCH(float, bf16_t);
  if (in_dtype == DN_BF16 && out_dtype == DN_BF16) DN_LAUNCH(bf16_t, bf16_t);
  if (in_dtype == DN_BF16 && out_dtype == DN_F32) DN_LAUNCH(bf16_t, float);
#undef DN_LAUNCH
  return DN_ERR_DTYPE;
}

// the fused projection of few rows: C and the pools have the operands' type
int run_qkv_of(int dtype, const void* A, int lda, const void* W, const float* bias, void* C, int ldc, int M, int N, int K,
               const int32_t* slot_map, void* k_pool, void* v_pool, int q_width, int Hkv, int dh, int page_size,
               float* work, long have, hipStream_t stream) {
  if (dtype == DN_F32) {
    KVRows<float> kv{slot_map, static_cast<float*>(k_pool), static_cast<float*>(v_pool), q_width, Hkv * dh, dh, page_size, Hkv};
    return run<float, float>(A, lda, W, bias, C, ldc, nullptr, 0, M, N, K, EPI_NONE, work, have, stream, kv);
  }
  if (dtype == DN_BF16) {
    KVRows<bf16_t> kv{slot_map, static_cast<bf16_t*>(k_pool), static_cast<bf16_t*>(v_pool), q_width, Hkv * dh, dh, page_size,
                      Hkv};
    return run<bf16_t, bf16_t>(A, lda, W, bias, C, ldc, nullptr, 0, M, N, K, EPI_NONE, work, have, stream, kv);
  }
  return DN_ERR_DTYPE;
}

// resid [M, N] += (part[0] + part[1] + ... in this order) + bias
void join_shares(const float* part, int shares, const float* bias, float* resid, int ldr, int M, int N, hipStream_t stream) {
  hipLaunchKernelGGL((join_kernel<float>), dim3((N + 255) / 256, M), dim3(256), 0, stream, part, shares, bias,
                     static_cast<float*>(nullptr), 0, resid, ldr, M, N, EPI_NONE, KVRows<float>{});
}
}  // namespace plain
