#include "gemm_common.h"

// ---------------------------------------------------------------------------------------
// Few rows (M <= 256), bfloat16: the decode step's products, bound by reading W once.
// A workgroup owns 8, 16, 32 or 64 output columns; its waves split K in steps of 32 (wave w takes
// steps w, w + WAVES, ...), each feeding v_mfma_f32_16x16x32_bf16 with one packed block of W per
// 16 columns straight from memory (16 bytes per lane) and the matching 16 bytes of up to four
// 16-row blocks of A (lane = row + 16 * (k / 8)).  The waves' sums meet in LDS and are added in
// wave order, so the result has one order of summation whatever M is.  No atomics.
// ---------------------------------------------------------------------------------------

namespace skinny {
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;

// The norm that stands between two such products of few rows runs inside them (NORM_OUT in the product before
// it, NORM_IN in the one after), so that it is no kernel of its own: a LayerNorm of a few rows is
// all launch and latency and no work.  With y = (x - mean) / sqrt(var + eps) * gamma + beta
// (crates/denno-engine/src/tensor.rs:1101-1112),
//     y . W^T + b = ((x * gamma) . W^T - mean * c1) / sqrt(var + eps) + c2,
//     c1[n] = sum_k gamma[k] W[n,k],  c2[n] = sum_k beta[k] W[n,k] + b[n]      (made once per weight),
// so the product itself runs on rows that are not normalised, and the norm is two numbers per row in
// the epilogue.  NORM_OUT: a product that adds into the residual stream also stores the updated rows
// times gamma (the next norm's), rounded to bfloat16, and, for each row, the mean and the sum of
// squared distances from it of its 16 columns.  NORM_IN: A is such a copy; each wave joins two to eight rows'
// N / 16 pairs (means are averaged; the squares add up with 16 times the squared distance of each
// block's mean from the row's: exact, and as stable as two passes over the row) while the operands
// travel, and wave 0 applies them at the end.  The rows are rounded to bfloat16 before the mean is
// taken off, not after: right where a row's mean is not large beside its spread.


// Mean and sum of squared distances of the 16 columns that lie in 16 lanes side by side, right in the first of them: the same sums in
// every kernel, so that the next norm is the same bits whichever kernel the product before it ran in.  (Eight columns a workgroup, 16 joined from
// two pairs of eights, rounds otherwise: steps of up to 8 rows would be 2 to 3 % faster by it, decoding one request at width 1,024 17.8 ms for 18.4.)
__device__ __forceinline__ float2 columns_stats(float x) {
#pragma clang fp contract(off)
  const float mean = group_reduce<16>(x, SumOp()) * (1.0f / 16.0f);
  const float d = x - mean;
  float sq = fmaf(d, d, dpp_move<DN_DPP_XOR1>(d * d));
  sq += dpp_move<DN_DPP_XOR2>(sq);
  sq += dpp_move<DN_DPP_HALF_MIRROR>(sq);
  sq += dpp_move<DN_DPP_MIRROR>(sq);
  return float2{mean, sq};
}

// what a kernel's last argument is (the plain kernels read none of it)
template <int END>
struct EndsFor {
  typedef Ends type;
};
template <>
struct EndsFor<END_PLAIN> {
  struct type {
    int none;
    __host__ explicit type(const Ends&) : none(0) {}
  };
};
template <int END>
using EndsOf = typename EndsFor<END>::type;

// The arguments of this file's kernels.  The first 14 words come in scalar registers with the launch, the others by a trip to memory that
// every wave makes before it can ask for anything they name (two cache lines of arguments more made a product 0.4 us slower): so what the first
// loads want stands in front; in gemm8_kernel and gemm16_kernel packed: `rows` is the rows and a flag; p is the statistics (NORM_IN), else what the results go to
// or are added to; q is the slot map (NORM_IN), else the leading dimension of p (a pointer in any case: through a pointer made from a number the
// compiler loads by instructions that are waited for one by one, 0.5 us more).
// In this order the operands' loads leave 0.2 to 0.5 us sooner, 8 rows: with the norm before, 3,072 x 1,024 4.3 -> 4.0 us, 5,120 x 1,280 6.6 -> 6.1,
// 6,400 x 1,600 7.6 -> 7.2; 50,257 x 1,024 23.8 -> 23.0; 8 columns a workgroup (with statistics, which that kernel left then), 1,024 x 1,024 3.1 -> 3.0,
// 1,280 x 5,120 6.4 -> 6.0, 1,600 x 6,400 8.1 -> 7.6.  64 rows: 4,800 x 1,600 8.4 -> 8.0, with the norm before 11.4 -> 11.1; with the norm after level.
constexpr int FIRST_ROWS = 255, FIRST_ADDS = 256;
template <int END>
struct Late {
  void* C;      // NORM_IN
  int ldc, epi;
  const float* c1;
  float eps;
  int no_mean;
  const float* gamma_out;
  bf16_t* copy_out;
  float* stats_out;
  int ldcopy;
  KVScatter kv;
  EndsOf<END> ends;
};

// Brings what the epilogue takes from `late` into scalar registers here, behind the first loads of the operands (left to the compiler these
// arguments were fetched where they are used, at the kernel's end, and the trip to memory came on top: a q | k | v of 4,800 columns 7.8 us for 7.2).
template <int NORM, bool KV, int END>
__device__ __forceinline__ void late_at_hand(const Late<END>& late) {
  if constexpr (NORM == NORM_IN) asm volatile("" ::"s"(late.C), "s"(late.ldc), "s"(late.eps), "s"(late.no_mean));
  if constexpr (NORM == NORM_OUT) asm volatile("" ::"s"(late.copy_out), "s"(late.stats_out), "s"(late.ldcopy));
  if constexpr (NORM != NORM_OUT) asm volatile("" ::"s"(late.epi));
  if constexpr (KV)
    asm volatile("" ::"s"(late.kv.k_pool), "s"(late.kv.v_pool), "s"(late.kv.q_width), "s"(late.kv.page_size), "s"(late.kv.c_cols));
  if constexpr (END == END_TWO) asm volatile("" ::"s"(late.ends.C2), "s"(late.ends.ldc2), "s"(late.ends.cols));
}

// What a load of W's step beyond K reads (no load is conditional): a packed block of zeros, so that the step adds nothing whatever the weights are.
// (A block of W's own times zeros of A would do for finite weights; one infinity in it, and every column of the product is not a number.)
__device__ uint4 zero_block[64];
__device__ __forceinline__ const bf16_t* no_step(int lane) { return reinterpret_cast<const bf16_t*>(&zero_block[lane]); }

// MB row blocks and NB column blocks of 16 per workgroup; U steps of K in flight per wave.
template <int MB, int NB, int WAVES, int U, typename TC, bool KV, int NORM = NORM_NONE, int END = END_PLAIN>
__global__ __launch_bounds__(WAVES * 64) void gemm_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int lda, int M, int N, int K, int packed,
                                                           int ldr, const void* __restrict__ first, const float* __restrict__ bias,
                                                           Late<END> late) {
  // (first: the statistics (NORM_IN), else the stream, or nullptr)
  float* resid = NORM == NORM_IN ? nullptr : static_cast<float*>(const_cast<void*>(first));
  const float* stats_in = static_cast<const float*>(first);
  const int blocks_in = K / 16;
  TC* C = static_cast<TC*>(late.C);
  constexpr int BLOCKS = MB * NB;                          // 16 x 16 blocks of C in this workgroup
  constexpr int PASSES = (BLOCKS + WAVES - 1) / WAVES;     // wave w finishes blocks w, w + WAVES, ...
  constexpr int SP = 2, SR = NORM == NORM_IN ? MB * 16 / WAVES : 0;      // (statistics: up to 64 SP pairs a row, SR rows a wave)
  __shared__ floatx4 red[WAVES][SR > BLOCKS ? SR : BLOCKS][64];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64), lane = threadIdx.x % 64;   // (a scalar: what follows from it is the scalar unit's work)
  const int col = lane % 16, g = lane / 16;
  const int n0 = blockIdx.x * (16 * NB);
  if constexpr (END == END_PAIR)
    if (n0 >= late.ends.cols) A += late.ends.a_shift;
  const int row0 = blockIdx.y * (MB * 16);     // the rows may be shared out among workgroups too (blockIdx.y)
  const int ksteps = (K + 31) / 32, nblocks = (N + 15) / 16;
  const bf16_t* wblk[NB];
#pragma unroll
  for (int nb = 0; nb < NB; ++nb) {
    // a block beyond N reads the last one again; its result is not stored
    const int blk = min(blockIdx.x * NB + nb, nblocks - 1);
    wblk[nb] = W + (static_cast<size_t>(blk) * ksteps * 64 + lane) * 8;
  }
  const bf16x8 zero = {0, 0, 0, 0, 0, 0, 0, 0};

  // what the epilogue will read (bias, the residual stream) is asked for first of all
  float epi_bias[PASSES];
  float epi_x[PASSES][4];
  int epi_slot[KV ? PASSES : 1][4];
  float2 epi_act[END != END_PLAIN ? PASSES : 1];
  float epi_norm[NORM != NORM_NONE ? PASSES : 1];          // NORM_IN: c1 of the lane's column; NORM_OUT: the next norm's gamma
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int blk = wave + p * WAVES;
    epi_bias[p] = 0.f;
    if constexpr (END != END_PLAIN) epi_act[p] = float2{0.f, 0.f};
#pragma unroll
    for (int r = 0; r < 4; ++r) epi_x[p][r] = 0.f;
    if constexpr (KV) {
#pragma unroll
      for (int r = 0; r < 4; ++r) epi_slot[p][r] = -1;
    }
    if (blk < BLOCKS) {
      const int mb = blk / NB, nb = blk % NB;
      const int nn = min(n0 + nb * 16 + col, N - 1);
      if (bias) epi_bias[p] = bias[nn];
      if (resid) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          const int m = min(row0 + mb * 16 + g * 4 + r, M - 1);
          epi_x[p][r] = resid[static_cast<size_t>(m) * ldr + nn];
        }
      }
    }
  }
  // NORM_IN: wave w joins the statistics of rows SR w .. SR w + SR - 1.  Their pairs are asked for now, before the operands, and go
  // straight into LDS, a row's 1 KB where this wave's sums will lie at the end, so no barrier stands between.  In registers they stood beside a round's
  // operands (with all else as it is here, 64 rows of 4,800 x 1,600 with a cache write 12.0 us for 11.0, 5,120 x 1,280 9.1 for 8.0).
  __shared__ float rowstat[NORM == NORM_IN ? MB * 16 : 1][2];
  if constexpr (NORM == NORM_IN) {
    if (blocks_in % 2 == 0 && reinterpret_cast<uintptr_t>(stats_in) % 16 == 0) {
#pragma unroll
      for (int t = 0; t < SR; ++t) {
        const int row = min(row0 + wave * SR + t, M - 1);
        load_to_lds(stats_in + (static_cast<size_t>(row) * blocks_in + min(2 * lane, blocks_in - 2)) * 2, red[wave][t]);
      }
    } else {      // (rows of an odd number of pairs are no multiples of 16 bytes)
#pragma unroll
      for (int t = 0; t < SR; ++t) {
        const float* row = stats_in + static_cast<size_t>(min(row0 + wave * SR + t, M - 1)) * blocks_in * 2;
#pragma unroll
        for (int i = 0; i < SP; ++i)
          reinterpret_cast<float2*>(red[wave][t])[lane + 64 * i] = *reinterpret_cast<const float2*>(row + min(lane + 64 * i, blocks_in - 1) * 2);
      }
    }
    // (no load of the first round in front of these: `join_stats` counts on their order)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  }
  // Loads are never conditional and nothing uses a loaded value before all loads of a round are
  // issued (a predicated load, or a use in between, makes each load wait for the one before it).
  // A step beyond K reads zeros (no_step) and meets a zeroed piece of A.
  // The first round of W is on its way while the rest of the prologue works.
  bf16x8 b[U][NB], a[U][MB];
  auto ask_w = [&](int p0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ks = 2 * (p0 + (u / 2) * WAVES) + u % 2;
#pragma unroll
      for (int nb = 0; nb < NB; ++nb)
        b[u][nb] = *reinterpret_cast<const bf16x8*>(ks < ksteps ? wblk[nb] + ks * 512 : no_step(lane));
    }
  };
  ask_w(wave);
  // what the epilogue reads by arguments that do not come with the launch: behind the first round of W
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int blk = min(wave + p * WAVES, BLOCKS - 1);
    const int nn = min(n0 + blk % NB * 16 + col, N - 1);
    if constexpr (NORM != NORM_NONE) epi_norm[p] = NORM == NORM_IN ? late.c1[nn] : late.gamma_out[nn];
    if constexpr (END != END_PLAIN) epi_act[p] = end_numbers<TC, END>(late.ends, nn);
    if constexpr (KV) {
#pragma unroll
      for (int r = 0; r < 4; ++r) epi_slot[p][r] = late.kv.slot_map[min(row0 + blk / NB * 16 + g * 4 + r, M - 1)];
    }
  }
  late_at_hand<NORM, KV>(late);

  // A in rows, or packed like W (PACKED_A): then a wave reads 1 KB in one piece per block
  const bf16_t* arow[MB];
  const bf16_t* asafe[MB];
  bool a_ok[MB];
  const int astep = (packed & PACKED_A) ? 512 : 32;
#pragma unroll
  for (int mb = 0; mb < MB; ++mb) {
    int row = row0 + mb * 16 + col;
    a_ok[mb] = row < M;
    // (a block of rows beyond M, where MB is more than the rows need, reads the last one again: packed
    // rows end with the block that holds row M - 1)
    arow[mb] = (packed & PACKED_A) ? A + (static_cast<size_t>(min(static_cast<int>(blockIdx.y) * MB + mb, (M + 15) / 16 - 1)) * ksteps * 64 + lane) * 8
                                   : A + static_cast<size_t>(a_ok[mb] ? row : 0) * lda + g * 8;
    // where a step's piece lies beyond K the load goes to an address that is surely inside A instead: the start
    // of the row (with K < 32 the row's piece g itself may lie beyond the row, and the last row's beyond A)
    asafe[mb] = (packed & PACKED_A) ? arow[mb] : A + static_cast<size_t>(a_ok[mb] ? row : 0) * lda;
  }
  // NORM_IN: the rows' means and 1 / sqrt(var + eps), joined while the first round of operands travels (a
  // wave does it in its first turn of the loop below, which every wave has: K >= 1024); the finishing
  // waves meet them behind the barrier further down.  The sums of several rows go through the lanes side by side, with no branch between them, and the
  // last steps are lane t's for the wave's row t.  Row by row, each with divisions, a square root and stores of its own, a wave's eight rows took longer than
  // the operands (before -> with the statistics in LDS and the later rounds' loads together, 24, 40 and 64 rows: 4,800 x 1,600 with a cache write 9.2 -> 8.5,
  // 10.7 -> 9.7, 13.0 -> 11.0 us; 6,400 x 1,600 with GELU 8.7 -> 7.8, 10.1 -> 8.8, 11.4 -> 9.8; 3,840 x 1,280 7.7 -> 7.2, 9.0 -> 8.2, 11.3 -> 9.3; 4,096 x
  // 1,024 5.9 -> 5.4, 7.4 -> 6.2, 9.1 -> 7.2).
  auto join_stats = [&]() {
    const float blocks = static_cast<float>(blocks_in);      // pairs of statistics a row, 16 columns a pair
    // The first round's U (MB + NB) loads are behind the statistics' (a barrier to the compiler stands between) and in front of this wait (the wave asked
    // for both already), so with that many out the statistics are there; no load may move across.  The compiler sets no wait of its own between such loads and reads of LDS.
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_waitcnt vmcnt(%0)" ::"n"(U * (MB + NB)) : "memory");
    __builtin_amdgcn_sched_barrier(0);
    constexpr int TOGETHER = SR % 4 == 0 ? 4 : 3;      // rows whose sums go through the lanes side by side
    float row_mean = 0.f, row_sq = 0.f;                // (lane t: of the wave's row t)
#pragma unroll
    for (int t0 = 0; t0 < SR; t0 += TOGETHER) {
      float2 st[TOGETHER][SP];
      float mean[TOGETHER], sq[TOGETHER];
#pragma unroll
      for (int t = 0; t < TOGETHER; ++t)
#pragma unroll
        for (int i = 0; i < SP; ++i) st[t][i] = reinterpret_cast<const float2*>(red[wave][t0 + t])[lane + 64 * i];
#pragma unroll
      for (int t = 0; t < TOGETHER; ++t) {
        mean[t] = sq[t] = 0.f;
#pragma unroll
        for (int i = 0; i < SP; ++i) mean[t] += lane + 64 * i < blocks_in ? st[t][i].x : 0.f;
      }
#pragma unroll
      for (int t = 0; t < TOGETHER; ++t) mean[t] = wave_sum(mean[t]);
#pragma unroll
      for (int t = 0; t < TOGETHER; ++t) {
        mean[t] = late.no_mean ? 0.f : mean[t] / blocks;      // (without it the squares are taken about 0)
#pragma unroll
        for (int i = 0; i < SP; ++i) {
          const float d = st[t][i].x - mean[t];
          const float more = sq[t] + (st[t][i].y + 16.f * d * d);
          sq[t] = lane + 64 * i < blocks_in ? more : sq[t];
        }
      }
#pragma unroll
      for (int t = 0; t < TOGETHER; ++t) sq[t] = wave_sum(sq[t]);
#pragma unroll
      for (int t = 0; t < TOGETHER; ++t)
        if (lane == t0 + t) row_mean = mean[t], row_sq = sq[t];
    }
    if (lane < SR) {
      const int row = wave * SR + lane;
      rowstat[row][0] = row0 + row < M ? row_mean : 0.f;
      rowstat[row][1] = row0 + row < M ? 1.0f / sqrtf(row_sq / (16.f * blocks) + late.eps) : 0.f;
    }
  };
  floatx4 acc[MB][NB];
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[mb][nb] = floatx4{0.f, 0.f, 0.f, 0.f};
  // the steps go to the waves in pairs: wave w takes steps 2w, 2w + 1, 2 (w + WAVES), ... (the same
  // shares as in gemm16_kernel, so that both sum in the same order)
  auto ask_a = [&](int p0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ks = 2 * (p0 + (u / 2) * WAVES) + u % 2;
      const bool ok = ks < ksteps && ks * 32 + g * 8 < K;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        a[u][mb] = *reinterpret_cast<const bf16x8*>(ok ? arow[mb] + ks * astep : asafe[mb]);
    }
  };
  auto use = [&](int p0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int ks = 2 * (p0 + (u / 2) * WAVES) + u % 2;
      const bool ok = ks < ksteps && ks * 32 + g * 8 < K;
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
        if (!(ok && a_ok[mb])) a[u][mb] = zero;
    }
#pragma unroll
    for (int u = 0; u < U; ++u)
#pragma unroll
      for (int mb = 0; mb < MB; ++mb)
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
          acc[mb][nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u][mb], b[u][nb], acc[mb][nb], 0, 0, 0);
  };
  // A later round's loads of W stand together behind one branch: a branch for each step, among A's loads, made each of them wait for every load
  // before it.  Not so (`BY_STEP`) where a round's loads of W are many, so that a first step waits long for the last step's: with four column blocks (together ->
  // a branch a step: 17 and 32 rows of 50,304 x 768 21.4 -> 20.3 and 22.4 -> 21.2 us; 24 of 33,000 x 2,080 41.2 -> 37.8, 64 56.4 -> 50.1), with two and four
  // steps (250 rows of 1,600 x 3,104 11.6 -> 11.0), and with twelve row blocks (160 rows of 1,600 x 4,128 19.9 -> 18.5; of 4,800 x 1,632, where K is no
  // multiple of 32, 11.9 -> 13.1).  Nor, with eight steps, where the norm's statistics are left (33 rows of 1,600 x 4,096 8.4 -> 8.1, of 1,024 x 4,096 6.5 -> 6.4, no other K differs).
  constexpr bool BY_STEP = (NORM == NORM_OUT && U == 8) || (NORM == NORM_NONE && (NB == 4 || (NB == 2 && U == 4) || (MB == 12 && WAVES == 8)));
  for (int p0 = wave; 2 * p0 < ksteps; p0 += WAVES * (U / 2)) {
    if constexpr (BY_STEP) {
#pragma unroll
      for (int u = 0; u < U; ++u) {
        const int ks = 2 * (p0 + (u / 2) * WAVES) + u % 2;
        const bool ok = ks < ksteps && ks * 32 + g * 8 < K;
        if (p0 != wave) {
#pragma unroll
          for (int nb = 0; nb < NB; ++nb)
            b[u][nb] = *reinterpret_cast<const bf16x8*>(ks < ksteps ? wblk[nb] + ks * 512 : no_step(lane));
        }
#pragma unroll
        for (int mb = 0; mb < MB; ++mb)
          a[u][mb] = *reinterpret_cast<const bf16x8*>(ok ? arow[mb] + ks * astep : asafe[mb]);
      }
    } else {
      if (p0 != wave) ask_w(p0);
      ask_a(p0);
    }
    if constexpr (NORM == NORM_IN) {
      if (p0 == wave) join_stats();
    }
    use(p0);
  }
#pragma unroll
  for (int mb = 0; mb < MB; ++mb)
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) red[wave][mb * NB + nb][lane] = acc[mb][nb];
  __syncthreads();
  // acc[mb][nb][r] of lane (col, g) is row mb*16 + g*4 + r, column n0 + nb*16 + col
#pragma unroll
  for (int p = 0; p < PASSES; ++p) {
    const int blk = wave + p * WAVES;
    if (blk >= BLOCKS) break;
    const int mb = blk / NB, nb = blk % NB;
    const int nn = n0 + nb * 16 + col;
    floatx4 s = red[0][blk][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) s += red[w][blk][lane];
    if constexpr (NORM == NORM_OUT) {
      // a row's 16 columns of this block lie in the 16 lanes of a row of lanes (N is a multiple of 16)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = epi_x[p][r] + (s[r] + epi_bias[p]);
        const float2 stats = columns_stats(x);
        const int m = row0 + mb * 16 + g * 4 + r;
        if (col == 0 && m < M)
          *reinterpret_cast<float2*>(late.stats_out + (static_cast<size_t>(m) * nblocks + blockIdx.x * NB + nb) * 2) = stats;
      }
    }
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      int m = row0 + mb * 16 + g * 4 + r;
      if (m >= M || nn >= N) continue;
      float v = s[r] + epi_bias[p];
      if constexpr (NORM == NORM_IN) v = (s[r] - rowstat[m - row0][0] * epi_norm[p]) * rowstat[m - row0][1] + epi_bias[p];
      if (resid) {
        resid[static_cast<size_t>(m) * ldr + nn] = epi_x[p][r] + v;
        if constexpr (NORM == NORM_OUT)
          late.copy_out[late.ldcopy > 0 ? static_cast<size_t>(m) * late.ldcopy + nn : packed_index(m, nn, N / 32)] =
              from_float<bf16_t>((epi_x[p][r] + v) * epi_norm[p]);
      } else {
        TC cv = from_float<TC>(end_value<TC, END>(v, late.epi, nn, late.ends, epi_act[END != END_PLAIN ? p : 0]));
        if constexpr (END == END_TWO) {
          if (nn < late.ends.cols)
            late.ends.C2[static_cast<size_t>(m) * late.ends.ldc2 + nn] = from_float<bf16_t>(v);
          else
            C[static_cast<size_t>(m) * late.ldc + nn - late.ends.cols] = cv;
          continue;
        }
        if (!KV || nn < late.kv.c_cols)
          C[(packed & PACKED_C) ? packed_index(m, nn, N / 32) : static_cast<size_t>(m) * late.ldc + nn] = cv;
        if constexpr (KV) scatter_kv_at(late.kv, epi_slot[p][r], nn, cv);
      }
    }
  }
}

struct First {
  int rows;
  const void* p;
  const void* q;
};
static First first_of(const Call& c, const NormIO& nio, int norm) {
  if (norm == NORM_IN)
    return First{c.M, nio.stats_in, c.kv ? c.kv->slot_map : nullptr};
  return First{c.M | (c.resid ? FIRST_ADDS : 0), c.resid ? static_cast<const void*>(c.resid) : c.C, reinterpret_cast<const void*>(static_cast<uintptr_t>(c.resid ? c.ldr : c.ldc))};
}
template <int END>
static Late<END> late_of(const Call& c, const NormIO& nio) {
  return Late<END>{c.C, c.ldc, c.epi, nio.c1, nio.eps, nio.no_mean, nio.gamma_out, nio.copy_out, nio.stats_out, nio.ldcopy,
                   c.kv ? *c.kv : KVScatter{}, EndsOf<END>(c.ends)};
}

// Up to 16 rows of A in rows.  In the operands' layout 16 lanes are 16 rows, and a load of A from
// memory touches as many cache lines (four times as many lookups as the packed W costs, and they
// were what this product of 8 rows waited for).  Here a wave takes the steps of K in pairs
// (wave w: steps 2w, 2w + 1, then 2 (w + WAVES), ...), so that a row's share of a pair is one cache
// line of 128 bytes; it loads A eight lanes to a row, turns each pair round through a piece of LDS
// of its own (no barrier: a wave's LDS operations keep their order) and reads the operands from
// there, two pairs at a time through two such pieces, so that the way into LDS and out of it is
// waited for once per two pairs.  16 columns per workgroup, sums joined through LDS in wave order, as in gemm_kernel.
template <int WAVES, int U, typename TC, bool KV, int NORM, bool TWO, int END = END_PLAIN, bool SHORT = false>
__global__ __launch_bounds__(WAVES * 64) void gemm16_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int lda, int rows, int N,
                                                             int K, const void* __restrict__ p, const float* __restrict__ bias, const void* __restrict__ q,
                                                             Late<END> late) {
  typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
  const int M = rows & FIRST_ROWS;
  TC* C = static_cast<TC*>(NORM == NORM_IN ? late.C : const_cast<void*>(p));
  float* resid = NORM != NORM_IN && (rows & FIRST_ADDS) ? static_cast<float*>(const_cast<void*>(p)) : nullptr;
  const int ldc = NORM == NORM_IN ? late.ldc : static_cast<int>(reinterpret_cast<uintptr_t>(q)), ldr = ldc;
  const float* stats_in = static_cast<const float*>(p);
  const int32_t* slot_map = NORM == NORM_IN ? static_cast<const int32_t*>(q) : late.kv.slot_map;
  constexpr int ROW = 9 * 8;                               // elements per row of a wave's piece: 8 chunks and one of padding
  __shared__ floatx4 red[WAVES][64];
  constexpr int PIECES = U < 2 ? 1 : 2;                    // pairs turned round at a time
  __shared__ __attribute__((aligned(16))) bf16_t turn[WAVES][PIECES][16 * ROW];
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int col = lane % 16, g = lane / 16;
  const int n0 = blockIdx.x * 16;
  if constexpr (END == END_PAIR)
    if (n0 >= late.ends.cols) A += late.ends.a_shift;
  const int ksteps = (K + 31) / 32, npairs = (ksteps + 1) / 2, nblocks = (N + 15) / 16;
  const bf16_t* wblk = W + (static_cast<size_t>(min(static_cast<int>(blockIdx.x), nblocks - 1)) * ksteps * 64 + lane) * 8;
  // (TWO: rows 8 .. 15 need a second load per pair)
  // NORM_IN: the rows' pairs of statistics are asked for before the operands (loads come back in the
  // order asked): wave w joins rows w, w + WAVES, ...; a lane holds up to SP pairs of a row
  // (SHORT: K = 2,048 at most, so no load of a place that cannot be there)
  constexpr int SP = SHORT ? 2 : 4, SR = (TWO ? 16 : 8) / WAVES;
  __shared__ float rowstat[16][2];
  // what the epilogue will read is asked for first of all (wave 0 finishes the block)
  float epi_bias = 0.f;
  float epi_x[4] = {0.f, 0.f, 0.f, 0.f};
  int epi_slot[4] = {-1, -1, -1, -1};
  float2 epi_act{0.f, 0.f};
  const int blocks_in = K / 16;      // (NORM_IN)
  if (wave == 0) {
    const int nn = min(n0 + col, N - 1);
    if (bias) epi_bias = bias[nn];
    if constexpr (KV) {
#pragma unroll
      for (int r = 0; r < 4; ++r) epi_slot[r] = g * 4 + r < M ? slot_map[g * 4 + r] : -1;
    }
    if (resid) {
#pragma unroll
      for (int r = 0; r < 4; ++r) epi_x[r] = resid[static_cast<size_t>(min(g * 4 + r, M - 1)) * ldr + nn];
    }
  }
  // (after the epilogue's loads and before the operands': they are back before the operands are)
  float2 st[SR][SP];
  float epi_c1 = 0.f, epi_gamma = 1.f;
  if constexpr (NORM == NORM_IN) {
#pragma unroll
    for (int t = 0; t < SR; ++t) {
      const size_t row = static_cast<size_t>(min(wave + t * WAVES, M - 1)) * blocks_in;
#pragma unroll
      for (int i = 0; i < SP; ++i) st[t][i] = *reinterpret_cast<const float2*>(stats_in + (row + min(lane + 64 * i, blocks_in - 1)) * 2);
    }
  }
  // never a conditional load; a step beyond K reads zeros and meets zeros of A
  const int lrow = lane / 8, lch = lane % 8;               // as loader: row and 16-byte chunk of the pair's 128 bytes
  const bf16_t* a0 = A + static_cast<size_t>(min(lrow, M - 1)) * lda + lch * 8;
  const bf16_t* a1 = A + static_cast<size_t>(min(lrow + 8, M - 1)) * lda + lch * 8;
  // a chunk beyond K is not loaded; its load goes to the start of the row instead, which is surely inside A (a0
  // itself is not where K < 64: chunk lch of a row of 32 elements lies in the next row, the last row's beyond A)
  const bf16_t* asafe = A + static_cast<size_t>(min(lrow, M - 1)) * lda;
  bf16_t* mine = turn[wave][0];
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  // a round: U pairs of steps per wave, all its loads issued at once (asking for the next round
  // before this one is used, into a second set of registers, was slower)
  auto ask = [&](int p0, bf16x8 (*b)[2], u32x4 (*al)[2]) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * WAVES, ks = 2 * p;
      b[u][0] = *reinterpret_cast<const bf16x8*>(ks < ksteps ? wblk + ks * 512 : no_step(lane));
      b[u][1] = *reinterpret_cast<const bf16x8*>(ks + 1 < ksteps ? wblk + (ks + 1) * 512 : no_step(lane));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int p = p0 + u * WAVES;
      const bool ok = p * 64 + lch * 8 < K;
      al[u][0] = *reinterpret_cast<const u32x4*>(ok ? a0 + p * 64 : asafe);
      if constexpr (TWO) al[u][1] = *reinterpret_cast<const u32x4*>(ok ? a1 + p * 64 : asafe);
    }
  };
  auto use = [&](int p0, const bf16x8 (*b)[2], const u32x4 (*al)[2]) {
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += PIECES) {
#pragma unroll
      for (int i = 0; i < PIECES && u0 + i < U; ++i) {
        const int p = p0 + (u0 + i) * WAVES;
        const bool ok = p < npairs && p * 64 + lch * 8 < K;
        bf16_t* piece = mine + i * 16 * ROW;
        *reinterpret_cast<u32x4*>(piece + lrow * ROW + lch * 8) = ok ? al[u0 + i][0] : zero4;
        if constexpr (TWO) *reinterpret_cast<u32x4*>(piece + (lrow + 8) * ROW + lch * 8) = ok ? al[u0 + i][1] : zero4;
      }
      // as operand: lane (row col, chunk g) of each of a pair's two steps
      bf16x8 f[PIECES][2];
#pragma unroll
      for (int i = 0; i < PIECES && u0 + i < U; ++i) {
        const bf16_t* piece = mine + i * 16 * ROW;
        f[i][0] = *reinterpret_cast<const bf16x8*>(piece + col * ROW + g * 8);
        f[i][1] = *reinterpret_cast<const bf16x8*>(piece + col * ROW + (4 + g) * 8);
      }
#pragma unroll
      for (int i = 0; i < PIECES && u0 + i < U; ++i) {
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[i][0], b[u0 + i][0], acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[i][1], b[u0 + i][1], acc, 0, 0, 0);
      }
    }
  };
  bf16x8 b0[U][2];
  u32x4 al0[U][2];
  // NORM_IN: the first round is asked for by every wave, with or without steps of its own (so that the
  // wait for the statistics, which were asked for before, counts these loads exactly and depends on
  // no branch), and the rows' statistics are joined while it travels
  if (NORM == NORM_IN || wave < npairs) ask(wave, b0, al0);
  // what the epilogue reads by arguments that do not come with the launch (`Late`): behind the operands, which do not wait for those
  const int late_column = min(n0 + col, N - 1);
  if constexpr (NORM == NORM_IN) epi_c1 = late.c1[late_column];
  if constexpr (NORM == NORM_OUT) epi_gamma = late.gamma_out[late_column];
  if constexpr (END != END_PLAIN) epi_act = end_numbers<TC, END>(late.ends, late_column);
  late_at_hand<NORM, KV>(late);
  if constexpr (NORM == NORM_IN) {
    // the rows' means and 1 / sqrt(var + eps) for wave 0, which meets them behind the barrier further down
    const float blocks = static_cast<float>(blocks_in);      // of 16 columns
#pragma unroll
    for (int t = 0; t < SR; ++t) {
      const int row = wave + t * WAVES;
      float sm = 0.f;
#pragma unroll
      for (int i = 0; i < SP; ++i)
        if (lane + 64 * i < blocks_in) sm += st[t][i].x;
      const float mean = late.no_mean ? 0.f : wave_sum(sm) / blocks;      // (without it the squares are taken about 0)
      float sq = 0.f;
#pragma unroll
      for (int i = 0; i < SP; ++i)
        if (lane + 64 * i < blocks_in) {
          const float d = st[t][i].x - mean;
          sq += st[t][i].y + 16.f * d * d;
        }
      const float var = wave_sum(sq) / (16.f * blocks);
      if (lane == 0) {
        rowstat[row][0] = row < M ? mean : 0.f;
        rowstat[row][1] = row < M ? 1.0f / sqrtf(var + late.eps) : 0.f;
      }
    }
  }
  for (int p0 = wave; p0 < npairs; p0 += WAVES * U) {
    if (p0 != wave) ask(p0, b0, al0);
    use(p0, b0, al0);
  }
  red[wave][lane] = acc;
  __syncthreads();
  // acc[r] of lane (col, g) is row g*4 + r, column n0 + col
  if (wave == 0) {
    const int nn = n0 + col;
    floatx4 sm = red[0][lane];
#pragma unroll
    for (int w = 1; w < WAVES; ++w) sm += red[w][lane];
#pragma unroll
    for (int r = 0; r < 4; ++r) {
      const int m = g * 4 + r;
      if (m >= M || nn >= N) continue;
      float v = sm[r] + epi_bias;
      if constexpr (NORM == NORM_IN) v = (sm[r] - rowstat[m][0] * epi_c1) * rowstat[m][1] + epi_bias;
      if (resid) {
        resid[static_cast<size_t>(m) * ldr + nn] = epi_x[r] + v;
        if constexpr (NORM == NORM_OUT)
          late.copy_out[static_cast<size_t>(m) * late.ldcopy + nn] = from_float<bf16_t>((epi_x[r] + v) * epi_gamma);
      } else {
        const TC cv = from_float<TC>(end_value<TC, END>(v, late.epi, nn, late.ends, epi_act));
        if constexpr (END == END_TWO) {
          if (nn < late.ends.cols)
            late.ends.C2[static_cast<size_t>(m) * late.ends.ldc2 + nn] = from_float<bf16_t>(v);
          else
            C[static_cast<size_t>(m) * ldc + nn - late.ends.cols] = cv;
          continue;
        }
        if (!KV || nn < late.kv.c_cols) C[static_cast<size_t>(m) * ldc + nn] = cv;
        if constexpr (KV) scatter_kv_at(late.kv, epi_slot[r], nn, cv);
      }
    }
    if constexpr (NORM == NORM_OUT) {
      // a row's 16 columns of this block lie in the 16 lanes of a row of lanes (N is a multiple of 16)
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const float x = epi_x[r] + (sm[r] + epi_bias);
        const float2 stats = columns_stats(x);
        const int m = g * 4 + r;
        if (col == 0 && m < M)
          *reinterpret_cast<float2*>(late.stats_out + (static_cast<size_t>(m) * nblocks + blockIdx.x) * 2) = stats;
      }
    }
  }
}


constexpr int ROW_ROTATE_8 = 0x128;      // (DPP: lane i of each 16 takes from lane i - 8 of the same 16)

// Up to 8 rows of a product with few columns: gemm16_kernel with 8 columns a workgroup.  A CU takes 50 to 60 GB/s of what its XCD's L2 does not
// hold, whatever it asks for ahead, so a workgroup of 16 columns waits for its own share of W (205 KB at K = 6,400) while half of the
// CUs have none.  A pair of steps is one load of W: lanes l % 16 < 8 bring 8 columns of the first step, the others the same
// columns of the second.  The product of the second step takes them with the halves of every 16 lanes exchanged; what columns 8 .. 15 of the
// results add up to is nothing and is dropped.  A column's sums are gemm16_kernel's, in its order: the same bits.  A lane ends one element.
template <int WAVES, int U, typename TC>
__global__ __launch_bounds__(WAVES * 64) void gemm8_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int lda, int rows, int N, int K,
                                                            const void* __restrict__ p, const float* __restrict__ bias, const void* __restrict__ q,
                                                            Late<END_PLAIN> late) {
  typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
  const int M = rows & FIRST_ROWS, ldc = static_cast<int>(reinterpret_cast<uintptr_t>(q)), ldr = ldc;
  TC* C = static_cast<TC*>(const_cast<void*>(p));
  float* resid = rows & FIRST_ADDS ? static_cast<float*>(const_cast<void*>(p)) : nullptr;
  constexpr int ROW = 9 * 8;                               // elements per row of a wave's piece: 8 chunks and one of padding
  constexpr int PIECES = U < 2 ? 1 : 2;                    // pairs turned round at a time
  __shared__ floatx4 red[WAVES][64];
  __shared__ __attribute__((aligned(16))) bf16_t turn[WAVES][PIECES][8 * ROW];
  // (the wave's number not as a scalar: the compiler then puts a pair's loads behind a branch, and each is waited for by itself)
  const int wave = threadIdx.x / 64, lane = threadIdx.x % 64;
  const int col = lane % 16, g = lane / 16, second = col / 8;
  const int n0 = blockIdx.x * 8, nn = n0 + lane % 8, mm = lane / 8;      // (the element that a lane of the first wave ends)
  const int ksteps = (K + 31) / 32, npairs = (ksteps + 1) / 2;
  const bf16_t* wblk = W + (static_cast<size_t>(blockIdx.x / 2) * ksteps * 64 + g * 16 + (blockIdx.x % 2) * 8 + col % 8) * 8;
  // what the epilogue will read is asked for first of all
  float epi_bias = 0.f, epi_x = 0.f;
  if (wave == 0) {
    const int c = min(nn, N - 1);
    if (bias) epi_bias = bias[c];
    if (resid) epi_x = resid[static_cast<size_t>(min(mm, M - 1)) * ldr + c];
  }
  // never a conditional load; a step beyond K reads zeros and meets zeros of A, whose chunks beyond K come from the row's start
  const int lrow = lane / 8, lch = lane % 8;               // as loader: row and 16-byte chunk of the pair's 128 bytes
  const bf16_t* asafe = A + static_cast<size_t>(min(lrow, M - 1)) * lda;
  const bf16_t* a0 = asafe + lch * 8;
  bf16_t* mine = turn[wave][0];
  const u32x4 zero4 = {0u, 0u, 0u, 0u};
  floatx4 acc = {0.f, 0.f, 0.f, 0.f};
  u32x4 b[U], al[U];
  auto ask = [&](int p0) {
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int step = 2 * (p0 + u * WAVES) + second;
      b[u] = *reinterpret_cast<const u32x4*>(step < ksteps ? wblk + static_cast<size_t>(step) * 512 : no_step(lane));
    }
#pragma unroll
    for (int u = 0; u < U; ++u) {
      const int at = p0 + u * WAVES;
      al[u] = *reinterpret_cast<const u32x4*>(at * 64 + lch * 8 < K ? a0 + at * 64 : asafe);
    }
  };
  if (wave < npairs) ask(wave);
  // behind the operands, as in gemm16_kernel
  late_at_hand<NORM_NONE, false>(late);
  for (int p0 = wave; p0 < npairs; p0 += WAVES * U) {
    if (p0 != wave) ask(p0);
#pragma unroll
    for (int u0 = 0; u0 < U; u0 += PIECES) {
#pragma unroll
      for (int i = 0; i < PIECES && u0 + i < U; ++i) {
        const int pair = p0 + (u0 + i) * WAVES;
        *reinterpret_cast<u32x4*>(mine + i * 8 * ROW + lrow * ROW + lch * 8) = pair < npairs && pair * 64 + lch * 8 < K ? al[u0 + i] : zero4;
      }
      // as operand: lane (row col, chunk g) of each of a pair's two steps; rows 8 .. 15 are the others again, their results nothing's
      bf16x8 f[PIECES][2];
#pragma unroll
      for (int i = 0; i < PIECES && u0 + i < U; ++i) {
        const bf16_t* piece = mine + i * 8 * ROW + (col % 8) * ROW;
        f[i][0] = *reinterpret_cast<const bf16x8*>(piece + g * 8);
        f[i][1] = *reinterpret_cast<const bf16x8*>(piece + (4 + g) * 8);
      }
#pragma unroll
      for (int i = 0; i < PIECES && u0 + i < U; ++i) {
        u32x4 other;
#pragma unroll
        for (int e = 0; e < 4; ++e)
          other[e] = static_cast<uint32_t>(__builtin_amdgcn_update_dpp(0, static_cast<int>(b[u0 + i][e]), ROW_ROTATE_8, 0xf, 0xf, true));
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[i][0], __builtin_bit_cast(bf16x8, b[u0 + i]), acc, 0, 0, 0);
        acc = __builtin_amdgcn_mfma_f32_16x16x32_bf16(f[i][1], __builtin_bit_cast(bf16x8, other), acc, 0, 0, 0);
      }
    }
  }
  red[wave][lane] = acc;
  __syncthreads();
  // acc[r] of lane (col, g) is row g*4 + r, column n0 + col
  if (wave > 0) return;
  const float* at = reinterpret_cast<const float*>(&red[0][(mm / 4) * 16 + lane % 8]) + mm % 4;
  float sum = at[0];
#pragma unroll
  for (int w = 1; w < WAVES; ++w) sum += at[w * 64 * 4];
  const float v = sum + epi_bias;
  if (mm >= M || nn >= N) return;
  if (resid) {
    resid[static_cast<size_t>(mm) * ldr + nn] = epi_x + v;
  } else {
    C[static_cast<size_t>(mm) * ldc + nn] = from_float<TC>(apply_epilogue_fast(v, late.epi));
  }
}


template <int MB, int NB, int WAVES, int U, typename TC, bool KV, int END = END_PLAIN>
static void launch_one(const Call& c, hipStream_t stream) {
  // (MB row blocks per workgroup: where the rows need more, the second grid dimension shares them out)
  dim3 grid((c.N + 16 * NB - 1) / (16 * NB), ((c.M + 15) / 16 + MB - 1) / MB), block(WAVES * 64);
  hipLaunchKernelGGL((gemm_kernel<MB, NB, WAVES, U, TC, KV, NORM_NONE, END>), grid, block, 0, stream,
                     static_cast<const bf16_t*>(c.A), static_cast<const bf16_t*>(c.W), c.lda, c.M, c.N, c.K, c.packed, c.ldr, c.resid, c.bias,
                     late_of<END>(c, NormIO{}));
}

// the same with the norm before the product (NORM_IN: bfloat16 out) or after it (NORM_OUT: into the
// residual stream), for 17 to 64 rows
template <int MB, int NB, int WAVES, int U>
static void launch_norm(const Call& c, const NormIO& nio, int norm, hipStream_t stream) {
  dim3 grid((c.N + 16 * NB - 1) / (16 * NB), ((c.M + 15) / 16 + MB - 1) / MB), block(WAVES * 64);
#define DN_LN(TC, KV, NORM)                                                                                        \
  hipLaunchKernelGGL((gemm_kernel<MB, NB, WAVES, U, TC, KV, NORM>), grid, block, 0, stream,                       \
                     static_cast<const bf16_t*>(c.A), static_cast<const bf16_t*>(c.W), c.lda, c.M, c.N, c.K, c.packed, c.ldr, \
                     NORM == NORM_IN ? static_cast<const void*>(nio.stats_in) : c.resid, c.bias, late_of<END_PLAIN>(c, nio))
  if (norm == NORM_OUT) {
    DN_LN(float, false, NORM_OUT);
  } else if constexpr (U <= 8) {      // (K of 2,048 at most: four pairs a wave)
    if (c.kv)
      DN_LN(bf16_t, true, NORM_IN);
    else
      DN_LN(bf16_t, false, NORM_IN);
  }
#undef DN_LN
}

// 17 to 64 rows with a norm inside: the shapes that launch_mb picks for these rows (8 waves: K >= 1024)
void launch_mb_norm(const Call& c, const NormIO& nio, int norm, hipStream_t stream) {
  const int mb = (c.M + 15) / 16;
  if (c.N >= 2560) {
    switch (mb) {
      // (four steps in flight a wave; with six and the statistics in LDS, 64 rows of 3,840 x 1,280 9.3 -> 10.3 us, 4,800 x 1,600 level)
      case 2: return launch_norm<2, 2, 8, 4>(c, nio, norm, stream);
      case 3: return launch_norm<3, 2, 8, 4>(c, nio, norm, stream);
      default: return launch_norm<4, 2, 8, 4>(c, nio, norm, stream);
    }
  }
  // (few columns: the rows in two halves, so that there are workgroups for all CUs)
  // A wave's share of K in whole rounds of five pairs where it is that many (64 rows of 1,280 x 5,120, two rounds for three: 10.7 -> 9.5 us), else in rounds of four.
  if (norm == NORM_OUT && ((c.K + 63) / 64 + 7) / 8 % 5 == 0) return launch_norm<2, 1, 8, 10>(c, nio, norm, stream);
  return launch_norm<2, 1, 8, 8>(c, nio, norm, stream);
}

template <int MB, int NB, int WAVES, int U>
static void launch(const Call& c, hipStream_t stream) {
  if constexpr (MB <= 4) {      // (up to 64 rows: what the entry points take)
    if (c.end == END_ACT && c.out_dtype == DN_BF16) return launch_one<MB, NB, WAVES, U, bf16_t, false, END_ACT>(c, stream);
    if (c.end == END_ACT) return launch_one<MB, NB, WAVES, U, float, false, END_ACT>(c, stream);
    if (c.end == END_TWO) return launch_one<MB, NB, WAVES, U, float, false, END_TWO>(c, stream);
    if (c.end == END_PAIR) return launch_one<MB, NB, WAVES, U, float, false, END_PAIR>(c, stream);
  }
  if (c.kv) return launch_one<MB, NB, WAVES, U, bf16_t, true>(c, stream);
  if (c.out_dtype == DN_BF16) return launch_one<MB, NB, WAVES, U, bf16_t, false>(c, stream);
  return launch_one<MB, NB, WAVES, U, float, false>(c, stream);
}

// the pairs in flight per wave that make its share of K whole rounds of at most `most` (loads of what is not there cost as much as the
// others)
template <int WAVES>
static int pairs_ahead(int K, int most) {
  const int share = ((K + 63) / 64 + WAVES - 1) / WAVES, rounds = (share + most - 1) / most;
  return (share + rounds - 1) / rounds;
}

// Four pairs ahead at most.  (Always four before -> as many as the share wants, 8 rows: 4,096 x 1,024 4.3 -> 4.0 us, 50,257 x 1,024 27.5 -> 23.8,
// x 1,280 31.8 -> 28.7, 32,000 x 1,024 18.7 -> 16.0; with the norm before, 3,072 x 1,024 4.6 -> 4.3, 5,120 x 1,280 6.9 -> 6.6; K = 1,600 and 2,048 level.)
template <int WAVES, int U, typename TC, bool KV, int NORM, int END>
static void launch16_ahead(const Call& c, const NormIO& nio, hipStream_t stream) {
  const First f = first_of(c, nio, NORM);
#define DN_L16(TWO, SHORT)                                                                                               \
  hipLaunchKernelGGL((gemm16_kernel<WAVES, U, TC, KV, NORM, TWO, END, SHORT>), dim3((c.N + 15) / 16), dim3(WAVES * 64), 0,       \
                     stream, static_cast<const bf16_t*>(c.A), static_cast<const bf16_t*>(c.W), c.lda, f.rows, c.N, c.K,   \
                     f.p, c.bias, f.q, late_of<END>(c, nio))
  if (c.M > 8)
    DN_L16(true, false);
  else if (NORM == NORM_IN && c.K <= 2048)
    DN_L16(false, NORM == NORM_IN);
  else
    DN_L16(false, false);
#undef DN_L16
}

template <int WAVES, typename TC, bool KV, int NORM = NORM_NONE, int END = END_PLAIN>
static void launch16_one(const Call& c, const NormIO& nio, hipStream_t stream) {
  const int ahead = pairs_ahead<WAVES>(c.K, 4);
  if constexpr (WAVES == 4) {      // (eight waves: K of 1,024 and more, at least two pairs each)
    if (ahead == 1) return launch16_ahead<WAVES, 1, TC, KV, NORM, END>(c, nio, stream);
  }
  switch (ahead) {
    case 2: return launch16_ahead<WAVES, 2, TC, KV, NORM, END>(c, nio, stream);
    case 3: return launch16_ahead<WAVES, 3, TC, KV, NORM, END>(c, nio, stream);
    default: return launch16_ahead<WAVES, 4, TC, KV, NORM, END>(c, nio, stream);
  }
}

// Where gemm8_kernel runs: up to 8 rows of at most 2,048 columns, whose 256 workgroups the chip has CUs for (beyond, 16 columns a workgroup
// give every CU its own too, and read A half as often: 2,304 columns from K = 9,216 at 8 rows 13.6 us so, 16 to 17 in eights).
static bool eight_columns(int M, int N) { return M <= 8 && N <= 2048; }

// The pairs in flight per wave are as many as make its share of K whole rounds: loads of what is not there cost as much as the others
// (with statistics, at 8 rows, 1,024 x 1,024 3.1 us with 2, 3.5 with 4, 4.2 with 8; 1,024 x 4,096 5.1, 4.8, 4.8; 1,600 x 6,400 9.3, 9.2, 8.3 and 8.1 with 6).
// gemm16_kernel -> this, into the stream, 1 and 8 rows: 1,024 x 1,024 3.0 -> 2.8 and 3.6 -> 2.9 us, 1,600 x 1,600 3.6 -> 3.5 and 4.4 -> 3.7,
// 1,024 x 4,096 5.0 -> 4.7 and 6.0 -> 5.3, 1,280 x 5,120 6.4 -> 5.4 and 7.7 -> 5.9, 1,600 x 6,400 8.4 -> 7.1 and 9.6 -> 7.9, 2,048 x 8,192 9.7 -> 9.1 and 12.7 -> 9.7.
template <int WAVES, typename TC>
static void launch8(const Call& c, hipStream_t stream) {
  const First f = first_of(c, NormIO{}, NORM_NONE);
#define DN_L8(U)                                                                                                          \
  case U:                                                                                                                 \
    hipLaunchKernelGGL((gemm8_kernel<WAVES, U, TC>), dim3((c.N + 7) / 8), dim3(WAVES * 64), 0, stream,                    \
                       static_cast<const bf16_t*>(c.A), static_cast<const bf16_t*>(c.W), c.lda, f.rows, c.N, c.K, f.p,    \
                       c.bias, f.q, late_of<END_PLAIN>(c, NormIO{}));                                                     \
    break
  const int ahead = pairs_ahead<WAVES>(c.K, 8);
  if constexpr (WAVES == 4) {      // (K below 1,024: at most four pairs a wave; eight waves have at least two)
    switch (ahead) {
      DN_L8(1);
      DN_L8(2);
      DN_L8(3);
      DN_L8(4);
    }
  } else {
    switch (ahead) {
      DN_L8(2);
      DN_L8(3);
      DN_L8(4);
      DN_L8(5);
      DN_L8(6);
      DN_L8(7);
      DN_L8(8);
    }
  }
#undef DN_L8
}

// the same with the norm before the product (NORM_IN: bfloat16 out) or after it (NORM_OUT: into the residual stream)
template <int WAVES>
static void launch16_norm(const Call& c, const NormIO& nio, int norm, hipStream_t stream) {
  if (norm == NORM_OUT) return launch16_one<WAVES, float, false, NORM_OUT>(c, nio, stream);
  if (c.kv) return launch16_one<WAVES, bf16_t, true, NORM_IN>(c, nio, stream);
  return launch16_one<WAVES, bf16_t, false, NORM_IN>(c, nio, stream);
}

template <int WAVES>
static void launch16(const Call& c, hipStream_t stream) {
  const NormIO none{};
  if (c.end == END_ACT && c.out_dtype == DN_BF16) return launch16_one<WAVES, bf16_t, false, NORM_NONE, END_ACT>(c, none, stream);
  if (c.end == END_ACT) return launch16_one<WAVES, float, false, NORM_NONE, END_ACT>(c, none, stream);
  if (c.end == END_TWO) return launch16_one<WAVES, float, false, NORM_NONE, END_TWO>(c, none, stream);
  if (c.end == END_PAIR) return launch16_one<WAVES, float, false, NORM_NONE, END_PAIR>(c, none, stream);
  if (c.kv) return launch16_one<WAVES, bf16_t, true>(c, none, stream);
  if (c.out_dtype == DN_BF16) return launch16_one<WAVES, bf16_t, false>(c, none, stream);
  return launch16_one<WAVES, float, false>(c, none, stream);
}

// With more than 16 rows every workgroup reads all of A (16 cache lines per load and 16 lanes,
// as A lies in rows), so wider workgroups read less in total, as long as enough of them remain
// to keep the memory system busy: 2 column blocks per workgroup from 2,560 columns on (with 2,304 columns
// that way was the slower), 4 from 32,768 on, else 1.
template <int WAVES>
static void launch_mb(const Call& c, hipStream_t stream) {
  const int mb = (c.M + 15) / 16;
  // 65 to 256 rows of a product with few columns and a short K (an output projection): four row blocks and two
  // column blocks per workgroup, the rows shared out among workgroups (at 1,600 x 1,600: 6.7 us at 128 rows and 8.0
  // at 256, where sixteen row blocks x one column block took 7.7 and 12.6: every workgroup read all rows)
  if (mb > 4 && c.N < 2048 && c.K < 4096) return launch<4, 2, WAVES, 4>(c, stream);
  if (mb == 1 && !(c.packed & (PACKED_A | PACKED_C)) && eight_columns(c.M, c.N) && !c.kv && c.end == END_PLAIN) {
    if (c.out_dtype == DN_BF16 && !c.resid) return launch8<WAVES, bf16_t>(c, stream);
    return launch8<WAVES, float>(c, stream);
  }
  // (one row too, since this kernel asks for whole rounds only: 50,257 x 1,024 27.3 -> 22.1 us, 32,000 x 1,024 18.4 -> 15.1, 4,096 x 1,024 4.0 -> 3.9)
  if (mb == 1 && !(c.packed & (PACKED_A | PACKED_C))) return launch16<WAVES>(c, stream);
  if (mb == 1) return launch<1, 1, WAVES, 8>(c, stream);
  if (mb > 4) {
    // 65 to 256 rows: 16 columns per workgroup, the waves' sums for all row blocks through LDS
    // (the tiled kernel has too few tiles to fill the chip at so few rows, and walks a long K in
    // as many steps whatever M is)
    if (mb <= 6) return launch<6, 1, WAVES, 2>(c, stream);
    if (mb <= 8) return launch<8, 1, WAVES, 2>(c, stream);
    if (mb <= 12) return launch<12, 1, WAVES, 2>(c, stream);
    return launch<16, 1, WAVES, 2>(c, stream);
  }
  if (c.N >= 32768) {
    switch (mb) {
      case 2: return launch<2, 4, WAVES, 4>(c, stream);
      case 3: return launch<3, 4, WAVES, 4>(c, stream);
      default: return launch<4, 4, WAVES, 4>(c, stream);
    }
  }
  if (c.N >= 2560) {
    // (six steps in flight a wave: with K = 1,600 a wave's seven steps are one round and a step, where four in
    // flight made two rounds: 4,800 and 6,400 columns at 64 rows 10.3 -> 9.6 and 10.0 -> 9.1 us)
    switch (mb) {
      case 2: return launch<2, 2, WAVES, 6>(c, stream);
      case 3: return launch<3, 2, WAVES, 6>(c, stream);
      default: return launch<4, 2, WAVES, 6>(c, stream);
    }
  }
  // (few columns: the rows in two halves, so that there are workgroups for all CUs)
  return launch<2, 1, WAVES, 8>(c, stream);
}

void run(const Call& c, hipStream_t stream) {
  if (c.K >= 1024)
    launch_mb<8>(c, stream);
  else
    launch_mb<4>(c, stream);
}

// A must allow 16-byte loads: in rows with K and lda multiples of 8 and the base aligned, or packed
// (K a multiple of 32 then: nothing zeroes a packed block's columns beyond K); W is packed
bool takes(const void* A, int lda, const void* W, int M, int K, int packed) {
  if (M > 256 || reinterpret_cast<uintptr_t>(A) % 16 != 0 || reinterpret_cast<uintptr_t>(W) % 16 != 0) return false;
  return (packed & PACKED_A) ? K % 32 == 0 : (K % 8 == 0 && lda % 8 == 0);
}

// up to 16 rows with a norm inside, by the number of waves a workgroup (8: K >= 1024, else 4)
void launch16_norm_of(int waves, const Call& c, const NormIO& nio, int norm, hipStream_t stream) {
  if (waves == 8)
    launch16_norm<8>(c, nio, norm, stream);
  else
    launch16_norm<4>(c, nio, norm, stream);
}
}  // namespace skinny
