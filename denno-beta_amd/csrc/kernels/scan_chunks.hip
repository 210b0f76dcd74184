// The recurrences of a matrix state per head, for portions of prompts: sixteen rows of a request at a time, on the matrix cores in 32-bit.
//   delta rule:      S <- w S;  e = beta (v - S^T k);  S <- S + k e^T;  o = S^T r        (S [dk, dv] per head, row after row of a request;
//   constant decay:  S <- w S + k v^T;  o = S^T r                                        w per row and key channel, per row, or constant)
// With S_0 the state before such a chunk and f(t, j) the product of the decays of the rows j + 1 .. t (of a channel), the rows of a chunk obey
//   e_t = beta_t (v_t - sum_i k_t,i f(t, -1)_i S_0,i - sum_{j<t} m(t, j) e_j),   m(t, j) = sum_i k_t,i f(t, j)_i k_j,i
// which is (I + M) E = diag(beta) V - diag(beta) (K o F) S_0 with M strictly lower triangular, so that with X = (I + M)^-1 diag(beta)
//   E = U - W S_0,   U = X V,   W = X (K o F)        (constant decay: E = V, no W)
//   o_t = (r_t o f(t, -1))^T S_0 + sum_{j<=t} P[t, j] e_j,   P[t, j] = sum_i r_t,i f(t, j)_i k_j,i
//   S   = f(15, -1) o S_0 + sum_t (k_t o f(15, t)) e_t^T
// Everything but S_0 is known before the walk: one kernel makes U, W, P, r o F, the weighed keys and the chunk's decay of all chunks side by
// side, a second walks a request's chunks in order.
// In the first kernel the products of decays (which run along the rows: never a quotient, so a decay of zero is one), the sums of P and M, X and
// U are 64-bit and rounded once; W is 32-bit, and so are P's and M's sums and U where a row has one decay.  (All of it in 32-bit: 2 us less of 30, outputs 1.04e-7 from the 64-bit ones for 0.88e-7.)  A
// chunk's decay goes on as two 32-bit numbers: rounded to one, a decay that is the same in every chunk would be off the same way in each of the
// hundreds that a state lives for (4.9e-7 for 0.7e-7).
// The walk's products are v_mfma_f32_16x16x4_f32: operands, sums and state are 32-bit.  Its sums are short (the key channels in four parts, a
// chunk's rows by themselves, the state touched once a chunk instead of sixteen times), so results are nearer to the 64-bit ones than a walk
// row by row.  2-norms of the distance, 64 x 128, 46 to 1,000 rows, in units of 1e-7, outputs and states: a decay per channel 0.85 to 0.90 and
// 0.9 to 1.0 for 0.90 to 1.12 and 1.1 to 1.4; constant ones 0.63 to 0.67 and 0.7 for 0.7 to 0.9 and 1.1 to 2.2.
// Lane l of a wave holds, of an A operand, row l % 16 and, in register i of four, column 4 (l / 16) + i of each 16; of a B operand
// the same of its transpose; of a result, rows 4 (l / 16) + i of column l % 16: a result serves as the B operand of the next product as it
// lies.  The first kernel writes every operand as the walk's lanes hold it, 16 bytes a lane.
#include "common.h"

namespace {

typedef __attribute__((__vector_size__(4 * sizeof(float)))) float f32x4;
constexpr int L = 16;                                       // rows of a chunk
enum { DELTA_WIDE = 0, DELTA_ROWS = 1, FADE_HEAD = 2 };     // a decay per row and channel, per row (made from its argument), one for the head

__device__ __forceinline__ f32x4 mfma(float a, float b, f32x4 c) { return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0); }

// what stands in LDS is read here, not earlier (all of a triangle's numbers read ahead take more registers than there are)
__device__ __forceinline__ void not_before() {
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// every wave's LDS traffic is done and no wave is behind; loads from memory stay on their way (__syncthreads would wait for them)
__device__ __forceinline__ void meet() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// The chunks of request s have the numbers from chunk_base(s) on: room for as many as its rows can make.
__device__ __forceinline__ int chunk_base(const int* row_start, int s) { return row_start[s] / L + s; }

struct ChunkArgs {
  const float *r, *k, *v, *zb, *w, *rate, *bias;      // (w: decays per channel; the decay's argument; a number per head)
  size_t ldr, ldk, ldv, ldb, ldw;
  float* state;
  size_t slot_stride;
  const int *row_start, *slots;
  int S, H, G, dk, dv, chunks, rows_min;      // (requests of fewer than rows_min rows are another kernel's)
  float* work;
  float* out;
  size_t ldo;
};

// What the first kernel leaves for a chunk and head, in floats: P, r o F, weighed keys, decay (and what its rounding left), W, U
template <int DB>
struct Record {
  static constexpr int DK = 16 * DB, P = 0, R = L * L, KT = R + L * DK, HI = KT + L * DK, LO = HI + DK, W = LO + DK, U = W + L * DK;
  __device__ __forceinline__ static size_t floats(int dv) { return U + static_cast<size_t>(L) * ((dv + 15) / 16 * 16); }
};
static long long record_floats(int dk, int dv) { return L * L + 3LL * L * dk + 2 * dk + static_cast<long long>(L) * ((dv + 15) / 16 * 16); }

template <int CTRL>
__device__ __forceinline__ double dpp_move64(double v) {
  const int2 h = __builtin_bit_cast(int2, v);
  return __builtin_bit_cast(double, int2{__builtin_amdgcn_update_dpp(0, h.x, CTRL, 0xf, 0xf, true), __builtin_amdgcn_update_dpp(0, h.y, CTRL, 0xf, 0xf, true)});
}

// A number of lane i's and one of lane i ^ d's, each lane keeping the half of what both have that its bit d names: over all four steps
// lane i of 16 is left with the sum of x[i]
template <int CTRL, int HALF>
__device__ __forceinline__ void share_out(double* x, bool upper) {
#pragma unroll
  for (int k = 0; k < HALF; ++k) {
    const double keep = upper ? x[k + HALF] : x[k], give = upper ? x[k] : x[k + HALF];
    x[k] = keep + dpp_move64<CTRL>(give);
  }
}
__device__ __forceinline__ double sums_of_16(double* x, int lane) {
  share_out<DN_DPP_MIRROR, 8>(x, lane & 8);
  share_out<DN_DPP_HALF_MIRROR, 4>(x, lane & 4);
  share_out<DN_DPP_XOR2, 2>(x, lane & 2);
  share_out<DN_DPP_XOR1, 1>(x, lane & 1);
  return x[0];
}

// Whether no lane of the wave has an infinity or what is no number.  Rows of a chunk that come before others have zeros in their places in X and P;
// a matrix product multiplies those too, and what is no number in a later row must not reach the rows before it: then sums go by the rows that a row has.
__device__ __forceinline__ bool all_numbers(f32x4 x) {
  const float inf = __builtin_huge_valf();
  return __ballot(!(fabsf(x[0]) < inf && fabsf(x[1]) < inf && fabsf(x[2]) < inf && fabsf(x[3]) < inf)) == 0;
}

// A workgroup a chunk and head.  The pairs (t, j) of rows: a wave takes four rows j, 16 lanes a row, which carry k_j along the rows t while
// it fades.  Then the first wave solves for X, a column a lane, while the others weigh queries and keys, a channel a thread; then the
// W and U are made, 16 columns a wave and time.
template <int DB, int MODE>
__global__ __launch_bounds__(256, 4) void chunk_parts_kernel(ChunkArgs a) {
  typedef Record<DB> Rec;
  constexpr int DK = 16 * DB;
  constexpr bool WIDE = MODE == DELTA_WIDE, ROWS = MODE == DELTA_ROWS, DELTA = MODE != FADE_HEAD;
  // (rows of LDS 16 bytes longer than a head: 16 rows are then read from different banks)
  __shared__ __attribute__((aligned(16))) float sk[L][DK + 4], sr[L][DK + 4], sw[WIDE ? L : 1][DK + 4], P[L][L + 4], X[L][L + 4];
  __shared__ __attribute__((aligned(16))) double MT[DELTA ? L : 1][L];
  __shared__ double beta[L], fade[L];
  const int id = blockIdx.x, h = blockIdx.y, tid = threadIdx.x, lane = tid % 64, wave = __builtin_amdgcn_readfirstlane(tid / 64);
  const int g = lane / 16, n = lane % 16;
  int s = -1;      // the last request whose numbers begin at or before id, 64 of them asked for at a time
  for (int s0 = 0; s0 < a.S; s0 += 64) {
    const unsigned long long before = __ballot(s0 + lane < a.S && chunk_base(a.row_start, min(s0 + lane, a.S - 1)) <= id);
    s += __popcll(before);
    if (before != ~0ull) break;
  }
  if (s < 0) return;
  const int base = chunk_base(a.row_start, s), begin = a.row_start[s], end = a.row_start[s + 1], row0 = begin + L * (id - base), rows = min(L, end - row0);
  if (rows <= 0 || end - begin < a.rows_min || a.slots[s] < 0) return;
  const int hq = h / (a.H / a.G), dv = a.dv, vblocks = (dv + 15) / 16;
  float* rec = a.work + (static_cast<size_t>(id) * a.H + h) * Rec::floats(dv);
  // rows beyond the last: r = 0, k = 0, w = 1, beta = 0, which change nothing
  {
    float tk[DB], tr[DB], tw[DB];
#pragma unroll
    for (int q = 0; q < DB; ++q) {
      const int at = tid + 256 * q, t = at / DK, i = at % DK;
      const size_t row = row0 + min(t, rows - 1);
      tk[q] = a.k[row * a.ldk + hq * DK + i];
      tr[q] = a.r[row * a.ldr + hq * DK + i];
      if constexpr (WIDE) tw[q] = a.w[row * a.ldw + static_cast<size_t>(h) * DK + i];
    }
    if (tid < L) {
      const size_t row = row0 + min(tid, rows - 1);
      const bool mine = tid < rows;
      double f = 1.0, b = 0.0;
      if constexpr (MODE == DELTA_ROWS) f = exp(static_cast<double>(-a.rate[h] * softplus_f(a.w[row * a.ldw + h] + (a.bias ? a.bias[h] : 0.f))));
      if constexpr (MODE == FADE_HEAD) f = a.w[h];
      if constexpr (DELTA) b = 1.0f / (1.0f + expf(-a.zb[row * a.ldb + h]));
      beta[tid] = mine ? b : 0.0;
      fade[tid] = mine ? f : 1.0;
    }
#pragma unroll
    for (int q = 0; q < DB; ++q) {
      const int at = tid + 256 * q, t = at / DK, i = at % DK;
      const bool ok = t < rows;
      sk[t][i] = ok ? tk[q] : 0.f;
      sr[t][i] = ok ? tr[q] : 0.f;
      if constexpr (WIDE) sw[t][i] = ok ? tw[q] : 1.f;
    }
  }
  meet();
  if constexpr (ROWS) {
    // (a decay that all channels share stands outside the sums, which the matrix cores then make)
    if (wave < 2) {
      f32x4 even = {0.f, 0.f, 0.f, 0.f}, odd = even;
#pragma unroll
      for (int b = 0; b < DB; ++b) {
        const f32x4 k = *reinterpret_cast<const f32x4*>(&sk[n][16 * b + 4 * g]), x = wave == 0 ? k : *reinterpret_cast<const f32x4*>(&sr[n][16 * b + 4 * g]);
#pragma unroll
        for (int i = 0; i < 4; i += 2) {
          even = mfma(x[i], k[i], even);
          odd = mfma(x[i + 1], k[i + 1], odd);
        }
      }
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const int t = 4 * g + i, j = n;
        double f = even[i] + odd[i];
#pragma unroll
        for (int q = 1; q < L; ++q) f *= q > j && q <= t ? fade[q] : 1.0;
        if (wave == 0)
          MT[j][t] = t > j ? beta[t] * f : 0.0;
        else
          P[t][j] = t >= j ? static_cast<float>(f) : 0.f;
      }
    }
  } else {
    const int j = 4 * g + wave, i0 = n * DB;
    double x[DB], m[L], p[L];
#pragma unroll
    for (int q = 0; q < DB; ++q) x[q] = sk[j][i0 + q];
#pragma unroll
    for (int t = 0; t < L; ++t) {
      m[t] = p[t] = 0.0;
      const double f = WIDE || t <= j ? 1.0 : fade[t];
#pragma unroll
      for (int q = 0; q < DB; ++q) {
        if constexpr (WIDE)
          x[q] *= t > j ? sw[t][i0 + q] : 1.f;
        else
          x[q] *= f;
        if constexpr (DELTA) m[t] = fma(static_cast<double>(sk[t][i0 + q]), x[q], m[t]);
        p[t] = fma(static_cast<double>(sr[t][i0 + q]), x[q], p[t]);
      }
      asm volatile("" : "+v"(m[t]), "+v"(p[t])::"memory");      // (sums are made here, or the operands of all of them are kept)
    }
    const double pt = sums_of_16(p, n);      // (row t = n)
    P[n][j] = n >= j ? static_cast<float>(pt) : 0.f;
    if constexpr (DELTA) {
      const double mt = sums_of_16(m, n);
      MT[j][n] = n > j ? beta[n] * mt : 0.0;
    }
  }
  // (the wave's first blocks of values are on their way while X is solved for; rows 4 g + i, a column a lane)
  constexpr int AHEAD = 2;
  auto values = [&](int block) {
    f32x4 x;
    const size_t col = static_cast<size_t>(h) * dv + min(block * 16 + n, dv - 1);
#pragma unroll
    for (int i = 0; i < 4; ++i) x[i] = a.v[(row0 + min(4 * g + i, rows - 1)) * a.ldv + col];
    return x;
  };
  f32x4 ahead[AHEAD];
#pragma unroll
  for (int q = 0; q < AHEAD; ++q) ahead[q] = values(min(wave + 4 * q, vblocks - 1));
  meet();
  if (DELTA && wave == 0) {
    // (the four groups of lanes do the same work and store the same)
    double x[L];
#pragma unroll
    for (int t = 0; t < L; ++t) x[t] = t == n ? 1.0 : 0.0;
#pragma unroll
    for (int j = 0; j < L - 1; ++j) {
#pragma unroll
      for (int t = j + 1; t < L; ++t) x[t] = fma(-MT[DELTA ? j : 0][t], x[j], x[t]);
      asm volatile("" : "+v"(x[L - 1]), "+v"(x[j + 1])::"memory");
    }
#pragma unroll
    for (int t = 0; t < L; ++t) X[t][n] = t >= n ? static_cast<float>(x[t] * beta[n]) : 0.f;      // (a later row's beta may be no number)
  } else if (tid >= 64 && tid - 64 < DK) {
    const int i = tid - 64, b = i / 16;
    double f = 1.0;
    float k[L];
#pragma unroll
    for (int t = 0; t < L; ++t) {
      f *= WIDE ? static_cast<double>(sw[WIDE ? t : 0][i]) : fade[t];
      k[t] = sk[t][i];
      sr[t][i] = static_cast<float>(sr[t][i] * f);
      if constexpr (DELTA) sk[t][i] = static_cast<float>(k[t] * f);
    }
    const float whole = static_cast<float>(f);
    rec[Rec::HI + i] = whole;
    rec[Rec::LO + i] = static_cast<float>(f - static_cast<double>(whole));
    f = 1.0;
    f32x4 kt[4];
#pragma unroll
    for (int t = L - 1; t >= 0; --t) {
      kt[t / 4][t % 4] = static_cast<float>(k[t] * f);
      f *= WIDE ? static_cast<double>(sw[WIDE ? t : 0][i]) : fade[t];
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) *reinterpret_cast<f32x4*>(rec + Rec::KT + (b * 64 + q * 16 + i % 16) * 4) = kt[q];
  }
  meet();
  if (wave == 3) *reinterpret_cast<f32x4*>(rec + Rec::P + lane * 4) = *reinterpret_cast<const f32x4*>(&P[n][4 * g]);
  for (int b = wave; b < DB; b += 4)
    *reinterpret_cast<f32x4*>(rec + Rec::R + (b * 64 + lane) * 4) = *reinterpret_cast<const f32x4*>(&sr[n][16 * b + 4 * g]);
  f32x4 xf;
  if constexpr (DELTA) {
    // (W is wanted turned round: weighed keys times X, both turned round)
    xf = *reinterpret_cast<const f32x4*>(&X[n][4 * g]);
    for (int b = wave; b < DB; b += 4) {
      f32x4 w = {0.f, 0.f, 0.f, 0.f}, k;
#pragma unroll
      for (int i = 0; i < 4; ++i) k[i] = sk[4 * g + i][16 * b + n];
      if (all_numbers(k)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) w = mfma(k[i], xf[i], w);
      } else {
#pragma unroll 1
        for (int j = 0; j <= n; ++j) w += X[n][j] * *reinterpret_cast<const f32x4*>(&sk[j][16 * b + 4 * g]);
      }
      *reinterpret_cast<f32x4*>(rec + Rec::W + (b * 64 + lane) * 4) = w;
    }
  }
  auto finish = [&](int block, f32x4 v) {
    f32x4 u;
#pragma unroll
    for (int i = 0; i < 4; ++i) v[i] = 4 * g + i < rows ? v[i] : 0.f;
    if constexpr (DELTA) {
      double e[4] = {0.0, 0.0, 0.0, 0.0};
      const bool plain = all_numbers(v);
      if (ROWS && plain) {
        u = f32x4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int i = 0; i < 4; ++i) u = mfma(xf[i], v[i], u);
      } else if (plain) {
#pragma unroll
        for (int j = 0; j < L; ++j) {
          const double vj = __shfl(v[j % 4], j / 4 * 16 + n);
#pragma unroll
          for (int i = 0; i < 4; ++i) e[i] = fma(static_cast<double>(X[4 * g + i][j]), vj, e[i]);
          asm volatile("" : "+v"(e[0]), "+v"(e[1]), "+v"(e[2]), "+v"(e[3]));
        }
      } else {
#pragma unroll 1
        for (int j = 0; j < L; ++j) {
          const double vj = __shfl(j % 4 == 0 ? v[0] : j % 4 == 1 ? v[1] : j % 4 == 2 ? v[2] : v[3], j / 4 * 16 + n);
#pragma unroll
          for (int i = 0; i < 4; ++i)
            if (j <= 4 * g + i) e[i] = fma(static_cast<double>(X[4 * g + i][j]), vj, e[i]);
        }
      }
      if (!ROWS || !plain) {
#pragma unroll
        for (int i = 0; i < 4; ++i) u[i] = static_cast<float>(e[i]);
      }
    } else {
      u = v;
    }
    *reinterpret_cast<f32x4*>(rec + Rec::U + (block * 64 + lane) * 4) = u;
  };
#pragma unroll
  for (int q = 0; q < AHEAD; ++q)
    if (wave + 4 * q < vblocks) finish(wave + 4 * q, ahead[q]);
  for (int b = wave + 4 * AHEAD; b < vblocks; b += 4) finish(b, values(b));
}

// The waves of a workgroup of the walk that hold the state: one for each 16 key channels up to 64, for each 32 beyond
template <int DB>
struct Walk {
  static constexpr int KB = (DB + 3) / 4, WAVES = (DB + KB - 1) / KB;
};

// A workgroup a head and 16 value columns of a request; a wave holds KB blocks of 16 key channels of the state in its registers, and one wave more
// makes the outputs.  A chunk is a chain: the waves' parts of W S_0 meet in LDS, E, the weighed keys times E, the state.  So a wave has as few of a chunk's
// products as four of them can have, r o F times S_0 is made while the parts meet, and the outputs a chunk behind the state; operands are asked for D
// chunks ahead (a trip to memory is as long as several chunks).
template <int DB, bool DELTA>
__global__ __launch_bounds__((Walk<DB>::WAVES + 1) * 64) void chunk_walk_kernel(ChunkArgs a) {
  typedef Record<DB> Rec;
  constexpr int DK = 16 * DB, KB = Walk<DB>::KB, WAVES = Walk<DB>::WAVES, D = 4;
  __shared__ f32x4 parts_e[2][WAVES][64], parts_o[2][WAVES][64];
  __shared__ float rows_e[L][L], rows_p[L][L], rows_x[L][L];
  const int h = blockIdx.x, s = blockIdx.z, lane = threadIdx.x % 64, wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int g = lane / 16, n = lane % 16;
  const int slot = a.slots[s];
  if (slot < 0) return;
  const int row0 = a.row_start[s], row1 = a.row_start[s + 1];
  if (row0 >= row1 || row1 - row0 < a.rows_min) return;
  const int dv = a.dv, col = blockIdx.y * 16 + n;
  const bool live = col < dv;
  const int chunks = (row1 - row0 + L - 1) / L;
  const size_t floats = Rec::floats(dv), stride = floats * a.H;
  const float* rec = a.work + static_cast<size_t>(chunk_base(a.row_start, s)) * stride + h * floats;
  const uint32_t mine4 = 4 * lane, group4 = 4 * g;
  const f32x4 zero = {0.f, 0.f, 0.f, 0.f};
  // (a scalar base, the lane's place in 32 bits: no address is worked out lane by lane)
  auto load = [](const float* p, uint32_t at) { return *reinterpret_cast<const f32x4*>(p + at); };
  auto record = [&](int m) { return rec + static_cast<size_t>(min(m, chunks - 1)) * stride; };
  // U less the waves' parts of W S_0, the same in every wave
  auto errors = [&](int m, f32x4 u) {
    if constexpr (DELTA) {
      f32x4 x = parts_e[m & 1][0][lane];
      if constexpr (WAVES == 2) x += parts_e[m & 1][1][lane];
      if constexpr (WAVES == 3) x = (x + parts_e[m & 1][1][lane]) + parts_e[m & 1][2][lane];
      if constexpr (WAVES == 4) x = (x + parts_e[m & 1][1][lane]) + (parts_e[m & 1][2][lane] + parts_e[m & 1][3][lane]);
      return u - x;
    }
    return u;
  };
  if (wave < WAVES) {
    struct Operands { f32x4 w[KB], r[KB], kt[KB], hi[KB], lo[KB], u; };
    f32x4 S[KB];      // S[b][i]: key channel 16 (wave KB + b) + 4 g + i of column n
    int blk[KB];
    bool mine[KB];
    float* sp = a.state + static_cast<size_t>(slot) * a.slot_stride + (static_cast<size_t>(h) * dv + min(col, dv - 1)) * DK + 4 * g;
#pragma unroll
    for (int b = 0; b < KB; ++b) {
      blk[b] = min(wave * KB + b, DB - 1);
      mine[b] = wave * KB + b < DB;      // (a block beyond the last: zeros that stay zeros)
      // (a head's state may begin at any number of floats)
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float x = sp[16 * blk[b] + i];
        S[b][i] = mine[b] ? x : 0.f;
      }
    }
    auto fetch = [&](int m) {
      Operands q;
      const float* p = record(m);
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        if constexpr (DELTA) q.w[b] = load(p + Rec::W + blk[b] * 256, mine4);
        q.r[b] = load(p + Rec::R + blk[b] * 256, mine4);
        q.kt[b] = load(p + Rec::KT + blk[b] * 256, mine4);
        q.hi[b] = load(p + Rec::HI + blk[b] * 16, group4);
        q.lo[b] = load(p + Rec::LO + blk[b] * 16, group4);
      }
      q.u = load(p + Rec::U + blockIdx.y * 256, mine4);
      return q;
    };
    Operands ring[D];
#pragma unroll
    for (int d = 0; d < D; ++d) {
      ring[d] = fetch(d);
      not_before();      // (in the order of their use)
    }
    auto step = [&](int m, Operands& q) {
      f32x4 o = zero;
      if constexpr (DELTA) {
        f32x4 e = zero;
#pragma unroll
        for (int b = 0; b < KB; ++b)
#pragma unroll
          for (int i = 0; i < 4; ++i) e = mfma(q.w[b][i], S[b][i], e);
        parts_e[m & 1][wave][lane] = e;
      }
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i) o = mfma(q.r[b][i], S[b][i], o);
      meet();
      const f32x4 E = errors(m, q.u);
#pragma unroll
      for (int b = 0; b < KB; ++b) {
        f32x4 x = zero;
#pragma unroll
        for (int i = 0; i < 4; ++i) x = mfma(q.kt[b][i], E[i], x);
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          // (Without the delta rule, which makes of an infinity what is no number, it stays one: as it is, times what the decay's rounding left, which may be
          // nothing or less, it would not.  The largest number in its place in that product: three requests of 2,136 rows 41.1 -> 42.4 us.)
          const float rest = DELTA ? S[b][i] : __builtin_amdgcn_fmed3f(S[b][i], -__FLT_MAX__, __FLT_MAX__), y = fmaf(S[b][i], q.hi[b][i], fmaf(rest, q.lo[b][i], x[i]));
          S[b][i] = mine[b] ? y : 0.f;
        }
      }
      parts_o[m & 1][wave][lane] = o;
      q = fetch(m + D);
    };
    // (whole rounds of D and a rest, no way out of the middle: where there is one the compiler takes it for a way round as well, and waits for
    // more operands than it must)
    int m0 = 0;
    for (; m0 + D <= chunks; m0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) step(m0 + d, ring[d]);
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
      if (m0 + d < chunks) step(m0 + d, ring[d]);
    meet();
    if (live) {
#pragma unroll
      for (int b = 0; b < KB; ++b)
#pragma unroll
        for (int i = 0; i < 4; ++i)
          if (mine[b]) sp[16 * blk[b] + i] = S[b][i];
    }
  } else {
    struct Operands { f32x4 p, u; } ring[D];
    auto fetch = [&](int m) {
      const float* p = record(m);
      return Operands{load(p + Rec::P, mine4), load(p + Rec::U + blockIdx.y * 256, mine4)};
    };
    f32x4 before = zero;      // the last chunk's share of its own rows
    // (stores without a branch, which those beyond the rows and columns miss: behind a branch the compiler no longer knows how many
    // operands are on their way, and waits for all)
    const int ldo = static_cast<int>(a.ldo), mine = live ? 4 * (4 * g * ldo + n) : INT32_MIN;
    auto finish = [&](int m) {
      f32x4 o = parts_o[m & 1][0][lane];
      if constexpr (WAVES == 2) o += parts_o[m & 1][1][lane];
      if constexpr (WAVES == 3) o = (o + parts_o[m & 1][1][lane]) + parts_o[m & 1][2][lane];
      if constexpr (WAVES == 4) o = (o + parts_o[m & 1][1][lane]) + (parts_o[m & 1][2][lane] + parts_o[m & 1][3][lane]);
      o += before;
      const int first = row0 + L * m, rows = min(L, row1 - first);
      float* to = a.out + static_cast<size_t>(first) * a.ldo + static_cast<size_t>(h) * dv + blockIdx.y * 16;
      const __amdgpu_buffer_rsrc_t there = __builtin_amdgcn_make_buffer_rsrc(to, 0, 4 * ((rows - 1) * ldo + min(16, dv - static_cast<int>(blockIdx.y) * 16)), 0x00020000);
#pragma unroll
      for (int i = 0; i < 4; ++i) __builtin_amdgcn_raw_buffer_store_b32(__float_as_uint(o[i]), there, mine + 4 * i * ldo, 0, 0);
    };
#pragma unroll
    for (int d = 0; d < D; ++d) {
      ring[d] = fetch(d);
      not_before();
    }
    auto step = [&](int m, Operands& q) {
      meet();
      if (m > 0) finish(m - 1);
      f32x4 E = errors(m, q.u);
      if (!live) E = zero;
      f32x4 x = zero;
      if (all_numbers(E)) {
#pragma unroll
        for (int i = 0; i < 4; ++i) x = mfma(q.p[i], E[i], x);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) rows_e[4 * g + i][n] = E[i], rows_p[n][4 * g + i] = q.p[i];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll 1
        for (int t = 4 * g; t < 4 * g + 4; ++t) {
          float y = 0.f;
#pragma unroll 1
          for (int j = 0; j <= t; ++j) y = fmaf(rows_p[t][j], rows_e[j][n], y);
          rows_x[t][n] = y;
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
        for (int i = 0; i < 4; ++i) x[i] = rows_x[4 * g + i][n];
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      }
      before = x;
      q = fetch(m + D);
    };
    int m0 = 0;
    for (; m0 + D <= chunks; m0 += D) {
#pragma unroll
      for (int d = 0; d < D; ++d) step(m0 + d, ring[d]);
    }
#pragma unroll
    for (int d = 0; d < D - 1; ++d)
      if (m0 + d < chunks) step(m0 + d, ring[d]);
    meet();
    finish(chunks - 1);
  }
}

template <int DB, int MODE>
void launch(const ChunkArgs& a, hipStream_t stream) {
  hipLaunchKernelGGL((chunk_parts_kernel<DB, MODE>), dim3(a.chunks, a.H), dim3(256), 0, stream, a);
  // (heads side by side: where they are as many as the XCDs, a head's workgroups, which read the same operands, share an L2)
  hipLaunchKernelGGL((chunk_walk_kernel<DB, MODE != FADE_HEAD>), dim3(a.H, (a.dv + 15) / 16, a.S), dim3((Walk<DB>::WAVES + 1) * 64), 0, stream, a);
}

template <int MODE>
int launch_of(const ChunkArgs& a, hipStream_t stream) {
  switch (a.dk) {
    case 16: launch<1, MODE>(a, stream); break;
    case 32: launch<2, MODE>(a, stream); break;
    case 48: launch<3, MODE>(a, stream); break;
    case 64: launch<4, MODE>(a, stream); break;
    case 80: launch<5, MODE>(a, stream); break;
    case 96: launch<6, MODE>(a, stream); break;
    case 112: launch<7, MODE>(a, stream); break;
    case 128: launch<8, MODE>(a, stream); break;
    default: return DN_ERR_SHAPE;
  }
  return dn_launch_status();
}

}  // namespace

extern "C" {

int dn_state_scan(const float* r, long long ldr, const float* k, long long ldk, const float* v, long long ldv, const float* w,
                  long long ldw, const float* u, const float* beta, long long ldb, const float* w_head, int G, float* state,
                  long long slot_stride, const int* row_start, const int* slots, int S, int T, int H, int dk, int dv, int mode,
                  int key_from_decay, int beta_logits, int w_rows, const float* w_rate, const float* w_bias, int rows_below, float* out,
                  long long ldo, hipStream_t stream);      // (sequence.hip)

// floats of scratch that dn_scan_chunks needs for a step of T rows of S requests
long long dn_scan_chunks_floats(int T, int S, int H, int dk, int dv) {
  return (static_cast<long long>(T) / L + S) * H * record_floats(dk, dv);
}

// r, k [T, G dk], v, out [T, H dv], 32-bit; dk a multiple of 16 up to 128; work: dn_scan_chunks_floats floats, at a multiple of 16 bytes.
// mode 0: the delta rule, beta = sigmoid(zb [T, H]), decays w [T, H dk]; 1: the same, log decay = -rate softplus(w [T, H] + bias);
// 2: a constant decay per head, w [H], no delta rule (zb none).  Requests of fewer than rows_min rows are walked row by row (0: none are) by a launch of
// dn_state_scan's kernel: in this call, since a call of its own for them cost a step outside the graphs 30 us a layer, most of it in checks on the host.
int dn_scan_chunks(const float* r, long long ldr, const float* k, long long ldk, const float* v, long long ldv, const float* zb, long long ldb,
                   const float* w, long long ldw, const float* rate, const float* bias, int mode, float* state, long long slot_stride,
                   const int* row_start, const int* slots, int S, int T, int H, int G, int dk, int dv, int rows_min, float* work, float* out,
                   long long ldo, hipStream_t stream) {
  if (dk < 16 || dk > 128 || dk % 16 != 0 || dv < 1 || H < 1 || G < 1 || H % G != 0 || S < 1 || S > 65535 || H > 65535 || (dv + 15) / 16 > 65535 ||
      reinterpret_cast<uintptr_t>(work) % 16 != 0 || slot_stride < static_cast<long long>(H) * dk * dv || ldo >= (1LL << 24) || rows_min < 0 || mode < DELTA_WIDE || mode > FADE_HEAD ||
      !w || (mode != FADE_HEAD) != (zb != nullptr) || (mode == DELTA_ROWS) != (rate != nullptr))
    return DN_ERR_SHAPE;
  if (T == 0) return 0;
  const ChunkArgs a{r, k, v, zb, w, rate, bias, static_cast<size_t>(ldr), static_cast<size_t>(ldk), static_cast<size_t>(ldv), static_cast<size_t>(ldb),
                    static_cast<size_t>(ldw), state, static_cast<size_t>(slot_stride), row_start, slots, S, H, G, dk, dv, T / L + S, rows_min, work, out,
                    static_cast<size_t>(ldo)};
  const int rc = mode == DELTA_WIDE ? launch_of<DELTA_WIDE>(a, stream) : mode == DELTA_ROWS ? launch_of<DELTA_ROWS>(a, stream) : launch_of<FADE_HEAD>(a, stream);
  if (rc != 0 || rows_min == 0) return rc;
  const bool head = mode == FADE_HEAD;
  return dn_state_scan(r, ldr, k, ldk, v, ldv, head ? nullptr : w, ldw, nullptr, zb, ldb, head ? w : nullptr, G, state, slot_stride, row_start, slots, S, T, H, dk,
                       dv, head ? 1 : 2, 0, !head, mode == DELTA_ROWS, rate, bias, rows_min, out, ldo, stream);
}

}  // extern "C"
