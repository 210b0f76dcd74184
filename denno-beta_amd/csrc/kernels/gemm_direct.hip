#include "gemm_common.h"

// ---------------------------------------------------------------------------------------
// Many rows, bfloat16, slabs carried from memory straight into LDS (global_load_lds_dwordx4: 16
// bytes per lane, lane l's at the wave's LDS address + 16 l, no register and no LDS store between).
// A slab of 32 along K is a list of 1 KB blocks in the packed layout, 16 rows x 32 columns each:
// a block of W is 1 KB of memory as it lies and is read back at 16 l by lane l; rows of A are put in place by the load
// itself, in an order of its own.  Where a stage has two slabs (K a multiple of 64), 1 KB of A is 8 rows x 128 bytes: whole cache
// lines.  From the L2 into LDS a CU takes 110 GB/s in pieces of 1 KB, 105 so, and 68 where a load takes 64 bytes from each of 16
// rows, which is what a stage of one slab leaves (16 lanes then take 64 bytes from each of four rows: with a lane per row the
// lookups, 52 per load on average, kept the vector cache busy for three quarters of the kernel's time).  64 bytes a row
// everywhere -> whole lines: 320 x 3,840 x 1,280 15.9 -> 13.7 us; 3,500 x 1,280 x 5,120 88.6 -> 70.0; 8,192 x 3,840 x 1,280
// 110.4 -> 98.4; 8,192 x 6,400 x 1,600 201.5 -> 194; 2,048 x 4,800 x 1,600 44.4 -> 42.8.  Tiles whose last rows are missing had
// their loads nearly free before (a missing row reads the last one again) and lose 1 to 8 % where K is a power of two
// (65 x 2,048 x 8,192 34.3 -> 36.7, 400 x 3,072 x 1,024 10.7 -> 11.1); whole tiles of the same widths gain 4 to 10 %.  Two slabs a
// stage for tiles of 192 and more columns with a long K too, against one slab in more stages: 8,192 x 1,600 x 6,400
// 169.5 -> 161.  The 16-byte pieces of a row are exchanged by the row's number so that the operand read (lane l wants row
// l % 16, piece l / 16) meets every bank once: LDS serves lanes 0-3, 12-15 and 20-27 together, 4-11, 16-19 and 28-31, and the
// same 32 lanes on (an order that is free of conflicts for 16 lanes in a row only was slower by 0.3 us a product of 512 rows).
// STAGES stages of KB slabs are in flight (vmcnt counts a wave's own loads; one barrier per stage publishes them and frees the
// stage read before).
//
// The MFMA takes W as its first operand and A as its second: a lane then holds four consecutive
// columns of one row of C, which it stores as 8 bytes (bfloat16) or adds as 16 (the 32-bit
// residual) without a turn through LDS; for the fused QKV product they are one key's or one
// value's four dims.
//
// What bounds these products here is not the matrix cores (busy 30 % of the time with eight waves a workgroup)
// but a wave's chain of loads, waits and barriers, and the rounding of tiles to 256 CUs.  Measured per tile and
// slab with eight waves: time = 2.26e-7 us x BM x BN (matrix cores at nine tenths of their peak) + 3.07e-5 us x
// (BM + BN) (loads), the two adding up rather than overlapping, + 1.9e-4 us x BM x BN for the stores at the end.
// (Measured with 64 bytes of a row of A a load; whole lines shorten the loads' share, by more for narrow tiles.)
// The tile is chosen per product from a list, by that model: the largest that still fills the chip in whole
// rounds (a tile count just above a multiple of 256 costs a whole further round); and the waves of a workgroup
// are as many as give every SIMD four (see `run`), so that one of them can issue while the others wait.
// ---------------------------------------------------------------------------------------
namespace direct {
typedef __attribute__((__vector_size__(8 * sizeof(__bf16)))) __bf16 bf16x8;
typedef __attribute__((__vector_size__(4 * sizeof(float)))) float floatx4;
typedef __attribute__((__vector_size__(4 * sizeof(uint32_t)))) uint32_t u32x4;
typedef floatx4 floatx4_at_4 __attribute__((aligned(4)));
constexpr int XCDS = 8, CUS = 256, LDS_PER_CU = 160 * 1024;

// element `which` (0..3, the lane's own choice) of the vector that lane E of this lane's quad holds
template <int E>
__device__ __forceinline__ float quad_pick(const floatx4& v, int which) {
  const float b0 = dpp_move<0x55 * E>(v[0]), b1 = dpp_move<0x55 * E>(v[1]), b2 = dpp_move<0x55 * E>(v[2]),
              b3 = dpp_move<0x55 * E>(v[3]);
  return which == 0 ? b0 : which == 1 ? b1 : which == 2 ? b2 : b3;
}

// four values rounded to bfloat16, as the 8 bytes of one store (built in registers: an array that
// is read back through a pointer of another type can end up in scratch memory)
__device__ __forceinline__ uint2 pack4(float a, float b, float c, float d) {
  return uint2{static_cast<uint32_t>(from_float<bf16_t>(a).bits) | static_cast<uint32_t>(from_float<bf16_t>(b).bits) << 16,
               static_cast<uint32_t>(from_float<bf16_t>(c).bits) | static_cast<uint32_t>(from_float<bf16_t>(d).bits) << 16};
}

template <int N>
__device__ __forceinline__ void wait_loads() {      // until at most N of this wave's loads are in flight
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(N) : "memory");
}

// Tiles in the order in which a run of them shares most: bands of about 1,024 rows, a band column by column.  Each of the 8 XCDs,
// among which workgroups go round, takes a run of that order, so that the 32 tiles that its CUs work on at a time are some four by
// eight and its L2 fetches their rows and columns once.  (With whole columns of tiles one after the other an XCD fetched all rows of A
// for every column: 8,192 x 1,280 x 5,120 brought 685 MB into the L2s, now 220; 112 -> 103 us, 8,192 x 6,400 x 1,600 222 -> 197.)
__device__ __forceinline__ void tile_at(int pid, int tiles_m, int tiles_n, int band, int& tm, int& tn) {
  const int total = tiles_m * tiles_n, each = total / XCDS, more = total % XCDS, x = pid % XCDS;
  pid = x * each + min(x, more) + pid / XCDS;
  if (tiles_m <= band) {      // (few rows: one band, and a division less in front of a short kernel)
    tm = pid % tiles_m;
    tn = pid / tiles_m;
    return;
  }
  const int in_band = band * tiles_n, b = pid / in_band, first = b * band, rows = min(band, tiles_m - first), i = pid - b * in_band;
  tm = first + i % rows;
  tn = i / rows;
}

// WM x WN waves, each TM x TN blocks of 16 x 16: the tile is 16 WM TM rows x 16 WN TN columns.
// PING: eight waves, two a SIMD, that take turns: while one reads a stage's operands from LDS and asks for a later stage, the other
// multiplies (the second half of the waves runs a barrier behind the first).  Without it all waves read at the same time and multiply at the same
// time, and neither LDS nor the matrix cores are busy for more than half of a stage: 256 x 160 tiles took 0.91 us a stage of 64
// along K with sixteen waves in step and take 0.76 with eight in turns.  `run` says from which K on that pays for the longer epilogue.  The
// other tiles of 256 rows do not take turns: with bfloat16 results and K up to 3,200 they are level to 15 % slower so (256 x 128: 2,048 x 4,096 x 1,024
// 26.0 -> 28.7 us; 256 x 224: 2,048 x 6,400 x 1,600 46.8 -> 52.6; 256 x 256: 8,192 x 4,096 x 1,024 79.6 -> 91.4; 192 and more columns with
// slabs of 32 a stage, since three stages of 64 do not fit in LDS).  Left open: from K = 5,120 on they would gain 3 to 12 % (8,192 x 2,048 x 8,192 225.6 -> 199.3).
// A_IN: A comes in rows (0), packed (1), or as `packed` says (2).  XIELU: the epilogue is that activation (a kernel of its own: its
// instructions beside the others' cost every product registers).
template <typename TC, int WM, int WN, int TM, int TN, int STAGES, bool KV, int KB = 1, bool PING = false, int A_IN = 2, bool XIELU = false>
__global__ __launch_bounds__(WM * WN * 64) void gemm_kernel(const bf16_t* __restrict__ A, const bf16_t* __restrict__ W, int lda, int M, int N, int K, int packed,
                                                           int tiles_m, int tiles_n, int split_slabs, const int32_t* __restrict__ slot_map,
                                                           const float* __restrict__ bias, TC* __restrict__ C, int ldc,
                                                           float* __restrict__ resid, int ldr, int epi, KVScatter kv,
                                                           float* __restrict__ part, const float* __restrict__ act) {
  constexpr int NW = WM * WN;
  const bool a_packed = A_IN == 2 ? (packed & PACKED_A) != 0 : A_IN == 1;
  constexpr int BM = WM * TM * 16, BN = WN * TN * 16;
  constexpr int AB = BM / 16, WB = BN / 16;              // 1 KB blocks per slab of 32 along K
  constexpr int PER = (AB + WB) * KB;                    // blocks per stage: KB slabs travel and are multiplied together
  constexpr int SLAB = PER * 64;                         // a stage, in u32x4
  constexpr int HI = (PER + NW - 1) / NW, REM = PER % NW;   // waves below REM load HI blocks, the others HI - 1
  static_assert((STAGES - 2) * HI < 64, "vmcnt has six bits");
  extern __shared__ u32x4 lds[];
  int tm, tn;
  tile_at(blockIdx.x, tiles_m, tiles_n, 1024 / BM, tm, tn);
  const int m0 = tm * BM, n0 = tn * BN;
  const int lane = threadIdx.x % 64;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x / 64);
  const int wmb = (wave / WN) * TM, wnb = (wave % WN) * TN;     // in blocks
  // part: K is shared out among the workgroups of blockIdx.y, split_slabs slabs each; a workgroup leaves
  // its sums in part[blockIdx.y][m][n] and a second kernel adds them in order and ends with the epilogue
  // (stages of KB slabs: the host launches KB > 1 only where K is a multiple of 32 KB; split_slabs counts stages)
  const int kall = K / 32, nblocks = (N + 15) / 16;
  // (the first 14 words of the arguments come in registers with the launch: all that the operands' first loads need, and the slots of a cache
  // write; the others by a trip to memory, see ARGS_EARLY)
  const int first = blockIdx.y * split_slabs;
  const int ksteps = min(split_slabs, kall / KB - first);
  // Where the 16 bytes of row lane % 16, columns 8 (lane / 16) .. of a block of A lie among its KB pieces of 1 KB (see the loads below).
  // (A packed A is in the operand's order already: lane l reads at 16 l.)
  int aslot[KB];
#pragma unroll
  for (int kb = 0; kb < KB; ++kb) {
    const int r = lane % 16, g = lane / 16;
    if (a_packed)
      aslot[kb] = kb * (AB + WB) * 64 + lane;
    else if constexpr (KB == 2)
      aslot[kb] = (r / 8) * (AB + WB) * 64 + 8 * (r % 8) + ((4 * kb + g) ^ (r / 2));
    else
      aslot[kb] = kb * (AB + WB) * 64 + 16 * (lane % 4) + 4 * (r / 4) + (g ^ (lane % 4));
  }

  // the tokens' slots, which the epilogue reads, are asked for before everything else: the row's, and those of the quad's four tokens
  // (8,192 rows of fused projections of 4,800 and 3,840 columns: 166 -> 160 and 115 -> 108 us)
  int kslot[KV ? TM : 1], vslot[KV ? TM : 1][4];
  if constexpr (KV) {
#pragma unroll
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + (wmb + i) * 16 + lane % 16, mq = m - lane % 4;
      kslot[i] = m < M ? slot_map[m] : -1;
#pragma unroll
      for (int e = 0; e < 4; ++e) vslot[i][e] = mq + e < M ? slot_map[mq + e] : -1;
    }
  }
  // The epilogue's arguments do not come with the launch.  With a cache write, and in tiles of four waves, they are brought into registers behind
  // the operands' first loads (ARGS_EARLY).  Elsewhere that held up the walk along K, and they come with the bias, asked for in front of the operands where
  // a tile leaves the registers for it (BIAS_FIRST): which of the two is measured, us, arguments in their old order -> both everywhere -> as it is:
  // four waves: GELU 65 x 1,024 x 4,096 20.1 -> 21.4 -> 19.8, 300 x 512 x 512 6.25 -> 6.36 -> 6.24; cache write: 203 x 3,840 x 1,280 10.7 -> 10.7 -> 10.4,
  // 65 x 4,800 x 1,600 11.5 -> 11.6 -> 11.1; sixteen waves: GELU 203 x 4,800 x 1,600 13.8 -> 13.5 -> 13.3, 203 x 4,096 x 1,024 7.95 -> 8.04 -> 7.76,
  // 1,000 x 1,024 x 1,024 8.05 -> 8.25 -> 7.79, into the stream 1,000 x 1,600 x 1,600 15.4 -> 15.0 -> 14.7.
  constexpr bool ARGS_EARLY = KV || NW == 4, BIAS_FIRST = !ARGS_EARLY && TN <= 4;
  floatx4 bvs[TN];
  auto ask_bias = [&]() {
#pragma clang loop unroll(full)
    for (int j = 0; j < TN; ++j) bvs[j] = floatx4{0.f, 0.f, 0.f, 0.f};
    if (bias) {
#pragma clang loop unroll(full)
      for (int j = 0; j < TN; ++j) bvs[j] = *reinterpret_cast<const floatx4*>(bias + min(n0 + (wnb + j) * 16 + (lane / 16) * 4, N - 4));
    }
  };
  if constexpr (BIAS_FIRST) ask_bias();
  floatx4 acc[TM][TN];
#pragma unroll
  for (int i = 0; i < TM; ++i)
#pragma unroll
    for (int j = 0; j < TN; ++j) acc[i][j] = floatx4{0.f, 0.f, 0.f, 0.f};

  // where this lane's share of each of the wave's blocks starts; a row beyond M or a block of
  // columns beyond N is replaced by the last inside (its results are not stored)
  const bf16_t* src[HI];
  int step[HI];
#pragma unroll
  for (int u = 0; u < HI; ++u) {
    const int q = min(wave + u * NW, PER - 1);
    const int b = q % (AB + WB), kb = q / (AB + WB);      // block b of the stage's slab kb
    if (b < AB) {
      if (a_packed) {      // a block of packed rows is 1 KB as it lies, like a block of W
        src[u] = A + static_cast<size_t>(min(m0 / 16 + b, (M + 15) / 16 - 1)) * kall * 512 + kb * 512 + lane * 8;
        step[u] = 512 * KB;
      } else if constexpr (KB == 2) {
        // a stage's columns are one cache line of a row: 1 KB is 8 rows x 128 bytes, rows 0 .. 7 of the block in the first
        // slab's place and 8 .. 15 in the second's
        const int r = 8 * kb + lane / 8, piece = (lane % 8) ^ (r / 2);
        src[u] = A + static_cast<size_t>(min(m0 + b * 16 + r, M - 1)) * lda + piece * 8;
        step[u] = 64;
      } else {
        // 16 lanes in a row take 64 bytes from each of four rows (g, g + 4, g + 8, g + 12 of the block):
        // four cache lines, where a lane per row would touch sixteen
        const int g = lane / 16, h = (lane % 16) / 4, piece = (lane % 4) ^ g;
        src[u] = A + static_cast<size_t>(min(m0 + b * 16 + 4 * h + g, M - 1)) * lda + kb * 32 + piece * 8;
        step[u] = 32 * KB;
      }
    } else {
      src[u] = W + static_cast<size_t>(min(n0 / 16 + b - AB, nblocks - 1)) * kall * 512 + kb * 512 + lane * 8;
      step[u] = 512 * KB;
    }
    src[u] += static_cast<size_t>(first) * step[u];
  }
  auto issue = [&](int kt) {
    u32x4* slab = lds + (kt % STAGES) * SLAB;
#pragma unroll
    for (int u = 0; u < HI; ++u) {
      const int q = wave + u * NW;
      if (u < HI - 1 || REM == 0 || wave < REM) load_to_lds(src[u] + static_cast<size_t>(kt) * step[u], slab + q * 64);
    }
  };
#pragma unroll
  for (int s = 0; s < STAGES - 1; ++s)
    if (s < ksteps) issue(s);
  // (here, not at the kernel's end)
  if constexpr (ARGS_EARLY) asm volatile("" ::"s"(C), "s"(ldc), "s"(resid), "s"(ldr), "s"(epi), "s"(part));
  if constexpr (KV) asm volatile("" ::"s"(kv.k_pool), "s"(kv.v_pool), "s"(kv.q_width), "s"(kv.kv_width), "s"(kv.dh), "s"(kv.page_size), "s"(kv.c_cols));
  // this wave's share of a stage has landed when only its loads of the STAGES - 2 stages after it are out
  auto landed = [&](bool more) {
    if (!more)
      wait_loads<0>();
    else if (REM == 0 || wave < REM)
      wait_loads<(STAGES - 2) * HI>();
    else
      wait_loads<(STAGES - 2) * (HI - 1)>();
  };
  if constexpr (PING) {
    static_assert(NW == 8 && STAGES >= 3, "two waves a SIMD; the stage that is read, the one that has landed, the one that is asked for");
    const bool late = wave >= NW / 2;
    landed(ksteps >= STAGES - 1);
    __builtin_amdgcn_s_barrier();
    if (late) __builtin_amdgcn_s_barrier();
    for (int kt = 0; kt < ksteps; ++kt) {
      // A stage is read a barrier after every wave has waited for its share of it.  Its place is asked for again one barrier after its last
      // reader was done: the late half has read stage kt - 1 (lgkmcnt(0)) in front of the barrier that ends the early half's turn kt - 1,
      // and right behind that barrier the early half asks for stage kt + STAGES - 1, which lies where kt - 1 lay.  There is none to spare.
      const u32x4* slab = lds + (kt % STAGES) * SLAB;
      bf16x8 af[KB][TM], wf[KB][TN];
#pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const u32x4* sl = slab + kb * (AB + WB) * 64;
#pragma unroll
        for (int i = 0; i < TM; ++i) af[kb][i] = __builtin_bit_cast(bf16x8, slab[(wmb + i) * 64 + aslot[kb]]);
#pragma unroll
        for (int j = 0; j < TN; ++j) wf[kb][j] = __builtin_bit_cast(bf16x8, sl[(AB + wnb + j) * 64 + lane]);
      }
      const bool more = kt + STAGES - 1 < ksteps;
      if (more) issue(kt + STAGES - 1);
      landed(more);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_s_setprio(1);
#pragma unroll
      for (int kb = 0; kb < KB; ++kb)
#pragma unroll
        for (int i = 0; i < TM; ++i)
#pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[kb][j], af[kb][i], acc[i][j], 0, 0, 0);
      __builtin_amdgcn_s_setprio(0);
      __builtin_amdgcn_sched_barrier(0);
      __builtin_amdgcn_s_barrier();
      __builtin_amdgcn_sched_barrier(0);
    }
    if (!late) __builtin_amdgcn_s_barrier();
  } else {
    for (int kt = 0; kt < ksteps; ++kt) {
      landed(kt + STAGES - 2 < ksteps);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();      // every wave's share of slab kt is there, and slab kt - 1 has been read
      if (kt + STAGES - 1 < ksteps) issue(kt + STAGES - 1);
      const u32x4* slab = lds + (kt % STAGES) * SLAB;
  #pragma unroll
      for (int kb = 0; kb < KB; ++kb) {
        const u32x4* sl = slab + kb * (AB + WB) * 64;
        bf16x8 af[TM], wf[TN];
  #pragma unroll
        for (int i = 0; i < TM; ++i) af[i] = __builtin_bit_cast(bf16x8, slab[(wmb + i) * 64 + aslot[kb]]);
  #pragma unroll
        for (int j = 0; j < TN; ++j) wf[j] = __builtin_bit_cast(bf16x8, sl[(AB + wnb + j) * 64 + lane]);
  #pragma unroll
        for (int i = 0; i < TM; ++i)
  #pragma unroll
          for (int j = 0; j < TN; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(wf[j], af[i], acc[i][j], 0, 0, 0);
      }
    }
  }
  // acc[i][j][r]: row m0 + 16 (wmb + i) + lane % 16, column n0 + 16 (wnb + j) + 4 (lane / 16) + r
  //
  // Where the fused projection's keys and values go is worked out once per row, outside the loop over
  // the column blocks (a slot's page and offset are divisions by numbers known only at run time; done
  // per block and lane they cost more than the product's own epilogue).  Keys: the lane's row.  Values:
  // in its page a value lies as [dim][offset], so four tokens whose slots follow one another from a
  // multiple of 4 are 8 bytes side by side for one dim: the four lanes of a quad, which hold four
  // tokens x four dims, exchange them (a 4 x 4 turn), and each stores four tokens of one dim.
  // A place is the row's (page and offset) plus the column's (head and dim); the latter without a division.  Only where a head is a
  // multiple of 16 dims, and keys and values begin at one, does a block of 16 columns have one place (`whole_blocks`: the keys of the staged way
  // below); elsewhere a lane's four columns have theirs, which are one head's and of one kind since all of these are multiples of 4.
  long long krow[KV ? TM : 1], vrow[KV ? TM : 1];      // of the row in the pools, -1: none
  uint32_t dh_inverse = 0;                             // 2^32 / dh, rounded up: c / dh is c times that (below 2^32 / dh)
  int page_numbers = 0;
  bool whole_blocks = false;
  if constexpr (KV) {
    whole_blocks = kv.dh % 16 == 0 && kv.q_width % 16 == 0;
    dh_inverse = 0xffffffffu / static_cast<uint32_t>(kv.dh) + 1;
    page_numbers = kv.Hkv * kv.page_size * kv.dh;
#pragma clang loop unroll(full)
    for (int i = 0; i < TM; ++i) {
      int page, off;
      page_and_offset(kv, max(kslot[i], 0), page, off);
      krow[i] = kslot[i] < 0 ? -1 : static_cast<long long>(page) * page_numbers + off * kv.dh;
      const int* sq = vslot[i];
      const bool run = kv.page_size % 4 == 0 && sq[0] >= 0 && sq[0] % 4 == 0 && sq[1] == sq[0] + 1 && sq[2] == sq[0] + 2 &&
                       sq[3] == sq[0] + 3;
      page_and_offset(kv, max(sq[0], 0), page, off);
      vrow[i] = run ? static_cast<long long>(page) * page_numbers + off : -1;
    }
  }
  // where keys lie in a page from this column on, to the end of their head
  auto key_place = [&](int column) {
    const uint32_t c = column - kv.q_width;
    return static_cast<int>(c + __umulhi(c, dh_inverse) * (kv.page_size - 1) * kv.dh);
  };
  if (part) {
#pragma clang loop unroll(full)
    for (int j = 0; j < TN; ++j) {
      const int n = n0 + (wnb + j) * 16 + (lane / 16) * 4;
      if (n >= N) continue;
#pragma clang loop unroll(full)
      for (int i = 0; i < TM; ++i) {
        const int m = m0 + (wmb + i) * 16 + lane % 16;
        if (m < M) *reinterpret_cast<floatx4*>(part + (static_cast<size_t>(blockIdx.y) * M + m) * N + n) = acc[i][j];
      }
    }
    return;
  }
  float act_a = 0.f, act_b = 0.f;
  if constexpr (XIELU) act_a = act[0], act_b = act[1];
  // every load of the epilogue before its first store: a wait for a load is a wait for the stores
  // issued before it as well (one counter), and a load per column block made the blocks take turns
  if constexpr (!BIAS_FIRST) ask_bias();
  // Results of 16 bits leave through LDS, 16 rows of the wave's columns at a time: 16 bytes a lane side by side, where a lane's four columns as they lie
  // are 32 bytes of each of 16 rows a store (2,048 x 6,400 x 64, all epilogue: 15.3 -> 11.5 us; with K = 1,600 and GELU 49.0 -> 47.1,
  // 2,048 x 4,800 x 1,600 36.1 -> 33.2, 8,192 x 6,400 x 1,600 181 -> 170).  A row's part is 16 bytes longer in LDS, so that the
  // rows' pieces meet different banks.  The values of a fused projection stay out of it: a store of theirs is a page's 512 bytes already
  // (fused projections, with the places in pages by row and block as above: 2,048 x 4,800 x 1,600 43.2 -> 39.9, 6,700 x 3,840 x 1,280 88 -> 84).
  constexpr int ROW = TN * 32 + 16, PIECES = 2 * TN;
  constexpr bool STAGED = sizeof(TC) == 2 && TN >= 2 && NW * 16 * ROW <= STAGES * SLAB * 16;
  bool staged = false;
  if constexpr (STAGED) {
    staged = !(packed & PACKED_C) && ldc % 8 == 0 && N % 8 == 0 && reinterpret_cast<uintptr_t>(C) % 16 == 0;
    if constexpr (KV) staged = staged && whole_blocks && kv.c_cols % 8 == 0 && reinterpret_cast<uintptr_t>(kv.k_pool) % 16 == 0;
    if (staged) {
      int place[KV ? TN : 1];      // of a block of keys in its page: the head's and the first dim's
      if constexpr (KV) {
#pragma clang loop unroll(full)
        for (int j = 0; j < TN; ++j) place[j] = key_place(max(n0 + (wnb + j) * 16, kv.q_width));
      }
      char* mine = reinterpret_cast<char*>(lds) + wave * (16 * ROW);
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
      __builtin_amdgcn_s_barrier();      // (the last stage has been read)
      // (what the wave's columns have none of costs it nothing: keys among queries, and columns that go elsewhere)
      const int first = n0 + wnb * 16, end = KV ? max(kv.q_width + kv.kv_width, kv.c_cols) : N;
      const bool keys = KV && first < kv.q_width + kv.kv_width && first + TN * 16 > kv.q_width;
#pragma clang loop unroll(full)
      for (int i = 0; i < TM; ++i) {
        if (first >= end) break;
#pragma clang loop unroll(full)
        for (int j = 0; j < TN; ++j) {
          const floatx4 v = acc[i][j] + bvs[j];
          auto finish = [&](float e) { return XIELU ? xielu_f(e, act_a, act_b) : apply_epilogue_fast(e, epi); };
          *reinterpret_cast<uint2*>(mine + (lane % 16) * ROW + j * 32 + (lane / 16) * 8) = pack4(finish(v[0]), finish(v[1]), finish(v[2]), finish(v[3]));
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma clang loop unroll(full)
        for (int it = 0; it < (16 * PIECES + 63) / 64; ++it) {
          const int u = it * 64 + lane, row = min(u / PIECES, 15), piece = u % PIECES;
          const int m = m0 + (wmb + i) * 16 + row, n = n0 + wnb * 16 + piece * 8;
          const u32x4 x = *reinterpret_cast<const u32x4*>(mine + row * ROW + piece * 16);
          const bool ok = u < 16 * PIECES && m < M && n < N;
          if (ok && (!KV || n < kv.c_cols)) *reinterpret_cast<u32x4*>(C + static_cast<size_t>(m) * ldc + n) = x;
          if (KV && keys) {
            const long long of_row = static_cast<long long>(static_cast<uint64_t>(static_cast<uint32_t>(__shfl(static_cast<int>(krow[i] >> 32), row))) << 32 |
                                                            static_cast<uint32_t>(__shfl(static_cast<int>(krow[i]), row)));
            int at = place[0];
#pragma clang loop unroll(full)
            for (int j = 1; j < TN; ++j) at = piece / 2 == j ? place[j] : at;
            if (ok && of_row >= 0 && n >= kv.q_width && n < kv.q_width + kv.kv_width)
              *reinterpret_cast<u32x4*>(kv.k_pool + of_row + at + piece % 2 * 8) = x;
          }
        }
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");      // (the next rows go where these lay)
      }
      if constexpr (!KV) return;
    }
  }
#pragma clang loop unroll(full)
  for (int j = 0; j < TN; ++j) {
    const int n = n0 + (wnb + j) * 16 + (lane / 16) * 4;
    if (n >= N) continue;
    const floatx4 bv = bvs[j];
    // (what a block has none of is known to the whole wave)
    const int block = n0 + (wnb + j) * 16;
    bool keys = false, values = false;
    int at = 0;      // of the block's first column among the values of a page
    if constexpr (KV) {
      keys = block + 16 > kv.q_width && block < kv.q_width + kv.kv_width;
      values = block + 16 > kv.q_width + kv.kv_width;
      at = (block - kv.q_width - kv.kv_width) * kv.page_size;
    }
#pragma clang loop unroll(full)
    for (int i = 0; i < TM; ++i) {
      const int m = m0 + (wmb + i) * 16 + lane % 16;
      if (m >= M || (STAGED && staged)) continue;
      const floatx4 v = acc[i][j] + bv;
      if (resid) {
        floatx4* x = reinterpret_cast<floatx4*>(resid + static_cast<size_t>(m) * ldr + n);
        *x = *x + v;
      } else if constexpr (sizeof(TC) == 4) {
        // (rows of any length and place, see `takes`: 16 bytes at a multiple of 4, a row's last one to three columns by themselves)
        floatx4 o;
#pragma clang loop unroll(full)
        for (int r = 0; r < 4; ++r) o[r] = apply_epilogue_fast(v[r], epi);
        TC* to = C + static_cast<size_t>(m) * ldc + n;
        if (n + 4 <= N) {
          *reinterpret_cast<floatx4_at_4*>(to) = o;
        } else {
#pragma clang loop unroll(full)
          for (int r = 0; r < 3; ++r)
            if (n + r < N) to[r] = o[r];
        }
      } else {
        auto finish = [&](float e) { return XIELU ? xielu_f(e, act_a, act_b) : apply_epilogue_fast(e, epi); };
        const uint2 cv = pack4(finish(v[0]), finish(v[1]), finish(v[2]), finish(v[3]));
        // (in packed rows, four columns from a multiple of 4 are 8 bytes side by side too)
        if (!KV || n < kv.c_cols)
          *reinterpret_cast<uint2*>(C + ((packed & PACKED_C) ? packed_index(m, n, N / 32) : static_cast<size_t>(m) * ldc + n)) = cv;
        if constexpr (KV) {
          // (with the place of whole blocks the scalar unit's: lane by lane for all of them the wide tiles' registers don't reach)
          if (keys && krow[i] >= 0 && n >= kv.q_width && n < kv.q_width + kv.kv_width) {
            const int place = whole_blocks ? key_place(block) + (lane / 16) * 4 : key_place(n);
            *reinterpret_cast<uint2*>(kv.k_pool + krow[i] + place) = cv;
          }
        }
      }
    }
    if constexpr (KV) {
      if (values) {
        const int q = lane % 4;       // this lane's dim of the four after the turn
#pragma clang loop unroll(full)
        for (int i = 0; i < TM; ++i) {
          const int mq = m0 + (wmb + i) * 16 + (lane % 16) / 4 * 4;      // the quad's first token
          const floatx4 v = acc[i][j] + bv;
          // token mq + e, dim d + q: lane e of the quad holds it in v[q]
          const float t0 = quad_pick<0>(v, q), t1 = quad_pick<1>(v, q), t2 = quad_pick<2>(v, q), t3 = quad_pick<3>(v, q);
          const int dim = (lane / 16) * 4 + q;
          if (n < kv.q_width + kv.kv_width) continue;
          if (vrow[i] >= 0) {
            *reinterpret_cast<uint2*>(kv.v_pool + vrow[i] + at + dim * kv.page_size) = pack4(t0, t1, t2, t3);
          } else {
#pragma clang loop unroll(full)
            for (int e = 0; e < 4; ++e) {
              const int slot = vslot[i][e];
              if (slot < 0) continue;
              int page, off;
              page_and_offset(kv, slot, page, off);
              kv.v_pool[static_cast<size_t>(page) * page_numbers + at + dim * kv.page_size + off] =
                  from_float<bf16_t>(e == 0 ? t0 : e == 1 ? t1 : e == 2 ? t2 : t3);
            }
          }
        }
      }
    }
  }
}

// Everything 16 bytes at a time: slabs of 32 along K, rows of A and C (or the residual) and the bias.  32-bit results without a bias may have
// rows of any length and place: a vocabulary's logits (203 rows of 50,257 x 1,280 in the few-rows kernel, which took them, 279 us, here 48;
// 65 rows 81 and 36; 1,024 rows, in the tiled kernel before, 200).
bool takes(const void* A, int lda, const void* W, const float* bias, const void* C, int ldc, const float* resid,
                  int ldr, int N, int K, int out_dtype, int packed) {
  auto aligned = [](const void* p, int a) { return reinterpret_cast<uintptr_t>(p) % a == 0; };
  const bool any_rows = out_dtype == DN_F32 && !resid && !bias && !(packed & PACKED_C);
  if (K % 32 != 0 || (N % 4 != 0 && !any_rows) || !aligned(A, 16) || !aligned(W, 16) || !aligned(bias, 16)) return false;
  if (!(packed & PACKED_A) && lda % 8 != 0) return false;
  if (resid) return ldr % 4 == 0 && aligned(resid, 16);
  if (packed & PACKED_C) return N % 32 == 0 && out_dtype == DN_BF16 && aligned(C, 8);
  if (any_rows) return aligned(C, 4);
  return ldc % 4 == 0 && aligned(C, out_dtype == DN_F32 ? 16 : 8);
}


template <typename TC, int WM, int WN, int TM, int TN, int STAGES, bool KV, int KB = 1, bool PING = false, int A_IN = 2, bool XIELU = false>
static int launch_kernel(const Args& a, hipStream_t stream) {
  constexpr int BM = WM * TM * 16, BN = WN * TN * 16;
  const int tiles_m = (a.M + BM - 1) / BM, tiles_n = (a.N + BN - 1) / BN;
  constexpr size_t lds = static_cast<size_t>(STAGES) * KB * (BM + BN) / 16 * 1024;
  if (a.K % (32 * KB) != 0) return DN_ERR_SHAPE;
  static bool raised = false;      // more than 64 KB of LDS has to be asked for once per kernel
  if (lds > 65536 && !raised) {
    hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(&gemm_kernel<TC, WM, WN, TM, TN, STAGES, KV, KB, PING, A_IN, XIELU>),
                                       hipFuncAttributeMaxDynamicSharedMemorySize, static_cast<int>(lds));
    if (e != hipSuccess) return static_cast<int>(e);
    raised = true;
  }
  const int shares = a.part ? a.splits : 1, split_slabs = (a.K / (32 * KB) + shares - 1) / shares;
  hipLaunchKernelGGL((gemm_kernel<TC, WM, WN, TM, TN, STAGES, KV, KB, PING, A_IN, XIELU>), dim3(tiles_m * tiles_n, shares),
                     dim3(WM * WN * 64), lds, stream, static_cast<const bf16_t*>(a.A), static_cast<const bf16_t*>(a.W),
                     a.lda, a.M, a.N, a.K, a.packed, tiles_m, tiles_n, split_slabs, a.kv ? a.kv->slot_map : nullptr, a.part ? nullptr : a.bias,
                     static_cast<TC*>(a.C), a.ldc, a.resid, a.ldr, a.epi, a.kv ? *a.kv : KVScatter{}, a.part, a.act);
  return 0;
}

template <typename TC, int WM, int WN, int TM, int TN, int STAGES, bool KV, int KB = 1, bool PING = false, int A_IN = 2>
static int launch(const Args& a, hipStream_t stream) {
  if constexpr (!KV && sizeof(TC) == 2) {
    if (a.epi == EPI_XIELU) return launch_kernel<TC, WM, WN, TM, TN, STAGES, KV, KB, PING, A_IN, true>(a, stream);
  }
  return launch_kernel<TC, WM, WN, TM, TN, STAGES, KV, KB, PING, A_IN>(a, stream);
}

template <int WM, int WN, int TM, int TN, int STAGES, int KB = 1>
static int launch_as(const Args& a, hipStream_t stream) {
  if (a.kv) return launch<bf16_t, WM, WN, TM, TN, STAGES, true, KB>(a, stream);
  if (a.out_dtype == DN_BF16 && !a.resid) return launch<bf16_t, WM, WN, TM, TN, STAGES, false, KB>(a, stream);
  return launch<float, WM, WN, TM, TN, STAGES, false, KB>(a, stream);
}

// (for steps of 65 to 256 rows: a kernel each for A in rows and for packed A, since the choice at run time stands in front of
// the first loads)
template <int WM, int WN, int TM, int TN, int STAGES, int KB, int A_IN>
static int launch_mid_a(const Args& a, hipStream_t stream) {
  if (a.kv) return launch<bf16_t, WM, WN, TM, TN, STAGES, true, KB, false, A_IN>(a, stream);
  if (a.out_dtype == DN_BF16 && !a.resid) return launch<bf16_t, WM, WN, TM, TN, STAGES, false, KB, false, A_IN>(a, stream);
  return launch<float, WM, WN, TM, TN, STAGES, false, KB, false, A_IN>(a, stream);
}

template <int WM, int WN, int TM, int TN, int STAGES, int KB>
static int launch_mid(const Args& a, hipStream_t stream) {
  return (a.packed & PACKED_A) ? launch_mid_a<WM, WN, TM, TN, STAGES, KB, 1>(a, stream) : launch_mid_a<WM, WN, TM, TN, STAGES, KB, 0>(a, stream);
}

// (for tiles that never write the cache: the variant with the cache write is not built)
template <int WM, int WN, int TM, int TN, int STAGES, int KB = 1, bool PING = false>
static int launch_without_kv(const Args& a, hipStream_t stream) {
  if (a.out_dtype == DN_BF16 && !a.resid) return launch<bf16_t, WM, WN, TM, TN, STAGES, false, KB, PING>(a, stream);
  return launch<float, WM, WN, TM, TN, STAGES, false, KB, PING>(a, stream);
}

// The tiles that `pick` chooses among: rows x columns, and the slabs in flight that its model counts LDS with.
// 128 and 256 rows: one workgroup per CU; the small ones (four waves) leave room for several workgroups per CU and
// are for products with few rows and a long K, whose larger tiles would leave most CUs idle.  (Tiles of 256 x 320
// were on the list while the others ran with eight waves a workgroup; no product chooses them now.)
constexpr Shape SHAPES[] = {{64, 128, 4}, {128, 128, 4}, {256, 128, 4}, {256, 160, 4}, {256, 192, 4},
                            {256, 224, 4}, {256, 256, 4}, {64, 64, 4}, {32, 64, 4}};
constexpr int PICKED = 9;

static double model_us(const Shape& s, int M, int N, int K) {
  const double tiles = static_cast<double>((M + s.bm - 1) / s.bm) * ((N + s.bn - 1) / s.bn);
  const size_t lds = static_cast<size_t>(s.stages) * (s.bm + s.bn) / 16 * 1024;
  // two workgroups that share a CU hide some of each other's waits (measured: 1.5 to 1.8 times one's time for two rounds)
  const double whole = static_cast<double>((static_cast<long>(tiles) + CUS - 1) / CUS);
  const double rounds = 2 * lds <= LDS_PER_CU && whole > 1 ? 0.9 * whole : whole;
  const double area = static_cast<double>(s.bm) * s.bn;
  return rounds * (K * (2.26e-7 * area + 3.07e-5 * (s.bm + s.bn)) + 1.9e-4 * area);
}

int pick(int M, int N, int K, bool kv) {
  int best = 0;
  double best_us = 1e30;
  for (int i = 0; i < PICKED; ++i) {
    double us = model_us(SHAPES[i], M, N, K);
    // (the model is of eight waves a workgroup; the tiles that run with sixteen, see `run`, take about three
    // quarters of its time, which moves the choice at 4,096 rows and more: the fused projection of 8,192 rows
    // 185 -> 165 us)
    if (i >= 1 && i <= 6 && !(kv && i >= 5)) us *= 0.75;
    if (us < best_us) best_us = us, best = i;
  }
  return best;
}

// 65 to 512 rows.  A tile's walk along K costs a wave some dozens of instructions a slab beside its four matrix
// instructions, and with one or two waves a SIMD nothing hides them: tiles of 64 x 64 take two slabs a stage
// which halves that and fills the chip from 65 rows on where the product is wide.  Measured on the
// four products of a layer 1,600 wide (rows and weights that no cache holds; us, before -> now):
//   128 rows: 4,800 columns 18.7 -> 15.7, 6,400 columns 15.3 -> 12.3, 1,600 columns from K = 6,400 19.4 -> 15.2
//   256 rows: 25.6 -> 23.2, 19.3 -> 18.0, 25.6 -> 21.4;  512 rows, 1,600 columns: K = 1,600 12.6 -> 10.7, K = 6,400 38.7 -> 35.4
// -> whether this kernel takes the product for its rows (wide ones in `wide_mid`'s tiles; else `pick` chooses, or the few-rows kernel runs)
bool mid_rows(int M, int N, int K) {
  if (M <= 64 || M > 512 || K % 64 != 0) return false;
  if (N < 2048) return K >= 4096 || M > 256;      // (few columns and a short K up to 256 rows: the few-rows kernel)
  return M <= 256;
}

// 17 to 64 rows of so many columns that tiles of 64 x 64 give most CUs one (a vocabulary): a workgroup of the few-rows kernel reads all rows anew for
// every 32 or 64 columns, and its waves wait for the rows.  Few-rows kernel -> here, packed rows, K = 1,024, 1,600 and 2,048: 17 rows of 12,288 columns 8.3 ->
// 7.3, 12.8 -> 11.9, 16.3 -> 14.0 us, of 50,257 30.5 -> 23.8, 44.9 -> 36.5, 54.2 -> 41.9; 64 rows 11.0 -> 7.9, 16.0 -> 13.7, 20.3 -> 15.1 and 43.5 ->
// 26.2, 63.4 -> 39.2, 74.1 -> 45.2; 8,192 columns stay (64 rows 7.1, 7.6 here; 17 rows 5.9, 7.1).  Where those tiles are more than
// the CUs, tiles of 64 x 128 (64 rows of 24,576 x 1,600 22.4 -> 20.3, of 20,480 x 1,024 13.9 -> 13.2).  A short K: 40 rows of 50,257 x 512 19.6 -> 16.7, of
// 12,288 x 512 6.7 -> 5.7; up to 32 rows level from 576 to 832 (17 rows x 50,257 x 768 20.6 and 20.7) and slower below (512 14.9, 15.7).
bool wide_few(int M, int N, int K) { return M > 16 && M <= 64 && N >= 12288 && K >= (M > 32 ? 512 : 1024) && K % 64 == 0; }

// Up to 256 rows the few-rows kernel takes the product too (both read and write packed rows): it stays ahead,
// or level, where the product has few columns and a short K; everywhere else from 65 rows on this kernel is
// the faster (`mid_rows`), and beyond 256 rows it is the only one.
// any_rows: 32-bit rows that only `takes`' allowance lets in (no multiple of 4 columns, or not at 16 bytes), up to 128 of them of fewer than 4,096 columns and up to
// 192, the few-rows kernel's next border, of up to 1,024, stay with the few-rows kernel, whose waves share K (there -> here: 65 rows of 2,049 x 1,024 5.0 and 6.7 us, of 3,001 x 2,048 7.1 and 10.1, of 257 x 4,096 10.0 and 18.2,
// 128 of 3,001 x 1,600 7.4 and 8.8, of 1,601 x 5,120 21.2 and 23.1; 65 of 4,099 x 1,024 7.9 and 6.7; 160 of 2,049 x 1,600 9.6 and 8.9; 129
// of 257 x 4,096 16.6 and 18.4, 192 of 1,001 x 4,096 18.3 and 18.6, of 257 x 8,192 31.2 and 33.1, of 1,999 x 8,192 45.8 and 37.1, 208 of 257 x 4,096 22.6 and 18.4).
bool beats_few_rows(int M, int N, int K, bool any_rows) {
  if (any_rows && (M <= 128 ? N < 4096 : M <= 192 && N <= 1024)) return false;
  return wide_few(M, N, K) || mid_rows(M, N, K) || (M > 104 && N >= 4096) || (M > 208 && N >= 2048);
}

// A long K beside few columns and few rows: the tiles are few and each walks all of K, a slab at a time,
// so K is shared out among several workgroups per tile (whole, such a product takes the same time whatever
// its rows up to 256, and a quarter of K less than a third of it).  The number of shares, 0 for none.  With
// fewer than 2,048 columns: 4 up to 128 rows, 2 up to 256, none beyond (1,600 columns, K = 6,400: 15.2, 21.4
// and 35.4 us at 128, 256 and 512 rows; with 8, 4 and 4 shares of smaller tiles 19.4, 25.6, 38.7).  From 2,048 columns: 8
// where the tiles of 32 x 64 are at most 96, else 4.
int shares_of_k(int M, int N, int K, int packed, bool kv) {
  if (kv || (packed & PACKED_C) || M <= 64 || M > 512 || N >= 4096 || K < 4096) return 0;
  if (N < 2048 && K % 64 == 0) return M <= 128 ? 4 : M <= 256 ? 2 : 0;
  return ((M + 31) / 32) * ((N + 63) / 64) <= 96 ? 8 : 4;
}

// A product into the residual stream whose sum a norm's kernel adds (dn_gemm_deferred): the shares of K that it
// is cut into, 0 if it is not worth it.  Few columns and 65 to 512 rows: the tiles are too few to fill the chip,
// and with the shares' sums left for the next kernel to add nothing has to join them here (1,600 x 1,600 at 128
// and 256 rows: 4.8 and 6.2 us where the whole product takes 6.7 and 8.0; K = 6,400: the kernel that adds the
// shares, 4.5 us, falls away).  Up to 256 rows a long K is cut as shares_of_k says, so that a row's sums do not depend on who adds the
// shares (left open for it, with the norm's kernel, 2 shares -> 4, us: 136 rows, 1,280 columns from K = 5,120 17.2 -> 13.1; 256 rows, 1,024 from
// 4,096 14.5 -> 12.3).  Beyond 256 rows: as many shares as make one round of 64 x 64 tiles, or, where that is one
// share of a long K, two rounds in three shares or more (with the norm's kernel, weights that no cache holds, whole -> in shares: 320
// rows x 1,280 columns, K = 5,120 31.6 -> 20.7 us in 2, 384 rows 31.8 -> 21.0, 512 rows 31.7 -> 24.8 in 3; 384 x 1,024, K = 4,096
// 22.7 -> 15.5; K = 1,280 12.0 -> 11.0 at 320 rows.  Not: 512 rows x 1,600 columns, K = 6,400, 37.5 and 37.6 in 2; 512 x 1,280, K = 1,280,
// 12.8 and 13.6).
int deferred_shares(int M, int N, int K) {
  if (M <= 64 || M > 512 || N >= 2048 || K % 64 != 0) return 0;
  if (M <= 256) {
    if (K >= 4096) return M <= 128 ? 4 : 2;
    return K / 64 >= 8 ? 2 : 0;
  }
  const int tiles = ((M + 63) / 64) * ((N + 63) / 64), one = CUS / tiles, two = 2 * CUS / tiles;
  if (K < 4096) return one >= 2 && K / 64 >= 16 ? 2 : 0;
  return one >= 2 ? min(one, 4) : two >= 3 ? 3 : 0;
}

static long tiles_of(int M, int N, int bm, int bn) { return static_cast<long>((M + bm - 1) / bm) * ((N + bn - 1) / bn); }
static long mid_tiles_64(int M, int N) { return tiles_of(M, N, 64, 64); }
// The tile of 65 to 512 rows of a wide product: the first of 64 x 64, 64 x 96 and 128 x 64 of which one round covers the product, 0 (`pick` chooses) where none
// does: beyond, larger tiles read the rows less often.  Sixteen waves a workgroup, eight for 64 x 96, each tile's walk along K being what a round takes.
// us, 64 x 96 for what ran before (128 x 64, beyond 256 rows what `pick` has): 203 and 256 rows of 4,800 x 1,600 with a cache write 15.3 -> 13.6 and
// 15.7 -> 13.9, of 5,120 x 1,280 with GELU 11.8 -> 11.0 and 12.0 -> 11.2, 136 of 6,400 x 1,600 13.7 -> 12.5; 320 of 3,840 x 1,280 13.1 -> 11.9, 384 of 3,072 x
// 1,024 11.5 -> 10.3; where 64 x 64 is one round, 203 of 3,840 x 1,280, 9.5 stays (11.6 so); where 64 x 96 is two, 288 of 5,120 x 1,280,
// 128 x 64 11.9 and 64 x 96 13.1.  128 x 64 beyond 256 rows: 320 of 5,120 x 1,280 12.5 -> 11.6, 448 of 4,096 x 1,024 10.5 -> 10.1.  Two rounds of
// 128 x 64 for what `pick` has: 203 rows of 9,216 x 1,600 26.5 and 16.9 us, 16,384 x 1,600 29.0 and 23.1, 50,257 x 1,280 78 and 48; 128 rows of
// 20,480 x 1,024 20.8 and 16.1, of 16,384, one round, 12.3 and 12.1.
static int wide_mid(int M, int N, int K) {
  if (M <= 64 || M > 512 || N < 2048 || K % 64 != 0) return 0;
  if (mid_tiles_64(M, N) <= CUS) return 64064;
  if (tiles_of(M, N, 64, 96) <= CUS) return 64096;
  return tiles_of(M, N, 128, 64) <= CUS ? 128064 : 0;
}

int run(const Args& a, hipStream_t stream) {
  if (wide_few(a.M, a.N, a.K) && !a.part)
    return mid_tiles_64(a.M, a.N) <= CUS ? launch_mid<4, 4, 1, 1, 4, 2>(a, stream) : launch_as<4, 4, 1, 2, 4, 2>(a, stream);
  // Wide products: sixteen waves a workgroup, four a SIMD, each with one 16 x 16 block of a 64 x 64 tile (a wave
  // of such a product waits on a counter for more than half of its life, and with one wave a SIMD nothing else
  // runs meanwhile: 16.0 -> 13.9 and 12.8 -> 11.3 us for 4,800 and 6,400 columns at 128 rows), or tiles with more blocks a wave (`wide_mid`).
  // The narrow ones, whose K is shared out, take no such way faster: four waves.
  if (!a.part) {
    switch (wide_mid(a.M, a.N, a.K)) {
      case 64064: return launch_mid<4, 4, 1, 1, 4, 2>(a, stream);
      case 64096: return launch_mid<4, 2, 1, 3, 4, 2>(a, stream);
      case 128064: return launch_mid<4, 4, 2, 1, 4, 2>(a, stream);
    }
  }
  if (((a.part || a.N < 2048) && mid_rows(a.M, a.N, a.K)) || (a.part && a.N < 2048 && a.K % 64 == 0)) return launch_mid<2, 2, 2, 2, 4, 2>(a, stream);
  // Tiles of 128 and 256 rows: sixteen waves a workgroup, four a SIMD, as 8 x 2 (a wave: 32 rows x a half of the
  // tile's columns) or 4 x 4, where eight waves as 4 x 2 with twice the rows each left the SIMDs waiting (a wave
  // waits on a counter for more than half of its life and the matrix cores were busy 30 % of the time).  At 2,048
  // rows of the XL layer: 56.1 -> 41.0, 25.2 -> 21.3, 57.1 -> 46.6 and 71.8 -> 56.9 us.  Two slabs a stage where K
  // allows it (whole cache lines of A's rows), else one in as many stages as fit in LDS.  The cache write's epilogue needs registers that sixteen
  // waves do not leave beside seven column blocks and more a wave: those keep eight waves.
  const bool sixteen = !a.part, two = a.K % 64 == 0;
  switch (pick(a.M, a.N, a.part ? a.K / a.splits : a.K, a.kv != nullptr)) {
    case 0:      // (the small tiles with sixteen waves too, where one round of them covers the product: several
                 // workgroups of four waves share a CU, one of sixteen has it alone)
      if (sixteen && two && tiles_of(a.M, a.N, 64, 128) <= CUS) return launch_as<4, 4, 1, 2, 4, 2>(a, stream);
      return launch_as<2, 2, 2, 4, 4>(a, stream);
    case 1: return sixteen && two ? launch_as<4, 4, 2, 2, 3, 2>(a, stream) : launch_as<4, 2, 2, 4, 4>(a, stream);
    case 2: return sixteen && two ? launch_as<8, 2, 2, 4, 3, 2>(a, stream) : launch_as<4, 2, 4, 4, 4>(a, stream);
    case 3:
      if (!sixteen || !two) return launch_as<4, 2, 4, 5, 4>(a, stream);
      // Eight waves in turns walk along K faster than sixteen in step and end slower, the more so the more the epilogue does: a wave
      // has twice the blocks to finish.  So a long K takes turns: from 1,600 on where the results are 32-bit, from 1,280 where they
      // are rounded to bfloat16 and leave through LDS (time of turns over time in step, K = 512, 1,024, 1,280, 1,600, 2,560: 1,500 x 6,400 with GELU
      // 1.05, 0.99, 0.98, 0.97, 0.96; 2,048 x 5,120 with GELU 1.06, 1.00, 0.99, 1.00, 0.95; 8,192 x 3,200 1.11, 1.03, 0.99, 0.98, 0.94; added into the
      // stream, 1,500 x 6,400, K = 1,024, 1,600, 2,560, 4,096: 1.03, 1.00, 0.98, 0.95), and the product with a cache write, whose
      // epilogue is the longest, never does (2,048 x 4,800 x 1,600 40.3 us in step, 46.6 in turns; 6,700 x 3,840 x 1,280 84 and 106).
      // GELU with the error function, the longest of the others', from 2,304 (in turns and in step: 2,048 x 5,120, K = 1,280 and 1,600 40.0 and 38.0, 44.4 and
      // 42.3 us; 3,000 x 3,072, K = 1,280, 2,048, 2,304 and 2,496 40.2 and 37.6, 49.1 and 47.4, 52.8 and 52.7, 55.5 and 56.8).
      if (!a.kv && a.K >= (a.out_dtype != DN_BF16 || a.resid ? 1600 : a.epi == EPI_GELU_ERF ? 2304 : 1280)) return launch_without_kv<4, 2, 4, 5, 3, 2, true>(a, stream);
      return launch_as<8, 2, 2, 5, 3, 2>(a, stream);
    case 4:
      if (!sixteen) return launch_as<4, 2, 4, 6, 4>(a, stream);
      return two ? launch_as<8, 2, 2, 6, 2, 2>(a, stream) : launch_as<8, 2, 2, 6, 3>(a, stream);
    case 5:
      if (a.kv || !sixteen) return launch_as<4, 2, 4, 7, 4>(a, stream);
      return two ? launch_without_kv<8, 2, 2, 7, 2, 2>(a, stream) : launch_without_kv<8, 2, 2, 7, 5>(a, stream);
    case 6:
      if (a.kv || !sixteen) return launch_as<4, 2, 4, 8, 4>(a, stream);
      return two ? launch_without_kv<8, 2, 2, 8, 2, 2>(a, stream) : launch_without_kv<8, 2, 2, 8, 3>(a, stream);
    case 7:
      if (sixteen && two && tiles_of(a.M, a.N, 64, 64) <= CUS) return launch_mid<4, 4, 1, 1, 4, 2>(a, stream);
      return launch_as<2, 2, 2, 2, 4>(a, stream);
    default: return launch_as<2, 2, 1, 2, 4>(a, stream);
  }
}

// the tile that a product of these sizes gets: rows * 1000 + columns; beyond 256 rows the one on the list, which runs where `wide_tile_of` is 0
int tile_of(int M, int N, int K, bool kv) {
  if (wide_few(M, N, K)) return mid_tiles_64(M, N) <= CUS ? 64064 : 64128;
  if (N < 2048 && mid_rows(M, N, K)) return 64064;
  if (const int tile = wide_mid(M, N, K); tile && M <= 256) return tile;
  const Shape& s = SHAPES[pick(M, N, K, kv)];
  return s.bm * 1000 + s.bn;
}
int wide_tile_of(int M, int N, int K) { return wide_mid(M, N, K); }
}  // namespace direct
