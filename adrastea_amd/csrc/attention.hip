// Fused attention for one layer: out = softmax(mask(scale * Q K^T) / temp) V per head, without
// the [heads, m, n] score tensor ever reaching memory.  It stands for the three launches at
// adrastea_models/src/llama.rs:541-554 (matmul_f16 with Scale + Causal, softmax_rows_inplace,
// matmul_f16), clip.rs:372-388 and whisper.rs:424-436, whose time on this part is the write and
// two reads of that tensor.  Scores and probabilities stay in fp32 registers (the three-launch
// path rounds both to fp16 in between), so results agree with that path to fp16 rounding, not
// bit for bit.
#include <math.h>

#include <algorithm>
#include <type_traits>

#include "adr_common.hpp"

namespace adr {

namespace {

#define ADR_LDS_PTR(p) ((__attribute__((address_space(3))) void*)(p))

struct AttnArgs {
  half_t* out;
  const half_t* q;
  const half_t* k;
  const half_t* v;
  int heads, m, n;  // query rows, key/value rows
  int so_y, so_z, sq_y, sq_z, sk_y, sk_z, sv_y, sv_z;  // element strides; the x strides are 1
  float c;          // scale * log2(e) / temperature
  uint32_t mask;
  int qblocks;      // ceil(m / 128)
  int upper;        // query blocks dealt out downwards before the others upwards (see the kernel)
  int splits;       // workgroups that share the keys of one query block
  float* part_o;    // splits > 1: [splits][heads][m][d] unnormalised sums
  float2* part_ml;  // splits > 1: [splits][heads][m] (maximum in log2 units, sum)
};

typedef float float2_t __attribute__((ext_vector_type(2)));

constexpr int BM = 128, BN = 64;  // query rows of a workgroup, keys of a tile

// K tile: [64 rows][CPR 16-byte chunks]; chunk kc of row r sits at position kc ^ (line & 15)
// of its 256-byte line (16 lanes reading the same chunk of 16 consecutive rows hit 16
// different bank groups).
template <int CPR>
__device__ __forceinline__ int k_chunk_off(int row, int kc) {
  const int idx = row * CPR + kc, line = idx >> 4, pos = idx & 15;
  return ((line << 4) | (pos ^ (line & (CPR - 1)))) << 4;
}
template <int CPR>
__device__ __forceinline__ void k_chunk_inv(int phys, int& row, int& kc) {
  const int line = phys >> 4, pos = (phys & 15) ^ (line & (CPR - 1));
  const int idx = (line << 4) | pos;
  row = idx / CPR;
  kc = idx % CPR;
}
// V tile: [64 rows][CPR chunks], chunk c of row r at position c ^ v_swz(r): a transposing read
// touches 4 consecutive rows x 4 consecutive chunks per 32 lanes, and the XOR spreads those 16
// chunks over the 16 bank groups (rows of 128 bytes share a 256-byte line in pairs).
template <int CPR>
__device__ __forceinline__ int v_swz(int row) {
  return CPR == 16 ? ((row & 3) << 2) : (((row >> 1) & 1) << 2);
}

// The same for transposing reads of 8 consecutive rows x 2 consecutive chunks per 32 lanes.
template <int CPR>
__device__ __forceinline__ int v_swz8(int row) {
  return CPR == 16 ? ((row & 7) << 1) : (((row >> 1) & 3) << 1);
}

// v_permlane32_swap exchanges the upper half of the first register with the lower half of the second,
// v_permlane16_swap the odd rows of 16 lanes of the first with the even rows of the second: with one
// value in both, a lane then holds its own and its partner's (lane ^ 32, lane ^ 16), without a trip
// through LDS.  The second result passes through an empty asm statement: without it the compiler
// folds a floating-point operation on the two results as if they were the same register.
__device__ __forceinline__ void swap_halves(float& x, float& y) {
  const auto r = __builtin_amdgcn_permlane32_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y), false, false);
  uint32_t r0 = r[0], r1 = r[1];
  asm volatile("" : "+v"(r1));
  x = __builtin_bit_cast(float, r0);
  y = __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ void swap_rows(float& x, float& y) {
  const auto r = __builtin_amdgcn_permlane16_swap(__builtin_bit_cast(uint32_t, x), __builtin_bit_cast(uint32_t, y), false, false);
  uint32_t r0 = r[0], r1 = r[1];
  asm volatile("" : "+v"(r1));
  x = __builtin_bit_cast(float, r0);
  y = __builtin_bit_cast(float, r1);
}
__device__ __forceinline__ float pair_max(float v) {
  float x = v, y = v;
  swap_halves(x, y);
  return fmaxf(x, y);
}
__device__ __forceinline__ float pair_sum(float v) {
  float x = v, y = v;
  swap_halves(x, y);
  return x + y;
}

// Global -> LDS transfers of 1 KiB (16 bytes per lane, lane l to lds + 16 l).  Assembly, so that the
// compiler does not make every LDS read of the other buffers wait for the transfers in flight;
// the waits are written out below.  The buffer form reads zeros past the end of its descriptor: rows
// beyond the last key need no clamp, and a descriptor of 0 bytes is no transfer at all.  It makes two
// transfers, the second one's offset of 1024 bytes counting on both sides.  (The s_nop: m0, and
// scalars that a vector instruction wrote, need wait states before a memory instruction reads them.)
template <int FIRST>
__device__ __forceinline__ void dma_buffer_pair(uint32_t lds, uint32_t voff0, uint32_t voff1, u32x4_t desc) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tbuffer_load_dwordx4 %1, %3, 0 offen offset:%4 lds\n\t"
               "buffer_load_dwordx4 %2, %3, 0 offen offset:%5 lds"
               :: "s"(lds), "v"(voff0), "v"(voff1), "s"(desc), "n"(FIRST * 1024), "n"(FIRST * 1024 + 1024) : "memory");
}
__device__ __forceinline__ void dma_global(uint32_t lds, const void* p) {
  asm volatile("s_mov_b32 m0, %0\n\ts_nop 4\n\tglobal_load_lds_dwordx4 %1, off"
               :: "s"(lds), "v"(p) : "memory");
}
template <int N>
__device__ __forceinline__ void wait_vm() {
  asm volatile("s_waitcnt vmcnt(%0)" :: "n"(N) : "memory");
}
// (A barrier alone: it does not wait for LDS reads in flight.  Whoever reads what another wavefront may
// overwrite behind the next barrier waits for the reads first.  Those issued ahead at the end of a half
// tile, read_v(cV, 0) and read_k(cK, 0) below, need not: they are used, hence waited for, before the
// next barrier, and their buffers are refilled behind that one.)
__device__ __forceinline__ void barrier() {
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_barrier" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// One group of four wavefronts takes 128 query rows of one head, wavefront w of it rows 32 w ...
// 32 w + 31.  Key and value rows stream through LDS in tiles of 64 by global -> LDS DMA, double
// buffered.  With G = 1 a workgroup is one group and two workgroups share a compute unit; with G = 2
// two groups of a workgroup take the same rows and every other key tile, and their results are merged
// through LDS at the end: for launches of at most one workgroup per compute unit.
//
// Per tile a wavefront computes S^T = K Q^T (MFMA 32x32x16, Q fragments resident in registers), so
// that every lane holds scores of ONE query row: the running maximum and sum are in-lane reductions
// plus one exchange with lane ^ 32.  The probabilities, narrowed to fp16, are already in the operand
// layout of the second product O^T = V^T P^T; its V^T fragments come from the row-major V tile by
// transposing LDS reads (ds_read_b64_tr_b16).
//
// What bounds it: issuing.  A wavefront issues an instruction every 5 clocks, an MFMA 32x32x16 holds
// the matrix pipe for 32 and of the softmax's instructions only v_dot2 waits for that pipe (in a loop
// of one MFMA and four others, 2 wavefronts per SIMD: 34 clocks with v_fma, v_max3, v_cvt_pk or v_perm,
// 44 with v_exp, 62 with v_dot2).  So the two products and the softmax between them are interleaved
// in one instruction stream -- while the scores of tile i + 1 are on the matrix cores, the vector ALU
// turns those of tile i into probabilities; while P.V of tile i is, it finds the maximum of tile
// i + 1 -- and everything else is kept out of it: transfers count their bytes in descriptors (no clamps,
// no address arithmetic) and go out in pairs, one wait covers four fragments, and whatever needs many
// scalar registers (they would be kept in vector registers and read back) is serialised.
//
// With the phases one after the other a tile took 3950 cycles of two wavefronts per SIMD; now 2800,
// where the MFMAs need 2048, and on random data the clock under this load is 1.5 GHz (2.1 on zeros): the
// rest is the power limit's.  32 heads of 128, 2048 x 2048: 79.5 -> 70 us = 980 TFLOP/s, causal
// 55.1 -> 48.5; 4096 x 4096 294 -> 262; 40 heads 1600 causal 51.9 -> 38; 20 heads of 64, 1500 x 1500
// 28.0 -> 20.0.  MFMA 16x16x32, which costs less power, was 4 % ahead at 4096 keys and 2 % behind at
// 2048 and under the mask (twice the MFMAs to issue, and registers spilled in the prologue); two
// groups half a tile apart, one in the MFMAs of a whole tile while the other is in its softmax, took
// 82 us: alone on its SIMD's vector ALU a wavefront issues at half the rate.
// HD = 128 keeps 22 vector registers in scratch memory (WIDE 42), HD = 64 none: all of them in the
// straight-line halves behind the main loop, none in it.
template <int HD, int G, bool WIDE>
__global__ __launch_bounds__(256 * G, 2) void attention_fwd_kernel(AttnArgs a) {
  constexpr int CPR = HD / 8;
  constexpr int TILE = BN * HD * 2;   // bytes of one K or V tile
  constexpr int NI = TILE / 1024 / 4; // DMA instructions per wavefront and tile
  constexpr int DS = HD / 16;         // MFMA k-steps over the head dimension
  constexpr int DT = HD / 32;         // 32-wide output column tiles
  constexpr int ROWB = HD * 2;        // bytes per tile row
  static_assert(CPR == 16 || CPR == 8, "head dimension 128 or 64");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[G * 4 * TILE];  // K0 K1 V0 V1 of each group

  // (the wavefront index as a scalar: everything derived from it -- LDS stage addresses of the
  // transfers, role branches -- then stays out of the vector registers and the vector ALU)
  const int tid = threadIdx.x, lane = tid & 63, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int grp = G == 1 ? 0 : wave >> 2, w = wave & 3;
  const int frow = lane & 31, g = lane >> 5;
  const bool causal = a.mask == ADR_MASK_CAUSAL;

  // Workgroup -> (query block, unit), a unit being one of the `splits` parts of one head's keys.
  // Consecutive workgroup ids go to different dies; die x takes the units [x * units/8, (x+1) *
  // units/8) where that divides, so that the query blocks of a head (which share K and V) meet in
  // one L2.  Under the causal mask block b has 2b + 2 key tiles.  Where all workgroups are resident at
  // once, a die's own sequence runs through the upper half of the blocks downwards, then through the
  // lower half upwards: with 32 heads and 16 blocks the i-th and the (i+32)-th of the die share a
  // compute unit, and this order gives every unit a block b and its complement 15 - b.  With more
  // workgroups the blocks go downwards throughout: the heavy ones start first, the light ones fill in.
  const int units = a.heads * a.splits;
  int unit, j;
  if (units % 8 == 0) {
    const int ux = units >> 3, seq = blockIdx.x >> 3;
    unit = (blockIdx.x & 7) * ux + seq % ux;
    j = seq / ux;
  } else {
    unit = blockIdx.x % units;
    j = blockIdx.x / units;
  }
  const int qb = j < a.upper ? a.qblocks - 1 - j : j - a.upper;
  const int head = unit / a.splits, split = unit % a.splits;
  const int q0 = qb * BM, q0w = q0 + w * 32;

  const half_t* const Q = a.q + (int64_t)head * a.sq_z;
  const half_t* const K = a.k + (int64_t)head * a.sk_z;
  const half_t* const V = a.v + (int64_t)head * a.sv_z;

  int ntiles = (a.n + BN - 1) / BN;
  if (causal) ntiles = min(ntiles, (min(q0 + BM, a.m) - 1) / BN + 1);
  const int tile0 = (int)((int64_t)ntiles * split / a.splits);
  const int wg_tiles = (int)((int64_t)ntiles * (split + 1) / a.splits) - tile0;
  const int steps = (wg_tiles + G - 1) / G;  // of the workgroup: both groups pass every barrier
  // Tiles this wavefront computes (tile0 + grp + G i): none if its rows lie past the last, and under the
  // mask none whose first key lies beyond its last row.
  int active = q0w < a.m ? (wg_tiles - grp + G - 1) / G : 0;
  if (causal) active = max(0, min(active, ((q0w + 31) / BN - tile0 - grp + G) / G));
  // the first of them with keys that some row of the wavefront must not see
  int first_edge = (a.n / BN - tile0 - grp + G - 1) / G;
  if (causal) first_edge = min(first_edge, (q0w / BN - tile0 - grp + G - 1) / G);

  const uint32_t lds0 = (uint32_t)(uintptr_t)ADR_LDS_PTR(smem) + grp * 4 * TILE;
  const unsigned char* const sm = smem + grp * 4 * TILE;

  // Wavefront w transfers rows 16 w ... 16 w + 15 of a tile, 1 KiB at a time: lane l of transfer j
  // fills chunk (w NI + j) 64 + l, fetching whatever (row, chunk) the swizzle puts there.  koff, voff:
  // the byte offset of that chunk in the tile's rows, less the j KiB that the instruction adds.
  uint32_t koff[NI], voff[NI];
  int krow[NI], kcol[NI], vrow[NI], vcol[NI];
#pragma unroll
  for (int j = 0; j < NI; j++) {
    const int phys = (w * NI + j) * 64 + lane;
    int kc;
    k_chunk_inv<CPR>(phys, krow[j], kc);
    kcol[j] = kc * 8;
    vrow[j] = phys / CPR;
    vcol[j] = ((phys % CPR) ^ v_swz<CPR>(vrow[j])) * 8;
    koff[j] = ((uint32_t)krow[j] * (uint32_t)a.sk_y + kcol[j]) * 2 - j * 1024;
    voff[j] = ((uint32_t)vrow[j] * (uint32_t)a.sv_y + vcol[j]) * 2 - j * 1024;
  }
  // The group's next K and V tiles: address, and bytes from there to the end of the workgroup's keys
  // (0 past them).  WIDE: row numbers.
  const int row0 = (tile0 + grp) * BN, row_end = min(a.n, (tile0 + wg_tiles) * BN);
  struct Next {
    uint64_t p;
    int left, advance, row, stride;
  };
  auto first_tile = [&](const half_t* base, int stride) __attribute__((always_inline)) {
    Next t;
    t.p = (uint64_t)(base + (int64_t)row0 * stride);
    t.left = row_end > row0 ? (row_end - 1 - row0) * stride * 2 + HD * 2 : 0;
    t.advance = stride * (G * BN * 2);
    t.row = row0;
    t.stride = stride;
    return t;
  };
  Next nk = first_tile(K, a.sk_y), nv = first_tile(V, a.sv_y);
  auto advance = [&](Next& t) __attribute__((always_inline)) {
    t.p += t.advance;
    t.left = max(t.left - t.advance, 0);
    t.row += G * BN;
  };
  // Transfers 2 j and 2 j + 1 of the NI that bring a tile into buffer `buf` (0, 1: K; 2, 3: V).
  auto transfer = [&](const Next& t, auto is_k, int buf, auto pair) __attribute__((always_inline)) {
    constexpr bool IS_K = decltype(is_k)::value;
    constexpr int J = 2 * decltype(pair)::value;
    const uint32_t dst = lds0 + w * (NI * 1024) + buf * TILE;
    if constexpr (WIDE) {
      if (t.row >= row_end) return;
#pragma unroll
      for (int j = J; j < J + 2; j++) {
        const int row = min(t.row + (IS_K ? krow[j] : vrow[j]), a.n - 1);
        dma_global(dst + j * 1024, (IS_K ? K + kcol[j] : V + vcol[j]) + (int64_t)row * t.stride);
      }
    } else {
      const u32x4_t desc = {(uint32_t)t.p, (uint32_t)(t.p >> 32) & 0xffffu, (uint32_t)t.left, 0x00020000u};
      if constexpr (IS_K) dma_buffer_pair<J>(dst, koff[J], koff[J + 1], desc);
      else dma_buffer_pair<J>(dst, voff[J], voff[J + 1], desc);
    }
  };
  const std::true_type is_k{};
  const std::false_type is_v{};
  const std::integral_constant<int, 0> pair0{};
  const std::integral_constant<int, NI / 2 - 1> pair1{};  // (the last pair; HD = 64 has one)
  auto tile_transfers = [&](Next& t, auto k, int buf) __attribute__((always_inline)) {
    transfer(t, k, buf, pair0);
    if constexpr (NI > 2) transfer(t, k, buf, pair1);
    advance(t);
  };

  // What is waited for at the end of each half: all transfers but those issued in it.
  auto wait_landed = [&]() __attribute__((always_inline)) { wait_vm<WIDE ? 0 : NI>(); };

  // Q fragments (operand B of S^T = K Q^T): lane -> query row frow, head-dim group g.  They come by way
  // of the V buffers in the K tiles' layout, so that whole rows are fetched: wavefront w brings and
  // reads its own 32 rows.
  half8_t qf[DS];
  constexpr int QI = 2 * NI;           // transfers of a wavefront's 32 rows
  if constexpr (WIDE) {
    const half_t* qrow = Q + (int64_t)min(q0w + frow, a.m - 1) * a.sq_y + g * 8;
#pragma unroll
    for (int ds = 0; ds < DS; ds++) qf[ds] = *(const half8_t*)(qrow + ds * 16);
  } else {
    const uint64_t p = (uint64_t)(Q + (int64_t)q0w * a.sq_y);
    const u32x4_t desc = {(uint32_t)p, (uint32_t)(p >> 32) & 0xffffu,
                          q0w < a.m ? (uint32_t)((a.m - 1 - q0w) * a.sq_y * 2 + HD * 2) : 0u, 0x00020000u};
#pragma unroll
    for (int j = 0; j < QI; j += 2) {
      uint32_t off[2];
#pragma unroll
      for (int e = 0; e < 2; e++) {
        int row, kc;
        k_chunk_inv<CPR>(w * (32 * CPR) + (j + e) * 64 + lane, row, kc);
        off[e] = ((uint32_t)(row - w * 32) * (uint32_t)a.sq_y + kc * 8) * 2 - e * 1024;
      }
      dma_buffer_pair<0>(lds0 + 2 * TILE + w * (32 * ROWB) + j * 1024, off[0], off[1], desc);
    }
  }
  tile_transfers(nk, is_k, 0);
  tile_transfers(nk, is_k, 1);

  // LDS fragment offsets.  K: lane -> tile row frow (+32), chunk 2*ds + g.
  int offK[DS];
#pragma unroll
  for (int ds = 0; ds < DS; ds++) offK[ds] = k_chunk_off<CPR>(frow, ds * 2 + g);
  if constexpr (WIDE) {
#pragma unroll
    for (int ds = 0; ds < DS; ds++) asm volatile("" : "+v"(qf[ds]));
    wait_vm<0>();
  } else {
    wait_vm<2 * NI>();  // Q has landed
#pragma unroll
    for (int ds = 0; ds < DS; ds++) qf[ds] = *(const half8_t*)(sm + 2 * TILE + w * (32 * ROWB) + offK[ds]);
    // The first K tile has landed too, and the fragments are read before the barrier behind which any
    // wavefront may transfer the first V tile over them (one without rows of its own does so at once).
    asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" :: "n"(NI) : "memory");
  }
  // V (transposing read): in each group of 16 lanes, lanes 4r..4r+3 address 16 consecutive
  // halves of tile row r, and lane i of the group receives column i of that 4 x 16 block.
  // Group b = (lane / 16) % 2 takes columns 16b.. of the 32-column tile, g the rows 4g..4g+3.
  int offV[DT];
  {
    const int s = lane & 15, b = (lane >> 4) & 1, r = s >> 2;
    const int row = 4 * g + r;  // + 32*kt + 16*t + 8*h, all multiples of 8: row & 3 == r
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
      const int chunk = 4 * dt + 2 * b + ((s & 3) >> 1);
      offV[dt] = row * ROWB + ((chunk ^ v_swz<CPR>(row)) << 4) + (s & 1) * 8;
    }
  }

  float16_t o[DT], sa[2], sb[2];  // sums of P.V; scores of two tiles in turn
  u32x4_t pf[2][2];                 // probabilities, two to a register
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int r = 0; r < 16; r++) o[dt][r] = 0.0f;
  float m_run = -1.0e30f, l_run = 0.0f;  // running maximum (log2 units) and this lane's sum

  typedef short short4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) short4_t lds_short4_t;
  // A half tile is NG groups of four MFMAs.  A group's fragments are read a group ahead, and used in
  // the opposite order, so that one wait covers all four.
  constexpr int NG = DS / 2;
  half8_t kf[NG][4], vf[NG][4];

  auto read_k = [&](const unsigned char* cK, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; j++) kf[c][j] = *(const half8_t*)(cK + offK[2 * c + (j >> 1)] + (j & 1) * 32 * ROWB);
  };
  // which of the products with V the j-th of group c is: keys 32 kt + 16 t ..., columns 32 dt ...
  auto pv_of = [](int c, int j, int& kt, int& t, int& dt) __attribute__((always_inline)) {
    const int p = 4 * c + j;
    kt = p / (2 * DT), t = p / DT % 2, dt = p % DT;
  };
  auto read_v = [&](const unsigned char* cV, int c) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < 4; j++) {
      int kt, t, dt;
      pv_of(c, j, kt, t, dt);
      const unsigned char* p0 = cV + offV[dt] + (32 * kt + 16 * t) * ROWB;
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)ADR_LDS_PTR(p0));
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)ADR_LDS_PTR(p0 + 8 * ROWB));
      vf[c][j] = __builtin_shufflevector(__builtin_bit_cast(half4_t, lo), __builtin_bit_cast(half4_t, hi),
                                         0, 1, 2, 3, 4, 5, 6, 7);
    }
  };

  // First half of tile i: the scores of tile i + 1 on the matrix cores (K buffer KB), and the
  // probabilities of tile i on the vector ALU.
  auto half1 = [&](auto do_s, auto do_p, auto do_pv, auto kbuf, float16_t (&cur)[2], float16_t (&nxt)[2])
                   __attribute__((always_inline)) {
    constexpr bool S = decltype(do_s)::value, P = decltype(do_p)::value;
    constexpr int KB = decltype(kbuf)::value, VB = 1 - KB;
    const unsigned char* const cK = sm + KB * TILE;
    const unsigned char* const cV = sm + (2 + VB) * TILE;
    // Piece k of the softmax: VP scores, in three stages that run a piece apart, so that no instruction
    // waits for the one before it: exponents (k + 1), powers of two (k), rounding and sum (k - 1).
    // (The empty assembly keeps the stages where they are.  Sums by v_dot2 would be half the
    // instructions, but those wait for the matrix cores.)
    constexpr int NP = 4 * NG, VP = 32 / NP;
    float sum[2] = {l_run, 0.0f};
    float ex[VP], pw[VP];
    auto stage_exponent = [&](int k) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < VP; e++) ex[e] = fmaf(cur[k * VP >> 4][(k * VP & 15) + e], a.c, -m_run);
    };
    auto stage_power = [&]() __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < VP; e++) pw[e] = __builtin_amdgcn_exp2f(ex[e]);
    };
    auto stage_round = [&](int k) __attribute__((always_inline)) {
#pragma unroll
      for (int e = 0; e < VP; e += 2) {
        const int x = k * VP + e;
        const float2_t e2 = {pw[e], pw[e + 1]};
        uint32_t bits = __builtin_bit_cast(uint32_t, __builtin_convertvector(e2, half2_t));
        sum[0] += pw[e];
        sum[1] += pw[e + 1];
        asm volatile("" : "+v"(bits), "+v"(sum[0]), "+v"(sum[1]));
        pf[x >> 4][x >> 3 & 1][(x & 7) / 2] = bits;
      }
    };
    if constexpr (HD == 128) __builtin_amdgcn_s_setprio(1);
    if constexpr (P) stage_exponent(0);
    if constexpr (S) {
#pragma unroll
      for (int kt = 0; kt < 2; kt++)
#pragma unroll
        for (int r = 0; r < 16; r++) nxt[kt][r] = 0.0f;
    }
#pragma unroll
    for (int c = 0; c < NG; c++) {
      if constexpr (S) {
        if (c + 1 < NG) read_k(cK, c + 1);
      }
      if constexpr (decltype(do_pv)::value) {
        if (c + 1 == NG) read_v(cV, 0);
      }
      if (c == 0) transfer(nv, is_v, 2 + KB, pair0);
      if constexpr (NI > 2) {
        if (c == NG / 2) transfer(nv, is_v, 2 + KB, pair1);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if constexpr (S) {
          constexpr int last = 3;
          const int f = last - j;
          nxt[f & 1] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf[c][f], qf[2 * c + (f >> 1)], nxt[f & 1], 0, 0, 0);
        }
        if constexpr (P) {
          const int k = 4 * c + j;
          if (k > 0) stage_round(k - 1);
          stage_power();
          if (k + 1 < NP) stage_exponent(k + 1);
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (P) {
      stage_round(NP - 1);
      l_run = sum[0] + sum[1];
      asm volatile("" : "+v"(l_run));
    }
    if constexpr (HD == 128) __builtin_amdgcn_s_setprio(0);
    advance(nv);
    wait_landed();
    barrier();
  };

  // Second half of tile i: P.V of tile i on the matrix cores (V buffer VB), and the maximum of the
  // scores of tile i + 1 on the vector ALU.
  auto half2 = [&](int i, auto do_pv, auto do_max, auto do_s, auto vbuf, float16_t (&nxt)[2])
                   __attribute__((always_inline)) {
    constexpr bool PV = decltype(do_pv)::value, MAX = decltype(do_max)::value;
    constexpr int VB = decltype(vbuf)::value, KB = VB;  // K buffer of tile i + 2
    const unsigned char* const cV = sm + (2 + VB) * TILE;
    const unsigned char* const cK = sm + KB * TILE;
    if constexpr (MAX) {
      if (i + 1 >= first_edge) {
        // this lane's first masked key, counted from its own first one
        int end = (causal ? min(a.n, q0w + frow + 1) : a.n) - (tile0 + grp + G * (i + 1)) * BN - 4 * g;
#pragma unroll
        for (int kt = 0; kt < 2; kt++)
#pragma unroll
          for (int r = 0; r < 16; r++) {
            asm volatile("" : "+v"(end));  // (one comparison at a time: 32 would take as many scalar register pairs)
            if (32 * kt + 8 * (r >> 2) + (r & 3) >= end) nxt[kt][r] = -INFINITY;
          }
      }
    }
    // (the maximum from the second group on, when the scores are there; done before the last one)
    constexpr int FIRST = NG == 4 ? 4 : 2, PER = NG == 4 ? 2 : 4;
    float mx2[2] = {-1.0e30f, -1.0e30f}, mx = 0.0f;
#pragma unroll
    for (int c = 0; c < NG; c++) {
      if constexpr (PV) {
        if (c + 1 < NG) read_v(cV, c + 1);
      }
      if constexpr (decltype(do_s)::value) {
        if (c + 1 == NG) read_k(cK, 0);
      }
      if (c == 0) transfer(nk, is_k, 1 - KB, pair0);
      if constexpr (NI > 2) {
        if (c == NG / 2) transfer(nk, is_k, 1 - KB, pair1);
      }
#pragma unroll
      for (int j = 0; j < 4; j++) {
        if constexpr (PV) {
          constexpr int last = 3;
          const int f = last - j;
          int kt, t, dt;
          pv_of(c, f, kt, t, dt);
          o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf[c][f], __builtin_bit_cast(half8_t, pf[kt][t]), o[dt], 0, 0, 0);
        }
        if constexpr (MAX) {
          const int first = (4 * c + j - FIRST) * PER * 2;
          if (first >= 0 && first < 32) {
#pragma unroll
            for (int e = 0; e < PER; e++) {
              const int x = first + 2 * e;
              mx2[e & 1] = fmaxf(fmaxf(mx2[e & 1], nxt[x >> 4][x & 15]), nxt[x >> 4][(x & 15) + 1]);
            }
          }
          if (first == 32) mx = pair_max(fmaxf(mx2[0], mx2[1])) * a.c;  // in log2 units (c > 0)
        }
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    if constexpr (MAX) {
      // The exponent reference m_run follows the row maximum lazily: it moves only when some row
      // of the wavefront outgrew it by more than 2^8 (probabilities up to 256 are as exact in fp16
      // as those below 1), which after the first tiles is rare; the accumulator is rescaled only then.
      if (__builtin_amdgcn_ballot_w64(mx > m_run + 8.0f) != 0) {
        const float m_new = fmaxf(m_run, mx);
        const float alpha = __builtin_amdgcn_exp2f(m_run - m_new);
        m_run = m_new;
        l_run *= alpha;
#pragma unroll
        for (int dt = 0; dt < DT; dt++)
#pragma unroll
          for (int r = 0; r < 16; r++) o[dt][r] *= alpha;
      }
    }
    advance(nk);
    wait_landed();
    barrier();
  };
  auto idle = [&](int i) __attribute__((always_inline)) {
    tile_transfers(nv, is_v, 2 + ((i + 1) & 1));
    wait_landed();
    barrier();
    tile_transfers(nk, is_k, (i + 1) & 1);
    wait_landed();
    barrier();
  };

  const std::true_type yes{};
  const std::false_type no{};
  const std::integral_constant<int, 0> even{};
  const std::integral_constant<int, 1> odd{};

  barrier();               // the first K tile has landed for every wavefront
  if (grp == 1) barrier(); // group 1 runs half a tile behind
  int i = -1;
  if (active > 0) {
    read_k(sm, 0);
    half1(yes, no, no, even, sb, sa);
    half2(-1, no, yes, yes, odd, sa);
    for (i = 0; i + 2 < active; i += 2) {
      half1(yes, yes, yes, odd, sa, sb);
      half2(i, yes, yes, yes, even, sb);
      half1(yes, yes, yes, even, sb, sa);
      half2(i + 1, yes, yes, yes, odd, sa);
    }
    if (i + 1 < active) {
      half1(yes, yes, yes, odd, sa, sb);
      half2(i, yes, yes, no, even, sb);
      half1(no, yes, yes, even, sb, sa);
      half2(i + 1, yes, no, no, odd, sa);
    } else {
      half1(no, yes, yes, odd, sa, sb);
      half2(i, yes, no, no, even, sb);
    }
    i = active;
  }
  for (; i < steps; i++) idle(i);  // tiles this wavefront has no part in
  if (G == 2 && grp == 0) barrier();
  wait_vm<0>();            // (transfers of no bytes write zeros)
  barrier();               // every read of K and V tiles is done: LDS is free

  // Each group keeps HD / G of the output columns, from dt0 on; with two groups it hands the others over.
  constexpr int OT = DT / G;
  constexpr int XO = G == 1 ? 0 : 2 * 4 * OT * 16 * 64 * 4, XML = G == 1 ? 0 : 2 * 4 * 64 * 8;
  float16_t out[OT];
  float l_tot;
  if constexpr (G == 1) {
#pragma unroll
    for (int d = 0; d < OT; d++) out[d] = o[d];
    l_tot = pair_sum(l_run);
  } else {
    float* const xo = (float*)smem;              // [group][w][OT * 16][64]
    float2* const xml = (float2*)(smem + XO);    // [group][w][64]
    auto hand_over = [&](auto own) __attribute__((always_inline)) {
      constexpr int G0 = decltype(own)::value;
#pragma unroll
      for (int d = 0; d < OT; d++)
#pragma unroll
        for (int r = 0; r < 16; r++) xo[((G0 * 4 + w) * OT * 16 + d * 16 + r) * 64 + lane] = o[(1 - G0) * OT + d][r];
#pragma unroll
      for (int d = 0; d < OT; d++) out[d] = o[G0 * OT + d];
    };
    if (grp == 0) hand_over(even);
    else hand_over(odd);
    xml[(grp * 4 + w) * 64 + lane] = make_float2(m_run, l_run);
    __syncthreads();
    const float2 other = xml[((1 - grp) * 4 + w) * 64 + lane];
    const float m_all = fmaxf(m_run, other.x);
    const float f_own = __builtin_amdgcn_exp2f(m_run - m_all), f_other = __builtin_amdgcn_exp2f(other.x - m_all);
    const float* const recv = xo + ((1 - grp) * 4 + w) * OT * 16 * 64 + lane;
#pragma unroll
    for (int d = 0; d < OT; d++)
#pragma unroll
      for (int r = 0; r < 16; r++) out[d][r] = out[d][r] * f_own + recv[(d * 16 + r) * 64] * f_other;
    m_run = m_all;
    l_tot = pair_sum(l_run * f_own + other.y * f_other);
  }
  const int qi = q0w + frow, col0 = grp * (HD / G);
  if (a.splits == 1) {
    // out[q][32d + 8i + 4g + j] = out[d][4i + j] / l, by way of LDS, so that whole rows are stored
    constexpr int OROWB = ROWB / G, OCPR = CPR / G, PITCH = OROWB + 16;
    static_assert(XO + XML + G * 4 * 32 * PITCH <= G * 4 * TILE, "the output's slots fit the LDS");
    unsigned char* const slot = smem + XO + XML + wave * (32 * PITCH);
    const float inv = 1.0f / l_tot;
#pragma unroll
    for (int d = 0; d < OT; d++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        half4_t r;
#pragma unroll
        for (int j = 0; j < 4; j++) r[j] = (half_t)(out[d][4 * i + j] * inv);
        *(half4_t*)(slot + frow * PITCH + (32 * d + 8 * i + 4 * g) * 2) = r;
      }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the slot is the wavefront's own)
    constexpr int RPI = 64 / OCPR;  // rows of a store instruction
    const int row = lane / OCPR, col = lane % OCPR;
    half_t* const orow = a.out + (int64_t)head * a.so_z + (int64_t)(q0w + row) * a.so_y + col0 + col * 8;
#pragma unroll
    for (int i = 0; i < 32 / RPI; i++) {
      const half8_t r = *(const half8_t*)(slot + (row + i * RPI) * PITCH + col * 16);
      if (q0w + row + i * RPI < a.m) *(half8_t*)(orow + (int64_t)(i * RPI) * a.so_y) = r;
    }
  } else if (qi < a.m) {
    const int64_t prow = ((int64_t)split * a.heads + head) * a.m + qi;
    float* const po = a.part_o + prow * HD + col0 + 4 * g;
#pragma unroll
    for (int d = 0; d < OT; d++)
#pragma unroll
      for (int i = 0; i < 4; i++) {
        float4_t r;
#pragma unroll
        for (int j = 0; j < 4; j++) r[j] = out[d][4 * i + j];
        *(float4_t*)(po + 32 * d + 8 * i) = r;
      }
    if (grp == 0 && g == 0) a.part_ml[prow] = make_float2(m_run, l_tot);
  }
}

// A single tile of keys and few rows: the same arithmetic, in the same order (so the same bits), with
// nothing to overlap -- a workgroup per head, one trip to memory for Q, K and V together, one barrier,
// any strides.  Bound by that trip and the launch.  In the kernel above such a call passes the code of all
// four kinds of halves, waits for V behind the scores and takes Q and the output by way of LDS, which
// pays from about 96 rows on: in a graph, us, this kernel against that one: 32 heads of 128, 64 keys, 17
// rows 3.9 / 4.6, 64 4.7 / 4.9, 96 5.3 / 5.0, 300 6.1 / 5.5; 12 heads of 64 3.1 / 3.7, 3.5 / 3.8, 3.8 / 3.8, 4.1 / 3.9.
template <int HD>
__global__ __launch_bounds__(256, 2) void attention_tile_kernel(AttnArgs a) {
  constexpr int CPR = HD / 8, ROWB = HD * 2, TILE = BN * ROWB, NI = TILE / 1024 / 4, DS = HD / 16, DT = HD / 32;
  __shared__ __attribute__((aligned(1024))) unsigned char smem[2 * TILE];  // K, V

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int frow = lane & 31, g = lane >> 5;
  const int head = blockIdx.x, qi = w * 32 + frow;
  const bool causal = a.mask == ADR_MASK_CAUSAL;

  half8_t qf[DS];
  const half_t* const qrow = a.q + (int64_t)head * a.sq_z + (int64_t)min(qi, a.m - 1) * a.sq_y + g * 8;
#pragma unroll
  for (int ds = 0; ds < DS; ds++) qf[ds] = *(const half8_t*)(qrow + ds * 16);
  // (rows past the last key fetch that one; their scores are masked)
  const uint32_t lds0 = (uint32_t)(uintptr_t)ADR_LDS_PTR(smem) + w * (NI * 1024);
#pragma unroll
  for (int j = 0; j < NI; j++) {
    int row, kc;
    k_chunk_inv<CPR>((w * NI + j) * 64 + lane, row, kc);
    dma_global(lds0 + j * 1024, a.k + (int64_t)head * a.sk_z + (int64_t)min(row, a.n - 1) * a.sk_y + kc * 8);
  }
#pragma unroll
  for (int j = 0; j < NI; j++) {
    const int phys = (w * NI + j) * 64 + lane, row = phys / CPR, c = (phys % CPR) ^ v_swz<CPR>(row);
    dma_global(lds0 + TILE + j * 1024, a.v + (int64_t)head * a.sv_z + (int64_t)min(row, a.n - 1) * a.sv_y + c * 8);
  }
  int offV[DT];
  {
    const int c = lane & 15, b = (lane >> 4) & 1, row = 4 * g + (c >> 2);
#pragma unroll
    for (int dt = 0; dt < DT; dt++)
      offV[dt] = row * ROWB + (((4 * dt + 2 * b + ((c & 3) >> 1)) ^ v_swz<CPR>(row)) << 4) + (c & 1) * 8;
  }
#pragma unroll
  for (int ds = 0; ds < DS; ds++) asm volatile("" : "+v"(qf[ds]));
  wait_vm<0>();
  barrier();
  if (w * 32 >= a.m) return;

  float16_t s[2], o[DT];
#pragma unroll
  for (int r = 0; r < 16; r++) {
    s[0][r] = s[1][r] = 0.0f;
#pragma unroll
    for (int dt = 0; dt < DT; dt++) o[dt][r] = 0.0f;
  }
#pragma unroll
  for (int c = 0; c < DS; c++) {
    const int ds = c ^ 1;
#pragma unroll
    for (int kt = 1; kt >= 0; kt--) {
      const half8_t kf = *(const half8_t*)(smem + k_chunk_off<CPR>(frow, ds * 2 + g) + kt * 32 * ROWB);
      s[kt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(kf, qf[ds], s[kt], 0, 0, 0);
    }
  }
  float mx = -1.0e30f;
  const int end = (causal ? min(a.n, qi + 1) : a.n) - 4 * g;  // this lane's first masked key
#pragma unroll
  for (int kt = 0; kt < 2; kt++)
#pragma unroll
    for (int r = 0; r < 16; r++) {
      if (32 * kt + 8 * (r >> 2) + (r & 3) >= end) s[kt][r] = -INFINITY;
      mx = fmaxf(mx, s[kt][r]);
    }
  const float m_row = fmaxf(-1.0e30f, pair_max(mx) * a.c);
  float sum[2] = {0.0f, 0.0f};
  u32x4_t pf[2][2];
#pragma unroll
  for (int x = 0; x < 32; x += 2) {
    float2_t e;
#pragma unroll
    for (int j = 0; j < 2; j++) {
      e[j] = __builtin_amdgcn_exp2f(fmaf(s[x >> 4][(x & 15) + j], a.c, -m_row));
      sum[j] += e[j];
    }
    pf[x >> 4][x >> 3 & 1][(x & 7) / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e, half2_t));
  }
  typedef short short4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) short4_t lds_short4_t;
#pragma unroll
  for (int x = 0; x < 4; x++) {
    const int y = HD == 64 ? x ^ 1 : x, kt = y >> 1, t = y & 1;
#pragma unroll
    for (int dt = 0; dt < DT; dt++) {
      const unsigned char* const p0 = smem + TILE + offV[dt] + (32 * kt + 16 * t) * ROWB;
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)ADR_LDS_PTR(p0));
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)ADR_LDS_PTR(p0 + 8 * ROWB));
      const half8_t vf = __builtin_shufflevector(__builtin_bit_cast(half4_t, lo), __builtin_bit_cast(half4_t, hi),
                                                 0, 1, 2, 3, 4, 5, 6, 7);
      o[dt] = __builtin_amdgcn_mfma_f32_32x32x16_f16(vf, __builtin_bit_cast(half8_t, pf[kt][t]), o[dt], 0, 0, 0);
    }
  }
  const float inv = 1.0f / pair_sum(sum[0] + sum[1]);
  if (qi >= a.m) return;
  half_t* const orow = a.out + (int64_t)head * a.so_z + (int64_t)qi * a.so_y + 4 * g;
#pragma unroll
  for (int dt = 0; dt < DT; dt++)
#pragma unroll
    for (int i = 0; i < 4; i++) {
      half4_t r;
#pragma unroll
      for (int j = 0; j < 4; j++) r[j] = (half_t)(o[dt][4 * i + j] * inv);
      *(half4_t*)(orow + 32 * dt + 8 * i) = r;
    }
}

// At most sixteen query rows (generation, cross attention) against all keys, no mask: a read of K and
// V.  A workgroup takes one head and one of `splits` parts of its keys; its four wavefronts walk
// tiles of 32 keys in turn, each through two tiles' worth of LDS of its own, so that up to 128 KiB of
// transfers are in flight per compute unit at any time and the loop has no barrier.  The arithmetic is
// that of the kernel above on 16x16x32 MFMAs: S^T = K Q^T, so that a lane holds scores of one query
// row, and O^T = V^T P^T.  The four partial results meet in LDS.
// Bound by the path into a compute unit (69 GB/s) where one workgroup has a head to itself, by memory
// where the parts fill the chip: 32 heads of 128, K and V from HBM, one row against 2047 keys 42 -> 12.7 us
// in eight parts (27 in one; 33.5 MB), against 500 keys 13.2 -> 9.9 in one, against 8192 156 -> 31.
template <int HD>
__global__ __launch_bounds__(256) void attention_rows_kernel(AttnArgs a) {
  constexpr int CPR = HD / 8, KEYS = 32;
  constexpr int ROWB = HD * 2, TILE = KEYS * ROWB;  // bytes of a tile row, of a K or V tile
  constexpr int NI = TILE / 1024;                   // transfers per tile
  constexpr int KS = HD / 32, DB = HD / 16;         // k-steps of S, blocks of 16 output columns
  constexpr int WAVE = 4 * TILE;                    // K0 K1 V0 V1 of a wavefront
  constexpr int PITCH = HD + 4;                     // of the partial results' rows, in floats
  static_assert(4 * 16 * (PITCH + 2) * 4 <= 4 * WAVE, "the partial results fit the tiles' LDS");
  __shared__ __attribute__((aligned(1024))) unsigned char smem[4 * WAVE];

  const int tid = threadIdx.x, lane = tid & 63, w = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int frow = lane & 15, g = lane >> 4;
  const int head = blockIdx.x / a.splits, split = blockIdx.x % a.splits;
  const half_t* const Q = a.q + (int64_t)head * a.sq_z;
  const half_t* const K = a.k + (int64_t)head * a.sk_z;
  const half_t* const V = a.v + (int64_t)head * a.sv_z;

  const int all = (a.n + KEYS - 1) / KEYS;
  const int tile0 = (int)((int64_t)all * split / a.splits), tile1 = (int)((int64_t)all * (split + 1) / a.splits);
  const int row_end = min(a.n, tile1 * KEYS);
  const int tiles = max(0, (tile1 - tile0 - w + 3) >> 2);  // of this wavefront: tile0 + w + 4 i

  const uint32_t lds0 = (uint32_t)(uintptr_t)ADR_LDS_PTR(smem) + w * WAVE;
  const unsigned char* const sm = smem + w * WAVE;
  uint32_t koff[NI], voff[NI];
#pragma unroll
  for (int j = 0; j < NI; j++) {
    int krow, kc;
    k_chunk_inv<CPR>(j * 64 + lane, krow, kc);
    const int vrow = (j * 64 + lane) / CPR, vc = (lane % CPR) ^ v_swz8<CPR>(vrow);
    koff[j] = ((uint32_t)krow * (uint32_t)a.sk_y + kc * 8) * 2 - (j & 1) * 1024;
    voff[j] = ((uint32_t)vrow * (uint32_t)a.sv_y + vc * 8) * 2 - (j & 1) * 1024;
  }
  // (Tiles that exist: a transfer of no bytes takes the address path's time all the same.  With three such
  // tiles of a wavefront asked for, one row against 64 keys of 32 heads of 128 took 4.2 us in a graph, 3.4 now;
  // 3.8 with the kernel above before this one was there.)
  auto fetch = [&](int i) __attribute__((always_inline)) {
    const int key0 = (tile0 + w + 4 * i) * KEYS, rows = row_end - key0;
    const uint64_t pk = (uint64_t)(K + (int64_t)key0 * a.sk_y), pv = (uint64_t)(V + (int64_t)key0 * a.sv_y);
    const u32x4_t dk = {(uint32_t)pk, (uint32_t)(pk >> 32) & 0xffffu,
                        (uint32_t)((rows - 1) * a.sk_y * 2 + ROWB), 0x00020000u};
    const u32x4_t dv = {(uint32_t)pv, (uint32_t)(pv >> 32) & 0xffffu,
                        (uint32_t)((rows - 1) * a.sv_y * 2 + ROWB), 0x00020000u};
#pragma unroll
    for (int j = 0; j < NI; j += 2) dma_buffer_pair<0>(lds0 + (i & 1) * TILE + j * 1024, koff[j], koff[j + 1], dk);
#pragma unroll
    for (int j = 0; j < NI; j += 2) dma_buffer_pair<0>(lds0 + (2 + (i & 1)) * TILE + j * 1024, voff[j], voff[j + 1], dv);
  };

  half8_t qf[KS];
  const half_t* const qrow = Q + (int64_t)min(frow, a.m - 1) * a.sq_y + g * 8;
#pragma unroll
  for (int ks = 0; ks < KS; ks++) qf[ks] = *(const half8_t*)(qrow + ks * 32);
  if (tiles > 0) fetch(0);
  if (tiles > 1) fetch(1);
  int offK[KS], offV[DB];
#pragma unroll
  for (int ks = 0; ks < KS; ks++) offK[ks] = k_chunk_off<CPR>(frow, ks * 4 + g);
  {
    const int c = lane & 15, row = 4 * g + (c >> 2);
#pragma unroll
    for (int db = 0; db < DB; db++)
      offV[db] = row * ROWB + (((2 * db + ((c & 3) >> 1)) ^ v_swz8<CPR>(row)) << 4) + (c & 1) * 8;
  }
  typedef short short4_t __attribute__((ext_vector_type(4)));
  typedef __attribute__((address_space(3))) short4_t lds_short4_t;

  float4_t o[DB];
  float m_run = -1.0e30f, l_run = 0.0f;
#pragma unroll
  for (int db = 0; db < DB; db++) o[db] = float4_t{0.0f, 0.0f, 0.0f, 0.0f};
  // Tile i; `next`: there is a tile i + 1, `more`: and a tile i + 2.
  auto tile = [&](int i, auto next, auto more) __attribute__((always_inline)) {
    wait_vm<decltype(next)::value ? 2 * NI : 0>();  // tile i has landed (tile i + 1 may be in flight)
    const unsigned char* const cK = sm + (i & 1) * TILE;
    const unsigned char* const cV = sm + (2 + (i & 1)) * TILE;
    float4_t s[2] = {{0.0f, 0.0f, 0.0f, 0.0f}, {0.0f, 0.0f, 0.0f, 0.0f}};
#pragma unroll
    for (int ks = 0; ks < KS; ks++)
#pragma unroll
      for (int kb = 0; kb < 2; kb++) {
        const half8_t kf = *(const half8_t*)(cK + offK[ks] + kb * 16 * ROWB);
        s[kb] = __builtin_amdgcn_mfma_f32_16x16x32_f16(kf, qf[ks], s[kb], 0, 0, 0);
      }
    half8_t vf[DB];
#pragma unroll
    for (int db = 0; db < DB; db++) {
      const unsigned char* const p0 = cV + offV[db];
      const short4_t lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)ADR_LDS_PTR(p0));
      const short4_t hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((lds_short4_t*)ADR_LDS_PTR(p0 + 16 * ROWB));
      vf[db] = __builtin_shufflevector(__builtin_bit_cast(half4_t, lo), __builtin_bit_cast(half4_t, hi),
                                       0, 1, 2, 3, 4, 5, 6, 7);
    }
    const int left = row_end - (tile0 + w + 4 * i) * KEYS - 4 * g;  // keys of this lane from its first one on
    float mx = -1.0e30f;
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 4; r++) {
        if (16 * kb + r >= left) s[kb][r] = -INFINITY;
        mx = fmaxf(mx, s[kb][r]);
      }
    float x = mx, y = mx;  // over the four lanes that share a row
    swap_halves(x, y);
    x = fmaxf(x, y), y = x;
    swap_rows(x, y);
    const float m_new = fmaxf(m_run, fmaxf(x, y) * a.c), alpha = __builtin_amdgcn_exp2f(m_run - m_new);
    m_run = m_new;
    float sum = 0.0f;
    u32x4_t pf;
#pragma unroll
    for (int kb = 0; kb < 2; kb++)
#pragma unroll
      for (int r = 0; r < 4; r += 2) {
        float2_t e;
#pragma unroll
        for (int j = 0; j < 2; j++) e[j] = __builtin_amdgcn_exp2f(fmaf(s[kb][r + j], a.c, -m_new));
        sum += e[0] + e[1];
        pf[kb * 2 + r / 2] = __builtin_bit_cast(uint32_t, __builtin_convertvector(e, half2_t));
      }
    l_run = l_run * alpha + sum;
#pragma unroll
    for (int db = 0; db < DB; db++) {
      o[db] *= alpha;
      o[db] = __builtin_amdgcn_mfma_f32_16x16x32_f16(vf[db], __builtin_bit_cast(half8_t, pf), o[db], 0, 0, 0);
    }
    // (the tile has been read: its fragments are in registers)
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    if constexpr (decltype(more)::value) fetch(i + 2);
  };
  const std::true_type yes{};
  const std::false_type no{};
  int i = 0;
  for (; i + 2 < tiles; i++) tile(i, yes, yes);
  if (i + 1 < tiles) tile(i++, yes, no);
  if (i < tiles) tile(i, no, no);

  // Merge the four wavefronts' results: [wavefront][row][HD] sums, and (maximum, sum) of every row.
  wait_vm<0>();
  __syncthreads();
  float* const xo = (float*)smem;
  float2* const xml = (float2*)(smem + 4 * 16 * PITCH * 4);
  float x = l_run, y = x;
  swap_halves(x, y);
  x = x + y, y = x;
  swap_rows(x, y);
  if (g == 0) xml[w * 16 + frow] = make_float2(m_run, x + y);
#pragma unroll
  for (int db = 0; db < DB; db++) *(float4_t*)(xo + (w * 16 + frow) * PITCH + 16 * db + 4 * g) = o[db];
  __syncthreads();
  for (int e = tid; e < a.m * (HD / 4); e += 256) {
    const int row = e / (HD / 4), col = e % (HD / 4) * 4;
    float2 ml[4];
    float m_all = -1.0e30f, l = 0.0f;
#pragma unroll
    for (int x = 0; x < 4; x++) {
      ml[x] = xml[x * 16 + row];
      m_all = fmaxf(m_all, ml[x].x);
    }
    float4_t sum = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int x = 0; x < 4; x++) {
      const float f = __builtin_amdgcn_exp2f(ml[x].x - m_all);
      l += ml[x].y * f;
      sum += *(const float4_t*)(xo + (x * 16 + row) * PITCH + col) * f;
    }
    if (a.splits == 1) {
      half4_t r;
      const float inv = 1.0f / l;
#pragma unroll
      for (int j = 0; j < 4; j++) r[j] = (half_t)(sum[j] * inv);
      *(half4_t*)(a.out + (int64_t)head * a.so_z + (int64_t)row * a.so_y + col) = r;
    } else {
      const int64_t prow = ((int64_t)split * a.heads + head) * a.m + row;
      *(float4_t*)(a.part_o + prow * HD + col) = sum;
      if (col == 0) a.part_ml[prow] = make_float2(m_all, l);
    }
  }
}

constexpr int MAX_SPLITS = 32;

// Sums the parts of a row whose keys several workgroups shared: one wavefront per row, HD / 64
// columns per lane.  Its time is that of two trips to memory (the parts come from other dies), so
// lane x reads the x-th part's maximum and sum, and the parts themselves are requested eight at a time.
template <int HD>
__global__ __launch_bounds__(256) void attention_combine_kernel(AttnArgs a) {
  constexpr int C = HD / 64;
  typedef float vec_t __attribute__((ext_vector_type(C)));
  __shared__ float factor[4][MAX_SPLITS];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int rows = a.heads * a.m, row = min((int)blockIdx.x * 4 + w, rows - 1);
  const float2 ml = lane < a.splits ? a.part_ml[(int64_t)lane * rows + row] : make_float2(-1.0e30f, 0.0f);
  const float* const part = a.part_o + (int64_t)row * HD + lane * C;
  const int64_t step = (int64_t)rows * HD;
  float m_all = ml.x;
#pragma unroll
  for (int off = 1; off < MAX_SPLITS; off <<= 1) m_all = fmaxf(m_all, __shfl_xor(m_all, off, 64));
  float f = __builtin_amdgcn_exp2f(ml.x - m_all), l = ml.y * f;
#pragma unroll
  for (int off = 1; off < MAX_SPLITS; off <<= 1) l += __shfl_xor(l, off, 64);
  if (lane < MAX_SPLITS) factor[w][lane] = f / l;
  __syncthreads();
  vec_t acc = 0.0f;
  for (int s = 0; s < a.splits; s += 8) {
    vec_t v[8];
#pragma unroll
    for (int j = 0; j < 8; j++) v[j] = *(const vec_t*)(part + min(s + j, a.splits - 1) * step);
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (s + j < a.splits) acc += v[j] * factor[w][s + j];
  }
  typedef half_t hvec_t __attribute__((ext_vector_type(C)));
  half_t* const o = a.out + (int64_t)(row / a.m) * a.so_z + (int64_t)(row % a.m) * a.so_y + lane * C;
  if ((int)blockIdx.x * 4 + w < rows) *(hvec_t*)o = __builtin_convertvector(acc, hvec_t);
}

}  // namespace

// The buffer transfers count the bytes of a head, and of two tiles, in 31 bits, and take rows to be no
// closer than they are long.
static bool attention_wide(const AttentionShape& t) {
  const int64_t far = t.sk_y > t.sv_y ? t.sk_y : t.sv_y;
  return t.sq_y < t.d || t.sk_y < t.d || t.sv_y < t.d || far >= 1 << 22 || t.n * far >= (int64_t)1 << 30 ||
         (int64_t)t.m * t.sq_y >= (int64_t)1 << 30;
}

// Fewer query blocks than compute units leave units idle, so the keys are then shared: by two groups of
// wavefronts inside the workgroup, or by several workgroups, whose parts a second launch adds up.
AttentionPlan attention_plan(const AttentionShape& t, int cus, int64_t avail) {
  AttentionPlan p;
  p.cus = cus;
  p.wide = attention_wide(t);
  p.rows = t.m <= 16 && t.mask == ADR_MASK_NONE && !p.wide;
  // (no row sees a key past the last row's own)
  const int n = t.mask == ADR_MASK_CAUSAL ? std::min(t.n, t.m) : t.n;
  p.tile = !p.rows && n <= BN && t.m <= 80;  // (between 65 rows, where that kernel still is ahead, and 96)
  const int64_t rows = (int64_t)t.heads * t.m, blocks = (int64_t)t.heads * ((t.m + BM - 1) / BM);
  // (rows beyond what all parts of can be counted in 31 bits fill the chip many times over)
  const int most = rows <= 0x7fffffff / MAX_SPLITS ? MAX_SPLITS : 1;
  const int64_t part = most > 1 ? rows * (t.d * 4 + 8) : 0;
  // One workgroup per compute unit at most: two groups take 9.5 us per 1000 keys where one takes 14
  // (two such workgroups per unit take as long as one of two groups), and half a microsecond to merge,
  // which pays from six tiles on (20 heads of 64, 1500 x 1500: 25.3 -> 21.2 us, 12 x 1000 causal
  // 15.3 -> 12.7; 12 x 256 6.2 -> 6.3).
  p.groups = !p.rows && !p.wide && blocks <= cus && n > 5 * BN ? 2 : 1;
  // Under the mask also with up to half as many blocks again, from 1024 keys on: the heavy blocks start first and
  // the light ones fill in behind them, and none is left to a single group alone on its unit (us, one
  // group / two: 32 heads of 128, 1100 24.9 / 22.1, 1280 26.6 / 23.4, 1500 29.8 / 28.1; 20 of 64, 1700 22.1 / 17.6,
  // 2048 25.1 / 21.1).  With more blocks the second round is as long as what it saves (32 heads, 2048 43.8 / 42.9, 40
  // heads, 1300 28.0 / 29.5, 1600 36.9 / 40.8), with fewer keys the merges are (64 heads, 513 13.6 / 16.6).
  p.two_rounds = !p.rows && !p.wide && t.mask == ADR_MASK_CAUSAL && blocks > cus && 2 * blocks <= 3 * (int64_t)cus && n >= 1024;
  if (p.two_rounds) p.groups = 2;
  p.splits = 1;
  // Times beyond what every launch takes, in us, fitted to 40 shapes of 12-40 heads, 1-448 query rows
  // and 64-8192 keys with every number of parts: the rows kernel reads 69 GB/s per compute unit; parts
  // cost a launch (and the host its issue: more than a short read takes) and their way through memory.
  double best = 1e30;
  for (int s = 1; s <= most && s * 64 <= n + 63 && (s == 1 || s * part <= avail); s++) {
    const double keys = (double)n / s;
    double us;
    if (p.rows) {
      us = ceil((double)t.heads * s / cus) * keys * t.d * (4.0 / 69e3);
      if (s > 1) us += 4.0;
    } else if (s == 1 && p.groups == 2 && !p.two_rounds) {
      us = keys * 0.0095 + 0.5;
    } else {
      us = ceil((double)blocks * s / cus) * keys * 0.014;
      if (s > 1) us += 2.5;
    }
    if (s > 1) us += s * part / 1.35e6;
    if (us < best * 0.97) best = us, p.splits = s;
    // Under some 500 keys the second launch is time the host does not have: a call of two takes it 10 us,
    // and one walk over all keys is over before (17 rows, 16 heads of 64: 257 keys 7.3 us unshared, 10.2
    // shared; 500 keys 8.0, 10.2; at 640 8.1, 9.9, but 8.1, 7.4 on the device; 2 heads of 128: 384 keys 8.6,
    // 10.0; 500 9.9, 10.0; 640 10.9, 9.9).
    if (!p.rows && s == 1 && us < 5.5) break;
  }
  if (p.splits > 1) p.groups = 1, p.two_rounds = false;
  p.workspace_bytes = p.splits > 1 ? p.splits * part : 0;
  return p;
}

template <int HD>
static void attention_launches(hipStream_t stream, const AttnArgs& a, const AttentionPlan& p) {
  const dim3 block(256), grid((unsigned)(a.heads * (p.rows ? 1 : a.qblocks) * a.splits));
  if (p.rows) hipLaunchKernelGGL(attention_rows_kernel<HD>, grid, block, 0, stream, a);
  else if (p.tile) hipLaunchKernelGGL(attention_tile_kernel<HD>, grid, block, 0, stream, a);
  else if (p.wide) hipLaunchKernelGGL(HIP_KERNEL_NAME(attention_fwd_kernel<HD, 1, true>), grid, block, 0, stream, a);
  else if (p.groups == 2) hipLaunchKernelGGL(HIP_KERNEL_NAME(attention_fwd_kernel<HD, 2, false>), grid, dim3(512), 0, stream, a);
  else hipLaunchKernelGGL(HIP_KERNEL_NAME(attention_fwd_kernel<HD, 1, false>), grid, block, 0, stream, a);
  if (a.splits > 1) {
    const int64_t rows = (int64_t)a.heads * a.m;
    hipLaunchKernelGGL(attention_combine_kernel<HD>, dim3((unsigned)((rows + 3) / 4)), block, 0, stream, a);
  }
}

hipError_t launch_attention(hipStream_t stream, half_t* out, const half_t* q, const half_t* k, const half_t* v,
                            const AttentionShape& t, const AttentionPlan& p, float scale, float temp, void* workspace) {
  AttnArgs a;
  a.out = out; a.q = q; a.k = k; a.v = v;
  a.heads = t.heads; a.m = t.m; a.n = t.n;
  a.so_y = t.so_y; a.so_z = t.so_z; a.sq_y = t.sq_y; a.sq_z = t.sq_z;
  a.sk_y = t.sk_y; a.sk_z = t.sk_z; a.sv_y = t.sv_y; a.sv_z = t.sv_z;
  // the three-call sequence multiplies by the scale rounded to fp16 (matmul.cu:60-74)
  a.c = (float)(half_t)scale * 1.44269504088896340736f / temp;
  a.mask = t.mask;
  a.splits = p.splits;
  const int64_t rows = (int64_t)t.heads * t.m;
  a.part_o = (float*)workspace;
  a.part_ml = (float2*)((float*)workspace + (a.splits > 1 ? a.splits * rows * t.d : 0));
  a.qblocks = (t.m + BM - 1) / BM;
  a.upper = !p.two_rounds && (int64_t)t.heads * a.qblocks * a.splits <= 2 * p.cus ? (a.qblocks + 1) / 2 : a.qblocks;
  // (parts are shared only where their rows can be counted: no product here runs over)
  if ((int64_t)t.heads * a.qblocks * a.splits > 0x7fffffffLL) return hipErrorInvalidConfiguration;
  if (t.d == 128) attention_launches<128>(stream, a, p);
  else attention_launches<64>(stream, a, p);
  return hipGetLastError();
}

}  // namespace adr
