// gemm.h — dense K-contraction on CDNA4 matrix cores (family G).
//
// The reference lowers C[m,n] = sum_k A[m,k] B[k,n] as a CTA-wide
// WarpReducer collective per output element (a shuffle tree per Reduce and
// two barriers per Combine; .planning/quick/261030-uai-.../after-cu/gemm.cu:
// 59-90). Here the contraction runs on MFMA:
//   bf16 inputs : v_mfma_f32_16x16x32_bf16 (gfx950): large planes of whole
//                 256x256 tiles on gemm_bf16_4w (K % 64 == 0 and K >= 256)
//                 or gemm_bf16_256_w8, everything else on gemm16_any;
//                 fp32 accumulate (f16 inputs: the same kernels with the
//                 _f16 MFMAs)
//   fp32 inputs : v_mfma_f32_32x32x2f32 (gemm_f32_4w on whole tiles from
//                 M, N >= 4096 on, else gemm_f32_any), fp32 accumulate
//   output planes of at most 2^20 elements: gemm_small
// The any-shape kernels stage slices of K through registers into LDS with
// unguarded, possibly unaligned 16-byte loads (gemm16_tile, gemm32_tile).
//
// v_mfma_f32_32x32x2f32 operand/result lane layout (CDNA3/CDNA4 ISA):
//   A operand: lane l supplies row (l % 32), k = l / 32
//   B operand: lane l supplies col (l % 32), same k
//   result   : lane l, element i -> row 8*(i/4) + 4*(l/32) + (i%4), col l%32
#ifndef TCA_HIP_GEMM_H_
#define TCA_HIP_GEMM_H_

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>
#include <utility>

namespace tca {
namespace hip {

typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));

// The 16-bit contractions below move raw 16-bit values (as bf16x8 registers)
// through memory, LDS and registers; F16 selects the MFMA that reads them as
// IEEE half (v_mfma_f32_*_f16) instead of bfloat16. The fp32 accumulation,
// the operand layout and every data movement are the same for both.
template <bool F16, typename Acc>
__device__ __forceinline__ Acc mfma_16x16x32_16b(const bf16x8& a, const bf16x8& b, const Acc& c) {
  if constexpr (F16)
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c, 0, 0, 0);
  else
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, b, c, 0, 0, 0);
}
typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));

// Maps the linear workgroup id to a (tile_m, tile_n) pair. Workgroups are
// dealt round-robin over the 8 XCDs; regrouping so that each XCD receives a
// contiguous run of tiles (and walking those runs in GROUP_M-row bands) keeps
// the A row panels and B column panels a run touches inside one XCD's L2.
// `tile` is the linear tile index: the workgroup id, or for a batched
// contraction the workgroup id within its batch (the emitted kernel passes it).
__device__ __forceinline__ void gemm_tile_coords(uint32_t tiles_m, uint32_t tiles_n, uint32_t* tm, uint32_t* tn,
                                                 uint32_t tile) {
  const uint32_t total = tiles_m * tiles_n;
  uint32_t b = tile;
  if (total % 8u == 0u) b = (b % 8u) * (total / 8u) + b / 8u;
  const uint32_t kGroup = 8u;
  const uint32_t band = kGroup * tiles_n;
  const uint32_t g = b / band;
  const uint32_t first_m = g * kGroup;
  const uint32_t rows = (tiles_m - first_m) < kGroup ? (tiles_m - first_m) : kGroup;
  const uint32_t in = b % band;
  *tm = first_m + in % rows;
  *tn = in / rows;
}

// ----------------------------------------------- 16-bit path, any shape
// The thread index, computed where it is used: inside a loop over tiles the
// compiler would otherwise keep every lane address of every tile shape in
// registers across the loop, and spill them.
__device__ __forceinline__ uint32_t thread_here() {
  uint32_t t = threadIdx.x;
  asm volatile("" : "+v"(t));
  return t;
}
// ... and the lane, counted, so that not even the thread index is kept.
__device__ __forceinline__ uint32_t lane_here() {
  uint32_t lane;
  asm volatile("v_mbcnt_lo_u32_b32 %0, -1, 0\n\tv_mbcnt_hi_u32_b32 %0, -1, %0" : "=v"(lane));
  return lane;
}

// Between the writes and the reads of LDS that lanes of one wave exchange, and
// between those reads and the next writes. The hardware completes the LDS
// operations of one wave in order, so this costs no instruction; it tells the
// compiler, which sees one thread only, that other lanes' values are read.
__device__ __forceinline__ void wave_exchange() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront", "local");
  __builtin_amdgcn_wave_barrier();
}

// Unaligned 16-byte accesses: gfx950 serves a 16-byte vector load or store
// at any element address (the amdhsa unaligned access mode), so rows whose
// length is not a multiple of the vector still move 16 bytes per lane.
typedef uint32_t u32x4_a2 __attribute__((ext_vector_type(4), aligned(2)));
typedef float f32x4_a4 __attribute__((ext_vector_type(4), aligned(4)));
__device__ __forceinline__ u32x4 load16_any(const uint16_t* p) { return *reinterpret_cast<const u32x4_a2*>(p); }

// The eight 16-bit values of v moved down by n places (zeros shifted in; all
// zero from n = 8 on): a chunk that would run past the end of its row is
// loaded from 8 elements before that end instead, so the load stays inside
// the row, and moved into place.
__device__ __forceinline__ u32x4 shift_down16(u32x4 v, uint32_t n) {
  uint64_t lo = v[0] | (static_cast<uint64_t>(v[1]) << 32), hi = v[2] | (static_cast<uint64_t>(v[3]) << 32);
  const uint32_t b = 16u * (n & 3u);
  if (n & 4u) {
    lo = hi;
    hi = 0u;
  }
  lo = b ? (lo >> b) | (hi << (64u - b)) : lo;
  hi >>= b;
  if (n >= 8u) lo = hi = 0u;
  return u32x4{static_cast<uint32_t>(lo), static_cast<uint32_t>(lo >> 32), static_cast<uint32_t>(hi),
               static_cast<uint32_t>(hi >> 32)};
}

typedef short i16x4 __attribute__((ext_vector_type(4)));
typedef __attribute__((address_space(3))) void lds_void;

// s_waitcnt immediate for gfx9: vmcnt[3:0] | expcnt[6:4] (7 = no wait) |
// lgkmcnt[11:8] | vmcnt[5:4] at [15:14].
constexpr int waitcnt_imm(int vm, int lgkm) { return (vm & 15) | (7 << 4) | ((lgkm & 15) << 8) | ((vm >> 4) << 14); }

// Whether the whole 256x256 tiles of `batch` planes run on the direct-to-LDS
// kernels (one workgroup per CU, so in rounds of 256 tiles) rather than on
// gemm16_any's 128x128 tiles. Measured at K = 4096 (time grows with K on both
// sides): a round of 256x256 tiles takes 95 us, 128x128 tiles 0.16 us each,
// and the ragged edges, which gemm16_any takes afterwards, 40 us. Planes that
// are whole tiles throughout compare the first two: from WHOLE_MIN elements
// on (128 tiles; the times cross at 150, but with that bound 2304 x 4096 x 4096
// took 109 us against 84; the plan's guards carry the same bound, and skip
// gemm16_any there); planes with edges also pay the third. WHOLE_MIN 0: always.
template <uint64_t WHOLE_MIN>
__host__ __device__ __forceinline__ bool gemm16_on_whole_tiles(uint32_t M, uint32_t N, uint32_t batch) {
  if constexpr (WHOLE_MIN == 0u) return true;
  if (static_cast<uint64_t>(M) * N * batch < WHOLE_MIN) return false;
  if (M % 256u == 0u && N % 256u == 0u) return true;
  const uint64_t whole = static_cast<uint64_t>(M / 256u) * (N / 256u) * batch;
  const uint64_t t128 = static_cast<uint64_t>((M - 1u) / 128u + 1u) * ((N - 1u) / 128u + 1u) * batch;
  return (whole + 255u) / 256u * 600u + 250u <= t128;
}
// K and row alignments the direct-to-LDS kernels take: K a positive multiple
// of 32, [K][N] / [N][K] rows 16-byte aligned.
__host__ __device__ __forceinline__ bool gemm16_direct_k(uint32_t N, uint32_t K) { return K % 32u == 0u && N % 8u == 0u && K > 0u; }
// The (tile_m, tile_n) of tile index `tile` among the whole 256x256 tiles of
// one plane; false past them (the edges are gemm16_any's).
__device__ __forceinline__ bool gemm16_whole_coords(uint32_t M, uint32_t N, uint32_t tile, uint32_t* tm, uint32_t* tn) {
  const uint32_t tiles_m = M / 256u, tiles_n = N / 256u;
  if (tile >= tiles_m * tiles_n) return false;
  gemm_tile_coords(tiles_m, tiles_n, tm, tn, tile);
  return true;
}

__device__ __forceinline__ uint32_t swz_rows32(uint32_t row, uint32_t cg) {
  return row * 32u + ((cg ^ (((row >> 3) & 1u) << 1)) << 3);
}
__device__ __forceinline__ uint32_t swz_rows64(uint32_t row, uint32_t g) { return row * 64u + ((g ^ (row & 6u)) << 3); }
// The 16-byte slot of a [K][BN] slice's row k is XORed with this (measured
// bank cycles at gemm_bf16_256_w8): rows of 256 bytes and more cover the 64
// banks, rows of 128 bytes pair up by the parity of k.
template <uint32_t BN>
__device__ __forceinline__ uint32_t kn_slot_xor(uint32_t k) {
  if constexpr (BN >= 128u) return ((k & 3u) | (((k >> 3) & 1u) << 2)) << 1;
  else if constexpr (BN == 64u) return (((k >> 1) & 1u) | (((k >> 3) & 1u) << 1)) << 1;
  else return ((k >> 3) & 1u) << 1;  // 64-byte rows: four to the banks
}
template <uint32_t BN>
__device__ __forceinline__ uint32_t swz_kn(uint32_t k, uint32_t n) {
  return k * BN + (((n >> 3) ^ kn_slot_xor<BN>(k)) << 3) + (n & 7u);
}

// B operand of v_mfma_f32_16x16x32_bf16 (lane l: column n_col0 + l%16,
// k = k_row0 + 8(l/16) .. +8) from a [K][BN] slice with the gfx950
// transposing read ds_read_b64_tr_b16: within each 16-lane group, lane j
// points at four consecutive values R_j of one k row and lane i receives
// [R_{i/4}[i%4], R_{4+i/4}[i%4], R_{8+i/4}[i%4], R_{12+i/4}[i%4]]. With lane j
// addressing row kb + j/4, columns n_col0 + 4(j%4), lane i gets
// B[kb + e][n_col0 + i] for e = 0..3; a second read at kb + 4 completes its 8.
template <uint32_t BN>
__device__ __forceinline__ bf16x8 frag_b16_tr(const uint16_t* Bs, uint32_t n_col0, uint32_t lane, uint32_t k_row0 = 0u) {
  const uint32_t g = lane >> 4, j = lane & 15u;
  const uint32_t k = k_row0 + 8u * g + (j >> 2), n = n_col0 + 4u * (j & 3u);
  const i16x4 lo =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(Bs + swz_kn<BN>(k, n)));
  const i16x4 hi =
      __builtin_amdgcn_ds_read_tr16_b64_v4i16((__attribute__((address_space(3))) i16x4*)(Bs + swz_kn<BN>(k + 4u, n)));
  typedef short i16x8 __attribute__((ext_vector_type(8)));
  const i16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
  return __builtin_bit_cast(bf16x8, v);
}

// One BM x BN tile of C at (m0, n0), every shape: ragged edges, K of any
// length, rows of any alignment. KG groups of WGM x WGN waves each hold the
// whole tile, a wave (BM/WGM) x (BN/WGN) of it as blocks of
// v_mfma_f32_16x16x32, and take every KG-th 64-deep slice of K; their sums
// meet in LDS in group order. A slice goes global memory -> registers (16
// bytes per lane, D of the group's slices ahead) -> LDS (two buffers per
// group, one barrier per slice) -> fragments.
// No load is guarded: rows past the end re-read the last row (their results
// are not stored), and a chunk past the end of its row is loaded from 8
// elements before it and moved into place on its way into LDS
// (shift_down16), so the K tail adds zeros. With guarded loads and one wave
// per SIMD the kernel before took 269 us for 1001 x 1501 x 1003 (13 now) and
// 362 for 257 x 4096 x 4096 (31); 1000 x 4096 x 1024 went from 97 to 15 us.
// What bounds it: the waves of a workgroup load, write and compute in step,
// so the 0.27 us of MFMAs and fragment reads of a 128x128 slice and the 0.3 us
// of its loads and LDS writes overlap little (0.5-0.6 us a slice). Measured
// at 2048 x 2048 x 4096 and not better than the 44 us here: 4 waves per
// workgroup and two workgroups per CU 47, two groups of 4 waves on
// alternate slices 43 (but 106 against 94 at 3000^3), the same with the groups half a turn
// apart 44, operands loaded straight into a 4-deep LDS ring 45 (8 waves) and
// 55 (4 waves). `TINY` (K-contiguous rows or
// [K][N] rows shorter than one chunk) loads those element by element.
// PAIRS: the two 32-deep products of a slice start from zero, their sum is added
// to the accumulators, and every 8 turns these to a second set (in the long loop
// the second product adds to the first). A matrix instruction that adds to a
// running sum rounds it worse than an addition does, so chains of them show where
// K is short. Distance from 64 bits, 1e-8, by 16 waves' sums / chains of 8
// instructions / pairs: 32 batches of 500 x 500, K = 64 4.02 / 4.23 / 3.91, K = 256
// 7.39 / 8.55 / 5.63; 1000 x 1000, K = 1000 8.87 / 9.29 / 7.49, K = 4096 11.5 / 10.6 /
// 8.57. Many batches pay up to 5% of their time for it (64 x 1024 x 1024 x 32 76.6 us
// by chains, 80.3).
// `lds` holds KG * 2 * 64 * (BM + BN) values; `thread` is threadIdx.x.
template <uint32_t BM, uint32_t BN, uint32_t WGM, uint32_t WGN, uint32_t KG, int D, bool B_NK, bool F16, bool TINY,
          bool PAIRS = false, typename Epi>
__device__ __forceinline__ void gemm16_tile(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                            float* __restrict__ C, uint32_t M, uint32_t N, uint32_t K, Epi epi,
                                            uint32_t m0, uint32_t n0, uint16_t* lds, uint32_t thread) {
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr uint32_t THREADS = 64u * WGM * WGN, TM = BM / WGM, TN = BN / WGN;
  constexpr int IM = TM / 16, JN = TN / 16, CA = BM * 8 / THREADS, CB = BN * 8 / THREADS;
  static_assert(CA >= 1 && CB >= 1 && (D == 1 || D % 2 == 0), "whole chunks per thread; the buffer of a slice is static");
  constexpr uint32_t ASL = BM * 64u, BUF = ASL + BN * 64u;
  const uint32_t lane = thread & 63u, wave_id = __builtin_amdgcn_readfirstlane(thread >> 6);
  const uint32_t grp = wave_id / (WGM * WGN), wave = wave_id % (WGM * WGN), tid = wave * 64u + lane;
  const uint32_t wm = (wave / WGN) * TM, wn = (wave % WGN) * TN;
  uint16_t* glds = lds + grp * (2u * BUF);
  // Chunk i of this thread: row (i * THREADS + tid) / 8 of a K-contiguous
  // panel at k chunk tid % 8, or row k = (i * THREADS + tid) / (BN / 8) of a
  // [K][N] slice at column chunk tid % (BN / 8).
  const uint32_t kch = (tid & 7u) * 8u, row0 = tid >> 3;
  const uint32_t bk0 = tid / (BN / 8u), bn = n0 + (tid % (BN / 8u)) * 8u;
  const uint16_t* pa[CA];
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const uint32_t r = m0 + row0 + i * (THREADS / 8u);
    pa[i] = A + static_cast<uint64_t>(r < M ? r : M - 1u) * K;
  }
  const uint16_t* pb[B_NK ? CB : 1];
  uint32_t bsh = 0u;  // [K][N]: places this thread's chunks move down (columns past N)
  if constexpr (B_NK) {
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      const uint32_t r = n0 + row0 + i * (THREADS / 8u);
      pb[i] = B + static_cast<uint64_t>(r < N ? r : N - 1u) * K;
    }
  } else {
    const uint32_t last = N >= 8u ? N - 8u : 0u, at = bn < last ? bn : last;
    bsh = bn - at;
    pb[0] = B + at;
  }
  auto load_k = [&](const uint16_t* row, uint32_t k0) -> u32x4 {  // a chunk of a K-contiguous row
    const uint32_t k = k0 + kch;
    if constexpr (TINY) {
      if (K < 8u) {
        u32x4 v = {0u, 0u, 0u, 0u};
        for (uint32_t e = 0; e < 8u; ++e)
          if (k + e < K) v[e >> 1] |= static_cast<uint32_t>(row[k + e]) << (16u * (e & 1u));
        return v;
      }
    }
    return load16_any(row + (k < K - 8u ? k : K - 8u));
  };
  auto load_n = [&](uint32_t k) -> u32x4 {  // a chunk of row k of a [K][N] operand
    const uint16_t* row = pb[0] + static_cast<uint64_t>(k < K ? k : K - 1u) * N;
    if constexpr (TINY) {
      if (N < 8u) {
        u32x4 v = {0u, 0u, 0u, 0u};
        for (uint32_t e = 0; e < 8u; ++e)
          if (bn + e < N) v[e >> 1] |= static_cast<uint32_t>(row[bn + e]) << (16u * (e & 1u));
        return v;
      }
    }
    return load16_any(row);
  };
  u32x4 ra[D][CA], rb[D][CB];
  auto load = [&](int d, uint32_t k0) {
#pragma unroll
    for (int i = 0; i < CA; ++i) ra[d][i] = load_k(pa[i], k0);
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      if constexpr (B_NK) rb[d][i] = load_k(pb[i], k0);
      else rb[d][i] = load_n(k0 + bk0 + i * (THREADS / (BN / 8u)));
    }
  };
  const bool edge_n = !B_NK && n0 + BN > N && !(TINY && N < 8u);
  auto write = [&](auto last, int d, uint32_t buf, uint32_t k0) {
    constexpr bool kLast = decltype(last)::value;  // may be the last, short slice
    uint16_t* As = glds + buf * BUF;
    uint16_t* Bs = As + ASL;
    if (kLast && k0 + 64u > K && !(TINY && K < 8u)) {
      const uint32_t k = k0 + kch, n = k - (k < K - 8u ? k : K - 8u);
#pragma unroll
      for (int i = 0; i < CA; ++i) ra[d][i] = shift_down16(ra[d][i], n);
      if constexpr (B_NK) {
#pragma unroll
        for (int i = 0; i < CB; ++i) rb[d][i] = shift_down16(rb[d][i], n);
      }
    }
    if constexpr (!B_NK) {
      if (edge_n) {
#pragma unroll
        for (int i = 0; i < CB; ++i) rb[d][i] = shift_down16(rb[d][i], bsh);
      }
      if (kLast && k0 + 64u > K) {
#pragma unroll
        for (int i = 0; i < CB; ++i)
          if (k0 + bk0 + i * (THREADS / (BN / 8u)) >= K) rb[d][i] = u32x4{0u, 0u, 0u, 0u};
      }
    }
#pragma unroll
    for (int i = 0; i < CA; ++i)
      *reinterpret_cast<u32x4*>(&As[swz_rows64(row0 + i * (THREADS / 8u), tid & 7u)]) = ra[d][i];
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      if constexpr (B_NK)
        *reinterpret_cast<u32x4*>(&Bs[swz_rows64(row0 + i * (THREADS / 8u), tid & 7u)]) = rb[d][i];
      else
        *reinterpret_cast<u32x4*>(&Bs[swz_kn<BN>(bk0 + i * (THREADS / (BN / 8u)), (tid % (BN / 8u)) * 8u)]) = rb[d][i];
    }
  };
  f32x4 acc[IM][JN];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j) acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
  f32x4 sum[PAIRS ? IM : 1][PAIRS ? JN : 1];
  if constexpr (PAIRS) {
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j) sum[i][j] = acc[i][j];
  }
  auto flush = [&]() {
    if constexpr (PAIRS) {
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j) {
          sum[i][j] += acc[i][j];
          acc[i][j] = f32x4{0.0f, 0.0f, 0.0f, 0.0f};
        }
    }
  };
  auto compute = [&](auto last, uint32_t buf) {
    const uint16_t* As = glds + buf * BUF;
    const uint16_t* Bs = As + ASL;
    f32x4 pair[PAIRS ? IM : 1][PAIRS ? JN : 1];
#pragma unroll
    for (uint32_t h = 0; h < 2u; ++h) {
      bf16x8 fa[IM], fb[JN];
#pragma unroll
      for (int i = 0; i < IM; ++i)
        fa[i] = *reinterpret_cast<const bf16x8*>(&As[swz_rows64(wm + i * 16u + (lane & 15u), 4u * h + (lane >> 4))]);
#pragma unroll
      for (int j = 0; j < JN; ++j) {
        if constexpr (B_NK)
          fb[j] = *reinterpret_cast<const bf16x8*>(&Bs[swz_rows64(wn + j * 16u + (lane & 15u), 4u * h + (lane >> 4))]);
        else
          fb[j] = frag_b16_tr<BN>(Bs, wn + j * 16u, lane, 32u * h);
      }
      // Operand-swapped: the MFMA computes the C^T block, so a lane holds
      // four consecutive columns of one row of C.
#pragma unroll
      for (int j = 0; j < JN; ++j)
#pragma unroll
        for (int i = 0; i < IM; ++i) {
          if constexpr (PAIRS) {
            // The long loop: the second product adds to the first.
            constexpr bool kChain = !decltype(last)::value;
            const f32x4 from = kChain && h == 1u ? pair[i][j] : f32x4{0.0f, 0.0f, 0.0f, 0.0f};
            const f32x4 v = mfma_16x16x32_16b<F16>(fb[j], fa[i], from);
            if (h == 0u) pair[i][j] = v;
            else acc[i][j] += kChain ? v : pair[i][j] + v;
          } else {
            acc[i][j] = mfma_16x16x32_16b<F16>(fb[j], fa[i], acc[i][j]);
          }
        }
      if (PAIRS && h == 0u) __builtin_amdgcn_sched_barrier(0);
    }
  };
  // Turn t of a group (slice t * KG + grp) is written into LDS while turn t-1
  // is computed and loaded D turns earlier. The main loop's loads are
  // unconditional: with a load that may not have been issued the compiler
  // must wait for the younger ones too. (A slice past K re-reads the rows'
  // last chunk and is written as zeros.)
  using Body = std::false_type;
  using Last = std::true_type;
  const uint32_t ns = K / 64u + (K % 64u != 0u ? 1u : 0u), nt = ns / KG + (ns % KG != 0u ? 1u : 0u);
  constexpr int U = D == 1 ? 2 : D;  // turns per loop iteration: buffer and register set static
  auto k_of = [&](uint32_t t) { return (t * KG + grp) * 64u; };
  if (nt > 0u) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, k_of(d));
    write(Last{}, 0, 0u, k_of(0));
    load(0, k_of(D));
    __syncthreads();
  }
  uint32_t t0 = 0;
  for (; t0 + U + D < nt; t0 += U) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      write(Body{}, (i + 1) % D, (i + 1) & 1, k_of(t0 + i + 1u));
      load((i + 1) % D, k_of(t0 + i + 1u + D));
      compute(Body{}, i & 1);
      if (PAIRS && (t0 + i) % 8u == 7u) flush();
      __syncthreads();
    }
  }
  for (; t0 < nt; t0 += U) {
#pragma unroll
    for (int i = 0; i < U; ++i) {
      const uint32_t t = t0 + i;
      if (t < nt) {
        if (t + 1u < nt) write(Last{}, (i + 1) % D, (i + 1) & 1, k_of(t + 1u));
        if (t + 1u + D < nt) load((i + 1) % D, k_of(t + 1u + D));
        compute(Last{}, i & 1);
        if (PAIRS && t % 8u == 7u) flush();
        __syncthreads();
      }
    }
  }
  if constexpr (PAIRS) {
    flush();
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j) acc[i][j] = sum[i][j];
  }
  // Block (i, j) is finished by group (i * JN + j) / (IM * JN / KG): the
  // others hand it their sums through LDS (16 bytes per lane and block).
  constexpr int OWN = IM * JN / static_cast<int>(KG);
  if constexpr (KG > 1u) {
    static_assert(IM * JN % KG == 0u && KG * IM * JN * THREADS * 16u <= KG * 2u * BUF * 2u, "the sums fit the slices' LDS");
    f32x4* red = reinterpret_cast<f32x4*>(lds);
#pragma unroll
    for (int b = 0; b < IM * JN; ++b)
      if (static_cast<uint32_t>(b / OWN) != grp) red[(grp * (IM * JN) + b) * THREADS + tid] = acc[b / JN][b % JN];
    __syncthreads();
#pragma unroll
    for (int b = 0; b < IM * JN; ++b) {
      if (static_cast<uint32_t>(b / OWN) == grp) {
        f32x4 v = acc[b / JN][b % JN];
#pragma unroll
        for (uint32_t g = 0; g < KG; ++g)
          if (g != grp) v += red[(g * (IM * JN) + b) * THREADS + tid];
        acc[b / JN][b % JN] = v;
      }
    }
  }
  // acc[i][j][e] = C[m][n], m = m0 + wm + 16i + lane%16, n = n0 + wn + 16j + 4(lane/16) + e.
  const uint32_t last = lane_here();  // not kept through the loop
  const uint32_t mr = m0 + wm + (last & 15u), nc = n0 + wn + 4u * (last >> 4);
#pragma unroll
  for (int b = 0; b < IM * JN; ++b) {
    const int i = b / JN, j = b % JN;
    if (static_cast<uint32_t>(b / OWN) != grp) continue;
    const uint32_t m = mr + 16u * i, n = nc + 16u * j;
    if (m >= M) continue;
    float* c = C + static_cast<uint64_t>(m) * N + n;
    if (n + 4u <= N) {
      f32x4_a4 v;
#pragma unroll
      for (int e = 0; e < 4; ++e) v[e] = epi(acc[i][j][e], m, n + e);
      *reinterpret_cast<f32x4_a4*>(c) = v;
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e)
        if (n + e < N) c[e] = epi(acc[i][j][e], m, n + e);
    }
  }
}

// The contraction's tiles that gemm_bf16_4w and gemm_bf16_256_w8 do not
// take, 8 waves per workgroup: 128x128 of C, or, when 128x128 tiles would
// leave half the CUs without one (`parts` >= 2 workgroups were launched per
// tile) or M <= 64, 64x128 (1024 x 2048 x 4096: 31 us against 42, 1001 x 1501
// x 1003: 12 against 16; from 256 tiles on the taller tile reads less:
// 2048 x 2048 x 4096 44 us against 53).
template <bool B_NK, typename Epi, bool F16, uint64_t WHOLE_MIN>
__device__ __forceinline__ void gemm16_any(const __bf16* __restrict__ A, const __bf16* __restrict__ B,
                                           float* __restrict__ C, uint32_t M, uint32_t N, uint32_t K, Epi epi,
                                           uint32_t batch, uint32_t tile, uint32_t part, uint32_t parts) {
  __shared__ __attribute__((aligned(16))) uint16_t lds[2 * 64 * 256];
  const uint32_t tiles_m = (M - 1u) / 128u + 1u, tiles_n = (N - 1u) / 128u + 1u;
  uint32_t tm, tn;
  gemm_tile_coords(tiles_m, tiles_n, &tm, &tn, tile);
  const uint32_t m0 = tm * 128u + part * 64u, n0 = tn * 128u;
  if (part >= 2u || m0 >= M) return;
  if (tm / 2u < M / 256u && tn / 2u < N / 256u && gemm16_direct_k(N, K) && gemm16_on_whole_tiles<WHOLE_MIN>(M, N, batch))
    return;
  const uint16_t* A16 = reinterpret_cast<const uint16_t*>(A);
  const uint16_t* B16 = reinterpret_cast<const uint16_t*>(B);
  if (K < 8u || (!B_NK && N < 8u)) {
    if (part == 0u) gemm16_tile<128, 128, 2, 4, 1, 1, B_NK, F16, true>(A16, B16, C, M, N, K, epi, m0, n0, lds, threadIdx.x);
  } else if (parts >= 2u || M <= 64u) {
    gemm16_tile<64, 128, 2, 4, 1, 2, B_NK, F16, false>(A16, B16, C, M, N, K, epi, m0, n0, lds, threadIdx.x);
  } else {
    gemm16_tile<128, 128, 2, 4, 1, 2, B_NK, F16, false>(A16, B16, C, M, N, K, epi, m0, n0, lds, threadIdx.x);
  }
}

// -------------------------------------------- bf16 path, 8 waves per tile
// Whole tiles (gemm16_whole_coords), loaded straight into LDS: 512 threads, 2 waves per
// SIMD, each wave 128x64 of C as 8x4 blocks of v_mfma_f32_16x16x32_bf16
// (32 accumulators of 4, 225 VGPRs, no scratch).
//
// Why 16x16x32: the part is power-limited under dense MFMA load. On random
// bf16 operands an MFMA-only loop sustains 1.78 PFLOP/s with 32x32x16 (the
// clock drops to 1.81 GHz) and 2.04 PFLOP/s with 16x16x32 (2.05 GHz): half
// the accumulator traffic per flop. The operand bytes per flop, and so the
// LDS traffic, are the same for both shapes.
//
// K advances in 32-deep slices through a 4-slice ring of A [256][32] and
// [K][N] B [32][256] (or [N][K] B [256][32]) tiles, 32 KiB per slice,
// filled by global_load_lds_dwordx4 (lane i of a load writes bytes
// [16i, 16i + 16) of a 1 KiB LDS chunk, from any global address, so each
// lane's global address is the inverse of the LDS swizzle). Each slice is
// two halves of 16 MFMAs per wave:
//   half 0: A rows 0-63 of the wave x B; reads A rows 64-127 of the slice;
//   barrier (slice s+1 has landed, every wave is done with slice s-1);
//   half 1: A rows 64-127 x B; reads A rows 0-63 and B of slice s+1 into the
//           other B register set, and issues slice s+3 into slice s-1's
//           buffer, one load per quarter of the half (issued in a burst,
//           the 8 waves' loads stall their MFMA issue).
// Two slices per loop iteration, so the two B register sets alternate
// without copies; the last three slices, which load nothing, are a tail.
//
// LDS banks (measured with SQ_LDS_BANK_CONFLICT on gfx950): a 128-bit read
// is served per half-wave, in two 16-lane cycles split by the parity of
// lane bits 2^3^4; a 64-bit transposing read serves a half-wave per cycle.
// The swizzles below keep every cycle on 16 distinct 16-byte bank slots:
//   [rows][32] (64-byte rows): column group cg of row r at cg ^ 2*((r/8)%2);
//     a fragment read takes 16 rows x 4 groups (lane l: row l%16, group l/16);
//   [K][N] B (512-byte rows): 16-byte slot n/8 of row k at
//     (n/8) ^ 2*((k%4) + 4*((k/8)%2)); a transposing fragment read takes rows
//     8g..8g+3 (+4) of one 16-column block for lane group g.

// Every other tile returns at once: gemm16_any takes them.
// With K % 64 == 0 and K >= 256 the launch takes gemm_bf16_4w instead (4
// waves of 128x128, A in 64-deep slices, below).
template <bool B_NK, typename Epi, bool F16, uint64_t WHOLE_MIN, uint32_t STAGES = 4>
__device__ __forceinline__ void gemm_bf16_256_w8(const __bf16* __restrict__ A, const __bf16* __restrict__ B,
                                                 float* __restrict__ C, uint32_t M, uint32_t N, uint32_t K, Epi epi,
                                                 uint32_t batch, uint32_t tile) {
  static_assert(STAGES == 4 || STAGES == 5, "a ring of 4 or 5 slices (160 KiB of LDS at most)");
  typedef float f32x4 __attribute__((ext_vector_type(4)));
  constexpr uint32_t BM = 256, BN = 256, BK = 32, SLICE = 256u * BK;
  __shared__ __attribute__((aligned(16))) uint16_t lds[STAGES * 2 * SLICE];
  uint32_t tm, tn;
  if (!gemm16_direct_k(N, K) || !gemm16_on_whole_tiles<WHOLE_MIN>(M, N, batch) ||
      !gemm16_whole_coords(M, N, tile, &tm, &tn))
    return;  // gemm16_any takes it
  const uint32_t m0 = tm * BM, n0 = tn * BN;
  // The wave index is uniform over the wave: computed in a scalar register,
  // the LDS destination of every direct-to-LDS load (the m0 operand) is a
  // scalar value, with no readfirstlane per load.
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wm = (wave >> 2) * 128u, wn = (wave & 3u) * 64u;
  const uint16_t* __restrict__ A16 = reinterpret_cast<const uint16_t*>(A);
  const uint16_t* __restrict__ B16 = reinterpret_cast<const uint16_t*>(B);
  f32x4 acc[8][4];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0f;
  // Per-lane element offsets of the 2 chunks (of 16) this wave fills per
  // slice and operand: chunk ch = 2*wave + q covers LDS slots 64ch .. +63.
  uint32_t offa[2], offb[2];
#pragma unroll
  for (int q = 0; q < 2; ++q) {
    const uint32_t slot = (wave * 2u + q) * 64u + lane;
    const uint32_t r = slot >> 2, c = (slot & 3u) ^ (((r >> 3) & 1u) << 1);  // inverse of swz_rows32
    offa[q] = r * K + c * 8u;
    if constexpr (B_NK) {
      offb[q] = r * K + c * 8u;
    } else {
      const uint32_t k = slot >> 5, sp = slot & 31u;  // [32][256]: 32 slots per row
      offb[q] = k * N + ((sp ^ kn_slot_xor<256>(k)) << 3);
    }
  }
  uint16_t* ldsp = lds;
  auto a_slice = [&](uint32_t s) { return ldsp + s * 2u * SLICE; };
  auto b_slice = [&](uint32_t s) { return ldsp + s * 2u * SLICE + SLICE; };
  auto load = [&](int q, uint32_t s, uint32_t k0) {  // q even: A chunk q/2, q odd: B chunk q/2
    const uint32_t ch = wave * 2u + (q >> 1);
    if (q & 1) {
      const uint16_t* b0 = B_NK ? B16 + static_cast<uint64_t>(n0) * K + k0 : B16 + static_cast<uint64_t>(k0) * N + n0;
      __builtin_amdgcn_global_load_lds(b0 + offb[q >> 1], (lds_void*)(b_slice(s) + ch * 512u), 16, 0, 0);
    } else {
      const uint16_t* a0 = A16 + static_cast<uint64_t>(m0) * K + k0;
      __builtin_amdgcn_global_load_lds(a0 + offa[q >> 1], (lds_void*)(a_slice(s) + ch * 512u), 16, 0, 0);
    }
  };
  auto rd_a = [&](const uint16_t* As, uint32_t i) {  // A rows wm + 16i .. +16, all 32 k
    return *reinterpret_cast<const bf16x8*>(&As[swz_rows32(wm + i * 16u + (lane & 15u), lane >> 4)]);
  };
  auto rd_b = [&](const uint16_t* Bs, uint32_t j) {  // B columns wn + 16j .. +16, all 32 k
    if constexpr (B_NK)
      return *reinterpret_cast<const bf16x8*>(&Bs[swz_rows32(wn + j * 16u + (lane & 15u), lane >> 4)]);
    else
      return frag_b16_tr<256>(Bs, wn + j * 16u, lane);
  };
  bf16x8 fa[4], fh[4], fb0[4], fb1[4];  // A rows 0-63, A rows 64-127, the two B sets
  auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
  // The MFMA takes the B fragment as its first operand: it computes the C^T
  // block, so each lane ends up holding four consecutive columns of one row
  // of C (a 16-byte store). Each group below is fenced with sched_barrier:
  // left to itself the scheduler sinks the fragment reads behind the MFMAs.
  // MFMA number c of a half (0..15) takes block (i, j) in snake order,
  // j = c/4 and i = c%4 or 3 - c%4 for odd j, so consecutive MFMAs share an
  // operand register (measured: about 3% faster at 4096^3 than j-major,
  // the part being power-limited).
  auto blk_i = [](int c) { return ((c >> 2) & 1) ? 3 - (c & 3) : (c & 3); };
  auto half0 = [&](auto set, uint32_t s) {
    bf16x8* gb = decltype(set)::value == 0 ? fb0 : fb1;
    const uint16_t* As = a_slice(s);
    auto mf = [&](int c) {
      const int i = blk_i(c), j = c >> 2;
      acc[i][j] = mfma_16x16x32_16b<F16>(gb[j], fa[i], acc[i][j]);
      fence();
    };
    fence();
    mf(0);
    fh[0] = rd_a(As, 4); fh[1] = rd_a(As, 5); fence();
    mf(1);
    fh[2] = rd_a(As, 6); fh[3] = rd_a(As, 7); fence();
#pragma unroll
    for (int c = 2; c < 16; ++c) mf(c);
  };
  auto half1 = [&](auto set, uint32_t ns, bool dma, uint32_t ds, uint32_t dk) {
    bf16x8* gb = decltype(set)::value == 0 ? fb0 : fb1;
    bf16x8* nb = decltype(set)::value == 0 ? fb1 : fb0;
    const uint16_t* As = a_slice(ns);
    const uint16_t* Bs = b_slice(ns);
    auto mf = [&](int c) {
      const int i = blk_i(c), j = c >> 2;
      acc[4 + i][j] = mfma_16x16x32_16b<F16>(gb[j], fh[i], acc[4 + i][j]);
      fence();
    };
    auto dm = [&](int q) {
      if (dma) load(q, ds, dk);
      fence();
    };
    fence();
    mf(0);
    fa[0] = rd_a(As, 0); fa[1] = rd_a(As, 1); fence();
    mf(1);
    fa[2] = rd_a(As, 2); fa[3] = rd_a(As, 3); fence();
    mf(2);
    nb[0] = rd_b(Bs, 0); fence();
    mf(3);
    nb[1] = rd_b(Bs, 1); fence();
    mf(4);
    nb[2] = rd_b(Bs, 2); fence();
    mf(5);
    nb[3] = rd_b(Bs, 3); fence();
    mf(6); dm(0);
    mf(7);
    mf(8); dm(1);
    mf(9);
    mf(10); dm(2);
    mf(11);
    mf(12); dm(3);
    mf(13); mf(14); mf(15);
  };
  // The barrier waits only for the slice about to be read (vmcnt counts in
  // issue order, 4 loads per slice and lane); its lgkmcnt leaves half 0's 4
  // fragment reads in flight but guarantees that every earlier read, the
  // last ones of the buffer the next loads overwrite, has completed: LDS
  // reads complete in order.
  constexpr int kReads = 4;
  auto wait_slices = [](uint32_t d, bool keep_reads) {  // at most d slices of loads still in flight
    if (keep_reads) {
      if (d >= 3u) __builtin_amdgcn_s_waitcnt(waitcnt_imm(12, kReads));
      else if (d == 2u) __builtin_amdgcn_s_waitcnt(waitcnt_imm(8, kReads));
      else if (d == 1u) __builtin_amdgcn_s_waitcnt(waitcnt_imm(4, kReads));
      else __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, kReads));
    } else {
      if (d >= 3u) __builtin_amdgcn_s_waitcnt(waitcnt_imm(12, 0));
      else if (d == 2u) __builtin_amdgcn_s_waitcnt(waitcnt_imm(8, 0));
      else if (d == 1u) __builtin_amdgcn_s_waitcnt(waitcnt_imm(4, 0));
      else __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
    }
  };
  auto barrier = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  const uint32_t nk = K / BK;
  const uint32_t pre = nk < STAGES - 1 ? nk : STAGES - 1;
  for (uint32_t s = 0; s < pre; ++s)
    for (int q = 0; q < 4; ++q) load(q, s, s * BK);
  asm volatile("" ::: "memory");
  wait_slices(pre - 1u, false);  // slice 0 landed
  barrier();
  // Main slices kt < nk - (STAGES - 1) load slice kt + STAGES - 1: at the
  // barrier of slice kt, slices up to kt + STAGES - 2 were issued and kt+1
  // must have landed (STAGES - 3 newer slices may remain in flight).
  const uint32_t main_end = nk > STAGES - 1 ? nk - (STAGES - 1) : 0u;
  auto main_slice = [&](auto set, uint32_t kt) {
    half0(set, kt % STAGES);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_waitcnt(waitcnt_imm(4 * static_cast<int>(STAGES - 3), kReads));
    barrier();
    half1(set, (kt + 1) % STAGES, true, (kt + STAGES - 1) % STAGES, (kt + STAGES - 1) * BK);
  };
  auto tail_slice = [&](auto set, uint32_t kt) {
    half0(set, kt % STAGES);
    if (kt + 1 < nk) {
      asm volatile("" ::: "memory");
      wait_slices(nk - 2u - kt, true);
      barrier();
    }
    half1(set, (kt + 1) % STAGES, false, 0, 0);  // the last one reads a stale buffer whose values are unused
  };
  // Slice 0's B fragments go into the set that makes the paired loop start on set 0.
  const bool odd = (main_end & 1u) != 0u;
  {
    const uint16_t* As = a_slice(0);
    const uint16_t* Bs = b_slice(0);
#pragma unroll
    for (int i = 0; i < 4; ++i) fa[i] = rd_a(As, i);
    if (odd) {
#pragma unroll
      for (int j = 0; j < 4; ++j) fb1[j] = rd_b(Bs, j);
    } else {
#pragma unroll
      for (int j = 0; j < 4; ++j) fb0[j] = rd_b(Bs, j);
    }
  }
  uint32_t kt = 0;
  if (odd) {
    main_slice(Set1{}, 0);
    kt = 1;
  }
  for (; kt < main_end; kt += 2) {
    main_slice(Set0{}, kt);
    main_slice(Set1{}, kt + 1);
  }
  if (main_end < nk) tail_slice(Set0{}, main_end);
  if (main_end + 1 < nk) tail_slice(Set1{}, main_end + 1);
  if (main_end + 2 < nk) tail_slice(Set0{}, main_end + 2);
  if (STAGES > 4 && main_end + 3 < nk) tail_slice(Set1{}, main_end + 3);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));  // nothing in flight past the loop
  // acc[i][j][e] = C[m][n], m = m0 + wm + 16i + lane%16, n = n0 + wn + 16j + 4(lane/16) + e.
  const uint32_t mr = m0 + wm + (lane & 15u), nc = n0 + wn + 4u * (lane >> 4);
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const uint32_t m = mr + 16u * i, n = nc + 16u * j;
      float4 v;
      v.x = epi(acc[i][j][0], m, n + 0);
      v.y = epi(acc[i][j][1], m, n + 1);
      v.z = epi(acc[i][j][2], m, n + 2);
      v.w = epi(acc[i][j][3], m, n + 3);
      *reinterpret_cast<float4*>(C + static_cast<uint64_t>(m) * N + n) = v;
    }
}

// ------------------------------------- bf16 path, 4 waves, 128x128 per wave
// Whole 256x256 tiles with K % 64 == 0 and K >= 256 (the launch guards pick
// this kernel): 256 threads, one wave per SIMD, each wave a 128x128 sub-tile
// of C as 8x8 blocks of v_mfma_f32_16x16x32_bf16, accumulators in AGPRs
// (256 per lane), 160 VGPRs. Against 8 waves of 128x64 this reads a third
// less LDS per flop (each A and B fragment feeds 8 blocks instead of 4 or 8
// and 4), which leaves more of the power budget to the MFMAs: measured
// interleaved with the 8-wave kernel on one box, 4096^3 with rotated inputs
// 105.0-105.6 against 107.9-112.4 us, 8192^3 1356-1371 against 1335-1344
// TFLOP/s, K = 16384 +2%, results bitwise equal.
// LDS: A in 64-deep slices ([256][64], 128-byte rows, whole cache lines per
// direct-to-LDS load) in a 3-buffer ring, B in 32-deep slices in a 4-buffer
// ring, 160 KiB in all; slot s (32 deep) is k half s%2 of A slice s/2 and B
// slice s.
// Step kt: wait until slot kt+1 has landed and every read of slot kt has
// completed, one barrier, then 64 MFMAs on the fragments of slot kt (read
// during step kt-1) while this step reads all fragments of slot kt+1 into
// the other register set and loads part kt%2 of A slice kt/2+2 (into the
// buffer of A slice kt/2-1, last read during step kt-2) and B slice kt+4
// (into slot kt's buffer).
// The MFMAs are inline asm with the accumulator tied to one AGPR quad: the
// compiler's own MFMA, given 256 accumulators, splits them between AGPRs and
// VGPRs and moves them inside the loop (or spills). The hazards its
// recogniser does not see for inline asm are covered here:
//   the zero-initialised AGPRs are fixed (an empty asm per accumulator, so
//   no zero is re-materialised later) and 16 wait states separate the last
//   write from the first MFMA (VALU write -> MFMA SrcC read);
//   24 wait states separate the last MFMA from the epilogue's AGPR reads
//   (an 8-pass XDL write -> VALU/VMEM read);
//   the MFMA A/B operands are ds_read results only (a host test checks the
//   assembly: no VALU writes an MFMA source register), whose completion
//   s_waitcnt covers; an MFMA's accumulator is written again only by the
//   64th MFMA after it.
template <bool F16 = false>
__device__ __forceinline__ void mfma16_bf16_acc(f32x4_t& c, const bf16x8& b, const bf16x8& a) {
  if constexpr (F16)
    asm volatile("v_mfma_f32_16x16x32_f16 %0, %1, %2, %0" : "+a"(c) : "v"(b), "v"(a));
  else
    asm volatile("v_mfma_f32_16x16x32_bf16 %0, %1, %2, %0" : "+a"(c) : "v"(b), "v"(a));
}

template <bool B_NK, typename Epi, bool F16, uint64_t WHOLE_MIN>
__device__ __forceinline__ void gemm_bf16_4w(const __bf16* __restrict__ A, const __bf16* __restrict__ B,
                                             float* __restrict__ C, uint32_t M, uint32_t N, uint32_t K, Epi epi,
                                             uint32_t batch, uint32_t tile) {
  constexpr uint32_t BM = 256, BN = 256, ASL = 256u * 64u, BSL = 256u * 32u;
  __shared__ __attribute__((aligned(16))) uint16_t lds[3 * ASL + 4 * BSL];
  uint32_t tm, tn;
  if (!gemm16_direct_k(N, K) || K % 64u != 0u || K < 256u || !gemm16_on_whole_tiles<WHOLE_MIN>(M, N, batch) ||
      !gemm16_whole_coords(M, N, tile, &tm, &tn))
    return;  // gemm16_any takes it
  const uint32_t m0 = tm * BM, n0 = tn * BN;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wm = (wave >> 1) * 128u, wn = (wave & 1u) * 128u;
  const uint16_t* __restrict__ A16 = reinterpret_cast<const uint16_t*>(A);
  const uint16_t* __restrict__ B16 = reinterpret_cast<const uint16_t*>(B);
  f32x4_t acc[8][8];
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j)
#pragma unroll
      for (int e = 0; e < 4; ++e) acc[i][j][e] = 0.0f;
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) asm volatile("" : "+a"(acc[i][j]));
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // Per-lane element offsets of the 4 chunks this wave fills per A part
  // (16 chunks of 8 rows x 128 bytes; wave w: chunks 4w .. 4w+3) and per B
  // slice (16 chunks of 64 16-byte slots).
  uint32_t offa[4], offb[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t row = 32u * wave + 8u * q + (lane >> 3);
    offa[q] = row * K + (((lane & 7u) ^ (row & 6u)) << 3);  // inverse of swz_rows64
    const uint32_t slot = (wave * 4u + q) * 64u + lane;
    if constexpr (B_NK) {
      const uint32_t r = slot >> 2, c = (slot & 3u) ^ (((r >> 3) & 1u) << 1);  // inverse of swz_rows32
      offb[q] = r * K + c * 8u;
    } else {
      const uint32_t k = slot >> 5, sp = slot & 31u;  // [32][256]: 32 slots per row
      offb[q] = k * N + ((sp ^ kn_slot_xor<256>(k)) << 3);
    }
  }
  uint16_t* ldsp = lds;
  auto a_buf = [&](uint32_t j) { return ldsp + (j % 3u) * ASL; };
  auto b_buf = [&](uint32_t s) { return ldsp + 3u * ASL + (s & 3u) * BSL; };
  auto load_b = [&](int q, uint32_t s) {
    const uint32_t k0 = s * 32u;
    const uint16_t* b0 = B_NK ? B16 + static_cast<uint64_t>(n0) * K + k0 : B16 + static_cast<uint64_t>(k0) * N + n0;
    __builtin_amdgcn_global_load_lds(b0 + offb[q], (lds_void*)(b_buf(s) + (wave * 4u + q) * 512u), 16, 0, 0);
  };
  auto load_a = [&](int q, uint32_t j, uint32_t p) {  // part p (rows 128p .. +127) of A slice j
    const uint16_t* a0 = A16 + static_cast<uint64_t>(m0 + 128u * p) * K + j * 64u;
    __builtin_amdgcn_global_load_lds(a0 + offa[q], (lds_void*)(a_buf(j) + (16u * p + wave * 4u + q) * 512u), 16, 0, 0);
  };
  auto rd_a = [&](uint32_t s, uint32_t i) {  // slot s: A rows wm + 16i .. +16
    const uint16_t* As = a_buf(s >> 1);
    return *reinterpret_cast<const bf16x8*>(&As[swz_rows64(wm + i * 16u + (lane & 15u), 4u * (s & 1u) + (lane >> 4))]);
  };
  auto rd_b = [&](uint32_t s, uint32_t j) {  // slot s: B columns wn + 16j .. +16
    const uint16_t* Bs = b_buf(s);
    if constexpr (B_NK)
      return *reinterpret_cast<const bf16x8*>(&Bs[swz_rows32(wn + j * 16u + (lane & 15u), lane >> 4)]);
    else
      return frag_b16_tr<256>(Bs, wn + j * 16u, lane);
  };
  bf16x8 a0s[8], b0s[8], a1s[8], b1s[8];  // two fragment sets: this step's and the next one's
  auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
  auto barrier = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  // MFMA c (0..63) takes block (i, j) with j = c/8 and i snaking over 0..7,
  // so consecutive MFMAs share an operand register. The operand-swapped
  // MFMA computes the C^T block: each lane ends up holding four consecutive
  // columns of one row of C (a 16-byte store).
  // wait_vm: the loads that may remain in flight at the start of the step
  // (-1: no wait and no barrier, the last step).
  auto step = [&](auto set, uint32_t kt, int wait_vm, bool rd, bool ld) {
    bf16x8* ca = decltype(set)::value == 0 ? a0s : a1s;
    bf16x8* cb = decltype(set)::value == 0 ? b0s : b1s;
    bf16x8* na = decltype(set)::value == 0 ? a1s : a0s;
    bf16x8* nb = decltype(set)::value == 0 ? b1s : b0s;
    if (wait_vm >= 0) {
      asm volatile("" ::: "memory");
      if (wait_vm == 16) __builtin_amdgcn_s_waitcnt(waitcnt_imm(16, 0));
      else if (wait_vm == 8) __builtin_amdgcn_s_waitcnt(waitcnt_imm(8, 0));
      else __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
      barrier();
    }
    const uint32_t ns = kt + 1u;
    auto mf = [&](int c) {
      const int j = c >> 3, i = (j & 1) ? 7 - (c & 7) : (c & 7);
      mfma16_bf16_acc<F16>(acc[i][j], cb[j], ca[i]);
      fence();
    };
    auto da = [&](int q) { if (ld) load_a(q, (kt >> 1) + 2u, kt & 1u); fence(); };
    auto db = [&](int q) { if (ld) load_b(q, kt + 4u); fence(); };
    fence();
    if (rd) {
#pragma unroll
      for (int c = 0; c < 8; ++c) { mf(c); na[c] = rd_a(ns, c); fence(); }
#pragma unroll
      for (int c = 0; c < 8; ++c) { mf(8 + c); nb[c] = rd_b(ns, c); fence(); }
    } else {
#pragma unroll
      for (int c = 0; c < 16; ++c) mf(c);
    }
#pragma unroll
    for (int q = 0; q < 4; ++q) {
      mf(16 + 8 * q); mf(17 + 8 * q); mf(18 + 8 * q); mf(19 + 8 * q); da(q);
      mf(20 + 8 * q); mf(21 + 8 * q); mf(22 + 8 * q); mf(23 + 8 * q); db(q);
    }
#pragma unroll
    for (int c = 48; c < 64; ++c) mf(c);
  };
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  const uint32_t nk = K / 32u;
  // Prologue: A0 (8 loads), B0 (4), B1 (4), A1 (8), B2 (4), B3 (4); A0 and B0 landed: 20 newer may remain.
  for (int q = 0; q < 4; ++q) load_a(q, 0, 0);
  for (int q = 0; q < 4; ++q) load_a(q, 0, 1);
  for (int q = 0; q < 4; ++q) load_b(q, 0);
  for (int q = 0; q < 4; ++q) load_b(q, 1);
  for (int q = 0; q < 4; ++q) load_a(q, 1, 0);
  for (int q = 0; q < 4; ++q) load_a(q, 1, 1);
  for (int q = 0; q < 4; ++q) load_b(q, 2);
  for (int q = 0; q < 4; ++q) load_b(q, 3);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(20, 0));
  barrier();
#pragma unroll
  for (int i = 0; i < 8; ++i) a0s[i] = rd_a(0, i);
#pragma unroll
  for (int j = 0; j < 8; ++j) b0s[j] = rd_b(0, j);
  // Loads run while kt < nk - 4 (8 per step). At the start of step kt slot
  // kt+1 must have landed: for even kt the loads of step kt-3 (16 newer may
  // remain), for odd kt the A part of step kt-2 (8 newer); in the prologue's
  // place the same counts are conservative. vmcnt counts in issue order.
  const uint32_t main_end = nk - 4u;  // even: K % 64 == 0
  for (uint32_t kt = 0; kt < main_end; kt += 2) {
    step(Set0{}, kt, 16, true, true);
    step(Set1{}, kt + 1, 8, true, true);
  }
  step(Set0{}, nk - 4u, 16, true, false);
  step(Set1{}, nk - 3u, 0, true, false);  // no loads after those of step nk-5
  step(Set0{}, nk - 2u, 0, true, false);
  step(Set1{}, nk - 1u, -1, false, false);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __builtin_amdgcn_sched_barrier(0);
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // acc[i][j][e] = C[m][n], m = m0 + wm + 16i + lane%16, n = n0 + wn + 16j + 4(lane/16) + e.
  const uint32_t mr = m0 + wm + (lane & 15u), nc = n0 + wn + 4u * (lane >> 4);
#pragma unroll
  for (int i = 0; i < 8; ++i)
#pragma unroll
    for (int j = 0; j < 8; ++j) {
      const uint32_t m = mr + 16u * i, n = nc + 16u * j;
      float4 v;
      v.x = epi(acc[i][j][0], m, n + 0);
      v.y = epi(acc[i][j][1], m, n + 1);
      v.z = epi(acc[i][j][2], m, n + 2);
      v.w = epi(acc[i][j][3], m, n + 3);
      *reinterpret_cast<float4*>(C + static_cast<uint64_t>(m) * N + n) = v;
    }
}

// ------------------------------------------------------- fp32 path, any shape
__device__ __forceinline__ f32x4_t load16_any(const float* p) { return *reinterpret_cast<const f32x4_a4*>(p); }

// The four values of v moved down by n places, zeros shifted in (shift_down16
// for 32-bit elements).
__device__ __forceinline__ f32x4_t shift_down32(f32x4_t v, uint32_t n) {
  const bool a = n & 1u, b = n & 2u;
  v = f32x4_t{a ? v[1] : v[0], a ? v[2] : v[1], a ? v[3] : v[2], a ? 0.0f : v[3]};
  v = f32x4_t{b ? v[2] : v[0], b ? v[3] : v[1], b ? 0.0f : v[2], b ? 0.0f : v[3]};
  return n >= 4u ? f32x4_t{0.0f, 0.0f, 0.0f, 0.0f} : v;
}

// LDS word of element (row, 16-byte chunk c) of a [rows][32] fp32 slice: a
// fragment read (32 rows, one chunk per half-wave) covers every bank slot
// once per 16-lane cycle (the cycles measured at gemm_bf16_256_w8).
__device__ __forceinline__ uint32_t swz32_rows(uint32_t row, uint32_t c) { return row * 32u + ((c ^ ((row >> 1) & 7u)) << 2); }
// ... of element (k, n) of a [32][BN] slice: the rows k and k + 4 that the
// halves of a wave read lie 32 banks apart.
template <uint32_t BN>
__device__ __forceinline__ uint32_t swz32_kn(uint32_t k, uint32_t n) {
  if constexpr (BN >= 64u) return k * BN + (n ^ ((k & 4u) << 3));
  else return (k ^ ((k >> 2) & 1u)) * BN + n;
}

// 8-deep steps of the 32-deep slice at k0 that hold any of K: the others are
// zeros throughout, and an fp32 step costs 256 cycles a block. Stepping through
// whole slices, 1500 x 8192 x 16 took 16.6 us (now 15.0; 12.9 on 128x128 tiles of
// 16-deep slices), 3 batches of 2048 x 2048 x 100 38.4 (34.6; 34.6) and 64 of 1024 x
// 1024 x 32, where two of four groups of waves only had zeros, 326 (228).
__host__ __device__ __forceinline__ uint32_t slice_steps32(uint32_t K, uint32_t k0) {
  return k0 >= K ? 0u : K - k0 >= 32u ? 4u : (K - k0 - 1u) / 8u + 1u;
}

// One BM x BN tile of C at (m0, n0), fp32, every shape: gemm16_tile's scheme on
// v_mfma_f32_32x32x2f32. KG groups of WGM x WGN waves take every KG-th 32-deep
// slice of K, loaded unguarded into registers while the slice before is
// computed, in NBUF LDS buffers per group (2: one barrier per slice); their
// sums meet in LDS. Four 2-deep MFMA steps take k = 8h + e on lanes 0-31 and
// k = 8h + 4 + e on lanes 32-63, one 16-byte read of a K-contiguous row each.
// fp32 MFMAs take 64 cycles per 32x32 block and 2 k, so small tiles do not
// starve them (a 64x64 tile needs a quarter of the L1 and LDS rates), and
// several workgroups per CU hide each other's waits.
// FLUSH: the accumulators are added to a second set every 8 k, for an error no
// larger than that of sums split over 16 waves.
// `lds` holds KG * NBUF * 32 * (BM + BN) floats; `thread` is threadIdx.x.
template <uint32_t BM, uint32_t BN, uint32_t WGM, uint32_t WGN, uint32_t KG, uint32_t NBUF, bool B_NK, bool TINY,
          bool FLUSH = false, typename Epi>
__device__ __forceinline__ void gemm32_tile(const float* __restrict__ A, const float* __restrict__ B,
                                            float* __restrict__ C, uint32_t M, uint32_t N, uint32_t K, Epi epi,
                                            uint32_t m0, uint32_t n0, float* lds, uint32_t thread) {
  constexpr uint32_t THREADS = 64u * WGM * WGN, TM = BM / WGM, TN = BN / WGN;
  constexpr int IM = TM / 32, JN = TN / 32, CA = BM * 8 / THREADS, CB = BN * 8 / THREADS;
  static_assert(CA >= 1 && CB >= 1 && (NBUF == 1 || NBUF == 2), "whole chunks per thread");
  constexpr uint32_t ASL = BM * 32u, BUF = ASL + BN * 32u;
  const uint32_t lane = thread & 63u, wave_id = __builtin_amdgcn_readfirstlane(thread >> 6);
  const uint32_t grp = wave_id / (WGM * WGN), wave = wave_id % (WGM * WGN), tid = wave * 64u + lane;
  const uint32_t wm = (wave / WGN) * TM, wn = (wave % WGN) * TN;
  float* glds = lds + grp * (NBUF * BUF);
  const uint32_t kch = (tid & 7u) * 4u, row0 = tid >> 3;
  const uint32_t bk0 = tid / (BN / 4u), bn = n0 + (tid % (BN / 4u)) * 4u;
  const float* pa[CA];
#pragma unroll
  for (int i = 0; i < CA; ++i) {
    const uint32_t r = m0 + row0 + i * (THREADS / 8u);
    pa[i] = A + static_cast<uint64_t>(r < M ? r : M - 1u) * K;
  }
  const float* pb[B_NK ? CB : 1];
  uint32_t bsh = 0u;
  if constexpr (B_NK) {
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      const uint32_t r = n0 + row0 + i * (THREADS / 8u);
      pb[i] = B + static_cast<uint64_t>(r < N ? r : N - 1u) * K;
    }
  } else {
    const uint32_t last = N >= 4u ? N - 4u : 0u, at = bn < last ? bn : last;
    bsh = bn - at;
    pb[0] = B + at;
  }
  auto load_k = [&](const float* row, uint32_t k0) -> f32x4_t {
    const uint32_t k = k0 + kch;
    if constexpr (TINY) {
      if (K < 4u) {
        f32x4_t v = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t e = 0; e < 4u; ++e)
          if (k + e < K) v[e] = row[k + e];
        return v;
      }
    }
    return load16_any(row + (k < K - 4u ? k : K - 4u));
  };
  auto load_n = [&](uint32_t k) -> f32x4_t {
    const float* row = pb[0] + static_cast<uint64_t>(k < K ? k : K - 1u) * N;
    if constexpr (TINY) {
      if (N < 4u) {
        f32x4_t v = {0.0f, 0.0f, 0.0f, 0.0f};
        for (uint32_t e = 0; e < 4u; ++e)
          if (bn + e < N) v[e] = row[bn + e];
        return v;
      }
    }
    return load16_any(row);
  };
  f32x4_t ra[CA], rb[CB];
  auto load = [&](uint32_t k0) {
#pragma unroll
    for (int i = 0; i < CA; ++i) ra[i] = load_k(pa[i], k0);
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      if constexpr (B_NK) rb[i] = load_k(pb[i], k0);
      else rb[i] = load_n(k0 + bk0 + i * (THREADS / (BN / 4u)));
    }
  };
  const bool edge_n = !B_NK && n0 + BN > N && !(TINY && N < 4u);
  auto write = [&](uint32_t buf, uint32_t k0) {
    float* As = glds + buf * BUF;
    float* Bs = As + ASL;
    if (k0 + 32u > K && !(TINY && K < 4u)) {  // the last, short slice
      const uint32_t k = k0 + kch, n = k - (k < K - 4u ? k : K - 4u);
#pragma unroll
      for (int i = 0; i < CA; ++i) ra[i] = shift_down32(ra[i], n);
      if constexpr (B_NK) {
#pragma unroll
        for (int i = 0; i < CB; ++i) rb[i] = shift_down32(rb[i], n);
      }
    }
    if constexpr (!B_NK) {
      if (edge_n) {
#pragma unroll
        for (int i = 0; i < CB; ++i) rb[i] = shift_down32(rb[i], bsh);
      }
      if (k0 + 32u > K) {
#pragma unroll
        for (int i = 0; i < CB; ++i)
          if (k0 + bk0 + i * (THREADS / (BN / 4u)) >= K) rb[i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
#pragma unroll
    for (int i = 0; i < CA; ++i)
      *reinterpret_cast<f32x4_t*>(&As[swz32_rows(row0 + i * (THREADS / 8u), tid & 7u)]) = ra[i];
#pragma unroll
    for (int i = 0; i < CB; ++i) {
      if constexpr (B_NK)
        *reinterpret_cast<f32x4_t*>(&Bs[swz32_rows(row0 + i * (THREADS / 8u), tid & 7u)]) = rb[i];
      else
        *reinterpret_cast<f32x4_t*>(&Bs[swz32_kn<BN>(bk0 + i * (THREADS / (BN / 4u)), (tid % (BN / 4u)) * 4u)]) = rb[i];
    }
  };
  f32x16 acc[IM][JN];
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < JN; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
  f32x16 sum[FLUSH ? IM : 1][FLUSH ? JN : 1];
  if constexpr (FLUSH) {
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j) sum[i][j] = acc[i][j];
  }
  auto flush = [&]() {
    if constexpr (FLUSH) {
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
#pragma unroll
          for (int e = 0; e < 16; ++e) {
            sum[i][j][e] += acc[i][j][e];
            acc[i][j][e] = 0.0f;
          }
    }
  };
  auto step = [&](const float* As, const float* Bs, uint32_t h, uint32_t lane) {
    const uint32_t l32 = lane & 31u, hf = lane >> 5;
    f32x4_t fa[IM], fb[JN];
#pragma unroll
    for (int i = 0; i < IM; ++i) fa[i] = *reinterpret_cast<const f32x4_t*>(&As[swz32_rows(wm + 32u * i + l32, 2u * h + hf)]);
#pragma unroll
    for (int j = 0; j < JN; ++j) {
      const uint32_t n = wn + 32u * j + l32;
      if constexpr (B_NK) {
        fb[j] = *reinterpret_cast<const f32x4_t*>(&Bs[swz32_rows(n, 2u * h + hf)]);
      } else {
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) fb[j][e] = Bs[swz32_kn<BN>(8u * h + 4u * hf + e, n)];
      }
    }
#pragma unroll
    for (int e = 0; e < 4; ++e)
#pragma unroll
      for (int i = 0; i < IM; ++i)
#pragma unroll
        for (int j = 0; j < JN; ++j)
          acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[i][e], fb[j][e], acc[i][j], 0, 0, 0);
    flush();
  };
  auto compute = [&](uint32_t buf) {
    const float* As = glds + buf * BUF;
    const float* Bs = As + ASL;
#pragma unroll
    for (uint32_t h = 0; h < 4u; ++h) step(As, Bs, h, lane);
  };
  // Turn t of a group is slice t * KG + grp; a slice past K re-reads the rows'
  // last chunk and is written as zeros.
  const uint32_t ns = K / 32u + (K % 32u != 0u ? 1u : 0u), nt = ns / KG + (ns % KG != 0u ? 1u : 0u);
  auto k_of = [&](uint32_t t) { return (t * KG + grp) * 32u; };
  if (nt > 0u) {
    load(k_of(0));
    write(0u, k_of(0));
    __syncthreads();
  }
  // Turns of whole slices in every group, then a short one, stepped through as
  // far as it goes (in the loop itself the test costs 3-8% everywhere).
  const uint32_t whole = K / 32u / KG;
  for (uint32_t t = 0; t < whole; ++t) {
    const bool more = t + 1u < nt;
    if (more) load(k_of(t + 1u));
    compute(NBUF == 2u ? t & 1u : 0u);
    if constexpr (NBUF == 1u) __syncthreads();
    if (more) write(NBUF == 2u ? (t + 1u) & 1u : 0u, k_of(t + 1u));
    __syncthreads();
  }
  if (whole < nt) {
    const float* As = glds + (NBUF == 2u ? (whole & 1u) * BUF : 0u);
    const uint32_t steps = slice_steps32(K, k_of(whole));
#pragma unroll 1
    for (uint32_t h = 0; h < steps; ++h) step(As, As + ASL, h, lane_here());
    __syncthreads();
  }
  if constexpr (FLUSH) {
#pragma unroll
    for (int i = 0; i < IM; ++i)
#pragma unroll
      for (int j = 0; j < JN; ++j) acc[i][j] = sum[i][j];
  }
  const uint32_t l32 = lane & 31u, hf = lane >> 5;
  // Four rows of a block (accumulator elements 4q .. 4q+3) are finished by
  // group (block * 4 + q) / (4 IM JN / KG): the others hand it their sums.
  constexpr int QUADS = IM * JN * 4, OWN = QUADS / static_cast<int>(KG);
  if constexpr (KG > 1u) {
    static_assert(QUADS % KG == 0u && KG * QUADS * THREADS * 4u <= KG * NBUF * BUF, "the sums fit the slices' LDS");
    f32x4_t* red = reinterpret_cast<f32x4_t*>(lds);
#pragma unroll
    for (int q = 0; q < QUADS; ++q) {
      const f32x16& c = acc[q / 4 / JN][q / 4 % JN];
      if (static_cast<uint32_t>(q / OWN) != grp)
        red[(grp * QUADS + q) * THREADS + tid] = f32x4_t{c[4 * (q % 4)], c[4 * (q % 4) + 1], c[4 * (q % 4) + 2], c[4 * (q % 4) + 3]};
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < QUADS; ++q) {
      if (static_cast<uint32_t>(q / OWN) == grp) {
        f32x16& c = acc[q / 4 / JN][q / 4 % JN];
#pragma unroll
        for (uint32_t g = 0; g < KG; ++g) {
          if (g == grp) continue;
          const f32x4_t v = red[(g * QUADS + q) * THREADS + tid];
#pragma unroll
          for (int e = 0; e < 4; ++e) c[4 * (q % 4) + e] += v[e];
        }
      }
    }
  }
  // acc[i][j][e] = C[r][c], r = m0 + wm + 32i + 8(e/4) + 4(lane/32) + e%4, c = n0 + wn + 32j + lane%32.
#pragma unroll
  for (int q = 0; q < QUADS; ++q) {
    if (static_cast<uint32_t>(q / OWN) != grp) continue;
    const int i = q / 4 / JN, j = q / 4 % JN;
#pragma unroll
    for (int e = 0; e < 4; ++e) {
      const uint32_t r = m0 + wm + 32u * i + 8u * (q % 4) + 4u * hf + e, c = n0 + wn + 32u * j + l32;
      if (r < M && c < N) C[static_cast<uint64_t>(r) * N + c] = epi(acc[i][j][4 * (q % 4) + e], r, c);
    }
  }
}

// Planes that gemm_f32_4w does not take: 64x64 of C per 256-thread workgroup,
// or 64x32 where 64x64 tiles would be fewer than three per CU (`parts` >= 2
// workgroups were launched per tile): the CUs' shares then differ less. The
// kernel before (128x128 tiles, element-wise guards on edges) took 147 us for
// 1000 x 1500 x 1001 (34 now), 317 for 1024 x 2048 x 4096 (158), 1052 for 4100
// x 4096 x 2048 on 256x256 tiles (610). MFMA-bound: 110-120 of the 150 TFLOP/s
// an MFMA loop reaches. 32 KiB of LDS keep five workgroups on a CU; with 48
// (two buffers for the halves) three, and 2048 x 2048 x 4096 took 308 us
// instead of 293. Sums are one chain over K (two, where 64x32 tiles deal the
// slices to two groups): 1000 x 1500 x 1001, in two, 4.0e-7 from 64 bits, 2000 x
// 3000 x 1001, in one, 5.7e-7, as the kernel before had at both.
template <bool B_NK, typename Epi>
__device__ __forceinline__ void gemm_f32_any(const float* __restrict__ A, const float* __restrict__ B,
                                             float* __restrict__ C, uint32_t M, uint32_t N, uint32_t K, Epi epi,
                                             uint32_t tile, uint32_t part, uint32_t parts) {
  __shared__ __attribute__((aligned(16))) float lds[2 * 32 * 128];
  const uint32_t tiles_m = (M - 1u) / 64u + 1u, tiles_n = (N - 1u) / 64u + 1u;
  uint32_t tm, tn;
  gemm_tile_coords(tiles_m, tiles_n, &tm, &tn, tile);
  const uint32_t m0 = tm * 64u, n0 = tn * 64u + part * 32u;
  if (part >= 2u || n0 >= N) return;
  if (K < 4u || (!B_NK && N < 4u)) {
    if (part == 0u) gemm32_tile<64, 64, 2, 2, 1, 2, B_NK, true>(A, B, C, M, N, K, epi, m0, n0, lds, threadIdx.x);
  } else if (parts >= 2u) {
    gemm32_tile<64, 32, 2, 1, 2, 1, B_NK, false>(A, B, C, M, N, K, epi, m0, n0, lds, threadIdx.x);
  } else {
    gemm32_tile<64, 64, 2, 2, 1, 2, B_NK, false>(A, B, C, M, N, K, epi, m0, n0, lds, threadIdx.x);
  }
}

// ------------------------------------- fp32 path, 4 waves, 128x128 per wave
// Whole 256x256 tiles with K % 32 == 0 and K >= 128 (the launch guards pick
// this kernel from M, N >= 4096 on): 256 threads, one wave per SIMD, each
// wave a 128x128 sub-tile of C as 4x4 blocks of v_mfma_f32_32x32x2f32,
// accumulators in AGPRs (256 per lane) through inline-asm MFMAs (the same
// scheme and hazard coverage as gemm_bf16_4w), about 150 VGPRs.
// LDS: a ring of 4 slots of 16-deep slices loaded straight from global
// memory (global_load_lds_dwordx4): A (and an [n][k] B) as [256][16] with
// the 16-byte chunk c of row r at c ^ ((r / 4) % 4), a [k][n] B as [16][264]
// (rows padded to 1056 bytes: the fragment read of rows k and k + 4 covers
// the 64 banks once). 133 KiB in all.
// Slice s: wait until slot s+1 has landed and every read of slot s has
// completed, one barrier, then 128 MFMAs on the fragments of slot s (read
// during slice s-1) while this slice reads all fragments of slot s+1 and
// loads slice s+4 into slot s's buffer.
// The 2-deep MFMA step (h, e) of a slice (h 0..1, e 0..3) takes k = 8h + e on
// lanes 0-31 and k = 8h + 4 + e on lanes 32-63, so a lane reads the four k
// of its row it needs for four steps with one 16-byte read (an [n][k] B
// too; a [k][n] B as four 4-byte reads). Every k of the slice is summed once;
// the order of the sums is the any-shape kernel's.
// Measured interleaved with a register-staged kernel of 16 waves of 64x64 in
// 256x256 tiles, k in order, at 4096^3 (rotated inputs, one box): 945-947 against 1030-1033 us, 145.3 against 133.3
// TFLOP/s; the error against a float64 sum of the same products 6.95e-5
// against 8.37e-5 on 64 sampled elements.
typedef float f32x16_t __attribute__((ext_vector_type(16)));
__device__ __forceinline__ void mfma32_f32_acc(f32x16_t& c, float a, float b) {
  asm volatile("v_mfma_f32_32x32x2_f32 %0, %1, %2, %0" : "+a"(c) : "v"(a), "v"(b));
}

// f(integral_constant<int, 0>) ... f(integral_constant<int, N-1>): a step's
// MFMAs with compile-time block indices (a loop over them is not unrolled
// by the compiler at this size, and run-time indices put the accumulators
// in scratch).
template <typename F, int... I>
__device__ __forceinline__ void static_for_impl(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, typename F>
__device__ __forceinline__ void static_for(F&& f) {
  static_for_impl(f, std::make_integer_sequence<int, N>{});
}

template <bool B_NK, typename Epi>
__device__ __forceinline__ void gemm_f32_4w(const float* __restrict__ A, const float* __restrict__ B,
                                            float* __restrict__ C, uint32_t M, uint32_t N, uint32_t K, Epi epi,
                                            uint32_t tile = ~0u) {
  constexpr uint32_t BM = 256, BN = 256, ASL = 256u * 16u, LDBK = 264u, BSL = B_NK ? 256u * 16u : 16u * LDBK;
  constexpr uint32_t SLOT = ASL + BSL;
  __shared__ __attribute__((aligned(16))) float lds[4 * SLOT];
  const uint32_t tiles_m = (M + BM - 1) / BM, tiles_n = (N + BN - 1) / BN;
  uint32_t tm, tn;
  gemm_tile_coords(tiles_m, tiles_n, &tm, &tn, tile == ~0u ? blockIdx.x : tile);
  const uint32_t m0 = tm * BM, n0 = tn * BN;
  if (m0 + BM > M || n0 + BN > N || K % 32u != 0u || K < 128u) return;
  const uint32_t tid = threadIdx.x, lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const uint32_t wm = (wave >> 1) * 128u, wn = (wave & 1u) * 128u;
  f32x16_t acc[4][4];
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.0f;
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j) asm volatile("" : "+a"(acc[i][j]));
  asm volatile("s_nop 7\n\ts_nop 7" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // A wave-load (1 KiB) fills 16 rows of a [256][16] slice, or one k row of
  // a [16][264] slice; wave w fills rows 16(4w) .. 16(4w+3)+15, or k rows
  // 4w .. 4w+3. Per-lane element offsets (the inverse of the chunk swizzle).
  uint32_t offa[4], offb[4];
#pragma unroll
  for (int q = 0; q < 4; ++q) {
    const uint32_t row = 16u * (4u * wave + q) + (lane >> 2);
    offa[q] = row * K + 4u * ((lane & 3u) ^ ((row >> 2) & 3u));
    if constexpr (B_NK) offb[q] = offa[q];
    else offb[q] = (4u * wave + q) * N + 4u * lane;
  }
  float* ldsp = lds;
  auto a_slot = [&](uint32_t s) { return ldsp + (s & 3u) * SLOT; };
  auto b_slot = [&](uint32_t s) { return ldsp + (s & 3u) * SLOT + ASL; };
  auto load = [&](int q, uint32_t s) {  // q 0..3: A rows, q 4..7: B rows
    const uint32_t k0 = s * 16u;
    if (q < 4) {
      const float* a0 = A + static_cast<uint64_t>(m0) * K + k0;
      __builtin_amdgcn_global_load_lds(a0 + offa[q], (lds_void*)(a_slot(s) + (4u * wave + q) * 256u), 16, 0, 0);
    } else if constexpr (B_NK) {
      const float* b0 = B + static_cast<uint64_t>(n0) * K + k0;
      __builtin_amdgcn_global_load_lds(b0 + offb[q - 4], (lds_void*)(b_slot(s) + (4u * wave + q - 4) * 256u), 16, 0, 0);
    } else {
      const float* b0 = B + static_cast<uint64_t>(k0) * N + n0;
      __builtin_amdgcn_global_load_lds(b0 + offb[q - 4], (lds_void*)(b_slot(s) + (4u * wave + q - 4) * LDBK), 16, 0, 0);
    }
  };
  auto rd_a = [&](uint32_t s, uint32_t i, uint32_t h) {  // rows wm + 32i + lane%32, k 8h + 4(lane/32) .. +3
    const float* As = a_slot(s);
    const uint32_t row = wm + 32u * i + (lane & 31u), c = 2u * h + (lane >> 5);
    return *reinterpret_cast<const f32x4_t*>(&As[row * 16u + 4u * (c ^ ((row >> 2) & 3u))]);
  };
  auto rd_b = [&](uint32_t s, uint32_t j, uint32_t h) {  // columns wn + 32j + lane%32, the same k
    const float* Bs = b_slot(s);
    const uint32_t col = wn + 32u * j + (lane & 31u);
    if constexpr (B_NK) {
      const uint32_t c = 2u * h + (lane >> 5);
      return *reinterpret_cast<const f32x4_t*>(&Bs[col * 16u + 4u * (c ^ ((col >> 2) & 3u))]);
    } else {
      const uint32_t k = 8u * h + 4u * (lane >> 5);
      f32x4_t v;
      v[0] = Bs[(k + 0u) * LDBK + col];
      v[1] = Bs[(k + 1u) * LDBK + col];
      v[2] = Bs[(k + 2u) * LDBK + col];
      v[3] = Bs[(k + 3u) * LDBK + col];
      return v;
    }
  };
  f32x4_t fa0[4][2], fb0[4][2], fa1[4][2], fb1[4][2];  // two fragment sets: this slice's and the next one's
  auto fence = []() { __builtin_amdgcn_sched_barrier(0); };
  auto barrier = [&]() {
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
  };
  auto step = [&](auto set, uint32_t s, int wait_vm, bool rd, bool ld) {
    auto& ca = decltype(set)::value == 0 ? fa0 : fa1;
    auto& cb = decltype(set)::value == 0 ? fb0 : fb1;
    auto& na = decltype(set)::value == 0 ? fa1 : fa0;
    auto& nb = decltype(set)::value == 0 ? fb1 : fb0;
    if (wait_vm >= 0) {
      asm volatile("" ::: "memory");
      if (wait_vm == 16) __builtin_amdgcn_s_waitcnt(waitcnt_imm(16, 0));
      else if (wait_vm == 8) __builtin_amdgcn_s_waitcnt(waitcnt_imm(8, 0));
      else __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
      barrier();
    }
    const uint32_t ns = s + 1u;
    fence();
    // MFMA c (0..127): 2-deep step t = c/16 (h = t/4, e = t%4), block (i, j)
    // snaking over 4x4. The next slot's 8 A and 8 B fragment reads follow
    // MFMAs 0..15, the 8 loads of slice s+4 MFMAs 55, 63, ..., 111.
    static_for<128>([&](auto ic) {
      constexpr int c = decltype(ic)::value;
      constexpr int t = c >> 4, h = t >> 2, e = t & 3, b = c & 15, i = b >> 2, j = (i & 1) ? 3 - (b & 3) : (b & 3);
      mfma32_f32_acc(acc[i][j], ca[i][h][e], cb[j][h][e]);
      fence();
      if constexpr (c < 16) {
        if (rd) {
          if constexpr (c < 8) na[c >> 1][c & 1] = rd_a(ns, c >> 1, c & 1);
          else nb[(c - 8) >> 1][(c - 8) & 1] = rd_b(ns, (c - 8) >> 1, (c - 8) & 1);
        }
        fence();
      }
      if constexpr (c >= 55 && (c - 55) % 8 == 0 && (c - 55) / 8 < 8) {
        if (ld) load((c - 55) / 8, s + 4u);
        fence();
      }
    });
  };
  using Set0 = std::integral_constant<int, 0>;
  using Set1 = std::integral_constant<int, 1>;
  const uint32_t nk = K / 16u;
  for (uint32_t s = 0; s < 4; ++s)
    for (int q = 0; q < 8; ++q) load(q, s);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(24, 0));  // slice 0 landed
  barrier();
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      fa0[i][h] = rd_a(0, i, h);
      fb0[i][h] = rd_b(0, i, h);
    }
  // At the start of slice s slot s+1 must have landed: the loads of slices
  // s+2 and s+3 may remain (16; vmcnt counts in issue order). The loop runs
  // at least once (K >= 128): a path around it kept the zeroed accumulators
  // live across an edge and spilled them.
  const uint32_t main_end = nk - 4u;  // even (K % 32 == 0), at least 4
  uint32_t s = 0;
  do {
    step(Set0{}, s, 16, true, true);
    step(Set1{}, s + 1, 16, true, true);
    s += 2;
  } while (s < main_end);
  step(Set0{}, nk - 4u, 16, true, false);
  step(Set1{}, nk - 3u, 8, true, false);
  step(Set0{}, nk - 2u, 0, true, false);
  step(Set1{}, nk - 1u, -1, false, false);
  __builtin_amdgcn_s_waitcnt(waitcnt_imm(0, 0));
  __builtin_amdgcn_sched_barrier(0);
  // 32 wait states: a 16-pass XDL write before the epilogue reads the AGPRs.
  asm volatile("s_nop 7\n\ts_nop 7\n\ts_nop 7\n\ts_nop 7" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  // acc[i][j][e] = C[r][c], r = m0 + wm + 32i + 8(e/4) + 4(lane/32) + e%4, c = n0 + wn + 32j + lane%32.
#pragma unroll
  for (int i = 0; i < 4; ++i)
#pragma unroll
    for (int j = 0; j < 4; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) {
        const uint32_t r = m0 + wm + i * 32u + 8u * (e >> 2) + 4u * (lane >> 5) + (e & 3);
        const uint32_t c = n0 + wn + j * 32u + (lane & 31u);
        C[static_cast<uint64_t>(r) * N + c] = epi(acc[i][j][e], r, c);
      }
}

// ------------------------------------------------ small contractions, K split
// The tile kernels above give one workgroup a 128x128 or 256x256 tile and
// the whole of K, so a contraction with few tiles (the reference suite's
// gemm, mlp, mm_* and qk_score have M, N <= 192: one or two workgroups) runs
// on one or two CUs, walking K alone (testing/kernels/tiling/mm_splitk.tca:1-2
// names the split-k schedule class for them). Here a workgroup of 16 waves
// owns a 32x32 tile of C and a chunk of K:
//   - the chunk's k steps (16 deep for f32, 32 for 16-bit inputs) are dealt
//     round-robin to the 16 waves; each wave accumulates the whole 32x32 tile;
//   - the waves' tiles meet in LDS and are summed in wave order;
//   - with P > 1 chunks (P = gemm_split_chunks(K, tiles, KCMIN, BLOCKS),
//     the formula of the launch plan's split record) the workgroup of chunk
//     p writes its sum to a partial scratch [P][tiles][1024] and a second
//     kernel (gemm_small_merge) adds the P partials in chunk order.
// Every order is fixed, so the result does not depend on the schedule.
// The waves of a workgroup read disjoint k, so nothing is shared inside it
// (small16_steps, small32_steps); neighbouring tiles share panels through the
// L2. Without a K split larger tiles are taken where they fill the CUs
// (gemm_small_form).
// f32 result element i of lane l is C[m0 + 8(i/4) + 4(l/32) + i%4][n0 + l%32];
// a wave's tile goes to LDS element-major (word i*64 + l: conflict-free) and
// thread t = i*64 + l of the workgroup sums word t over the waves.
// Tiles are numbered down the columns of tiles, and the workgroups of one
// XCD (every eighth) take a run of them: the tiles that read one panel of B
// share an L2.
constexpr uint32_t kSmallWaves = 16;

// P chunks of K for `tiles` output tiles: enough workgroups to reach
// `blocks`, each chunk at least kc_min deep (1 when K or tiles is 0). The
// launch plan's split record computes the same number (SplitChunks).
__host__ __device__ __forceinline__ uint32_t gemm_split_chunks(uint32_t k, uint32_t tiles, uint32_t kc_min,
                                                               uint32_t blocks) {
  if (k == 0u || tiles == 0u) return 1u;
  uint32_t p = (k - 1u) / kc_min + 1u;
  const uint32_t cap = blocks / tiles;
  if (p > cap) p = cap;
  return p ? p : 1u;
}

// Coordinates (row, column) inside a 32x32 tile of the value thread t holds
// after the wave merge: its word of the MFMA result for f32, row-major for
// 16-bit inputs.
template <bool H16>
__device__ __forceinline__ uint32_t small_row(uint32_t t) {
  if constexpr (H16) return t >> 5;
  const uint32_t i = t >> 6, l = t & 63u;
  return 8u * (i >> 2) + 4u * (l >> 5) + (i & 3u);
}
__device__ __forceinline__ uint32_t small_col(uint32_t t) { return t & 31u; }

// The tile that workgroup `i` of a chunk's T takes.
__device__ __forceinline__ uint32_t gemm_small_tile(uint32_t i, uint32_t T) {
  const uint32_t x = i & 7u, q = T >> 3, r = T & 7u;
  return x * q + (x < r ? x : r) + (i >> 3);
}

// A wave's 32-deep k steps (s_begin + wave, + 16, ...) of a 16 IM x 32 tile,
// 16-bit inputs. Four lanes load the 64 bytes of a row (loaded in the MFMA
// operand's layout, 16 rows to 16 consecutive lanes, every lane of a quad
// touches another line and the address unit takes 64 cycles per load instead
// of 16: 16 x 16384 x 16384 ran at 3.5-4.1 TB/s); the step goes through the
// wave's own 4 KiB of LDS (`stage`: 32 rows of A at a time, then B) into
// operand layout. No load is guarded (clamped and moved into place as in
// gemm16_tile; K >= 8, and N >= 8 for [K][N]). D steps are in flight; the main
// loop's loads are unconditional, as there.
template <int IM, int D, bool B_NK, bool F16>
__device__ __forceinline__ void small16_steps(const uint16_t* __restrict__ A, const uint16_t* __restrict__ B,
                                              uint32_t M, uint32_t N, uint32_t K, uint32_t m0, uint32_t n0,
                                              uint32_t s_begin, uint32_t s_end, uint16_t* stage, f32x4_t (&acc)[IM][2]) {
  const uint32_t thread = thread_here(), lane = thread & 63u, wave = __builtin_amdgcn_readfirstlane(thread >> 6);
  const uint32_t r = lane >> 2, kg = (lane & 3u) * 8u;  // as loaded
  const uint16_t *pa[IM], *pb[2];
  uint32_t bsh = 0u;
#pragma unroll
  for (int i = 0; i < IM; ++i) {
    const uint32_t m = m0 + r + 16u * i;
    pa[i] = A + static_cast<uint64_t>(m < M ? m : M - 1u) * K;
  }
  if constexpr (B_NK) {
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      const uint32_t n = n0 + r + 16u * j;
      pb[j] = B + static_cast<uint64_t>(n < N ? n : N - 1u) * K;
    }
  } else {
    const uint32_t n = n0 + kg, at = n < N - 8u ? n : N - 8u;
    bsh = n - at;
    pb[0] = pb[1] = B + at;
  }
  u32x4 xa[D][IM], xb[D][2];
  auto load = [&](int d, uint32_t s) {
    const uint32_t k = s * 32u + kg, kc = k < K - 8u ? k : K - 8u;
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (B_NK) {
        xb[d][j] = load16_any(pb[j] + kc);
      } else {
        const uint32_t kr = s * 32u + r + 16u * j;
        xb[d][j] = load16_any(pb[0] + static_cast<uint64_t>(kr < K ? kr : K - 1u) * N);
      }
    }
#pragma unroll
    for (int i = 0; i < IM; ++i) xa[d][i] = load16_any(pa[i] + kc);
  };
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j) acc[i][j] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
  const bool edge_n = !B_NK && n0 + 32u > N;
  auto mma = [&](auto last, int d, uint32_t s) {
    if (decltype(last)::value && s * 32u + 32u > K) {  // the short last step
      const uint32_t k = s * 32u + kg, n = k - (k < K - 8u ? k : K - 8u);
#pragma unroll
      for (int i = 0; i < IM; ++i) xa[d][i] = shift_down16(xa[d][i], n);
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        if constexpr (B_NK) xb[d][j] = shift_down16(xb[d][j], n);
        else if (s * 32u + r + 16u * j >= K) xb[d][j] = u32x4{0u, 0u, 0u, 0u};
      }
    }
    if constexpr (!B_NK) {
      if (edge_n) {
#pragma unroll
        for (int j = 0; j < 2; ++j) xb[d][j] = shift_down16(xb[d][j], bsh);
      }
    }
    // A region is rewritten behind the reads of what it held.
    uint16_t* bst = stage + 1024;
    wave_exchange();
#pragma unroll
    for (int j = 0; j < 2; ++j)
      *reinterpret_cast<u32x4*>(&bst[B_NK ? swz_rows32(r + 16u * j, lane & 3u) : swz_kn<32>(r + 16u * j, kg)]) = xb[d][j];
    auto stage_a = [&](int h) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        *reinterpret_cast<u32x4*>(&stage[swz_rows32(r + 16u * i, lane & 3u)]) = xa[d][2 * h + i];
    };
    stage_a(0);
    wave_exchange();
    bf16x8 fb[2];
#pragma unroll
    for (int j = 0; j < 2; ++j) {
      if constexpr (B_NK) fb[j] = *reinterpret_cast<const bf16x8*>(&bst[swz_rows32(16u * j + (lane & 15u), lane >> 4)]);
      else fb[j] = frag_b16_tr<32>(bst, 16u * j, lane);
    }
#pragma unroll
    for (int h = 0; h < IM / 2; ++h) {
      if (h > 0) {
        wave_exchange();
        stage_a(h);
        wave_exchange();
      }
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const bf16x8 fa = *reinterpret_cast<const bf16x8*>(&stage[swz_rows32(16u * i + (lane & 15u), lane >> 4)]);
#pragma unroll
        for (int j = 0; j < 2; ++j) acc[2 * h + i][j] = mfma_16x16x32_16b<F16>(fb[j], fa, acc[2 * h + i][j]);
      }
    }
  };
  constexpr uint32_t W = kSmallWaves;
  uint32_t s = s_begin + wave;
  if (s >= s_end) return;
  if (s + (2u * D - 1u) * W < s_end) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, s + d * W);
    do {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        mma(std::false_type{}, d, s + d * W);
        load(d, s + (D + d) * W);
      }
      s += D * W;
    } while (s + (2u * D - 1u) * W < s_end);
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (s + d * W < s_end) load(d, s + d * W);
  }
  for (; s < s_end; s += D * W) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (s + d * W < s_end) mma(std::true_type{}, d, s + d * W);
      if (s + (D + d) * W < s_end) load(d, s + (D + d) * W);
    }
  }
}

// Sums the 16 waves' 16 IM x 32 tiles, 32 rows at a time, in wave order, and
// hands `out` each element: out(row, column, sum). Rows go to LDS with their
// 16-byte groups XORed by the row, so the writes of 16 rows are conflict-free.
template <int IM, typename Out>
__device__ __forceinline__ void small16_sum(const f32x4_t (&acc)[IM][2], float* red, Out&& out) {
  const uint32_t tid = thread_here(), lane = tid & 63u, wave = tid >> 6;
  const uint32_t row = tid >> 5, word = row * 32u + ((((tid & 31u) >> 2) ^ ((row >> 1) & 7u)) << 2) + (tid & 3u);
#pragma unroll
  for (int h = 0; h < IM / 2; ++h) {
    if (h > 0) __syncthreads();
    else wave_exchange();  // the wave's rows held its operands
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int j = 0; j < 2; ++j) {
        const uint32_t rr = 16u * i + (lane & 15u), cg = 4u * j + (lane >> 4);
        *reinterpret_cast<f32x4_t*>(&red[wave * 1024u + rr * 32u + ((cg ^ ((rr >> 1) & 7u)) << 2)]) = acc[2 * h + i][j];
      }
    __syncthreads();
    float sum = red[word];
#pragma unroll
    for (uint32_t w = 1; w < kSmallWaves; ++w) sum += red[w * 1024u + word];
    out(32u * h + row, tid & 31u, sum);
  }
}

// small16_steps for fp32 inputs: 16-deep steps of a 32 IM x 32 tile (K >= 4, and
// N >= 4 for a [K][N] operand), 8 IM v_mfma_f32_32x32x2f32 each; four lanes load
// the 64 bytes of a row of A or [N][K] B, eight the 128 of a [K][N] row.
// HALVES: the 8-deep halves of the steps are dealt to the waves instead.
template <int IM, int D, bool B_NK, bool HALVES = false>
__device__ __forceinline__ void small32_steps(const float* __restrict__ A, const float* __restrict__ B, uint32_t M,
                                              uint32_t N, uint32_t K, uint32_t m0, uint32_t n0, uint32_t s_begin,
                                              uint32_t s_end, float* stage, f32x16 (&acc)[IM]) {
  const uint32_t thread = thread_here(), lane = thread & 63u, wave = __builtin_amdgcn_readfirstlane(thread >> 6);
  const uint32_t r = lane >> 2, kg = (lane & 3u) * 4u;      // rows of 16: row r (+ 16), k chunk
  // [K][N] rows of 32: row rn (+ 8), column chunk. Lane group q takes row q/2
  // + 4 (q%2), so that in LDS the rows k and k + 4 that the halves of a wave
  // read are neighbours: writes and reads go through the 64 banks in lane order.
  const uint32_t rn = (lane >> 4) + 4u * ((lane >> 3) & 1u), ng = (lane & 7u) * 4u;
  const float *pa[2 * IM], *pb[2];
  uint32_t bsh = 0u;
#pragma unroll
  for (int i = 0; i < 2 * IM; ++i) {
    const uint32_t m = m0 + r + 16u * i;
    pa[i] = A + static_cast<uint64_t>(m < M ? m : M - 1u) * K;
  }
  if constexpr (B_NK) {
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const uint32_t n = n0 + r + 16u * i;
      pb[i] = B + static_cast<uint64_t>(n < N ? n : N - 1u) * K;
    }
  } else {
    const uint32_t n = n0 + ng, at = n < N - 4u ? n : N - 4u;
    bsh = n - at;
    pb[0] = pb[1] = B + at;
  }
  f32x4_t xa[D][2 * IM], xb[D][2];
  auto load = [&](int d, uint32_t s) {
    const uint32_t k = s * 16u + kg, kc = k < K - 4u ? k : K - 4u;
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      if constexpr (B_NK) {
        xb[d][i] = load16_any(pb[i] + kc);
      } else {
        const uint32_t kr = s * 16u + rn + 8u * i;
        xb[d][i] = load16_any(pb[i] + static_cast<uint64_t>(kr < K ? kr : K - 1u) * N);
      }
    }
#pragma unroll
    for (int i = 0; i < 2 * IM; ++i) xa[d][i] = load16_any(pa[i] + kc);
  };
#pragma unroll
  for (int i = 0; i < IM; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.0f;
  // One block: the two 8-deep halves of a step sum apart (a shorter chain).
  f32x16 acc1 = acc[0];
  const bool edge_n = !B_NK && n0 + 32u > N;
  const auto rows16 = [](uint32_t row, uint32_t c) { return row * 16u + ((c ^ ((row >> 2) & 3u)) << 2); };
  const uint32_t hsel = wave & 1u;
  auto mma = [&](auto last, auto one, int d, uint32_t s) {
    constexpr bool kOne = decltype(one)::value;  // the 8-deep half hsel of the step only
    if (decltype(last)::value && s * 16u + 16u > K) {  // the short last step
      const uint32_t k = s * 16u + kg, n = k - (k < K - 4u ? k : K - 4u);
#pragma unroll
      for (int i = 0; i < 2 * IM; ++i) xa[d][i] = shift_down32(xa[d][i], n);
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        if constexpr (B_NK) xb[d][i] = shift_down32(xb[d][i], n);
        else if (s * 16u + rn + 8u * i >= K) xb[d][i] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
      }
    }
    if constexpr (!B_NK) {
      if (edge_n) {
#pragma unroll
        for (int i = 0; i < 2; ++i) xb[d][i] = shift_down32(xb[d][i], bsh);
      }
    }
    float* bst = stage + 512;
    wave_exchange();
#pragma unroll
    for (int i = 0; i < 2; ++i)
      *reinterpret_cast<f32x4_t*>(&bst[B_NK ? rows16(r + 16u * i, lane & 3u) : 256u * i + 4u * lane]) = xb[d][i];
    auto stage_a = [&](int b) {
#pragma unroll
      for (int i = 0; i < 2; ++i)
        *reinterpret_cast<f32x4_t*>(&stage[rows16(r + 16u * i, lane & 3u)]) = xa[d][2 * b + i];
    };
    stage_a(0);
    wave_exchange();
    const uint32_t l32 = lane & 31u, hf = lane >> 5;
    f32x4_t fb[2];
#pragma unroll
    for (uint32_t h = 0; h < 2u; ++h) {
      if constexpr (B_NK) {
        fb[h] = *reinterpret_cast<const f32x4_t*>(&bst[rows16(l32, 2u * h + hf)]);
      } else {
#pragma unroll
        for (uint32_t e = 0; e < 4u; ++e) fb[h][e] = bst[256u * h + 64u * e + lane];  // k = 8h + 4hf + e, column l32
      }
    }
#pragma unroll
    for (int b = 0; b < IM; ++b) {
      if (b > 0) {
        wave_exchange();
        stage_a(b);
        wave_exchange();
      }
#pragma unroll
      for (uint32_t h = 0; h < 2u; ++h) {
        if (kOne && h != hsel) continue;
        const f32x4_t fa = *reinterpret_cast<const f32x4_t*>(&stage[rows16(l32, 2u * h + hf)]);
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          f32x16& c = IM == 1 && h == 1u ? acc1 : acc[b];
          c = __builtin_amdgcn_mfma_f32_32x32x2f32(fa[e], fb[h][e], c, 0, 0, 0);
        }
      }
    }
  };
  using Body = std::false_type;
  using Last = std::true_type;
  if constexpr (HALVES) {
    for (uint32_t s = s_begin + (wave >> 1); s < s_end; s += kSmallWaves / 2u) {
      load(0, s);
      mma(Last{}, std::true_type{}, 0, s);
    }
    return;
  }
  constexpr std::false_type both{};
  constexpr uint32_t W = kSmallWaves;
  uint32_t s = s_begin + wave;
  if (s >= s_end) return;
  if (s + (2u * D - 1u) * W < s_end) {
#pragma unroll
    for (int d = 0; d < D; ++d) load(d, s + d * W);
    do {
#pragma unroll
      for (int d = 0; d < D; ++d) {
        mma(Body{}, both, d, s + d * W);
        load(d, s + (D + d) * W);
      }
      s += D * W;
    } while (s + (2u * D - 1u) * W < s_end);
  } else {
#pragma unroll
    for (int d = 0; d < D; ++d)
      if (s + d * W < s_end) load(d, s + d * W);
  }
  for (; s < s_end; s += D * W) {
#pragma unroll
    for (int d = 0; d < D; ++d) {
      if (s + d * W < s_end) mma(Last{}, both, d, s + d * W);
      if (s + (D + d) * W < s_end) load(d, s + (D + d) * W);
    }
  }
  if constexpr (IM == 1) {
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[0][e] += acc1[e];
  }
}

// Sums the 16 waves' blocks of 32x32 MFMA results, one block at a time, in wave
// order, and hands `out` each element: out(row, word, sum), word the
// element's place in the block's MFMA result.
template <int IM, typename Out>
__device__ __forceinline__ void small32_sum(const f32x16 (&acc)[IM], float* red, Out&& out) {
  const uint32_t tid = thread_here(), lane = tid & 63u, wave = tid >> 6;
#pragma unroll
  for (int b = 0; b < IM; ++b) {
    if (b > 0) __syncthreads();
    else wave_exchange();
#pragma unroll
    for (int i = 0; i < 16; ++i) red[wave * 1024u + static_cast<uint32_t>(i) * 64u + lane] = acc[b][i];
    __syncthreads();
    float sum = red[tid];
#pragma unroll
    for (uint32_t w = 1; w < kSmallWaves; ++w) sum += red[w * 1024u + tid];
    out(32u * b, tid, sum);
  }
}

// One 32x32 tile of C, over chunk p of P of K. `tile` is the tile within its
// contraction (column-major), `gtile` its index over all T tiles of the launch
// (batches included): the partial scratch is indexed by it.
template <bool H16, bool B_NK, typename Epi, bool F16 = false>
__device__ __forceinline__ void gemm_small(const void* __restrict__ Av, const void* __restrict__ Bv,
                                           float* __restrict__ C, float* __restrict__ part, uint32_t M, uint32_t N,
                                           uint32_t K, Epi epi, uint32_t tile, uint32_t gtile, uint32_t T, uint32_t p,
                                           uint32_t P) {
  __shared__ __attribute__((aligned(16))) float red[kSmallWaves * 1024u];
  const uint32_t tiles_m = (M - 1u) / 32u + 1u;
  const uint32_t m0 = (tile % tiles_m) * 32u, n0 = (tile / tiles_m) * 32u;
  const uint32_t tid = thread_here(), lane = tid & 63u, wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  if constexpr (H16) {
    if (__builtin_expect(K >= 8u && (B_NK || N >= 8u), 1)) {
      const uint32_t steps = (K - 1u) / 32u + 1u, per = P > 1u ? (steps - 1u) / P + 1u : steps;
      const uint32_t s_begin = p * per < steps ? p * per : steps;
      const uint32_t s_end = s_begin + per < steps ? s_begin + per : steps;
      f32x4_t acc[2][2];
      small16_steps<2, 4, B_NK, F16>(static_cast<const uint16_t*>(Av), static_cast<const uint16_t*>(Bv), M, N, K, m0, n0,
                                     s_begin, s_end, reinterpret_cast<uint16_t*>(red) + wave * 2048u, acc);
      small16_sum(acc, red, [&](uint32_t row, uint32_t col, float sum) {
        if (P > 1u) part[(static_cast<uint64_t>(p) * T + gtile) * 1024u + row * 32u + col] = sum;
        else if (m0 + row < M && n0 + col < N) C[static_cast<uint64_t>(m0 + row) * N + n0 + col] = epi(sum, m0 + row, n0 + col);
      });
      return;
    }
  }
  const auto store = [&](uint32_t, uint32_t t, float sum) {
    const uint32_t sr = small_row<false>(t), sc = small_col(t), m = m0 + sr, n = n0 + sc;
    if (P > 1u) part[(static_cast<uint64_t>(p) * T + gtile) * 1024u + (H16 ? sr * 32u + sc : t)] = sum;
    else if (m < M && n < N) C[static_cast<uint64_t>(m) * N + n] = epi(sum, m, n);
  };
  f32x16 acc[1];
  if constexpr (!H16) {
    if (__builtin_expect(K >= 4u && (B_NK || N >= 4u), 1)) {
      const uint32_t steps = (K - 1u) / 16u + 1u, per = P > 1u ? (steps - 1u) / P + 1u : steps;
      const uint32_t s_begin = p * per < steps ? p * per : steps;
      const uint32_t s_end = s_begin + per < steps ? s_begin + per : steps;
      small32_steps<1, 2, B_NK>(static_cast<const float*>(Av), static_cast<const float*>(Bv), M, N, K, m0, n0, s_begin,
                                s_end, red + wave * 1024u, acc);
      small32_sum(acc, red, store);
      return;
    }
  }
  // Rows shorter than a chunk: element by element, 2-deep MFMA steps of k =
  // step + lane / 32, dealt to the waves.
  const uint32_t am = m0 + (lane & 31u), bn = n0 + (lane & 31u);
  const uint32_t steps = K / 2u + K % 2u, per = steps / P + (steps % P != 0u ? 1u : 0u);
  const uint32_t s_begin = p * per < steps ? p * per : steps;
  const uint32_t s_end = s_begin + per < steps ? s_begin + per : steps;
  const auto value = [](const void* v, uint64_t i) -> float {
    if constexpr (!H16) return static_cast<const float*>(v)[i];
    else if constexpr (F16) return static_cast<float>(static_cast<const _Float16*>(v)[i]);
    else return static_cast<float>(static_cast<const __bf16*>(v)[i]);
  };
#pragma unroll
  for (int e = 0; e < 16; ++e) acc[0][e] = 0.0f;
  for (uint32_t s = s_begin + wave; s < s_end; s += kSmallWaves) {
    const uint32_t k = 2u * s + (lane >> 5);
    float a = 0.0f, b = 0.0f;
    if (am < M && k < K) a = value(Av, static_cast<uint64_t>(am) * K + k);
    if (bn < N && k < K) b = value(Bv, B_NK ? static_cast<uint64_t>(bn) * K + k : static_cast<uint64_t>(k) * N + bn);
    acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(a, b, acc[0], 0, 0, 0);
  }
  small32_sum(acc, red, store);
}

// The forms of the small kernel: TM x TN tiles of C, 128x128 (16-bit inputs),
// 64x64 or 64x32, all of K in one chunk. The plan picks the largest of which
// there are kSmallTilesMin (emit_hip.cpp), rows of a chunk and more; fewer
// tiles, or a K split over workgroups, stay 32x32 (gemm_small). A larger tile
// reads its operands fewer times: 64 x 8192 x 8192 (B as [K][N]) takes 73 us on
// 32x32 tiles, which read B twice, past what an L2 holds of it in flight, and
// 54 on 64x32; 1024 x 1024 x 4096 55 on 32x32 and 21 on 64x64; 32 batches of 500
// x 500 x 64 47 on 32x32 and 12 on 128x128. A 32x64 tile for M <= 32 was within
// 15% either way; fp32: 1024 x 1024 x 4096 127 us before, 85 on 64x64, 64 x 8192
// x 4096 81 before, 60 on 32x32, 52 on 64x32. What bounds a few rows against a
// large [K][N] B (16 x 16384 x 16384, 3.5 TB/s; 5.0 with [N][K]) is its 64-byte
// pieces of rows 32 KB apart.
// `wave` is the thread's, in a scalar register.
template <bool H16, bool B_NK, uint32_t TM, uint32_t TN, bool F16, typename Epi>
__device__ __forceinline__ void gemm_small_form(const void* __restrict__ Av, const void* __restrict__ Bv,
                                                float* __restrict__ C, uint32_t M, uint32_t N, uint32_t K, Epi epi,
                                                uint32_t tile, uint32_t wave) {
  static_assert((TM == 64u && (TN == 32u || TN == 64u)) || (H16 && TM == 128u && TN == 128u), "the small kernel's forms");
  __shared__ __attribute__((aligned(16))) float red[kSmallWaves * 1024u];
  const uint32_t tiles_m = (M - 1u) / TM + 1u;
  const uint32_t m0 = (tile % tiles_m) * TM, n0 = (tile / tiles_m) * TN;
  const uint32_t tid = wave * 64u + lane_here();
  if constexpr (H16) {
    const uint16_t* A = static_cast<const uint16_t*>(Av);
    const uint16_t* B = static_cast<const uint16_t*>(Bv);
    uint16_t* lds = reinterpret_cast<uint16_t*>(red);
    if constexpr (TN == 128u) {
      gemm16_tile<128, 128, 4, 4, 1, 2, B_NK, F16, false, true>(A, B, C, M, N, K, epi, m0, n0, lds, tid);
    } else if constexpr (TN == 64u) {
      gemm16_tile<64, 64, 2, 4, 2, 2, B_NK, F16, false, true>(A, B, C, M, N, K, epi, m0, n0, lds, tid);
    } else {
      f32x4_t acc[4][2];
      small16_steps<4, 2, B_NK, F16>(A, B, M, N, K, m0, n0, 0u, (K - 1u) / 32u + 1u, lds + wave * 2048u, acc);
      small16_sum(acc, red, [&](uint32_t row, uint32_t col, float sum) {
        if (m0 + row < M && n0 + col < N) C[static_cast<uint64_t>(m0 + row) * N + n0 + col] = epi(sum, m0 + row, n0 + col);
      });
    }
  } else {
    const float* A = static_cast<const float*>(Av);
    const float* B = static_cast<const float*>(Bv);
    if constexpr (TN == 64u) {
      gemm32_tile<64, 64, 2, 2, 4, 1, B_NK, false, true>(A, B, C, M, N, K, epi, m0, n0, red, tid);
    } else {
      f32x16 acc[2];
      const uint32_t steps = (K - 1u) / 16u + 1u;
      // Up to K = 144, where most waves get one half: more of them work, and no
      // chain of matrix instructions is longer than with sums of 8 k (60 x 8001 x
      // 64 4.2 us and 7.7e-8 from 64 bits; 6.2 us, 8.4e-8 by whole steps).
      if (steps <= 9u) small32_steps<2, 1, B_NK, true>(A, B, M, N, K, m0, n0, 0u, steps, red + wave * 1024u, acc);
      else small32_steps<2, 2, B_NK>(A, B, M, N, K, m0, n0, 0u, steps, red + wave * 1024u, acc);
      small32_sum(acc, red, [&](uint32_t row0, uint32_t t, float sum) {
        const uint32_t m = m0 + row0 + small_row<false>(t), n = n0 + small_col(t);
        if (m < M && n < N) C[static_cast<uint64_t>(m) * N + n] = epi(sum, m, n);
      });
    }
  }
}

// The P > 1 merge: one 1024-thread workgroup per tile, thread t adds word t
// of the tile's P partials in chunk order, applies the epilogue and stores.
template <bool H16, typename Epi>
__device__ __forceinline__ void gemm_small_merge(float* __restrict__ C, const float* __restrict__ part, uint32_t M,
                                                 uint32_t N, Epi epi, uint32_t tile, uint32_t gtile, uint32_t T,
                                                 uint32_t P) {
  const uint32_t tid = threadIdx.x, tiles_m = (M + 31u) / 32u;
  const uint32_t m = (tile % tiles_m) * 32u + small_row<H16>(tid), n = (tile / tiles_m) * 32u + small_col(tid);
  const float* q = part + static_cast<uint64_t>(gtile) * 1024u + tid;
  const uint64_t stride = static_cast<uint64_t>(T) * 1024u;
  float sum = q[0];
  uint32_t c = 1;
  for (; c + 4u <= P; c += 4u) {
    const float v0 = q[c * stride], v1 = q[(c + 1u) * stride], v2 = q[(c + 2u) * stride], v3 = q[(c + 3u) * stride];
    sum += v0;
    sum += v1;
    sum += v2;
    sum += v3;
  }
  for (; c < P; ++c) sum += q[c * stride];
  if (m < M && n < N) C[static_cast<uint64_t>(m) * N + n] = epi(sum, m, n);
}

}  // namespace hip
}  // namespace tca

#endif  // TCA_HIP_GEMM_H_
