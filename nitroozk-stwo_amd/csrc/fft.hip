// Circle FFT over batches of same-size M31 columns (PolyOps::interpolate / evaluate).
//
// Layer structure (prover/backend/cpu/circle.rs:28-80,190-228,295-335):
//   stage 0 (circle layer): pairs (2h, 2h+1), twiddle from line layer 0 pairs [x, y] -> [y,-y,-x,x]
//   stage s >= 1 (line layer s-1): pairs (idx, idx + 2^s), twiddle tree[len - 2^(K-s) + (idx >> (s+1))]
// interpolate runs stages 0..K-1 with inverse butterflies and inverse twiddles, then scales by
// 2^-K; evaluate runs stages K-1..0 with forward butterflies. Evaluating k coefficients onto a
// 2^b-times larger domain skips the top b stages: on zero-padded input they only copy, so the
// first pass reads the coefficient column with the index masked to 2^k.
//
// MI355X mapping, by transform size k (stages that run):
//   k >= 11   the low 11..15 stages in one pass over a tile in LDS, on doubles (fft_low_kernel);
//             the stages above in passes of at most 6 on register-resident words (fft_pass_reg_kernel)
//   k < 11    one or two passes on a tile in LDS (fft_pass_kernel)
#include <stdexcept>
#include "butterfly.h"
#include "field.h"
#include "kernels.h"

namespace sh {

// Column c (the same for a whole workgroup) of a transform's columns.
__device__ __forceinline__ const GLOBAL_AS uint32_t* col_in(const ColSet& s, uint32_t c) {
  return gmem(s.table ? s.table[c] : s.base + (int64_t)c * s.step);
}
__device__ __forceinline__ GLOBAL_AS uint32_t* col_out(const ColSet& s, uint32_t c) {
  return gmem(const_cast<uint32_t*>(s.table ? s.table[c] : s.base + (int64_t)c * s.step));
}

// Doubled circle twiddle of pair h (line layer 0 pairs [x, y] -> [y, -y, -x, x]).
__device__ __forceinline__ uint32_t circle_twiddle(const uint32_t* __restrict__ lt0, uint32_t h) {
  const uint32_t x = lt0[(h >> 2) * 2], y = lt0[(h >> 2) * 2 + 1];
  switch (h & 3) {
    case 0: return y;
    case 1: return neg_tw(y);
    case 2: return neg_tw(x);
    default: return x;
  }
}

// Doubled twiddle of the pair whose lower element has global index idx0 at stage s (see top of
// file); tree is a doubled tree.
__device__ __forceinline__ uint32_t stage_twiddle(const uint32_t* __restrict__ tree, uint32_t tree_len,
                                                  uint32_t log_n, uint32_t s, uint32_t idx0) {
  if (s == 0) return circle_twiddle(tree + tree_len - (1u << (log_n - 1)), idx0 >> 1);
  return tree[tree_len - (1u << (log_n - s)) + (idx0 >> (s + 1))];
}

// One round of R consecutive stages (local bits j0 .. j0+R-1 of t) on 2^R elements held in
// registers: 2^(R-1) * R butterflies, one twiddle per distinct butterfly block.
template <bool INV, int R>
__device__ __forceinline__ void radix_round(uint32_t* lds, uint32_t C, uint32_t c, uint32_t e, uint32_t j0,
                                            uint32_t base, uint32_t tile_n, const uint32_t* __restrict__ tree,
                                            uint32_t tree_len, uint32_t log_n) {
  constexpr uint32_t G = 1u << R;
  const uint32_t n_groups = tile_n >> R;
  for (uint32_t g = threadIdx.x; g < n_groups; g += blockDim.x) {
    uint32_t lo = g & (C - 1), r = g >> c;
    // t with R zero bits inserted at j0
    uint32_t t0 = ((r >> j0) << (j0 + R)) | (r & ((1u << j0) - 1));
    uint32_t v[G];
#pragma unroll
    for (uint32_t q = 0; q < G; ++q) v[q] = lds[(t0 | (q << j0)) * C + lo];
    const uint32_t idx_base = base | (t0 << e) | lo;
#pragma unroll
    for (int kk = 0; kk < R; ++kk) {
      const int k = INV ? kk : R - 1 - kk;  // bit within the group
      const uint32_t s = e + j0 + k;
      // the twiddle depends only on the group bits above k: 2^(R-1-k) distinct values
#pragma unroll
      for (uint32_t u = 0; u < (G >> (k + 1)); ++u) {
        uint32_t tw = stage_twiddle(tree, tree_len, log_n, s, idx_base | ((u << (k + 1)) << (j0 + e)));
#pragma unroll
        for (uint32_t l = 0; l < (1u << k); ++l) {
          uint32_t q = (u << (k + 1)) | l;
          bfly<INV>(v[q], v[q | (1u << k)], tw);
        }
      }
    }
#pragma unroll
    for (uint32_t q = 0; q < G; ++q) lds[(t0 | (q << j0)) * C + lo] = v[q];
  }
}

template <bool INV>
__global__ void __launch_bounds__(256) fft_pass_kernel(ColSet src, ColSet dst, uint32_t log_n,
                                                       uint32_t in_mask, uint32_t e, uint32_t S, uint32_t c,
                                                       const uint32_t* __restrict__ tree, uint32_t tree_len,
                                                       uint32_t scale, uint32_t prio) {
  if (prio) CRITICAL_PATH_WAVE();
  extern __shared__ uint32_t lds[];
  const uint32_t col = blockIdx.y;
  const GLOBAL_AS uint32_t* __restrict__ in = col_in(src, col);
  GLOBAL_AS uint32_t* __restrict__ out = col_out(dst, col);
  const uint32_t C = 1u << c;
  const uint32_t tile = blockIdx.x;
  const uint32_t lo_blk = tile & ((1u << (e - c)) - 1);
  const uint32_t hi = tile >> (e - c);
  const uint32_t base = (hi << (e + S)) | (lo_blk << c);
  const uint32_t tile_n = 1u << (S + c);
  for (uint32_t l = threadIdx.x; l < tile_n; l += blockDim.x) {
    uint32_t t = l >> c, lo = l & (C - 1);
    lds[l] = in[(base | (t << e) | lo) & in_mask];
  }
  __syncthreads();
  // stages in rounds of up to 3: ascending for the inverse transform, descending for the forward
  uint32_t done = 0;
  while (done < S) {
    uint32_t R = S - done < 3 ? S - done : 3;
    uint32_t j0 = INV ? done : S - done - R;
    if (R == 3) radix_round<INV, 3>(lds, C, c, e, j0, base, tile_n, tree, tree_len, log_n);
    else if (R == 2) radix_round<INV, 2>(lds, C, c, e, j0, base, tile_n, tree, tree_len, log_n);
    else radix_round<INV, 1>(lds, C, c, e, j0, base, tile_n, tree, tree_len, log_n);
    done += R;
    __syncthreads();
  }
  for (uint32_t l = threadIdx.x; l < tile_n; l += blockDim.x) {
    uint32_t t = l >> c, lo = l & (C - 1);
    uint32_t v = lds[l];
    out[base | (t << e) | lo] = scale ? mul_tw(v, scale) : v;
  }
}

// ---- high stages in registers ------------------------------------------------------------------
// Stages [e, e + S) of a transform whose low e >= 11 stages are done: a lane owns the 2^S values
// at hi 2^(e+S) + t 2^e + lo (t < 2^S) and runs all S stages on them in registers. The 64 lanes of
// a wave take 64 consecutive lo, so each of a lane's loads and stores is one 256-byte segment of the
// wave, and every twiddle (index (hi 2^(S-1-j)) + (t >> (j + 1)) at stage e + j) is the same for the
// whole wave: a scalar load. No LDS and no barrier.
template <bool INV, int S>
__global__ void __launch_bounds__(256) fft_pass_reg_kernel(ColSet src, ColSet dst, uint32_t log_n,
                                                           uint32_t in_mask, uint32_t e,
                                                           const uint32_t* __restrict__ tree, uint32_t tree_len,
                                                           uint32_t scale, uint32_t prio) {
  if (prio) CRITICAL_PATH_WAVE();
  const uint32_t col = blockIdx.y;
  const GLOBAL_AS uint32_t* __restrict__ in = col_in(src, col);
  GLOBAL_AS uint32_t* __restrict__ out = col_out(dst, col);
  const uint32_t g = blockIdx.x * blockDim.x + threadIdx.x;
  const uint32_t lo = g & ((1u << e) - 1);
  const uint32_t hi = __builtin_amdgcn_readfirstlane(g >> e);  // e >= 6: one value per wave
  const uint32_t base = (hi << (e + S)) | lo;
  uint32_t v[1 << S];
#pragma unroll
  for (uint32_t t = 0; t < (1u << S); ++t) v[t] = in[(base | (t << e)) & in_mask];
#pragma unroll
  for (int jj = 0; jj < S; ++jj) {
    const int j = INV ? jj : S - 1 - jj;  // the inverse ascends the stages, the forward descends
    const uint32_t* __restrict__ row = tree + (tree_len - (1u << (log_n - e - j)));
#pragma unroll
    for (uint32_t u = 0; u < (1u << (S - 1 - j)); ++u) {
      const uint32_t tw = row[(hi << (S - 1 - j)) | u];
#pragma unroll
      for (uint32_t l = 0; l < (1u << j); ++l) {
        const uint32_t q = (u << (j + 1)) | l;
        bfly<INV>(v[q], v[q | (1u << j)], tw);
      }
    }
  }
#pragma unroll
  for (uint32_t t = 0; t < (1u << S); ++t) {
    const uint32_t x = v[t];
    out[base | (t << e)] = scale ? mul_tw(x, scale) : x;
  }
}
constexpr uint32_t PASS_REG_MAX = 6;  // stages per register pass (2^S values per lane)

// ---- low stages of a 2^S-element block in one pass (11 <= S <= 15) ---------------------------
// A workgroup of 2^(S-5) threads owns one block (tile) of 2^S consecutive elements of one column
// and runs stages [0, S) on it as three rounds (bits 0-4, 5-9, 10..S-1); in a round each thread
// holds 32 elements in registers, as doubles (butterfly.h), and runs up to 5 stages on them. The
// first round reads its elements straight from global memory and the last round writes its results
// straight back; the hand-overs between rounds go through LDS as 32-bit words (pack_f64), where word
// e lives at e + e/32 so that every round's accesses are free of bank conflicts.
//
// In the rounds at bits 0 and 5 a wave owns the same 2048 consecutive elements, so the hand-over
// between them stays inside the wave: no workgroup barrier, only the one between the rounds at bits
// 5 and 10.
//
// Workgroups go to the 8 XCDs in turn (workgroup n to XCD n mod 8). Renumbering them so that each
// XCD takes a contiguous range of tiles keeps the tiles of one column on one XCD and its L2: when
// evaluation onto a larger domain makes every tile of a column read the same coefficients, only
// the first read reaches HBM.
__device__ __forceinline__ uint32_t lds_pad(uint32_t e) { return e + (e >> 5); }

// Threads per workgroup for a tile of 2^S elements, 32 per thread.
template <int S> constexpr uint32_t LOW_T = 1u << (S - 5);

// In the round at bit A a lane's register slot g 2^R + q holds the element
// lane_elem + g LOW_T + (q << A) (g > 0 in rounds at bit 10 of fewer than 5 stages only). All slots of a
// lane sit at fixed distances, in the tile and in LDS, so that an access is one base address and an
// immediate offset.
template <int A> __device__ __forceinline__ uint32_t lane_elem(uint32_t t) {
  return A == 0 ? t << 5 : A == 5 ? ((t >> 5) << 10) | (t & 31) : t;
}
template <int S, int A> __device__ __forceinline__ constexpr uint32_t slot_lds(uint32_t g, uint32_t q) {
  return g * (LOW_T<S> + (LOW_T<S> >> 5)) + q * (A == 0 ? 1u : (1u << A) + (1u << A >> 5));
}

// Orders a wave's LDS writes before its later LDS reads (other lanes' words): the LDS serves a wave's
// accesses in order, so only the compiler has to be held back.
__device__ __forceinline__ void wave_lds_fence() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

template <int S, int A, int R>
__device__ __forceinline__ void round_from_lds(double* w, const uint32_t* lds, uint32_t t) {
  const uint32_t* b = lds + lds_pad(lane_elem<A>(t));
#pragma unroll
  for (uint32_t g = 0; g < (1u << (5 - R)); ++g)
#pragma unroll
    for (uint32_t q = 0; q < (1u << R); ++q) w[(g << R) + q] = (double)b[slot_lds<S, A>(g, q)];
}
template <int S, int A, int R>
__device__ __forceinline__ void round_to_lds(const double* w, uint32_t* lds, uint32_t t) {
  uint32_t* b = lds + lds_pad(lane_elem<A>(t));
#pragma unroll
  for (uint32_t g = 0; g < (1u << (5 - R)); ++g)
#pragma unroll
    for (uint32_t q = 0; q < (1u << R); ++q) b[slot_lds<S, A>(g, q)] = pack_f64(w[(g << R) + q]);
}
// The round at bit 10 reads and writes its elements in rows of 2^(S-5) lanes: a buffer access takes
// the lane offset in a vector register and the slot's in a scalar one, with no vector address
// arithmetic.
// A raw buffer over `words` words at p: past them, loads read 0 and stores are dropped. Address and
// size are the same for the whole wave: said so, they stay in scalar registers.
__device__ __forceinline__ __amdgpu_buffer_rsrc_t tile_rsrc(const GLOBAL_AS uint32_t* p, uint32_t words) {
  const uint64_t a = (uint64_t)p;
  const uint64_t lo = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)a);
  const uint64_t hi = (uint32_t)__builtin_amdgcn_readfirstlane((uint32_t)(a >> 32));
  return __builtin_amdgcn_make_buffer_rsrc((void*)(hi << 32 | lo), (short)0,
                                           (int)__builtin_amdgcn_readfirstlane(words * 4u), 0x00020000);
}
template <int S>
__device__ __forceinline__ void load_round10(uint32_t* v, const GLOBAL_AS uint32_t* in, uint32_t t) {
  constexpr int R = S - 10;
  const __amdgpu_buffer_rsrc_t rs = tile_rsrc(in, 1u << S);
#pragma unroll
  for (uint32_t g = 0; g < (1u << (5 - R)); ++g)
#pragma unroll
    for (uint32_t q = 0; q < (1u << R); ++q)
      v[(g << R) + q] = __builtin_amdgcn_raw_buffer_load_b32(rs, t * 4u, (g * LOW_T<S> + (q << 10)) * 4u, 0);
}
template <int S>
__device__ __forceinline__ void store_round10(const uint32_t* v, GLOBAL_AS uint32_t* out, uint32_t out_words, uint32_t t) {
  constexpr int R = S - 10;
  const __amdgpu_buffer_rsrc_t rs = tile_rsrc(out, out_words);
#pragma unroll
  for (uint32_t g = 0; g < (1u << (5 - R)); ++g)
#pragma unroll
    for (uint32_t q = 0; q < (1u << R); ++q)
      __builtin_amdgcn_raw_buffer_store_b32(v[(g << R) + q], rs, t * 4u, (g * LOW_T<S> + (q << 10)) * 4u, 0);
}
// 16-byte accesses to columns that may be aligned to 4 bytes only: the device takes them at any word.
typedef u32x4 u32x4_w __attribute__((aligned(4)));
// The round at bit 0 reads 32 consecutive elements per lane.
__device__ __forceinline__ void load_round0(uint32_t* v, const GLOBAL_AS uint32_t* in, uint32_t t) {
  const GLOBAL_AS u32x4_w* b = reinterpret_cast<const GLOBAL_AS u32x4_w*>(in + (t << 5));
#pragma unroll
  for (uint32_t m = 0; m < 8; ++m) {
    const u32x4 x = b[m];
    v[4 * m] = x.x; v[4 * m + 1] = x.y; v[4 * m + 2] = x.z; v[4 * m + 3] = x.w;
  }
}
__device__ __forceinline__ void to_f64(double* w, const uint32_t* v) {
#pragma unroll
  for (uint32_t i = 0; i < 32; ++i) w[i] = (double)v[i];
}
// A last round's results, canonical; rot != 0 multiplies them by 2^rot, which rotates the 31-bit word
// (2^-log_n is 2^(31 - log_n)).
__device__ __forceinline__ void canon_words(uint32_t* v, const double* w, uint32_t rot) {
#pragma unroll
  for (uint32_t i = 0; i < 32; ++i) v[i] = canon_f64(w[i]);
  if (rot) {
#pragma unroll
    for (uint32_t i = 0; i < 32; ++i) v[i] = m31_rotl(v[i], rot);
  }
}
// The results of a last round at bit 0, canonical. A lane holds 32 consecutive words, and storing them
// from there would put 64 pieces of 16 bytes into 64 lines with every instruction. They cross the
// wave's own part of LDS instead (its 2048 words; 16-byte unit c of lane l at unit 8 l + (c ^ (l & 7)),
// free of bank conflicts both ways), so that an instruction stores 1 KB in a row: memory traffic alone,
// 497 MB, 92 us against 123. Streaming stores (aux 2): nothing of the tile is read again by this
// kernel, and the traffic alone takes 73 us.
__device__ __forceinline__ u32x4* wave_units(uint32_t* lds, uint32_t t) {
  return reinterpret_cast<u32x4*>(lds + lds_pad((t & ~63u) << 5));
}
__device__ __forceinline__ void round0_stage_out(const double* w, uint32_t* lds, uint32_t t) {
  uint32_t v[32];
  canon_words(v, w, 0);
  const uint32_t l = t & 63;
  u32x4* own = wave_units(lds, t);
#pragma unroll
  for (uint32_t c = 0; c < 8; ++c) own[8 * l + (c ^ (l & 7))] = u32x4{v[4 * c], v[4 * c + 1], v[4 * c + 2], v[4 * c + 3]};
  wave_lds_fence();
}
__device__ __forceinline__ void store_round0(uint32_t* lds, GLOBAL_AS uint32_t* out, uint32_t out_words, uint32_t t) {
  const uint32_t l = t & 63, r = l >> 3;  // unit (l & 7) of lane 8 k + r
  const u32x4* own = wave_units(lds, t);
  const __amdgpu_buffer_rsrc_t rs = tile_rsrc(out, out_words);
  const uint32_t base = __builtin_amdgcn_readfirstlane((t & ~63u) << 5);
#pragma unroll
  for (uint32_t k = 0; k < 8; ++k)
    __builtin_amdgcn_raw_buffer_store_b128(own[8 * (8 * k + r) + ((l & 7) ^ r)], rs, l * 16u, (base + 256 * k) * 4u, 2);
}

// Twiddles. Stage s >= 1 of the pair whose lower element is idx reads entry idx >> (s + 1) of the
// 2^(log_n - s) entries that end the tree (tree.end - 2^(log_n - s)).
//
// The round at bit 10: the lanes own bits below the round, so the workgroup shares its twiddles, and
// they come as doubles through the scalar cache.
template <bool INV, int S, int R>
__device__ __forceinline__ void round10_butterflies(double* w, uint32_t gbase, const double* __restrict__ td_end,
                                                    uint32_t log_n, double M) {
  constexpr uint32_t G = 1u << (5 - R), Q = 1u << R;
#pragma unroll
  for (int kk = 0; kk < R; ++kk) {
    const int k = INV ? kk : R - 1 - kk;
    const uint32_t s = 10 + k;
#pragma unroll
    for (uint32_t g = 0; g < G; ++g) {
      // group g's lanes: bits 0..9 and, for tiles below 2^15, none above the round (T G = 2^10)
      const double* tb = td_end - (1u << (log_n - s)) + __builtin_amdgcn_readfirstlane(gbase >> (s + 1));
#pragma unroll
      for (uint32_t u = 0; u < (Q >> (k + 1)); ++u) {
        const double tw = tb[u];
#pragma unroll
        for (uint32_t l = 0; l < (1u << k); ++l) {
          const uint32_t q = (u << (k + 1)) | l;
          bfly_f64<INV>(w[g * Q + q], w[g * Q + (q | (1u << k))], tw, M);
        }
      }
    }
  }
}

// The round at bit 5: 31 twiddles for each 2^10 consecutive elements, which are half a wave, kept in
// LDS: those of stage 5 + k of block b at [33 b + 2^(4-k), 33 b + 2^(5-k)). Each wave fills the entries
// of its own two blocks, one per lane, so no barrier is needed either.
constexpr uint32_t TW5_STRIDE = 33;
__device__ __forceinline__ double load_tw5(uint32_t gbase, const double* __restrict__ td_end, uint32_t log_n,
                                                uint32_t t) {
  const uint32_t b = t >> 5, j = t & 31;
  const uint32_t lg = j ? 31u - __builtin_clz(j) : 0u, s = 9 - lg;  // stage 5 + k with k = 4 - lg
  return gmem(td_end)[(int)((gbase >> (s + 1)) + (b << lg) + (j ? j - (1u << lg) : 0u)) - (1 << (log_n - s))];
}
__device__ __forceinline__ void store_tw5(double* tw5, double x, uint32_t t) {
  tw5[TW5_STRIDE * (t >> 5) + (t & 31)] = x;  // entry 0 of a block is not read
}
template <bool INV>
__device__ __forceinline__ void round5_butterflies(double* w, const double* tw5, double M, uint32_t t) {
  const double* tb = tw5 + TW5_STRIDE * (t >> 5);
#pragma unroll
  for (int kk = 0; kk < 5; ++kk) {
    const int k = INV ? kk : 4 - kk;
#pragma unroll
    for (uint32_t u = 0; u < (16u >> k); ++u) {
      const double tw = tb[(16u >> k) + u];
#pragma unroll
      for (uint32_t l = 0; l < (1u << k); ++l) {
        const uint32_t q = (u << (k + 1)) | l;
        bfly_f64<INV>(w[q], w[q | (1u << k)], tw, M);
      }
    }
  }
}

// The round at bit 0: a lane's own twiddles, as words (converted where they are used). Stage 0's pairs
// [x, y] (each for four circle pairs, whose twiddles are y, -y, -x, x: the negated ones become swapped
// additions), then those of stages 1..4 (8 + 4 + 2 + 1, stage k from 16 - 2^(5-k)).
struct Round0Tw {
  u32x4 c[2];
  u32x4 t1[2], t2;
  u32x2 t3;
  uint32_t t4;
};
__device__ __forceinline__ void load_round0_tw(Round0Tw& tw, uint32_t gbase, const uint32_t* __restrict__ t_end,
                                               uint32_t log_n, uint32_t t) {
  // the lane's first element is a multiple of 32, so every group of entries is aligned to its size
  const uint32_t idx = gbase | (t << 5);
  const auto at = [&](uint32_t s) { return gmem(t_end) - (1u << (log_n - s)) + (idx >> (s + 1)); };
  const GLOBAL_AS uint32_t* c = gmem(t_end) - (1u << (log_n - 1)) + 2 * (idx >> 3);
  tw.c[0] = *reinterpret_cast<const GLOBAL_AS u32x4*>(c);
  tw.c[1] = *reinterpret_cast<const GLOBAL_AS u32x4*>(c + 4);
  tw.t1[0] = *reinterpret_cast<const GLOBAL_AS u32x4*>(at(1));
  tw.t1[1] = *reinterpret_cast<const GLOBAL_AS u32x4*>(at(1) + 4);
  tw.t2 = *reinterpret_cast<const GLOBAL_AS u32x4*>(at(2));
  tw.t3 = *reinterpret_cast<const GLOBAL_AS u32x2*>(at(3));
  tw.t4 = *at(4);
}
template <bool INV>
__device__ __forceinline__ void round0_butterflies(double* w, const Round0Tw& tw, double M) {
#pragma unroll
  for (int kk = 0; kk < 5; ++kk) {
    const int k = INV ? kk : 4 - kk;
    if (k == 0) {
#pragma unroll
      for (uint32_t u = 0; u < 4; ++u) {
        const double x = (double)tw.c[u >> 1][2 * (u & 1)], y = (double)tw.c[u >> 1][2 * (u & 1) + 1];
        bfly_f64<INV, false>(w[8 * u], w[8 * u + 1], y, M);
        bfly_f64<INV, true>(w[8 * u + 2], w[8 * u + 3], y, M);
        bfly_f64<INV, true>(w[8 * u + 4], w[8 * u + 5], x, M);
        bfly_f64<INV, false>(w[8 * u + 6], w[8 * u + 7], x, M);
      }
      continue;
    }
#pragma unroll
    for (uint32_t u = 0; u < (16u >> k); ++u) {
      const double t = (double)(k == 1 ? tw.t1[u >> 2][u & 3] : k == 2 ? tw.t2[u & 3] : k == 3 ? tw.t3[u & 1] : tw.t4);
#pragma unroll
      for (uint32_t l = 0; l < (1u << k); ++l) {
        const uint32_t q = (u << (k + 1)) | l;
        bfly_f64<INV>(w[q], w[q | (1u << k)], t, M);
      }
    }
  }
}

// F64_ROUND31 in a vector register: a fused multiply-add takes one scalar operand, the twiddle.
__device__ __forceinline__ double round31_reg() {
  double M = F64_ROUND31;
  asm volatile("" : "+v"(M));
  return M;
}

// The kernel loops over tiles. A wave ends only when its stores are done, so with one tile per
// workgroup the stores of a CU's tiles held its slots (1264 columns of 2^15 onto 2^16: 205 us). In the
// loop a tile's loads are issued ahead of the previous tile's stores; vector memory operations complete
// in issue order, so the wait for the loads leaves the stores in flight, and both pass under the other
// waves' arithmetic: 184 us (the 32-bit kernel of before, its loads prefetched into registers: 243).
// Bound by the VALU: about 1870 issue slots per lane and tile of 2^15, 157 us of these 184 with loads
// and stores left out.
//
// The tiles are split into 8 contiguous ranges, one per XCD, and the workgroups of an XCD take its
// tiles in turn, so all waves of a workgroup meet the same barriers. 4 waves per SIMD: LDS holds 2^15
// values (and their padding), 32 a lane.
template <bool INV, int S>
__global__ void __launch_bounds__(LOW_T<S>, 4) fft_low_kernel(ColSet src, ColSet dst, uint32_t log_n,
                                                              uint32_t in_mask, const uint32_t* __restrict__ t_end,
                                                              const double* __restrict__ td_end, uint32_t rot,
                                                              uint32_t prio, uint32_t n_tiles) {
  if (prio) CRITICAL_PATH_WAVE();
  constexpr uint32_t N = 1u << S;
  __shared__ __align__(16) uint32_t lds[N + (N >> 5)];
  __shared__ double tw5[TW5_STRIDE * (LOW_T<S> >> 5)];
  const bool split = (gridDim.x & 7) == 0;
  const uint32_t step = split ? gridDim.x >> 3 : gridDim.x, xcd = blockIdx.x & 7;
  const uint32_t tile_end = split ? (uint32_t)(((uint64_t)n_tiles * (xcd + 1)) >> 3) : n_tiles;
  uint32_t tile = split ? (uint32_t)(((uint64_t)n_tiles * xcd) >> 3) + (blockIdx.x >> 3) : blockIdx.x;
  if (tile >= tile_end) return;
  const uint32_t blk_log = log_n - S, blk_mask = (1u << blk_log) - 1;
  const double M = round31_reg();
  // The previous tile's results: the inverse's in r, the forward's in LDS. Before the first tile the
  // stores run all the same, to a buffer of no words, which drops them: on a second path without them
  // the compiler could not count the stores that its waits may leave in flight.
  uint32_t r[32];
#pragma unroll
  for (uint32_t i = 0; i < 32; ++i) r[i] = 0;
  GLOBAL_AS uint32_t* out = col_out(dst, tile >> blk_log);
  uint32_t out_words = 0;
  const auto store = [&](uint32_t t) {
    if constexpr (INV) store_round10<S>(r, out, out_words, t);
    else store_round0(lds, out, out_words, t);
  };
  for (;; tile += step) {
    const uint32_t gbase = (tile & blk_mask) << S;
    const GLOBAL_AS uint32_t* in = col_in(src, tile >> blk_log) + (gbase & in_mask);  // in_mask >= 2^S - 1
    uint32_t t = threadIdx.x;
    asm volatile("" : "+v"(t));  // keeps the lane's addresses out of registers between the tiles
    double w[32];
    uint32_t v[32];
    Round0Tw tw;
    if constexpr (INV) {
      load_round0(v, in, t);
      load_round0_tw(tw, gbase, t_end, log_n, t);
    } else {
      load_round10<S>(v, in, t);
    }
    const double tw5_in = load_tw5(gbase, td_end, log_n, t);
    asm volatile("" ::: "memory");  // the loads stay ahead of the stores
    store(t);
    to_f64(w, v);
    store_tw5(tw5, tw5_in, t);
    __builtin_amdgcn_sched_barrier(0);
    if constexpr (INV) {
      round0_butterflies<true>(w, tw, M);
      __syncthreads();  // the last tile's reads in the round at bit 10 are done
      round_to_lds<S, 0, 5>(w, lds, t);
      wave_lds_fence();
      __builtin_amdgcn_sched_barrier(0);
      round_from_lds<S, 5, 5>(w, lds, t);
      round5_butterflies<true>(w, tw5, M, t);
      round_to_lds<S, 5, 5>(w, lds, t);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
      round_from_lds<S, 10, S - 10>(w, lds, t);
      round10_butterflies<true, S, S - 10>(w, gbase, td_end, log_n, M);
      canon_words(r, w, rot);
    } else {
      round10_butterflies<false, S, S - 10>(w, gbase, td_end, log_n, M);
      __syncthreads();  // the last tile's words have left LDS
      round_to_lds<S, 10, S - 10>(w, lds, t);
      __syncthreads();
      __builtin_amdgcn_sched_barrier(0);
      load_round0_tw(tw, gbase, t_end, log_n, t);
      round_from_lds<S, 5, 5>(w, lds, t);
      round5_butterflies<false>(w, tw5, M, t);
      round_to_lds<S, 5, 5>(w, lds, t);
      wave_lds_fence();
      __builtin_amdgcn_sched_barrier(0);
      round_from_lds<S, 0, 5>(w, lds, t);
      round0_butterflies<false>(w, tw, M);
      round0_stage_out(w, lds, t);
    }
    __builtin_amdgcn_sched_barrier(0);
    out = col_out(dst, tile >> blk_log) + gbase;
    out_words = N;
    if (tile + step >= tile_end) return store(t);
  }
}

// Foreground transforms run as many workgroups as the device holds at once, each looping over tiles;
// a background one has a workgroup per tile, so that the kernels beside it get CUs as its tiles end (a
// grid that holds every CU until the transform is done doubled the time of the trace's Merkle tree). Four
// contexts proving at once do not tell the two forms apart (694-718 proofs/s and p99 7.7-8.2 ms with the
// resident grid, 692-718 and 8.1-8.6 with a workgroup per tile); a lone one is 1-2 % faster with it.
template <bool INV, int S>
static void launch_low_tile(uint32_t n_cols, ColSet src, ColSet dst, uint32_t log_n,
                            uint32_t in_mask, const FftTree& tree, uint32_t rot, uint32_t prio, int cus,
                            hipStream_t stream) {
  const uint32_t n_tiles = n_cols << (log_n - S), resident = (uint32_t)(cus > 8 ? cus / 8 * 8 : 8) << (15 - S);
  const uint32_t grid = prio && n_tiles > resident ? resident : n_tiles;
  hipLaunchKernelGGL((fft_low_kernel<INV, S>), dim3(grid), dim3(LOW_T<S>), 0, stream, src, dst, log_n, in_mask,
                     tree.t + tree.len, tree.td_end, rot, prio, n_tiles);
}
template <bool INV>
static void launch_low(uint32_t S, uint32_t n_cols, ColSet src, ColSet dst, uint32_t log_n,
                       uint32_t in_mask, const FftTree& tree, uint32_t rot, uint32_t prio, int cus, hipStream_t stream) {
  switch (S) {
    case 11: return launch_low_tile<INV, 11>(n_cols, src, dst, log_n, in_mask, tree, rot, prio, cus, stream);
    case 12: return launch_low_tile<INV, 12>(n_cols, src, dst, log_n, in_mask, tree, rot, prio, cus, stream);
    case 13: return launch_low_tile<INV, 13>(n_cols, src, dst, log_n, in_mask, tree, rot, prio, cus, stream);
    case 14: return launch_low_tile<INV, 14>(n_cols, src, dst, log_n, in_mask, tree, rot, prio, cus, stream);
    default: return launch_low_tile<INV, 15>(n_cols, src, dst, log_n, in_mask, tree, rot, prio, cus, stream);
  }
}

// Host-side pass planning shared by interpolate and evaluate.
struct FftPass { uint32_t e, S, c; };
static std::vector<FftPass> plan_passes(uint32_t k, uint32_t K) {
  // stages [0, k) split into a contiguous first chunk and strided higher chunks
  std::vector<FftPass> p;
  const uint32_t TILE_LOG = 12;
  uint32_t first = k < TILE_LOG ? k : TILE_LOG;
  p.push_back({0, first, 0});
  uint32_t e = first;
  while (e < k) {
    uint32_t S = k - e;
    if (S > 8) S = 8;
    uint32_t c = TILE_LOG - S;
    if (c > e) c = e;
    // the tile must fit in the column: S + c <= K
    p.push_back({e, S, c});
    e += S;
  }
  (void)K;
  return p;
}

void launch_fft(bool inverse, ColSet src, ColSet dst, uint32_t n_cols, uint32_t log_in,
                uint32_t log_n, const FftTree& ft, int cus, hipStream_t stream, bool background, uint32_t low_log) {
  if (n_cols == 0) return;
  const uint32_t prio = background ? 0u : 1u;
  const uint32_t* const tree = ft.t2;
  const uint32_t tree_len = ft.len;
  const uint32_t k = inverse ? log_n : log_in;  // number of stages actually run
  const uint32_t inv_n = inverse ? 2 * m31_inv(1u << log_n) : 0;  // doubled, as the twiddles
  auto run_pass = [&](const FftPass& ps, const ColSet& from, uint32_t mask, uint32_t scale) {
    if (ps.c == ~0u) {  // a register pass (after the low stages: e >= 11, 2^(log_n - S) >= 256 lanes)
      const dim3 grid(1u << (log_n - ps.S - 8), n_cols), block(256);
#define PASS_REG(SS)                                                                                            \
  case SS:                                                                                                      \
    if (inverse)                                                                                                \
      hipLaunchKernelGGL((fft_pass_reg_kernel<true, SS>), grid, block, 0, stream, from, dst, log_n, mask, ps.e, \
                         tree, tree_len, scale, prio);                                                          \
    else                                                                                                        \
      hipLaunchKernelGGL((fft_pass_reg_kernel<false, SS>), grid, block, 0, stream, from, dst, log_n, mask,      \
                         ps.e, tree, tree_len, scale, prio);                                                    \
    break;
      switch (ps.S) {
        PASS_REG(1) PASS_REG(2) PASS_REG(3) PASS_REG(4) PASS_REG(5) PASS_REG(6)
        default: throw std::invalid_argument("launch_fft: register pass of more than 6 stages");
      }
#undef PASS_REG
      return;
    }
    const uint32_t tiles = 1u << (log_n - ps.S - ps.c), tile_n = 1u << (ps.S + ps.c);
    const uint32_t threads = tile_n / 2 < 64 ? 64 : (tile_n / 2 > 256 ? 256 : tile_n / 2);
    if (inverse)
      hipLaunchKernelGGL(fft_pass_kernel<true>, dim3(tiles, n_cols), dim3(threads), tile_n * 4, stream, from, dst,
                         log_n, mask, ps.e, ps.S, ps.c, tree, tree_len, scale, prio);
    else
      hipLaunchKernelGGL(fft_pass_kernel<false>, dim3(tiles, n_cols), dim3(threads), tile_n * 4, stream, from, dst,
                         log_n, mask, ps.e, ps.S, ps.c, tree, tree_len, scale, prio);
  };
  const uint32_t full = (1u << log_n) - 1, in_mask = inverse ? full : (1u << log_in) - 1;
  if (k >= 11) {
    // stages [0, S) in one pass of 2^S-element blocks; stages [S, k) in strided passes
    const uint32_t smax = k < 15 ? k : 15;
    if (low_log != 0 && (low_log < 11 || low_log > smax)) throw std::invalid_argument("launch_fft: low_log out of range");
    const uint32_t S = low_log ? low_log : smax;
    // the stages above the low tile: register passes of at most PASS_REG_MAX stages, as even as
    // the count allows (8 stages: 4 + 4, not 6 + 2)
    std::vector<FftPass> high;
    {
      const uint32_t rest = k - S, n_pass = (rest + PASS_REG_MAX - 1) / PASS_REG_MAX;
      for (uint32_t i = 0, e = S; i < n_pass; ++i) {
        const uint32_t st = (rest - (e - S) + (n_pass - i) - 1) / (n_pass - i);
        high.push_back({e, st, ~0u});
        e += st;
      }
    }
    if (inverse) {
      // 2^-log_n is 2^(31 - log_n): the low stages' own scaling is a rotation
      launch_low<true>(S, n_cols, src, dst, log_n, full, ft, high.empty() ? 31 - log_n : 0u, prio, cus, stream);
      for (size_t i = 0; i < high.size(); ++i)
        run_pass(high[i], dst, full, i + 1 == high.size() ? inv_n : 0u);
    } else {
      for (size_t ii = high.size(); ii-- > 0;)
        run_pass(high[ii], ii + 1 == high.size() ? src : dst,
                 ii + 1 == high.size() ? in_mask : full, 0u);
      launch_low<false>(S, n_cols, high.empty() ? src : dst, dst, log_n,
                        high.empty() ? in_mask : full, ft, 0u, prio, cus, stream);
    }
    return;
  }
  auto passes = plan_passes(k, log_n);
  if (inverse) {
    for (size_t i = 0; i < passes.size(); ++i)
      run_pass(passes[i], i == 0 ? src : dst, full, i + 1 == passes.size() ? inv_n : 0u);
  } else {
    for (size_t ii = passes.size(); ii-- > 0;) {
      const bool first = ii + 1 == passes.size();
      run_pass(passes[ii], first ? src : dst, first ? in_mask : full, 0u);
    }
  }
}

}  // namespace sh
