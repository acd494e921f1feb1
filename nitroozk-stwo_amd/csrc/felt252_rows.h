// Starknet's Poseidon permutation over the 16 lanes of a DPP row, for layers of few nodes: a node's
// hash is then not one lane's chain of 214 Montgomery products but one whose every product is spread over
// the row. Lane k holds limb k (k = 0..8, radix 2^29, signed: normalized limbs lie within 2^28 + 2^24 of
// zero), lanes 9..15 hold zero between products. Four nodes share a wave.
//
// A product's column k gathers in lane k: step i broadcasts a's limb i to the row and shifts b up by i
// lanes, so nine multiply-adds make columns 0..15 in 64-bit accumulators (column 16, one product, is kept
// in every lane). p = 1 + 17 2^192 + 2^251, so with signed limbs the Montgomery factor of column i is
// simply minus its content, and clearing columns 0..8 is no chain: they vanish, and what the factors add
// elsewhere (17 2^18 six columns up, 2^19 eight columns up) comes in two steps, first for columns 0..5,
// then for 6..8, which depend on them. Carries move by one lane, all lanes at once, between the steps:
// every value fits 32 bits after one of them. Products lie in (-p, p); a product is 65 instructions (57
// when the shifted operand is at hand) against 157 for one lane.
//
// Sums work limb by limb in every lane; carries move once before a product, and the partial rounds'
// recurrence (felt252.h) reduces one value a round. Ranges, checked over extreme limbs and whole
// permutations: accumulators below 2^59.4 (hi words of the first carry below 2^31), sums within 7.1 2^28.
#pragma once
#include "felt252.h"

namespace sh {
namespace f252 {

// Per lane of a row: the round constants, then R^2, the Montgomery forms of 1 and 2, 1, and the Montgomery
// forms of 1/2 and 1/4.
constexpr int ROWS_R2 = 107, ROWS_ONE = 108, ROWS_TWO = 109, ROWS_UNIT = 110,
              ROWS_HALF = 111, ROWS_QUARTER = 112, ROWS_N = 113;
struct RowTable { int32_t v[ROWS_N * 16]; };
constexpr void row_into(RowTable& t, int row, const M& m) {
  for (int i = 0; i < 9; ++i) t.v[16 * row + i] = m.w[i];
}
constexpr RowTable make_row_table() {
  RowTable t{};
  for (int i = 0; i < 107; ++i) row_into(t, i, RC.c[i]);
  row_into(t, ROWS_R2, R2M);
  row_into(t, ROWS_ONE, ONE);
  row_into(t, ROWS_TWO, TWO);
  row_into(t, ROWS_HALF, HALF);
  row_into(t, ROWS_QUARTER, QUARTER);
  t.v[16 * ROWS_UNIT] = 1;
  return t;
}

// DPP within rows of 16: lane k reads lane k - n (or k + n); past the row it reads zero.
template <int CTRL>
__device__ __forceinline__ int32_t row_dpp(int32_t x) {
  return __builtin_amdgcn_update_dpp(0, x, CTRL, 0xF, 0xF, true);
}
template <int N> __device__ __forceinline__ int32_t row_up(int32_t x) {  // from lane k - N
  if constexpr (N == 0) return x;
  else return row_dpp<0x110 + N>(x);
}
template <int N> __device__ __forceinline__ int32_t row_down(int32_t x) { return row_dpp<0x100 + N>(x); }
template <int N> __device__ __forceinline__ int32_t row_bcast(int32_t x) { return row_dpp<0x150 + N>(x); }

struct Row {
  static constexpr int32_t B28 = 1 << 28;
  const int32_t* tab;  // the lane's column of a RowTable
  uint32_t k;          // lane within the row
  int32_t p6a, p8a, p6b, p8b;  // minus p's limbs 6 and 8 in the lanes that take them in the two steps
  int32_t from6;               // all ones in lanes 6..15
  int32_t minus_b28;           // -2^28 in lanes 0..7
  int32_t minus_p;             // minus p's limb k
  uint32_t width;              // bits that a normalized limb keeps: all of the top one's
  int32_t round_up;            // half of what carries
  int32_t minus_p8;            // minus p's limb 8, kept from becoming a 64-bit shift and subtraction
  int64_t bias;                // 2^28, likewise one multiply-add's third operand

  __device__ __forceinline__ Row(const int32_t* table, uint32_t lane) : tab(table + lane), k(lane) {
    constexpr int32_t P6 = 17 << 18, P8 = 1 << 19;
    p6a = k >= 6 && k <= 11 ? -P6 : 0;
    p8a = k >= 8 && k <= 13 ? -P8 : 0;
    p6b = k >= 12 && k <= 14 ? -P6 : 0;
    p8b = k >= 14 ? -P8 : 0;
    from6 = k >= 6 ? -1 : 0;
    minus_b28 = k < 8 ? -B28 : 0;
    minus_p = k == 0 ? -1 : k == 6 ? -P6 : k == 8 ? -P8 : 0;
    width = k < 8 ? 29 : 31;
    round_up = k < 8 ? B28 : 1 << 30;
    minus_p8 = -P8;
    bias = B28;
    asm("" : "+v"(minus_p8), "+s"(bias));
  }
  __device__ __forceinline__ int32_t at(int row) const { return tab[16 * row]; }

  // Carries, by one lane, of limbs within 7 2^28 of zero; the top limb keeps everything.
  __device__ __forceinline__ int32_t carry(int32_t x) const {
    const int32_t lo = __builtin_amdgcn_sbfe(x, 0, width), hi = (x + round_up) >> width;
    return lo + row_up<1>(hi);
  }
  // reduce_top: minus the multiple of p that leaves the top limb near zero, then the carries, of limbs
  // within 7.5 2^28 of zero (the rounded shift in two steps, as adding half could overflow).
  __device__ __forceinline__ int32_t reduce(int32_t x) const {
    const int32_t h = row_bcast<8>((x + (1 << 18)) >> 19);
    const int32_t y = x + __mul24(h, minus_p);
    const int32_t lo = __builtin_amdgcn_sbfe(y, 0, width), hi = ((y >> (width - 1)) + 1) >> 1;
    return lo + row_up<1>(hi);
  }

  struct Shifted { int32_t s[9], top; };  // b moved up by 0..8 lanes, and its top limb in every lane
  __device__ __forceinline__ Shifted shifts(int32_t b) const {
    return {{b, row_up<1>(b), row_up<2>(b), row_up<3>(b), row_up<4>(b), row_up<5>(b), row_up<6>(b), row_up<7>(b),
             row_up<8>(b)}, row_bcast<8>(b)};
  }
  // a b 2^-261 (mod p)
  __device__ __forceinline__ int32_t mul(int32_t a, const Shifted& b) const {
    // every accumulator starts at 2^28, so that shifts and masks split off signed limbs
    int64_t acc = bias + (int64_t)row_bcast<0>(a) * b.s[0];
    acc += (int64_t)row_bcast<1>(a) * b.s[1];
    acc += (int64_t)row_bcast<2>(a) * b.s[2];
    acc += (int64_t)row_bcast<3>(a) * b.s[3];
    acc += (int64_t)row_bcast<4>(a) * b.s[4];
    acc += (int64_t)row_bcast<5>(a) * b.s[5];
    acc += (int64_t)row_bcast<6>(a) * b.s[6];
    acc += (int64_t)row_bcast<7>(a) * b.s[7];
    const int32_t a8 = row_bcast<8>(a);
    acc += (int64_t)a8 * b.s[8];
    int64_t c16 = bias + (int64_t)a8 * b.top;
    constexpr int32_t MASK = (1 << 29) - 1;
    const int32_t h1 = (int32_t)(acc >> 29);
    const int32_t c = ((int32_t)acc & MASK) + row_up<1>(h1);
    const int32_t h2 = c >> 29, db = (c & MASK) + row_up<1>(h2), d = db - B28;
    // the factors of columns 0..5
    const int64_t t = (int64_t)db + (int64_t)row_up<6>(d) * p6a + (int64_t)row_up<8>(d) * p8a;
    const int32_t h3 = (int32_t)(t >> 29) & from6, fb = ((int32_t)t & MASK) + row_up<1>(h3), f = fb - B28;
    // of columns 6..8, and what reaches column 16
    const int64_t g = (int64_t)fb + (int64_t)row_up<6>(f) * p6b + (int64_t)row_up<8>(f) * p8b;
    c16 += (int64_t)row_bcast<15>(h1 + h2 + h3);
    c16 += (int64_t)row_bcast<8>(f) * minus_p8;
    // columns 9..16 are the result's limbs 0..7, their last carry limb 8
    const int32_t glo = row_down<9>((int32_t)g), ghi = row_down<9>((int32_t)(g >> 32));
    const uint32_t rlo = k == 7 ? (uint32_t)c16 : (uint32_t)glo, rhi = k == 7 ? (uint32_t)(c16 >> 32) : (uint32_t)ghi;
    const int32_t h4 = (int32_t)__builtin_amdgcn_alignbit(rhi, rlo, 29);
    return (int32_t)(rlo & MASK) + row_up<1>(h4) + minus_b28;
  }
  __device__ __forceinline__ int32_t cube(int32_t x) const {
    const Shifted s = shifts(x);
    return mul(mul(x, s), s);
  }
  __device__ __forceinline__ void full_rounds(int32_t* s, int r) const {
#pragma unroll 1
    for (int i = 0; i < 4; ++i, r += 3) {
#pragma unroll
      for (int j = 0; j < 3; ++j) s[j] = cube(carry(s[j] + at(r + j)));
      const int32_t u = s[0] + s[1], d = s[0] - s[1];
      s[0] = u + s[2] + 2 * s[0];
      s[1] = d + s[2];
      s[2] = u - 2 * s[2];
    }
  }
  // poseidon_permute_comp, as permute() in felt252.h.
  __device__ __forceinline__ void permute(int32_t* s) const {
#pragma unroll
    for (int j = 0; j < 3; ++j) s[j] = carry(s[j]);
    full_rounds(s, 0);
    const int32_t s0 = carry(s[0]), s1 = carry(s[1]);
    int32_t w = mul(carry(s0 + s1), shifts(at(ROWS_HALF))), prev = mul(carry(s0 - s1), shifts(at(ROWS_QUARTER)));
    // w_{n+1} waits unreduced for the next round, whose product has idle slots for that
    int32_t rc = at(12);
#pragma unroll 1
    for (int r = 12; r < 95; ++r) {
      const int32_t next = at(r + 1), cur = reduce(w), x = cube(carry(s[2] + rc));
      s[2] = 2 * (cur - x);
      w = 2 * (2 * prev + cur) + x;
      prev = cur;
      rc = next;
    }
    const int32_t last = reduce(w);
    s[0] = last + 2 * prev;
    s[1] = last - 2 * prev;
    full_rounds(s, 95);
  }
  // Limb k of eight words in memory, and of eight words that every lane of the row holds; Montgomery form.
  __device__ __forceinline__ int32_t to_mont(int32_t limb) const { return mul(carry(limb), shifts(at(ROWS_R2))); }
  __device__ __forceinline__ int32_t limb_at(const uint32_t* __restrict__ p) const {
    const uint32_t w = (29 * k) >> 5, sh = (29 * k) & 31;
    const uint32_t lo = k < 9 ? gmem(p)[w] : 0u, hi = k < 8 ? gmem(p)[w + 1] : 0u;
    return (int32_t)(__builtin_amdgcn_alignbit(hi, lo, sh) & MASK29);
  }
  __device__ __forceinline__ int32_t limb_of(const F& f) const {
    const M m = to_radix29(f);
    uint32_t v = 0;
#pragma unroll
    for (uint32_t j = 0; j < 9; ++j) v = k == j ? (uint32_t)m.w[j] : v;
    return (int32_t)v;
  }
  // The canonical value of a state element, in every lane of the row.
  __device__ __forceinline__ F from_mont(int32_t x) const {
    const int32_t y = mul(carry(x), shifts(at(ROWS_UNIT))) - minus_p;  // above -p before p is added
    const M m{{row_bcast<0>(y), row_bcast<1>(y), row_bcast<2>(y), row_bcast<3>(y), row_bcast<4>(y), row_bcast<5>(y),
               row_bcast<6>(y), row_bcast<7>(y), row_bcast<8>(y)}};
    const F r = from_radix29(m);
    return geq_p(r) ? sub_p(r) : r;
  }
};

}  // namespace f252
}  // namespace sh
