// Additive masks for gfx950: what kind of mask it is, and the pair bits of a mask that only drops pairs.
//
// The eager branch adds its mask to the scaled logits (torchprime/torch_xla_models/attention.py:151-158).  The masks
// models build are causality, padding, or both: every entry is 0 or "minus infinity" (-inf, or the lowest value of the
// data type).  Evaluating such a mask element by element as a fp32 tensor in every tile of every head (the general
// attention kernels) cost five to ten times what the tiles themselves cost; as one bit per pair, with the tiles that
// hold no pair left out and those that hold all pairs unmasked, it costs the causal kernels' own time.
//
// A dropped pair must leave no trace in the softmax: its entry is at most Dropped<T>, and the row has a pair with entry
// 0 (a row of dropped finite entries only is a uniform distribution in the eager formula; the verdict sends such masks to
// the general kernels).  -1e30 is out of reach of any logit.  float16 has only -65504 to fill a mask with: there the
// pair drops out because the eager formula forms q.k in float16 before it scales by 1/sqrt(d), d >= 64: where that does
// not overflow, scaled logits lie within 65504 / 8 of 0, two of them differ by at most 16376, and exp(16376 - 65504) is
// 0 in float32 (callers take this only for float16 q / k and that scale).
#include "attn_common.hpp"

namespace tp {

template <typename T> constexpr float Dropped = -1e30f;
template <> constexpr float Dropped<f16_t> = -65504.f;
// flags[]: entries that are neither 0 nor dropped; entries that differ from the exact causal mask (0 / -inf); rows
// without a pair whose entries are not all -inf; pairs that are not the causal ones less rows and keys as a whole (padding)
constexpr int F_OTHER = 0, F_NOT_CAUSAL = 1, F_EMPTY_FINITE = 2, F_NOT_PADDED = 3;

// One wave per 64 x 64 block.  Lane r reads its row's 64 entries, 128 or 256 contiguous bytes, in 16-byte loads that are
// all in flight together, and builds the row's word; the columns' words are 64 ballots over the rows' words.  (A lane
// per column with 64 row reads one after the other, two bytes a lane, took 15-37 us at the sizes below.)  The last tile of
// a row is read the same way (entries one by one : this, us: 8 masks of 361 x 361 10.6 : 7.4, 4 of 1000 x 1000 9.9 : 6.9, 8 of
// 2041 x 2041 53 : 31).  Bound by latency below a few thousand rows; words are written 512 contiguous bytes at a time, in the
// order in which the attention kernels fetch them.
template <typename T>
__global__ __launch_bounds__(256) void mask_bits_kernel(const T* __restrict__ mask, int64_t bs, int64_t rs, int Sq, int Skv, int nqt,
                                                        int nkt, int nqb, int nkb, unsigned long long* __restrict__ qbits,
                                                        unsigned long long* __restrict__ kbits, unsigned short* __restrict__ qcls,
                                                        unsigned short* __restrict__ kcls, int* __restrict__ flags) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int kt = blockIdx.x * 4 + wave, qt = blockIdx.y, b = blockIdx.z;
  if (kt >= 2 * nkb) return;
  const int k0 = kt * 64, key = k0 + lane, q0 = qt * 64, row = q0 + lane;
  unsigned long long roww = 0ull;
  bool other = false, ncausal = false;
  if (row < Sq) {
    const T* mr = mask + b * bs + row * rs + k0;
    // entry at + j of the row's part in this tile, as bit j
    auto take = [&](T v, int j, int at, unsigned long long& w) {
      const float x = (float)v;
      const bool keep = !(x <= Dropped<T>);  // (a NaN is kept, and is not 0)
      w |= (unsigned long long)keep << j;
      other = other || (keep && x != 0.f);
      ncausal = ncausal || (k0 + at + j <= row ? x != 0.f : x != -INFINITY);
    };
    constexpr int PER = 16 / sizeof(T);
    typedef T Chunk __attribute__((ext_vector_type(PER), aligned(sizeof(T))));  // (rows are aligned to an entry only)
    if (k0 + 64 <= Skv) {
      Chunk c[64 / PER];
#pragma unroll
      for (int i = 0; i < 64 / PER; i++) c[i] = *(const Chunk*)(mr + i * PER);
#pragma unroll
      for (int j = 0; j < 64; j++) take(c[j / PER][j % PER], j, 0, roww);
    } else if (Skv >= PER && k0 < Skv) {
      // the row's end: no load leaves the row, the last one starts earlier instead (and brings entries again, which changes
      // nothing)
      const int n = Skv - k0, last = n - PER;
      Chunk c[64 / PER];
#pragma unroll
      for (int i = 0; i < 64 / PER; i++)
        if (i * PER < n) c[i] = *(const Chunk*)(mr + min(i * PER, last));
#pragma unroll
      for (int i = 0; i < 64 / PER; i++) {
        if (i * PER < n) {
          const int at = min(i * PER, last);
          unsigned long long w = 0ull;
#pragma unroll
          for (int e = 0; e < PER; e++) take(c[i][e], e, at, w);
          roww |= at >= 0 ? w << at : w >> -at;
        }
      }
    } else {
      for (int j = 0; j < Skv - k0; j++) take(mr[j], j, 0, roww);
    }
  }
  unsigned long long colw = 0ull;
#pragma unroll
  for (int j = 0; j < 64; j++) {
    const unsigned long long w = __ballot((roww >> j) & 1ull);
    colw = lane == j ? w : colw;
  }
  // words: rows up to the padding of the last block of 128
  if (kt < nkt) qbits[((int64_t)b * nkt + kt) * (nqb * 128) + row] = roww;
  if (qt < nqt) kbits[((int64_t)b * nqt + qt) * (nkb * 128) + key] = colw;
  // classes of the two halves of 32 rows: 0 no pair, 2 every pair (rows past the end do not count), 1 otherwise
  auto classes = [&](unsigned long long w, bool past) -> unsigned short {
    const unsigned long long any = __ballot(w != 0ull), full = __ballot(w == ~0ull || past);
    const unsigned a0 = (unsigned)any, a1 = (unsigned)(any >> 32), f0 = (unsigned)full, f1 = (unsigned)(full >> 32);
    return (unsigned short)((a0 == 0u ? 0 : f0 == ~0u ? 2 : 1) | ((a1 == 0u ? 0 : f1 == ~0u ? 2 : 1) << 8));
  };
  const unsigned short qc = classes(roww, row >= Sq), kc = classes(colw, key >= Skv);
  if (lane == 0) {
    if (kt < nkt) qcls[(((int64_t)b * nqb + (qt >> 1)) * nkt + kt) * 2 + (qt & 1)] = qc;
    if (qt < nqt) kcls[(((int64_t)b * nkb + (kt >> 1)) * nqt + qt) * 2 + (kt & 1)] = kc;
  }
  if (flags) {
    // (every writer stores the same value)
    if (__ballot(other) && lane == 0) flags[F_OTHER] = 1;
    if (__ballot(ncausal) && lane == 0) flags[F_NOT_CAUSAL] = 1;
  }
}

// One wave per row: a row without a pair must be -inf throughout; the others of a padded causal mask have no pair above the
// diagonal and, up to the row before, that row's keys (where it has any).
template <typename T>
__global__ __launch_bounds__(256) void mask_rows_kernel(const T* __restrict__ mask, int64_t bs, int64_t rs, int Sq, int Skv, int nkt, int nqb,
                                                        const unsigned long long* __restrict__ qbits, int* __restrict__ flags) {
  const int lane = threadIdx.x & 63, row = blockIdx.x * 4 + (threadIdx.x >> 6), b = blockIdx.y;
  if (row >= Sq) return;
  bool any = false, before = false, above = false, uneven = false;
  for (int t = lane; t < nkt; t += 64) {
    const unsigned long long* at = qbits + ((int64_t)b * nkt + t) * (nqb * 128) + row;
    const unsigned long long w = at[0], p = row > 0 ? at[-1] : 0ull;
    // the first n keys of the tile
    auto first = [](int n) { return n <= 0 ? 0ull : n >= 64 ? ~0ull : (1ull << n) - 1ull; };
    any = any || w != 0ull;
    before = before || p != 0ull;
    above = above || (w & ~first(row + 1 - 64 * t)) != 0ull;
    uneven = uneven || (w & first(row - 64 * t)) != p;
  }
  if (__ballot(any)) {
    const bool other = __ballot(above) || (__ballot(before) && __ballot(uneven));
    if (other && lane == 0) flags[F_NOT_PADDED] = 1;
    return;
  }
  bool finite = false;
  for (int j = lane; j < Skv; j += 64) finite = finite || (float)mask[b * bs + row * rs + j] != -INFINITY;
  if (__ballot(finite) && lane == 0) flags[F_EMPTY_FINITE] = 1;
}

template <typename T>
static int mask_typed(const void* mask, int Bm, int Sq, int Skv, const int64_t* st, void* pairs, bool verdict, hipStream_t stream) {
  const PairLayout l(Bm, Sq, Skv);
  unsigned char* p = (unsigned char*)pairs;
  int* flags = verdict ? (int*)p : nullptr;
  mask_bits_kernel<T><<<dim3((2 * l.nkb + 3) / 4, 2 * l.nqb, Bm), dim3(256), 0, stream>>>(
      (const T*)mask, st[0], st[1], Sq, Skv, l.nqt, l.nkt, l.nqb, l.nkb, (unsigned long long*)(p + l.qbits), (unsigned long long*)(p + l.kbits),
      (unsigned short*)(p + l.qcls), (unsigned short*)(p + l.kcls), flags);
  int rc = check_launch("tp_mask_pairs");
  if (rc || !verdict) return rc;
  mask_rows_kernel<T><<<dim3((Sq + 3) / 4, Bm), dim3(256), 0, stream>>>((const T*)mask, st[0], st[1], Sq, Skv, l.nkt, l.nqb,
                                                                        (const unsigned long long*)(p + l.qbits), flags);
  return check_launch("tp_mask_pairs(verdict)");
}

}  // namespace tp

using namespace tp;

extern "C" size_t tp_mask_pairs_bytes(int mask_batches, int Sq, int Skv) {
  if (mask_batches <= 0 || Sq <= 0 || Skv <= 0) return 0;
  return PairLayout(mask_batches, Sq, Skv).bytes;
}

extern "C" int tp_mask_pairs(const void* mask, const int64_t mask_strides[2], int mask_batches, int Sq, int Skv, int dtype, void* pairs,
                             int verdict, void* stream) {
  TP_REQUIRE(mask && mask_strides && pairs, TP_ERR_BAD_ARG, "tp_mask_pairs: null pointer");
  TP_REQUIRE(mask_batches > 0 && Sq > 0 && Skv > 0, TP_ERR_BAD_ARG, "tp_mask_pairs: non-positive size");
  TP_REQUIRE(mask_strides[0] >= 0 && mask_strides[1] >= 0, TP_ERR_BAD_ARG, "tp_mask_pairs: negative stride");
  TP_REQUIRE(aligned16(pairs), TP_ERR_BAD_ARG, "tp_mask_pairs: pairs must be 16-byte aligned");
  TP_REQUIRE(pair_mask_sizes_ok(mask_batches, Sq, Skv), TP_ERR_UNSUPPORTED, "tp_mask_pairs: mask too large");
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TP_BF16) return mask_typed<bf16_t>(mask, mask_batches, Sq, Skv, mask_strides, pairs, verdict != 0, st);
  if (dtype == TP_F16) return mask_typed<f16_t>(mask, mask_batches, Sq, Skv, mask_strides, pairs, verdict != 0, st);
  if (dtype == TP_F32) return mask_typed<float>(mask, mask_batches, Sq, Skv, mask_strides, pairs, verdict != 0, st);
  TP_REQUIRE(false, TP_ERR_UNSUPPORTED, "tp_mask_pairs: dtype %d", dtype);
}
