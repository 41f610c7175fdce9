// Small matrix products for gfx950: the projections of small models, several in one launch.
//
// What this is for: a projection of a few hundred tokens through a few hundred features is 0.05-0.5 GFLOP, microseconds
// of the matrix pipes, while a GEMM library call costs 18 us of host time for its heuristics and 6-10 us on the device,
// one launch each for q, k and v, for every dX and dW, and for the sums of dX's that meet.  Here up to four products go
// into one launch, and a product may sum over several (A, B) pairs, so that a group of projections with one input (q, k,
// v; gate, up) is one launch forward and one backward (all dW and the summed dX).  512 tokens through three 512 x 512
// weights, bf16: 62 -> 8 us forward, 296 -> 83 us with the backward (host included).  Large products stay with the
// library; the line is drawn where the torch operators choose (lin_max_work in torch_ops.cpp).
//
// C[m, n] = sum_seg sum_k A(m, k) B(n, k).  Either operand is given row-major with the contraction along the row
// (k-major rows: X and W forward, G in dX) or along the column (row k holds m or n contiguously: W in dX, G and X in dW).
// Workgroup = 4 waves = one 64 x 64 tile, a wave 32 x 32.  Per step 64 (16-bit) or 32 (fp32) values of k: two operand tiles
// of 8 KB, written to LDS by the loads themselves into a ring of four steps, three in flight, one barrier a step.  At
// these sizes the chip is latency-bound (64 to 500 workgroups of 1 to 32 steps): the depth of the ring is what matters,
// not the reuse per LDS byte.  The product is formed transposed (MFMA rows = n), so a lane ends up with four consecutive
// n of one row m and stores 8 or 16 bytes.
//
// Where even those workgroups do not cover the chip a few times (up to 1024 tiles of 32 x 32), a workgroup owns one 32 x 32
// tile and its four waves take the steps of the contraction in turn, each with tiles and a ring of its own in LDS and no
// barrier until their sums are added at the end: a quarter of the chain, four times the workgroups.  fp32 gains most (its
// MFMA takes 64 cycles for two values of k): backward of q, k, v (24 tokens, 512 features) 54 us with the 64 x 64 tiles.
#include "attn_common.hpp"

namespace tp {

constexpr int LIN_MAX = 4, LIN_SEGS = 3, LIN_TILE = 64, LIN_RING = 4;

struct LinSeg { const void* a; const void* b; int k, lda, ldb; };
struct LinProb {
  LinSeg seg[LIN_SEGS];
  void* c;
  int m, n, ldc, nseg, a_kmajor, b_kmajor, c_float, tiles_n, tile_end;  // tile_end: one past its last tile in the launch
};
struct LinArgs { LinProb p[LIN_MAX]; };

// four consecutive values of a row of c; c_float: rounded to the element type, stored as fp32 (a projection followed by
// .float(), without the pass in between)
template <typename E>
__device__ __forceinline__ void lin_store(const LinProb& p, int m, int n, float x0, float x1, float x2, float x3) {
  if (n >= p.n) return;
  const int64_t at = (int64_t)m * p.ldc + n;
  if constexpr (sizeof(E) == 2) {
    if (p.c_float) *(f32x4*)((float*)p.c + at) = f32x4{round_to<E>(x0), round_to<E>(x1), round_to<E>(x2), round_to<E>(x3)};
    else *(u32x2*)((E*)p.c + at) = pack4<E>(x0, x1, x2, x3);
  } else {
    *(f32x4*)((float*)p.c + at) = f32x4{x0, x1, x2, x3};
  }
}

// One operand's LDS tile of a step, 8 KB: its loads and its fragments.  E: element type; KM: rows hold the contraction.
//   KM:   64 rows (m or n) x 128 bytes of k, chunks of 16 bytes XOR-swizzled by the row (DmaTile)
//   !KM:  16-bit: 64 rows k x 64 columns, same swizzle, fragments by transposing reads;  fp32: 32 rows k x 64 columns, plain
typedef DmaTile<64, true> LT;
template <typename E, bool KM>
struct LinTile {
  static constexpr bool F32 = sizeof(E) == 4;
  static constexpr int BK = F32 ? 32 : 64;
  static constexpr int CPR = (F32 && !KM) ? 16 : 8;  // chunks per LDS row
  unsigned vo[2], koff[2];  // global byte offset of the lane's chunk inside a tile; KM: its first k as bytes, else unused

  __device__ __forceinline__ void init(int ld, int wave, int lane) {
#pragma unroll
    for (int i = 0; i < 2; i++) {
      const int slot = (wave * 2 + i) * 64 + lane, row = slot / CPR;
      const int c = (F32 && !KM) ? slot % CPR : (slot % CPR) ^ LT::swz(row);
      vo[i] = (unsigned)row * (unsigned)ld * (unsigned)sizeof(E) + (unsigned)c * 16u;
      koff[i] = (unsigned)c * 16u;
    }
  }
  // this wave's two loads of the step that starts at k0 of the tile that starts at row / column x0
  __device__ __forceinline__ void issue(u32x4 rs, int ld, int x0, int k0, int k, unsigned lds_tile, int wave_s) const {
    const unsigned so = KM ? (unsigned)x0 * (unsigned)ld * (unsigned)sizeof(E) + (unsigned)k0 * (unsigned)sizeof(E)
                           : (unsigned)k0 * (unsigned)ld * (unsigned)sizeof(E) + (unsigned)x0 * (unsigned)sizeof(E);
    const unsigned off = __builtin_amdgcn_readfirstlane(so);
    const unsigned left = (unsigned)(k - k0) * (unsigned)sizeof(E);
#pragma unroll
    for (int i = 0; i < 2; i++) {
      // (k past the row's end belongs to the next row: such chunks ask past the tensor and arrive as zeros)
      const unsigned v = KM && koff[i] >= left ? 0x7fffffffu : vo[i];
      asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                   :: "s"(__builtin_amdgcn_readfirstlane(lds_tile + (unsigned)(wave_s * 2 + i) * 1024u)), "v"(v), "s"(rs), "s"(off) : "memory", "m0");
    }
  }
  // 16-bit: operand of k-step ks (16 values of k, lane group g the values 8 g ..+7) of the wave's 32 rows / columns x
  template <typename V8>
  static __device__ __forceinline__ V8 frag16(unsigned tile, int x, int ks, int lane) {
    const int g = lane >> 5, ln = lane & 31;
    if constexpr (KM) {
      return *(const __attribute__((address_space(3))) V8*)(tile + (unsigned)LT::off(x + ln, 2 * ks + g));
    } else {
      const int cb = x / 16 + ((lane >> 4) & 1), r = 16 * ks + 8 * g;
      return tr_read8<V8>((const lds_byte*)(tile + (unsigned)LT::tr_off(r, cb, lane & 15)), (const lds_byte*)(tile + (unsigned)LT::tr_off(r + 4, cb, lane & 15)));
    }
  }
  // fp32: the values k = 8 j + 4 g ..+3
  static __device__ __forceinline__ f32x4 frag32(unsigned tile, int x, int j, int lane) {
    const int g = lane >> 5, ln = lane & 31;
    if constexpr (KM) {
      return *(const __attribute__((address_space(3))) f32x4*)(tile + (unsigned)LT::off(x + ln, 2 * j + g));
    } else {
      f32x4 r;
#pragma unroll
      for (int t = 0; t < 4; t++) r[t] = *(const __attribute__((address_space(3))) float*)(tile + (unsigned)((8 * j + 4 * g + t) * 256 + (x + ln) * 4));
      return r;
    }
  }
};

template <typename E, bool AK, bool BK_>
__device__ __forceinline__ void linear_tile(const LinProb& p, int tile, unsigned char* smem) {
  typedef LinTile<E, AK> TA;
  typedef LinTile<E, BK_> TB;
  constexpr int BK = TA::BK, TB_BYTES = 8192, STEP_BYTES = 2 * TB_BYTES;
  const int tid = threadIdx.x, lane = tid & 63, wave_s = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = tile / p.tiles_n * LIN_TILE, n0 = tile % p.tiles_n * LIN_TILE;
  const int wm = (wave_s >> 1) * 32, wn = (wave_s & 1) * 32;
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem);

  int steps = 0;
  for (int s = 0; s < p.nseg; s++) steps += (p.seg[s].k + BK - 1) / BK;

  // the cursor of the loads: segment, k inside it, its descriptors
  TA ta;
  TB tb;
  u32x4 ra, rb;
  int seg = 0, k0 = 0, lda = 0, ldb = 0, kk = 0;
  auto open = [&](int s) {
    const LinSeg& g = p.seg[s];
    lda = g.lda; ldb = g.ldb; kk = g.k;
    ta.init(lda, wave_s, lane);
    tb.init(ldb, wave_s, lane);
    // bytes from the base to one past the last element
    const int64_t ea = AK ? (int64_t)(p.m - 1) * lda + kk : (int64_t)(kk - 1) * lda + p.m;
    const int64_t eb = BK_ ? (int64_t)(p.n - 1) * ldb + kk : (int64_t)(kk - 1) * ldb + p.n;
    ra = make_rsrc_words(g.a, (unsigned)(ea * sizeof(E)));
    rb = make_rsrc_words(g.b, (unsigned)(eb * sizeof(E)));
  };
  open(0);
  int issued = 0;
  auto issue_next = [&]() {
    if (issued < steps) {
      const unsigned at = lds0 + (unsigned)(issued % LIN_RING) * STEP_BYTES;
      ta.issue(ra, lda, m0, k0, kk, at, wave_s);
      tb.issue(rb, ldb, n0, k0, kk, at + TB_BYTES, wave_s);
      k0 += BK;
      if (k0 >= kk && ++seg < p.nseg) { k0 = 0; open(seg); }
    }
    issued++;
  };
  f32x16 acc;
#pragma unroll
  for (int v = 0; v < 16; v++) acc[v] = 0.f;
  for (int i = 0; i < LIN_RING - 1; i++) issue_next();
  for (int s = 0; s < steps; s++) {
    // step s has landed (each step is four loads of this wave; two later steps may be in flight, fewer at the end), and
    // everybody is done with step s - 1, whose place step s + 3 takes
    const int after = min(steps - 1 - s, LIN_RING - 2);
    if (after >= 2) asm volatile("s_waitcnt vmcnt(8) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else if (after == 1) asm volatile("s_waitcnt vmcnt(4) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
    issue_next();
    const unsigned la = lds0 + (unsigned)(s % LIN_RING) * STEP_BYTES, lb = la + TB_BYTES;
    if constexpr (sizeof(E) == 2) {
      typedef typename MT<E>::v8 v8;
#pragma unroll
      for (int ks = 0; ks < 4; ks++)
        acc = MT<E>::mfma32(TB::template frag16<v8>(lb, wn, ks, lane), TA::template frag16<v8>(la, wm, ks, lane), acc);
    } else {
#pragma unroll
      for (int j = 0; j < 4; j++) {
        const f32x4 b = TB::frag32(lb, wn, j, lane), a = TA::frag32(la, wm, j, lane);
#pragma unroll
        for (int t = 0; t < 4; t++) acc = __builtin_amdgcn_mfma_f32_32x32x2f32(b[t], a[t], acc, 0, 0, 0);
      }
    }
  }
  // lane: row m, four consecutive n per group of values
  const int m = m0 + wm + (lane & 31), g = lane >> 5;
  if (m < p.m) {
#pragma unroll
    for (int vq = 0; vq < 4; vq++) lin_store<E>(p, m, n0 + wn + 8 * vq + 4 * g, acc[4 * vq], acc[4 * vq + 1], acc[4 * vq + 2], acc[4 * vq + 3]);
  }
}

// ---- 32 x 32 tiles, the contraction split over the waves ----
// One operand's tile of a step, 4 KB of a wave's own LDS:
//   KM:   32 rows (m or n) x 128 bytes of k, chunks XOR-swizzled by the row
//   !KM:  16-bit: 64 rows k x 32 columns;  fp32: 32 rows k x 32 columns; plain (a transposing read of 4 rows x 64 bytes is
//         256 contiguous bytes)
template <typename E, bool KM>
struct LinSplitTile {
  static constexpr bool F32 = sizeof(E) == 4;
  static constexpr int BK = F32 ? 32 : 64, CPR = KM ? 8 : F32 ? 8 : 4, ROWB = CPR * 16;
  unsigned vo[4], koff[4];

  __device__ __forceinline__ void init(int ld, int lane) {
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const int slot = i * 64 + lane, row = slot / CPR, c = KM ? (slot % CPR) ^ LT::swz(row) : slot % CPR;
      vo[i] = (unsigned)row * (unsigned)ld * (unsigned)sizeof(E) + (unsigned)c * 16u;
      koff[i] = (unsigned)c * 16u;
    }
  }
  __device__ __forceinline__ void issue(u32x4 rs, int ld, int x0, int k0, int k, unsigned lds_tile) const {
    const unsigned so = KM ? (unsigned)x0 * (unsigned)ld * (unsigned)sizeof(E) + (unsigned)k0 * (unsigned)sizeof(E)
                           : (unsigned)k0 * (unsigned)ld * (unsigned)sizeof(E) + (unsigned)x0 * (unsigned)sizeof(E);
    const unsigned off = __builtin_amdgcn_readfirstlane(so);
    const unsigned left = (unsigned)(k - k0) * (unsigned)sizeof(E);
#pragma unroll
    for (int i = 0; i < 4; i++) {
      const unsigned v = KM && koff[i] >= left ? 0x7fffffffu : vo[i];
      asm volatile("s_mov_b32 m0, %0\n\tbuffer_load_dwordx4 %1, %2, %3 offen lds"
                   :: "s"(__builtin_amdgcn_readfirstlane(lds_tile + (unsigned)i * 1024u)), "v"(v), "s"(rs), "s"(off) : "memory", "m0");
    }
  }
  template <typename V8>
  static __device__ __forceinline__ V8 frag16(unsigned tile, int ks, int lane) {
    const int g = lane >> 5, ln = lane & 31;
    if constexpr (KM) {
      return *(const __attribute__((address_space(3))) V8*)(tile + (unsigned)LT::off(ln, 2 * ks + g));
    } else {
      // lane 4 e + m of a group of 16: row r + e, columns 16 cb + 4 m ..+3 (see DmaTile::tr_off)
      const int cb = (lane >> 4) & 1, l16 = lane & 15, r = 16 * ks + 8 * g + (l16 >> 2), col = 16 * cb + 4 * (l16 & 3);
      const unsigned at = tile + (unsigned)(r * ROWB + col * 2);
      return tr_read8<V8>((const lds_byte*)at, (const lds_byte*)(at + 4 * ROWB));
    }
  }
  static __device__ __forceinline__ f32x4 frag32(unsigned tile, int j, int lane) {
    const int g = lane >> 5, ln = lane & 31;
    if constexpr (KM) {
      return *(const __attribute__((address_space(3))) f32x4*)(tile + (unsigned)LT::off(ln, 2 * j + g));
    } else {
      f32x4 r;
#pragma unroll
      for (int t = 0; t < 4; t++) r[t] = *(const __attribute__((address_space(3))) float*)(tile + (unsigned)((8 * j + 4 * g + t) * ROWB + ln * 4));
      return r;
    }
  }
};

template <typename E, bool AK, bool BK_>
__device__ __forceinline__ void linear_tile_split(const LinProb& p, int tile, unsigned char* smem) {
  typedef LinSplitTile<E, AK> TA;
  typedef LinSplitTile<E, BK_> TB;
  constexpr int BK = TA::BK, T_BYTES = 4096, STEP_BYTES = 2 * T_BYTES;
  const int tid = threadIdx.x, lane = tid & 63, wave_s = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int m0 = tile / p.tiles_n * 32, n0 = tile % p.tiles_n * 32;
  const unsigned lds0 = __builtin_amdgcn_readfirstlane((unsigned)(size_t)smem) + (unsigned)wave_s * 2u * STEP_BYTES;

  // the cursor of the loads: this wave's steps are wave, wave + 4, ... of all segments' steps in a row
  TA ta;
  TB tb;
  u32x4 ra, rb;
  int seg = -1, k0 = 0, lda = 0, ldb = 0, kk = 0, left = wave_s;  // left: steps to go from the segment's start
  bool more = true;
  auto open = [&](int s) {
    const LinSeg& g = p.seg[s];
    lda = g.lda; ldb = g.ldb; kk = g.k;
    ta.init(lda, lane);
    tb.init(ldb, lane);
    const int64_t ea = AK ? (int64_t)(p.m - 1) * lda + kk : (int64_t)(kk - 1) * lda + p.m;
    const int64_t eb = BK_ ? (int64_t)(p.n - 1) * ldb + kk : (int64_t)(kk - 1) * ldb + p.n;
    ra = make_rsrc_words(g.a, (unsigned)(ea * sizeof(E)));
    rb = make_rsrc_words(g.b, (unsigned)(eb * sizeof(E)));
  };
  auto seek = [&]() {  // to the step `left` steps after the current segment's start
    int steps = seg < 0 ? 0 : (kk + BK - 1) / BK;
    bool moved = false;
    while (left >= steps) {
      left -= steps;
      if (++seg >= p.nseg) { more = false; return; }
      steps = (p.seg[seg].k + BK - 1) / BK;
      moved = true;
    }
    if (moved) open(seg);
    k0 = left * BK;
  };
  auto issue_next = [&](int stage) -> bool {
    if (!more) return false;
    const unsigned at = lds0 + (unsigned)stage * STEP_BYTES;
    ta.issue(ra, lda, m0, k0, kk, at);
    tb.issue(rb, ldb, n0, k0, kk, at + T_BYTES);
    left += 4;
    seek();
    return true;
  };
  f32x16 acc[1];
#pragma unroll
  for (int v = 0; v < 16; v++) acc[0][v] = 0.f;
  seek();
  bool cur = issue_next(0), next = issue_next(1);
  for (int stage = 0; cur; stage ^= 1) {
    // (eight loads a step: the next step's may stay in flight)
    if (next) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    const unsigned la = lds0 + (unsigned)stage * STEP_BYTES, lb = la + T_BYTES;
    if constexpr (sizeof(E) == 2) {
      typedef typename MT<E>::v8 v8;
      v8 fa[4], fb[4];
#pragma unroll
      for (int ks = 0; ks < 4; ks++) { fb[ks] = TB::template frag16<v8>(lb, ks, lane); fa[ks] = TA::template frag16<v8>(la, ks, lane); }
      // (the fragments are in registers: the stage may be written again)
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa[0]), "+v"(fa[1]), "+v"(fa[2]), "+v"(fa[3]), "+v"(fb[0]), "+v"(fb[1]), "+v"(fb[2]), "+v"(fb[3]) :: "memory");
      cur = next;
      next = issue_next(stage);
#pragma unroll
      for (int ks = 0; ks < 4; ks++) acc[0] = MT<E>::mfma32(fb[ks], fa[ks], acc[0]);
    } else {
      f32x4 fa[4], fb[4];
#pragma unroll
      for (int j = 0; j < 4; j++) { fb[j] = TB::frag32(lb, j, lane); fa[j] = TA::frag32(la, j, lane); }
      asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa[0]), "+v"(fa[1]), "+v"(fa[2]), "+v"(fa[3]), "+v"(fb[0]), "+v"(fb[1]), "+v"(fb[2]), "+v"(fb[3]) :: "memory");
      cur = next;
      next = issue_next(stage);
#pragma unroll
      for (int j = 0; j < 4; j++)
#pragma unroll
        for (int t = 0; t < 4; t++) acc[0] = __builtin_amdgcn_mfma_f32_32x32x2f32(fb[j][t], fa[j][t], acc[0], 0, 0, 0);
    }
  }
  __syncthreads();  // every wave has read its last step: the LDS is free for the sums
  sum_waves(acc, (float*)smem, wave_s, lane);
  const int m = m0 + (lane & 31), g = lane >> 5;
  if (wave_s == 0 && m < p.m) {
#pragma unroll
    for (int vq = 0; vq < 4; vq++) lin_store<E>(p, m, n0 + 8 * vq + 4 * g, acc[0][4 * vq], acc[0][4 * vq + 1], acc[0][4 * vq + 2], acc[0][4 * vq + 3]);
  }
}

template <typename E, bool SPLIT>
__global__ __launch_bounds__(256) void linears_kernel(const LinArgs a) {
  __shared__ __align__(16) unsigned char smem[65536];
  static_assert(LIN_RING * 16384 == 65536, "four steps of two 8 KB tiles, or four waves' two steps of two 4 KB tiles");
  int i = 0, first = 0;
  while (i < LIN_MAX - 1 && (int)blockIdx.x >= a.p[i].tile_end) first = a.p[i++].tile_end;
  const LinProb& p = a.p[i];
  const int tile = (int)blockIdx.x - first;
  if constexpr (SPLIT) {
    if (p.a_kmajor && p.b_kmajor) linear_tile_split<E, true, true>(p, tile, smem);
    else if (p.a_kmajor) linear_tile_split<E, true, false>(p, tile, smem);
    else linear_tile_split<E, false, false>(p, tile, smem);
  } else {
    if (p.a_kmajor && p.b_kmajor) linear_tile<E, true, true>(p, tile, smem);
    else if (p.a_kmajor) linear_tile<E, true, false>(p, tile, smem);
    else linear_tile<E, false, false>(p, tile, smem);
  }
}

template <typename E>
static void linears_launch(const LinArgs& a, bool split, unsigned tiles, hipStream_t st) {
  if (split) linears_kernel<E, true><<<dim3(tiles), dim3(256), 0, st>>>(a);
  else linears_kernel<E, false><<<dim3(tiles), dim3(256), 0, st>>>(a);
}

}  // namespace tp

using namespace tp;

extern "C" int tp_linears(const tp_linear_problem* problems, int count_, int dtype, void* stream) {
  TP_REQUIRE(problems && count_ >= 1 && count_ <= LIN_MAX, TP_ERR_BAD_ARG, "tp_linears: 1 to %d problems, got %d", LIN_MAX, count_);
  TP_REQUIRE(dtype == TP_BF16 || dtype == TP_F16 || dtype == TP_F32, TP_ERR_UNSUPPORTED, "tp_linears: dtype %d", dtype);
  const int e = dtype == TP_F32 ? 4 : 2, vec = 16 / e;
  LinArgs a;
  auto count = [&](int t) {
    int64_t n = 0;
    for (int i = 0; i < count_; i++) n += (int64_t)((problems[i].m + t - 1) / t) * ((problems[i].n + t - 1) / t);
    return n;
  };
  const bool split = count(32) <= 1024;  // (four workgroups per CU)
  const int edge = split ? 32 : LIN_TILE;
  int64_t tiles = 0;
  for (int i = 0; i < LIN_MAX; i++) {
    LinProb& d = a.p[i];
    if (i >= count_) { d = a.p[count_ - 1]; continue; }
    const tp_linear_problem& s = problems[i];
    TP_REQUIRE(s.c && s.m > 0 && s.n > 0 && s.segments >= 1 && s.segments <= LIN_SEGS, TP_ERR_BAD_ARG, "tp_linears: null output or bad size");
    TP_REQUIRE(s.a_kmajor || !s.b_kmajor, TP_ERR_UNSUPPORTED, "tp_linears: no kernel for a row-k A with a k-major B");
    TP_REQUIRE(s.n % 4 == 0 && s.ldc >= s.n && s.ldc % 4 == 0 && aligned16(s.c), TP_ERR_BAD_ARG, "tp_linears: output rows must be a multiple of 4 values, 16-byte aligned");
    for (int j = 0; j < s.segments; j++) {
      const int64_t lda = s.lda[j], ldb = s.ldb[j], k = s.k[j];
      TP_REQUIRE(s.a[j] && s.b[j] && k > 0 && aligned16(s.a[j]) && aligned16(s.b[j]) && lda % vec == 0 && ldb % vec == 0, TP_ERR_BAD_ARG,
                 "tp_linears: operands must be 16-byte aligned rows");
      TP_REQUIRE(lda >= (s.a_kmajor ? k : s.m) && ldb >= (s.b_kmajor ? k : s.n), TP_ERR_BAD_ARG, "tp_linears: row stride below the row");
      TP_REQUIRE((!s.a_kmajor && !s.b_kmajor) || k % vec == 0, TP_ERR_BAD_ARG, "tp_linears: a k-major contraction must be a multiple of %d", vec);
      // (tiles reach up to 64 rows past the end, with 32-bit byte offsets)
      TP_REQUIRE(((s.a_kmajor ? s.m : k) + 64) * lda * e < (1ll << 31) && ((s.b_kmajor ? s.n : k) + 64) * ldb * e < (1ll << 31), TP_ERR_UNSUPPORTED,
                 "tp_linears: an operand spans 2 GiB or more");
      d.seg[j] = LinSeg{s.a[j], s.b[j], (int)k, (int)lda, (int)ldb};
    }
    for (int j = s.segments; j < LIN_SEGS; j++) d.seg[j] = d.seg[0];
    d.c = s.c; d.m = s.m; d.n = s.n; d.ldc = (int)s.ldc; d.nseg = s.segments; d.a_kmajor = s.a_kmajor != 0; d.b_kmajor = s.b_kmajor != 0; d.c_float = s.c_float != 0;
    d.tiles_n = (s.n + edge - 1) / edge;
    tiles += (int64_t)((s.m + edge - 1) / edge) * d.tiles_n;
    TP_REQUIRE(tiles < (1ll << 30), TP_ERR_UNSUPPORTED, "tp_linears: too many tiles");
    d.tile_end = (int)tiles;
  }
  hipStream_t st = (hipStream_t)stream;
  if (dtype == TP_BF16) linears_launch<bf16_t>(a, split, (unsigned)tiles, st);
  else if (dtype == TP_F16) linears_launch<f16_t>(a, split, (unsigned)tiles, st);
  else linears_launch<float>(a, split, (unsigned)tiles, st);
  return check_launch("tp_linears");
}
