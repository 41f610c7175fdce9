// Attention forward in fp32 for gfx950: fp32 operands and accumulation on v_mfma_f32_32x32x2_f32.
//
// The reference's eager branch on fp32 tensors (torchprime/torch_xla_models/attention.py:151-170: fp32 matmuls, fp32
// softmax) is what its own CPU tests run the small configurations in
// (torchprime/torch_xla_models/tests/test_llama.py:143-188); the 16-bit kernels cannot meet those tolerances.  This
// kernel is the same algorithm as attn_fwd.hip without any 16-bit rounding: causal / full, segment ids, GQA, explicit
// scale, LSE out.
//
// At the sizes this is used for (sequences of a few hundred, eight heads) there are few query rows to go round and the
// chain of kv tiles is what takes the time.  So a workgroup owns 32 query rows only, its four waves take the kv tiles in
// turn, each with an online softmax of its own, and the four partial results meet in LDS at the end; operands come
// straight from memory in the layout the MFMA wants (K and Q rows as contiguous pieces, V rows as coalesced columns: every
// byte of a line is used), so no wave waits for another inside the loop, and V's loads fly under the S products.
// B2 S128, 8 heads of 64: 22 us with 128 rows a workgroup and staged tiles, 10 us so.
//
// Where there are enough query rows to fill the chip anyway that costs more than it gives: every 32 rows fetch all keys and
// values, four times the reads, and the sums over the waves come on top.  STAGED is the layout for those: 128 rows a
// workgroup, 32 a wave, tiles of keys and values staged through LDS and read by all four waves, two barriers a tile
// (fwd_staged has the line and the figures).
//
// v_mfma_f32_32x32x2_f32 (wave64; ln = lane % 32, g = lane / 32):
//   A (32 x 2): lane holds row ln, k = g        B (2 x 32): lane holds column ln, k = g
//   C (32 x 32): lane holds column ln, rows 8*(v/4) + 4*g + v%4 for v = 0..15
// As in the 16-bit kernel the scores are computed transposed, S^T = K Q^T, so a lane owns one query column: row
// max / sum are per-lane scalars and exp(S^T) is directly the B operand of O^T += V^T P^T.  The hardware pairs A and
// B per k index, so the order of the contraction index is free as long as both operands agree: lane group g takes
// head-dim element g*D/2 + step for S^T (contiguous per lane, 16-byte LDS reads), and kv row 8*(v/4) + 4*g + v%4 at
// step v for P V (exactly the C layout of P^T).
#include "attn_common.hpp"

namespace tp {

struct FwdArgs32 {
  const float* q;
  const float* k;
  const float* v;
  const int32_t* seg;
  float* out;
  float* lse;
  int B, Hq, Hkv, Sq, Skv, n_rep;
  int64_t qs[3], ks[3], vs[3], os[3];
  float scale_log2;
  int causal;
  MaskExt mx;   // window / query positions / causal offset as a band of key positions per query row; soft cap
  float cap2;   // the soft cap in the scores' log2 units (0: none)
};

template <int D, bool STAGED>
__global__ __launch_bounds__(256) void attn_fwd_f32_kernel(const FwdArgs32 a) {
  constexpr int BN = 32, BM = STAGED ? 128 : 32, DB = D / 32, HD = D / 2;
  constexpr int KSTRIDE = D + 4;  // floats per LDS row of K: 16-byte aligned rows, consecutive rows 4 banks apart
  constexpr int VSTRIDE = D + 1;
  __shared__ __align__(16) float smem[STAGED ? BN * (KSTRIDE + VSTRIDE) : 2 * DB * 1024];  // K and V tile, or the waves' sums
  __shared__ float msm[4][64], lsm[4][64];
  __shared__ int ssm[BN];  // STAGED: the tile's segment ids
  float* const ksm = smem;
  float* const vsm = smem + BN * KSTRIDE;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, g = lane >> 5, ln = lane & 31;
  const int n_qt = (a.Sq + BM - 1) / BM;
  const int qt = n_qt - 1 - blockIdx.x % n_qt;  // the longest rows first
  const int bh = blockIdx.x / n_qt;
  const int h = bh % a.Hq, b = bh / a.Hq, hk = h / a.n_rep;
  const int q0 = qt * BM, wq0 = q0 + (STAGED ? wave * 32 : 0);
  const int Sq = a.Sq, Skv = a.Skv;
  const int qrow = wq0 + ln, qrow_c = min(qrow, Sq - 1);
  const float* kb = a.k + b * a.ks[0] + hk * a.ks[1];
  const float* vb = a.v + b * a.vs[0] + hk * a.vs[1];
  const int32_t* segb = a.seg ? a.seg + (int64_t)b * Skv : nullptr;
  const int segq = segb ? segb[qrow_c] : 0;
  // mask extensions: this lane's query row may see key positions qp - lo_off .. qp + hi_off (causality is part of
  // the band then, and a.causal is off)
  const int qp = a.mx.on ? (a.mx.qpos ? a.mx.qpos[qrow_c] : qrow) : 0;
  const int band_lo = a.mx.on ? qp - a.mx.lo_off : -BAND_INF, band_hi = a.mx.on ? qp + a.mx.hi_off : BAND_INF;
  const float* bias_row = a.mx.bias ? a.mx.bias + b * a.mx.bias_s[0] + h * a.mx.bias_s[1] + (int64_t)qrow_c * a.mx.bias_s[2] : nullptr;

  // Q^T fragments: lane (query column ln, group g) holds Q[q][g*HD + s] for s = 0..HD-1, pre-multiplied by the
  // scale in log2 units (an fp32 product: no precision is lost that the fp32 reference keeps)
  float qf[HD];
  load_row32(qf, a.q + b * a.qs[0] + h * a.qs[1] + (int64_t)qrow_c * a.qs[2] + g * HD);
#pragma unroll
  for (int s = 0; s < HD; s++) qf[s] *= a.scale_log2;

  f32x16 oacc[DB];
#pragma unroll
  for (int d = 0; d < DB; d++)
#pragma unroll
    for (int v = 0; v < 16; v++) oacc[d][v] = 0.f;
  float m_run = -INFINITY, l_run = 0.f;

  const int kv_end = a.causal ? min(Skv, q0 + BM) : Skv;
  const int ntiles = (kv_end + BN - 1) / BN;
  for (int t = STAGED ? 0 : wave; t < ntiles; t += STAGED ? 1 : 4) {
    const int kv0 = t * BN;
    f32x16 s;
#pragma unroll
    for (int v = 0; v < 16; v++) s[v] = 0.f;
    float vf[16][DB];  // (not STAGED)
    // S^T = K Q^T: row = kv (ln of the A operand), column = query
    if constexpr (STAGED) {
      __syncthreads();  // everyone is done with the previous tile
      // K and V rows kv0 .. kv0+31 (rows past Skv as zeros): 16-byte chunks, thread -> (row, chunk), both loads in flight
      for (int c = tid; c < BN * (D / 4); c += 256) {
        const int r = c / (D / 4), cc = (c % (D / 4)) * 4;
        f32x4 kvv = {0.f, 0.f, 0.f, 0.f}, vvv = {0.f, 0.f, 0.f, 0.f};
        if (kv0 + r < Skv) {
          kvv = *(const f32x4*)(kb + (int64_t)(kv0 + r) * a.ks[2] + cc);
          vvv = *(const f32x4*)(vb + (int64_t)(kv0 + r) * a.vs[2] + cc);
        }
        *(f32x4*)(ksm + r * KSTRIDE + cc) = kvv;
#pragma unroll
        for (int e = 0; e < 4; e++) vsm[r * VSTRIDE + cc + e] = vvv[e];
      }
      if (segb && tid < BN) ssm[tid] = segb[min(kv0 + tid, Skv - 1)];
      __syncthreads();
      if (a.causal && kv0 > wq0 + 31) continue;  // the whole tile lies above this wave's diagonal (uniform per wave)
      const float* kr = ksm + ln * KSTRIDE + g * HD;
#pragma unroll
      for (int st = 0; st < HD; st += 4) {
        const f32x4 k4 = *(const f32x4*)(kr + st);
#pragma unroll
        for (int e = 0; e < 4; e++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(k4[e], qf[st + e], s, 0, 0, 0);
      }
    } else {
      float kf[HD];
      load_row32(kf, kb + (int64_t)min(kv0 + ln, Skv - 1) * a.ks[2] + g * HD);
      load_cols32(vf, vb, a.vs[2], kv0, Skv, g, ln);
#pragma unroll
      for (int st = 0; st < HD; st++) s = __builtin_amdgcn_mfma_f32_32x32x2f32(kf[st], qf[st], s, 0, 0, 0);
    }
    // mask, online softmax (log2 units)
    float mx = -INFINITY;
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int kvl = 8 * (v / 4) + 4 * g + (v % 4), kv = kv0 + kvl;
      const bool ok = kv < Skv && (!a.causal || kv <= qrow) && (!segb || (STAGED ? ssm[kvl] : segb[min(kv, Skv - 1)]) == segq) && kv >= band_lo && kv <= band_hi;
      if (a.cap2 != 0.f) s[v] = a.cap2 * tanhf(s[v] / a.cap2);  // cap * tanh(score / cap), in log2 units
      if (bias_row) s[v] += LOG2E * bias_row[min(kv, Skv - 1)];  // additive mask (-inf stays -inf)
      s[v] = ok ? s[v] : -INFINITY;
      mx = fmaxf(mx, s[v]);
    }
    mx = half_max(mx);
    const float m_new = fmaxf(m_run, mx);
    const float m_use = (m_new == -INFINITY) ? 0.f : m_new;
    const float alpha = (m_run == -INFINITY) ? 0.f : exp2f(m_run - m_use);
    float rs = 0.f;
#pragma unroll
    for (int v = 0; v < 16; v++) {
      s[v] = exp2f(s[v] - m_use);
      rs += s[v];
    }
    l_run = l_run * alpha + rs;
    m_run = m_new;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int v = 0; v < 16; v++) oacc[d][v] *= alpha;
    // O^T += V^T P^T: step v pairs kv row 8*(v/4) + 4*g + v%4 of V with the lane's value v of P^T
#pragma unroll
    for (int v = 0; v < 16; v++) {
      const int kvl = 8 * (v / 4) + 4 * g + (v % 4);
#pragma unroll
      for (int d = 0; d < DB; d++)
        oacc[d] = __builtin_amdgcn_mfma_f32_32x32x2f32(STAGED ? vsm[kvl * VSTRIDE + d * 32 + ln] : vf[v][d], s[v], oacc[d], 0, 0, 0);
    }
  }

  float m_all = m_run, l = l_run;
  if constexpr (!STAGED) {
    // the waves' shares: brought to the largest of the four maxima, then added
    msm[wave][lane] = m_run;
    __syncthreads();
    m_all = fmaxf(fmaxf(msm[0][lane], msm[1][lane]), fmaxf(msm[2][lane], msm[3][lane]));
    const float share = m_run == -INFINITY ? 0.f : exp2f(m_run - m_all);
    lsm[wave][lane] = l_run * share;
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int v = 0; v < 16; v++) oacc[d][v] *= share;
    sum_waves(oacc, smem, wave, lane);
    if (wave != 0) return;
    l = (lsm[0][lane] + lsm[2][lane]) + (lsm[1][lane] + lsm[3][lane]);
  }

  // epilogue: lane = query, value v of block d is output column d*32 + 8*(v/4) + 4*g + v%4
  l = half_sum(l);
  const float inv = l > 0.f ? 1.f / l : 0.f;
  if (qrow < Sq) {
    if (g == 0) a.lse[((int64_t)b * a.Hq + h) * Sq + qrow] = l > 0.f ? (m_all + log2f(l)) * LN2 : -INFINITY;
    float* op = a.out + b * a.os[0] + h * a.os[1] + (int64_t)qrow * a.os[2];
#pragma unroll
    for (int d = 0; d < DB; d++)
#pragma unroll
      for (int vq = 0; vq < 4; vq++) {
        const f32x16& o = oacc[d];
        *(f32x4*)(op + d * 32 + 8 * vq + 4 * g) = f32x4{o[4 * vq] * inv, o[4 * vq + 1] * inv, o[4 * vq + 2] * inv, o[4 * vq + 3] * inv};
      }
  }
}

// Which layout: staged where its workgroups of 128 rows fill the CUs by themselves.  Head dim 128 keeps one workgroup a CU
// busy with its MFMAs, so rounds count whole; at head dim 64 two share a CU, and staging pays from two of them on.  Not for
// long causal sequences (the 128 rows of a workgroup wait for its last ones, and four times fewer workgroups balance the
// triangle worse), nor where a workgroup would have rows for one wave only.  us, 32 rows : staged, B Hq/Hkv S:
//   64, full:    1 8/8 4096  470 : 640;  2 32/8 768  149 : 169;  2 32/8 1024  254 : 225;  64 8/8 100  53 : 34;  2 32/8 4096  3560 : 2930
//   64, causal:  16 8/8 384  72 : 79;  4 32/8 512  130 : 113;  64 8/8 640  543 : 433;  16 8/8 900  265 : 392;  4 32/8 2048  1380 : 1521
//   128, full:   2 8/8 1024  148 : 251;  2 32/8 512  155 : 134;  2 32/8 768  327 : 382;  4 32/32 256  96 : 69;  4 32/8 2048  4573 : 4114
//   128, causal: 16 8/8 384  149 : 162;  64 8/8 128  111 : 75;  4 32/8 768  489 : 494;  4 32/8 1024  1118 : 973;  2 32/8 2048  1673 : 1898
static bool fwd_staged(int D, int64_t workgroups, int Sq, bool causal) {
  return Sq > 32 && (!causal || staged_triangle(Sq)) && (D == 64 ? workgroups >= 2 * CUS : full_rounds(workgroups));
}

// called by tp_attn_fwd for TP_F32 inputs (arguments already validated there)
int attn_fwd_f32(const void* q, const void* k, const void* v, const int32_t* seg, void* out, float* lse, int B, int Hq, int Hkv,
                 int Sq, int Skv, int Dqk, int Dv, const int64_t* qs, const int64_t* ks, const int64_t* vs, const int64_t* os,
                 float sm_scale, int causal, hipStream_t st, const MaskExt& mx) {
  TP_REQUIRE(Dqk == Dv && (Dqk == 64 || Dqk == 128), TP_ERR_UNSUPPORTED,
             "tp_attn_fwd: fp32 attention is built for head dims 64 and 128 (got qk=%d, v=%d)", Dqk, Dv);
  FwdArgs32 a;
  a.q = (const float*)q; a.k = (const float*)k; a.v = (const float*)v; a.seg = seg; a.out = (float*)out; a.lse = lse;
  a.B = B; a.Hq = Hq; a.Hkv = Hkv; a.Sq = Sq; a.Skv = Skv; a.n_rep = Hq / Hkv;
  bool ok = aligned16(q) && aligned16(k) && aligned16(v) && aligned16(out);
  for (int i = 0; i < 3; i++) {
    a.qs[i] = qs[i]; a.ks[i] = ks[i]; a.vs[i] = vs[i]; a.os[i] = os[i];
    ok = ok && qs[i] % 4 == 0 && ks[i] % 4 == 0 && vs[i] % 4 == 0 && os[i] % 4 == 0;
  }
  TP_REQUIRE(ok, TP_ERR_BAD_ARG, "tp_attn_fwd: fp32 pointers and strides must keep rows 16-byte aligned");
  a.scale_log2 = sm_scale * LOG2E;
  a.causal = mx.on ? 0 : causal;
  a.mx = mx;
  a.cap2 = mx.cap_in != 0.f ? mx.cap_out * sm_scale * LOG2E : 0.f;
  const int64_t blocks = (int64_t)B * Hq * ((Sq + 31) / 32);
  TP_REQUIRE(blocks < (1ll << 31), TP_ERR_UNSUPPORTED, "tp_attn_fwd: too many workgroups");
  const int64_t staged_blocks = (int64_t)B * Hq * ((Sq + 127) / 128);
  const bool staged = fwd_staged(Dqk, staged_blocks, Sq, a.causal);
  const dim3 grid((unsigned)(staged ? staged_blocks : blocks)), block(256);
  if (Dqk == 64 && staged) attn_fwd_f32_kernel<64, true><<<grid, block, 0, st>>>(a);
  else if (Dqk == 64) attn_fwd_f32_kernel<64, false><<<grid, block, 0, st>>>(a);
  else if (staged) attn_fwd_f32_kernel<128, true><<<grid, block, 0, st>>>(a);
  else attn_fwd_f32_kernel<128, false><<<grid, block, 0, st>>>(a);
  return check_launch("tp_attn_fwd(fp32)");
}

}  // namespace tp
