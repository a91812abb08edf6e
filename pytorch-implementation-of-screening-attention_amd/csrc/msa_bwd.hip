// Backward path of fused Screening Attention on gfx950.
//
// Gradients of the dense math in attention.py:142-200 / norm.py:23-25, written
// out for the normalised operands (same derivation as the reference's
// screening_bwd.py:6-18) plus the per-head terms the reference fused path
// drops (attention_triton.py:44):
//   dh_i   = TanhNorm'(h_i)^T dy_i
//   dP_ij  = dh_i . v^_j                        (pair weight p_ij = a_ij^2 m_ij)
//   dv^_j  = sum_i p_ij dh_i
//   ds_ij  = 2 a_ij r m_ij dP_ij  [a_ij > 0]
//   dq^_i  = sum_j ds_ij k^_j,   dk^_j = sum_i ds_ij q^_i
//   dr     = -sum 2 a (1-s) m dP,  dw = sum a^2 dP dm/dw
//   dx     = (dx^ - x^ (x^.dx^)) / |x|   (|x| > eps),  dx^/eps otherwise
// Only the 32x32 units the forward marked live in its bitmap are revisited;
// each wave walks its bitmap row/column.  MFMA operands are the raw q, k, v
// values (exact in bf16), staged in LDS a unit at a time and read in row and in
// column order, and the 1/|x|
// factors are applied in fp32 to the products, so no normalised copy is
// rounded; dh is formed on the fly from y, dy and |h|.  Per-row scale
// factors reach register order through a small LDS vector.  Key padding
// (attention.py:185-188) enters as a zero 1/|k|, which gives s = 0 and so
// alpha = 0 for those keys.
//
//   dq_kernel   : wave per 32-query unit over its live key units; writes dq
//                 and the unit's (dr, dw) share, and leaves dh and 1/|q| of
//                 its rows for dkdv_kernel.
//   dkdv_kernel : wave per 32-key unit; accumulates dv^, dk^ in MFMA
//                 registers over its live query units and writes dk, dv; one
//                 wave per head also sums the (dr, dw) shares in a fixed
//                 order into dr, dw.
// No atomics anywhere, so every gradient is bitwise reproducible.
#include "msa_device.h"
#include "msa_internal.h"

namespace msa {

// G(n) = F'(n)/n with F(n) = tanh(n)/n.  Series below 0.25 (the closed form
// cancels there): F = 1 - n^2/3 + 2n^4/15 - 17n^6/315 + 62n^8/2835.
__device__ inline float tanhnorm_g(float n, float t) {
  if (n < 0.25f) {
    const float n2 = n * n;
    return -2.0f / 3.0f + n2 * (8.0f / 15.0f + n2 * (-34.0f / 105.0f + n2 * (496.0f / 2835.0f)));
  }
  return ((1.0f - t * t) / n - t / (n * n)) / n;
}

// dh = F dy + G (h.dy) h with h = y/F  ->  dh = c1 dy + c2 (y.dy) y
__device__ inline void tanhnorm_coefs(float n, float eps, float& c1, float& c2) {
  if (n > eps) {
    const float t = tanhf(n);
    c1 = t / n;
    c2 = tanhnorm_g(n, t) / (c1 * c1);
  } else {
    c1 = tanhf(eps) / eps;
    c2 = 0.0f;
  }
}

struct BwdKArgs {
  const void* q; Strides3 qs;
  const void* k; Strides3 ks;
  const void* v; Strides3 vs;
  const uint8_t* kpm;
  const void* y; const void* dy; const float* hnorm;
  const float* r; const float* w;
  const uint32_t* bits;
  void* dq; void* dk; void* dv; float* dr; float* dw;
  float* part;  // workspace: (dr, dw) shares per (b, h, query unit), [2][b*h][2*nqt]
  // workspace: dh [b*h][Tq_pad][DP] (T), 1/|q| [b*h][Tq_pad] (fp16: negative for
  // rows whose ds may come within a factor 2 of fp16's range)
  void* dh; float* iqs;
  int B, H, Tq, Tk, D, nqt, nkt, nku_words, causal;
  int64_t Tq_pad;
  float eps;
  Dropout drop;
};

// Query-side rows for row i of head (b,h), in two steps so that other memory
// traffic can be issued between them: load raw q, y, dy and |h|; then finish
// 1/|q| and dh (rounded to T, as the MFMA operand it becomes).  Rows past Tq
// read row 0 and are zeroed.
template <typename T, int DP>
struct QueryRows {
  PRow<T, DP> q, y, dh;
  float hn;
  bool ok;
  __device__ inline void load(const BwdKArgs& a, int b, int h, int bh, int i, int half) {
    ok = i < a.Tq;
    const int ii = ok ? i : 0;
    const int64_t yoff = (((int64_t)b * a.Tq + ii) * a.H + h) * a.D;
    q.load((const T*)a.q + b * a.qs.sb + (int64_t)ii * a.qs.st + h * a.qs.sh, ok, a.D, half);
    y.load((const T*)a.y + yoff, ok, a.D, half);
    dh.load((const T*)a.dy + yoff, ok, a.D, half);
    hn = a.hnorm[(int64_t)bh * a.Tq + ii];
  }
  // returns 1/|q|; dh holds TanhNorm'(h)^T dy afterwards
  __device__ inline float finish(float eps) {
    const float iq = q.inv_norm(eps);
    const float ydot = y.dot(dh);
    float c1, c2;
    tanhnorm_coefs(ok ? hn : 0.0f, eps, c1, c2);
    dh.axpby(c1, c2 * ydot, y);
    return iq;
  }
};

// Key-side rows for key j of head (b,h), load then finish as for the query
// side: raw k with 1/|k| (0 for padded or masked keys), raw v with 1/|v|.
template <typename T, int DP>
struct KeyRows {
  PRow<T, DP> k, v;
  bool ok, masked;
  __device__ inline void load(const BwdKArgs& a, int b, int h, int j, int half) {
    ok = j < a.Tk;
    const int jj = ok ? j : 0;
    k.load((const T*)a.k + b * a.ks.sb + (int64_t)jj * a.ks.st + h * a.ks.sh, ok, a.D, half);
    v.load((const T*)a.v + b * a.vs.sb + (int64_t)jj * a.vs.st + h * a.vs.sh, ok, a.D, half);
    masked = a.kpm != nullptr && a.kpm[(int64_t)b * a.Tk + jj] != 0;
  }
  __device__ inline void finish(float eps, float& ik, float& iv) const {
    ik = (ok && !masked) ? k.inv_norm(eps) : 0.0f;
    iv = v.inv_norm(eps);
  }
};

// D = 16 (DP = 32): rows of the product past D come from the repeated columns
// of the staged rows; they are dropped here.
template <typename T, int DP>
__device__ inline void zero_past_d(f32x16 (&acc)[DP / 32], int D) {
  if constexpr (DP == 32) {
#pragma unroll
    for (int r = 0; r < 16; ++r)
      if (Mma<T>::KS * creg_ks<T>(0, r) >= D) acc[0][r] = 0.0f;
  }
}

// Writes dx = normalise-backward(dx^, x) (attention.py:156-158 under
// autograd) for one row: dx^ in C-layout registers acc[dblk] whose rows are
// tcol-ordered columns, x as the lane's raw operand fragments of the same row
// (the operands the kernel already holds, so nothing is re-read).
//   |x| > eps:  dx = (dx^ - x^ (x^ . dx^)) / |x|;   otherwise dx = dx^ / eps.
template <typename T, int DP>
__device__ inline void write_norm_bwd(const f32x16 (&acc)[DP / 32], const typename Mma<T>::frag (&x)[DP / Mma<T>::KS],
                                      bool valid, int D, float eps, int half, T* out) {
  using M = Mma<T>;
  constexpr int NDH = DP / 32, NKS = DP / M::KS;
  const float ss = half_sum(row_dot<T>(x, x));
  const float nx = sqrtf(ss);
  const float ix = 1.0f / fmaxf(nx, eps);
  float dot = 0.0f;
#pragma unroll
  for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
    for (int r = 0; r < 16; ++r) dot += M::get(x[creg_ks<T>(dblk, r)], creg_e<T>(r)) * ix * acc[dblk][r];
  dot = half_sum(dot);
  const float proj = nx > eps ? dot : 0.0f;
  if (!valid) return;
  store_creg_row<T, NDH>(out, D, half, [&](int dblk, int r) {
    const float xn = M::get(x[creg_ks<T>(dblk, r)], creg_e<T>(r)) * ix;
    return (acc[dblk][r] - xn * proj) * ix;
  });
}

// ---------------------------------------------------------------------------
// dQ (runs first).  One wave (a 64-thread block) per query unit: 32
// consecutive queries of head (b,h), lane -> query i = 32*qu + l%32,
// registers -> keys.  The wave walks its row of the live-unit bitmap; each
// live key unit's raw K and V rows are staged in the wave's LDS (UnitTile),
// the next unit's copies in flight behind the current one.  It forms S^T = K
// Q^T and dP^T = V dH^T, scales them by 1/|k|, 1/|v| (exchanged in register
// order through a 32-float LDS vector), and accumulates dq^T += K^T (ds/|k|)^T
// with K^T read transposed from the staged rows.  Side output for dkdv_kernel:
// dh (rounded to T, as the operand it becomes) and 1/|q| of the unit's rows,
// written by every unit with a live key unit (the only rows dkdv_kernel
// reads).  S > 1: as in the live pass, S waves share the row's live units and
// wave 0 adds their partial dq, dr and dw in wave order.
// ---------------------------------------------------------------------------
template <typename T, int DP>
constexpr int dq_waves() { return sizeof(T) * DP <= 64 ? 3 : (sizeof(T) * DP <= 128 ? 2 : 1); }
// fp32 rows of D = 128: the K columns are read from the staged rows only where
// they are used, and K's next copy waits for that; held across the pair terms as
// in the other cases they spill 68 registers, and each reload waits behind the
// copies in flight.  With one or two waves a row the dh fragments stay in
// registers too, so that a CU's LDS holds four waves instead of three or two;
// four waves a row fit it once either way and share the copy in LDS.  us a
// launch, columns held -> columns late -> dh in registers too: B=4 H=8, T=4096
// (one wave) 4257 -> 2531 -> 2256, T=2048 (two) 1542 -> 1134 -> 687, T=1000 (four)
// 412 -> 239 -> 258.
template <typename T, int DP>
constexpr bool kLateK = sizeof(T) * DP > 256;

template <typename T, int DP, int S, bool DROP>
__global__ __launch_bounds__(64 * S) __attribute__((amdgpu_waves_per_eu(dq_waves<T, DP>())))
void dq_kernel(BwdKArgs a) {
  using M = Mma<T>;
  using frag = typename M::frag;
  using U = UnitTile<T, DP>;
  constexpr int KS = M::KS, PER = M::PER, NKS = DP / KS, NDH = DP / 32, NC = 32 / KS;
  // per wave:
  __shared__ __attribute__((aligned(16))) float sk_w[S][32];  // 1/|k| (0 if padded or masked) of the unit's key rows
  __shared__ __attribute__((aligned(16))) float sv_w[S][32];  // 1/|v|
  __shared__ float mtab_w[S][128];  // soft-mask table of the current unit, then its dm/dw table (unit_mask_table)
  __shared__ __attribute__((aligned(16))) float sw_w[kPow2Rows<T> ? S : 1][32];   // fp16: the w of 1/|k| (Pow2Split)
  __shared__ __attribute__((aligned(16))) f16 sc_w[kPow2Rows<T> ? S : 1][2][32];  // fp16: its powers of two
  __shared__ __attribute__((aligned(1024))) char stage[S][2 * U::BYTES];  // the unit's K and V rows; then the partial dq
  static_assert(NDH * 16 * kWave * 4 <= 2 * U::BYTES, "the partial dq fits the staged rows");
  constexpr bool kDhRegs = kLateK<T, DP> && S < 4;
  __shared__ frag hsh[kDhRegs ? 1 : NKS][kWave];  // own dh operand fragments (each wave writes the same ones)
  const int lane = (int)(threadIdx.x & 63), half = lane >> 5, l32 = lane & 31;
  const int wave = S > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
  float* sk = sk_w[wave];
  float* sv = sv_w[wave];
  float* mtab = mtab_w[wave];
  char* kt = stage[wave];
  char* vt = kt + U::BYTES;
  LdsChar* const kt_at = (LdsChar*)&stage[0][0] + wave * 2 * U::BYTES;
  LdsChar* const vt_at = kt_at + U::BYTES;
  int qu, bh;
  float head_r, head_w;
  xcd_interleave_ranked(a.r, a.w, a.H, qu, bh, head_r, head_w);
  const int b = bh / a.H, h = bh % a.H;
  const bool causal = a.causal != 0;
  const HeadParams hp = head_params_rw(head_r, head_w, causal);
  const int i = qu * kUnit + l32;
  const bool valid = i < a.Tq;
  auto dqrow = [&]() { return (T*)a.dq + (((int64_t)b * a.Tq + (valid ? i : 0)) * a.H + h) * a.D; };

  int ku_lo, ku_hi;
  {
    const int64_t qa = (int64_t)qu * kUnit, qb = qa + kUnit - 1 < a.Tq - 1 ? qa + kUnit - 1 : a.Tq - 1;
    int64_t jlo = qa - hp.wc + 1;
    int64_t jhi = causal ? qb : qb + hp.wc - 1;
    if (jlo < 0) jlo = 0;
    if (jhi > a.Tk - 1) jhi = a.Tk - 1;
    ku_lo = (int)(jlo / kUnit);
    ku_hi = jhi >= jlo ? (int)(jhi / kUnit) : ku_lo - 1;
  }
  const uint32_t* brow = a.bits + ((int64_t)bh * 2 * a.nqt + qu) * a.nku_words;
  RowWalk walk(brow, ku_lo, ku_hi);
  int cur = walk.next();
  const int64_t nbh = (int64_t)a.B * a.H;
  const int nqu = 2 * a.nqt;
  if (cur < 0) {  // block-uniform: no live key unit, dq = 0 and no share of dr, dw
    if (wave != 0) return;
    if (valid)
#pragma unroll
      for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int d = 32 * dblk + 8 * g + 4 * half;
          if (d < a.D) store4(dqrow() + d, 0.0f, 0.0f, 0.0f, 0.0f);
        }
    if (lane == 0) {
      a.part[(int64_t)bh * nqu + qu] = 0.0f;
      a.part[nbh * nqu + (int64_t)bh * nqu + qu] = 0.0f;
    }
    return;
  }
  // a row of one unit, the usual one at initialisation, is wave 0's alone: the
  // others leave, and there is nothing to add up (B=8 T=241 x 269 D=64 bf16, us:
  // one wave a row 9.2, four 14.9, four with the others gone 10.2; B=2 T=298 7.6,
  // 9.7, 7.8).  Not for fp32, whose rows of one unit gained from the split as it is,
  // and where the branch cost dense rows 3% (B=2 T=1500 D=64 117 -> 120).
  const bool alone = S > 1 && sizeof(T) == 2 && walk.ended();
  if (alone && wave != 0) return;
  for (int w = 0; w < wave && cur >= 0; ++w) cur = walk.next();  // S > 1: the wave's first unit

  // key row of this lane in unit u: 32u + perm_row(l32)
  const int m = perm_row(l32);
  const typename U::Source ksrc((const T*)a.k + b * a.ks.sb + h * a.ks.sh, a.ks.st, a.Tk, a.D, lane);
  const typename U::Source vsrc((const T*)a.v + b * a.vs.sb + h * a.vs.sh, a.vs.st, a.Tk, a.D, lane);
  const uint32_t rb = U::row_base(lane), cb = U::col_base(lane);
  // D = 16: the staged columns past D repeat the first ones
  auto zero_tail = [&](frag (&f)[NKS]) {
    if constexpr (DP == 32) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        if (KS * ks >= a.D) f[ks] = M::zero();
    }
  };
  // 1/|k| is 0 for keys past Tk and for masked keys
  auto key_mask = [&](int u) -> unsigned {  // the mask byte, tested when the unit is computed
    const int j = u * kUnit + m;
    return a.kpm != nullptr && j < a.Tk ? a.kpm[(int64_t)b * a.Tk + j] : 0u;
  };

  // own queries' rows first, then the first key unit's copies behind them
  frag qf[NKS];  // raw q operand fragments; those of dh are kept in LDS (read back per unit)
  frag hreg[kDhRegs ? NKS : 1];
  float iql;
  // fp16: dh's row enters as dh p, p the power of two that makes its largest
  // element (times the dropout scale) 2^10 .. 2^11.  The packed ds (without 2r)
  // is then at most 2 * 2^11 sqrt(D) < 2^16, and the row's whole range has
  // fp16's full precision however small or large the gradient is.
  float ip = 1.0f;  // 1/p
  unsigned kmask = 0u;
  {
    QueryRows<T, DP> qr;
    qr.load(a, b, h, bh, i, half);
    if (cur >= 0) {
      ksrc.issue(kt_at, cur);
      vsrc.issue(vt_at, cur);
      kmask = key_mask(cur);
    }
    iql = qr.finish(a.eps);
    float p = 1.0f;
    bool big = false;  // 2r a m dP w, w < 2, may leave fp16's range
    if constexpr (kPow2Rows<T>) {
      float mx = 0.0f;
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
#pragma unroll
        for (int e = 0; e < PER; ++e) mx = fmaxf(mx, fabsf(qr.dh.get(ks, e)));
      mx = half_max(mx) * (DROP ? a.drop.scale : 1.0f);
      p = row_pow2(mx);
      ip = 1.0f / p;
      big = !(4.0f * hp.r * mx * (DP == 128 ? 11.32f : (DP == 64 ? 8.0f : 5.66f)) < 65504.0f);  // |dP| <= sqrt(D) mx
    }
    // dh and 1/|q| of this unit's rows for dkdv_kernel (zero past Tq)
    T* dst = (T*)a.dh + ((int64_t)bh * a.Tq_pad + i) * DP;
#pragma unroll
    for (int ks = 0; ks < NKS; ++ks) {
      qf[ks] = qr.q.f[ks];
      if (wave == 0) *reinterpret_cast<frag*>(dst + KS * ks + PER * half) = qr.dh.f[ks];
      if constexpr (kPow2Rows<T>) {
        f32x16 t;
#pragma unroll
        for (int e = 0; e < PER; ++e) t[e] = qr.dh.get(ks, e) * p;
        hsh[ks][lane] = M::pack(t, 0);
      } else if constexpr (kDhRegs) {
        hreg[ks] = qr.dh.f[ks];
      } else {
        hsh[ks][lane] = qr.dh.f[ks];
      }
    }
    if (wave == 0 && half == 0) a.iqs[(int64_t)bh * a.Tq_pad + i] = !valid ? 0.0f : (big ? -iql : iql);
  }
  const float thq = hp.thr / iql;  // s > thr  <=>  (q . k)/|k| > thr |q|
  float dr_acc = 0.0f, dw_acc = 0.0f;  // this unit's share of dr, dw
  f32x16 adq[NDH];
#pragma unroll
  for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
    for (int r = 0; r < 16; ++r) adq[dblk][r] = 0.0f;

  while (cur >= 0) {
    const int k0 = cur * kUnit;
    // the unit's mask tables first, while few values are live (the LDS sync
    // after the products below covers these writes too; this iteration's
    // writes follow the previous one's reads in the wave's LDS order)
    unit_mask_table<true>(mtab, mtab + 64, qu * kUnit - k0 - 31, hp, lane);
    wait_vmcnt<0>();  // the unit's rows have landed
    // register r -> key k0 + rowof(r, half), lane -> query i
    f32x16 s, slo, dp;  // fp32: s + slo
    float ikl, iv;  // 1/|k|, 1/|v| of this lane's key row m
    frag ka[kLateK<T, DP> ? 1 : NDH * NC];
    {
      float s2k, s2v;
      {
        frag kf[NKS];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) kf[ks] = U::row_frag(kt, rb, ks);
        zero_tail(kf);
        s = unit_product<T>(kf, qf, &slo);
        s2k = row_dot<T>(kf, kf);
        guard_run(kf, s);
      }
      __builtin_amdgcn_sched_barrier(0);
      {
        frag vf[NKS], hf[NKS];
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) vf[ks] = U::row_frag(vt, rb, ks);
#pragma unroll
        for (int ks = 0; ks < NKS; ++ks) hf[ks] = kDhRegs ? hreg[kDhRegs ? ks : 0] : hsh[kDhRegs ? 0 : ks][lane];
        zero_tail(vf);
        dp = unit_product<T>(vf, hf);
        s2v = row_dot<T>(vf, vf);
        guard_run(vf, dp);
        guard_keep(hf);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (!kLateK<T, DP>)
#pragma unroll
        for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
          for (int c = 0; c < NC; ++c) ka[dblk * NC + c] = U::col_frag(kt, cb, dblk, c);
      ikl = k0 + m < a.Tk && kmask == 0u ? inv_len_of<T>(half_sum(s2k), a.eps) : 0.0f;
      iv = inv_len_of<T>(half_sum(s2v), a.eps);
    }
    // every read of the staged rows has returned (kLateK: of the V rows): the
    // next unit's copies run behind the rest of this unit's work
    int nxt = -1;  // this wave's next unit: S positions on in the row's walk
    for (int w = 0; w < S; ++w) {
      nxt = walk.next();
      if (nxt < 0) break;
    }
    wave_lds_sync();
    if (nxt >= 0) {
      if constexpr (!kLateK<T, DP>) ksrc.issue(kt_at, nxt);
      vsrc.issue(vt_at, nxt);
      kmask = key_mask(nxt);
    }
    if (half == 0) {
      sk[m] = ikl;
      sv[m] = iv;
    }
    bool two = false;  // fp16: some K row takes a second power of two
    if constexpr (kPow2Rows<T>) {
      const Pow2Split p(ikl);
      two = p.two_factors();
      if (half == 0) {
        sw_w[wave][m] = p.w;
        sc_w[wave][0][m] = (f16)p.c1;
        sc_w[wave][1][m] = (f16)p.c2;
      }
    }
    wave_lds_sync();
    // the K columns' second power of two, rarely needed.  At D <= 32 it is branched
    // off here, where few values are live: beside the first one, below, the branch
    // splits the straight-line part and 22 registers spill (three waves a SIMD),
    // 149 -> 98 us at B=4 T=2048; D = 64 takes 148 us either way, D = 128 169
    // here and 165 below.
    auto scale_cols = [&](auto p) {  // fp16 only
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int dblk = 0; dblk < NDH; ++dblk) scale_slots(ka[dblk * NC + c], sc_w[wave][p], c, half);
    };
    if constexpr (kPow2Rows<T> && DP == 32)
      if (two) scale_cols(1);
    // scaled in place: s = (q . k)/|k|, dp = dH . v^
    {
      float sc[16];
      read_row_scales(sk, half, sc);
#pragma unroll
      for (int r = 0; r < 16; ++r) scale_pair<T>(s, slo, r, sc[r]);
      __builtin_amdgcn_sched_barrier(0);
      read_row_scales(sv, half, sc);
#pragma unroll
      for (int r = 0; r < 16; ++r) dp[r] *= sc[r];
      __builtin_amdgcn_sched_barrier(0);
    }
    // every lane forms its pair's terms branch-free (a = 0 below the
    // threshold, the mask and dm/dw, 0 outside the window, from the unit's
    // tables: entry l32 - 8half + 31 - 16(r/8) - r%8 for register r), for
    // every register; with dropout, only for the registers where some lane
    // may pass a conservative gate on the products (s > thr |q|), so the
    // pair hash runs there only
    {
      // entry 23 - (16(r/8) + r%8) of each table: constant offsets from one base
      const float* mrow = mtab + (l32 - 8 * half + 8);
      // (rows past Tq hold q = 0, so s = 0 and a = 1 - r <= 0: no term)
      // with um = a m dP: ds = 2r um (2r enters once, in the epilogue), dr
      // = -2 um (1 - s) = -(2/r) um (1 - a), dw = a^2 dP dm/dw
      auto body = [&](int r) {
        const int off = 16 * (r >> 3) + (r & 7);
        const float av = pair_root<T>(s[r], slo[r], iql, hp.r);
        float u = av * dp[r];
        if constexpr (DROP) u *= dropout_factor(a.drop, bh, i, k0 + 8 * half + off);
        const float um = u * mrow[23 - off];
        dr_acc = fmaf(um, 1.0f - av, dr_acc);
        dw_acc = fmaf(u * av, mrow[64 + 23 - off], dw_acc);
        dp[r] = um;
      };
      if constexpr (DROP) {  // the pair's hash only where some lane may pass
        const uint32_t pm0 = pass_mask(s, thq);
        for_each_set(pm0, body);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (((pm0 >> r) & 1u) == 0u) dp[r] = 0.0f;
      } else {  // every register: a = 0 gives no term, and no mask or branches
#pragma unroll
        for (int r = 0; r < 16; ++r) body(r);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // dq^T[d][i] += sum_j K^T[d][j] (ds/|k|)^T[j][i] (fp16: 1/|k|'s power of
    // two goes to the K columns, the rest to ds)
    {
      float ksc[16];
      if constexpr (kPow2Rows<T>) read_row_scales(sw_w[wave], half, ksc);
      else read_row_scales(sk, half, ksc);
#pragma unroll
      for (int r = 0; r < 16; ++r) dp[r] *= ksc[r];
    }
    if constexpr (kPow2Rows<T>) {
      scale_cols(0);
      if (DP > 32 && two) scale_cols(1);
    }
    frag db[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) db[c] = M::pack(dp, c * PER);
    if constexpr (kLateK<T, DP>) {
#pragma unroll
      for (int dblk = 0; dblk < NDH; ++dblk) {
        frag f[NC];
#pragma unroll
        for (int c = 0; c < NC; ++c) f[c] = U::col_frag(kt, cb, dblk, c);
#pragma unroll
        for (int c = 0; c < NC; ++c) adq[dblk] = M::mma_ng(f[c], db[c], adq[dblk]);
        guard_run(f, adq[dblk]);
      }
      guard_keep(db);
      wave_lds_sync();
      if (nxt >= 0) ksrc.issue(kt_at, nxt);
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int dblk = 0; dblk < NDH; ++dblk) adq[dblk] = M::mma_ng(ka[dblk * NC + c], db[c], adq[dblk]);
      guard_run(ka, adq[NDH - 1]);
      guard_keep(db);
    }
    cur = nxt;
  }
  dr_acc = wave_sum(dr_acc * ip) * (-2.0f / hp.r);
  dw_acc = wave_sum(dw_acc * ip);
  if (S > 1 && !alone) {
    auto part = [&](int w) { return reinterpret_cast<float(*)[kWave]>(stage[w]); };
    if (wave > 0) {
#pragma unroll
      for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
        for (int r = 0; r < 16; ++r) part(wave)[dblk * 16 + r][lane] = adq[dblk][r];
      if (lane == 0) { sk[0] = dr_acc; sv[0] = dw_acc; }
    }
    __syncthreads();
    if (wave > 0) return;
    for (int w = 1; w < S; ++w) {
#pragma unroll
      for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
        for (int r = 0; r < 16; ++r) adq[dblk][r] += part(w)[dblk * 16 + r][lane];
      dr_acc += sk_w[w][0];
      dw_acc += sv_w[w][0];
    }
  }
#pragma unroll
  for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
    for (int r = 0; r < 16; ++r) adq[dblk][r] *= 2.0f * hp.r * ip;
  zero_past_d<T, DP>(adq, a.D);
  write_norm_bwd<T, DP>(adq, qf, valid, a.D, a.eps, half, dqrow());
  if (lane == 0) {
    a.part[(int64_t)bh * nqu + qu] = dr_acc;
    a.part[nbh * nqu + (int64_t)bh * nqu + qu] = dw_acc;
  }
}

// ---------------------------------------------------------------------------
// dK, dV (runs after dq_kernel).  One wave (a 64-thread block) per key unit:
// 32 consecutive keys of head (b,h), lane -> key j = 32*ku + l%32 of the C
// blocks, registers -> queries.  The wave walks its column of the live-unit
// bitmap; each live query unit's raw Q rows and the dh rows that dq_kernel
// left in the workspace are staged in the wave's LDS (UnitTile), the next
// unit's copies in flight behind the current one.  It forms S = Q K^T and dP =
// dH V^T with its own raw K, V rows as B operands, and accumulates dv^T +=
// dH^T P and dk^T += Q^T (ds/|q|) with dH^T, Q^T read transposed from the
// staged rows.  1/|q| reaches register order through a 32-float LDS vector.
// S > 1: S waves share the column's live units; wave 0 adds their partial dk,
// dv in wave order.
// ---------------------------------------------------------------------------
// Waves per SIMD: two where both accumulators, the unit's fragments and their
// transposes fit 256 registers a lane.
template <typename T, int DP>
constexpr int dkdv_waves() { return sizeof(T) * DP <= 128 ? 2 : 1; }
template <typename T>
constexpr bool kLateColumns = sizeof(T) == 4;

template <typename T, int DP, int S, bool DROP>
__global__ __launch_bounds__(64 * S) __attribute__((amdgpu_waves_per_eu(dkdv_waves<T, DP>())))
void dkdv_kernel(BwdKArgs a) {
  using M = Mma<T>;
  using frag = typename M::frag;
  using U = UnitTile<T, DP>;
  constexpr int KS = M::KS, PER = M::PER, NKS = DP / KS, NDH = DP / 32, NC = 32 / KS;
  // per wave:
  __shared__ __attribute__((aligned(16))) float sq_w[S][32];  // 1/|q| of the current query unit's rows
  __shared__ float mt_w[S][64];  // soft-mask table of the current unit (unit_mask_table)
  __shared__ __attribute__((aligned(16))) float sw_w[kPow2Rows<T> ? S : 1][32];   // fp16: the w of 1/|q| (Pow2Split)
  __shared__ __attribute__((aligned(16))) f16 sc_w[kPow2Rows<T> ? S : 1][2][32];  // fp16: its powers of two
  __shared__ __attribute__((aligned(1024))) char stage[S][2 * U::BYTES];  // the unit's Q and dh rows; then partial dk, dv
  static_assert(NDH * 16 * kWave * 4 <= 2 * U::BYTES, "a partial dk fits the staged rows");
  const int lane = (int)(threadIdx.x & 63), half = lane >> 5, l32 = lane & 31;
  const int wave = S > 1 ? __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)) : 0;
  float* sq = sq_w[wave];
  float* mt = mt_w[wave];
  char* qt = stage[wave];
  char* ht = qt + U::BYTES;
  LdsChar* const qt_at = (LdsChar*)&stage[0][0] + wave * 2 * U::BYTES;
  LdsChar* const ht_at = qt_at + U::BYTES;
  int ku, bh;
  float head_r, head_w;
  xcd_interleave_ranked(a.r, a.w, a.H, ku, bh, head_r, head_w);
  // a key unit's live query units lie after it (its window runs forward), so
  // under a causal mask the lowest key units carry the most work: they go first
  if (a.causal) ku = (int)gridDim.x - 1 - ku;
  const int b = bh / a.H, h = bh % a.H;
  const bool causal = a.causal != 0;
  const HeadParams hp = head_params_rw(head_r, head_w, causal);
  const int k0 = ku * kUnit;
  const int j = k0 + l32;
  const bool jvalid = j < a.Tk;
  const int jj = jvalid ? j : 0;
  const int64_t orow = (((int64_t)b * a.Tk + jj) * a.H + h) * a.D;
  if (ku == 2 * a.nkt - 1 && bh < a.H && wave == 0) {
    // one wave per head: dr, dw from dq_kernel's per-query-unit shares
    // (complete: dq_kernel ran first), summed in a fixed order
    const int64_t nbh = (int64_t)a.B * a.H;
    const int nqu = 2 * a.nqt;
    float ar = 0.0f, aw = 0.0f;
    for (int64_t idx = lane; idx < (int64_t)a.B * nqu; idx += kWave) {
      const int bb = (int)(idx / nqu), u = (int)(idx % nqu);
      const int64_t o = ((int64_t)bb * a.H + bh) * nqu + u;
      ar += a.part[o];
      aw += a.part[nbh * nqu + o];
    }
    ar = wave_sum(ar);
    aw = wave_sum(aw);
    if (lane == 0) {
      a.dr[bh] = ar;
      a.dw[bh] = aw;
    }
  }

  int qu_lo, qu_hi;
  {
    const int64_t klast = k0 + kUnit - 1 < a.Tk - 1 ? k0 + kUnit - 1 : a.Tk - 1;
    int64_t ilo = causal ? (int64_t)k0 : (int64_t)k0 - hp.wc + 1;
    int64_t ihi = klast + hp.wc - 1;
    if (ilo < 0) ilo = 0;
    if (ihi > a.Tq - 1) ihi = a.Tq - 1;
    qu_lo = (int)(ilo / kUnit);
    qu_hi = ihi >= ilo && k0 < a.Tk ? (int)(ihi / kUnit) : qu_lo - 1;
  }
  const uint32_t* bcol = a.bits + (int64_t)bh * 2 * a.nqt * a.nku_words + (ku >> 5);
  ColWalk walk(bcol, a.nku_words, ku & 31, qu_lo, qu_hi);
  int cur = walk.next();
  if (cur < 0) {  // block-uniform: no live query unit, dk = dv = 0
    if (jvalid && wave == 0)
#pragma unroll
      for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
        for (int g = 0; g < 4; ++g) {
          const int d = 32 * dblk + 8 * g + 4 * half;
          if (d < a.D) {
            store4((T*)a.dk + orow + d, 0.0f, 0.0f, 0.0f, 0.0f);
            store4((T*)a.dv + orow + d, 0.0f, 0.0f, 0.0f, 0.0f);
          }
        }
    return;
  }
  const bool alone = S > 1 && sizeof(T) == 2 && walk.ended();  // as in dq_kernel
  if (alone && wave != 0) return;
  for (int w = 0; w < wave && cur >= 0; ++w) cur = walk.next();  // S > 1: the wave's first unit

  // Raw q rows past Tq read row Tq-1; their 1/|q| and dh rows (workspace,
  // zero past Tq) are 0, so they contribute nothing.
  const typename U::Source qsrc((const T*)a.q + b * a.qs.sb + h * a.qs.sh, a.qs.st, a.Tq, a.D, lane);
  const typename U::Source hsrc((const T*)a.dh + (int64_t)bh * a.Tq_pad * DP, DP, (int)a.Tq_pad, DP, lane);
  const float* iq0 = a.iqs + (int64_t)bh * a.Tq_pad;
  uint32_t rb = U::row_base(lane), cb = U::col_base(lane);
  // D = 16: the staged columns past D repeat the first ones (dh rows hold DP)
  auto zero_tail = [&](frag (&f)[NKS]) {
    if constexpr (DP == 32) {
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks)
        if (KS * ks >= a.D) f[ks] = M::zero();
    }
  };

  // own keys as raw B operands (lane -> key), with 1/|k| (0 if padded or
  // masked) and 1/|v|; their loads go first, the first query unit's behind
  KeyRows<T, DP> kr;
  float ikl, ivl, iqv = 0.0f;
  kr.load(a, b, h, j, half);
  if (cur >= 0) {
    qsrc.issue(qt_at, cur);
    hsrc.issue(ht_at, cur);
    iqv = iq0[(int64_t)cur * kUnit + l32];  // lanes l and l+32 read the same row
  }
  kr.finish(a.eps, ikl, ivl);
  // what dp takes of the key's side: 2r/|v|, in the epilogue; in fp16 before ds is
  // packed, as small gradients would be subnormal there without 2r and large ones
  // out of range without 1/|v|
  const float kfac = 2.0f * hp.r * ivl;
  f32x16 acc_k[NDH], acc_v[NDH];
#pragma unroll
  for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
    for (int r = 0; r < 16; ++r) { acc_k[dblk][r] = 0.0f; acc_v[dblk][r] = 0.0f; }
  const float thk = hp.thr / ikl;  // s > thr  <=>  (q . k)/|q| > thr |k|  (+inf for masked keys)

  while (cur >= 0) {
    const int q0 = cur * kUnit;
    if constexpr (!__is_same(T, bf16)) {
      rederive(rb);
      rederive(cb);
    }
    wait_vmcnt<0>();  // the unit's rows have landed
    if (half == 0) sq[l32] = kPow2Rows<T> ? fabsf(iqv) : iqv;
    bool two = false;  // fp16: some Q row takes a second power of two
    if constexpr (kPow2Rows<T>) {
      const Pow2Split p(iqv);
      two = p.two_factors();
      if (half == 0) {
        sw_w[wave][l32] = p.w;
        sc_w[wave][0][l32] = (f16)p.c1;
        sc_w[wave][1][l32] = (f16)p.c2;
      }
    }
    unit_mask_table<false>(mt, nullptr, q0 - k0 - 31, hp, lane);
    // register r -> query q0 + rowof(r, half), lane -> key j
    f32x16 s, slo, dp;  // fp32: s + slo
    {
      frag f[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) f[ks] = U::row_frag(qt, rb, ks);
      zero_tail(f);
      s = unit_product<T>(f, kr.k.f, &slo);
      guard_run(f, s);
    }
    __builtin_amdgcn_sched_barrier(0);
    {
      frag f[NKS];
#pragma unroll
      for (int ks = 0; ks < NKS; ++ks) f[ks] = U::row_frag(ht, rb, ks);
      dp = unit_product<T>(f, kr.v.f);
      guard_run(f, dp);
    }
    __builtin_amdgcn_sched_barrier(0);
    int nxt = -1;  // this wave's next unit: S positions on in the column's walk
    for (int w = 0; w < S; ++w) {
      nxt = walk.next();
      if (nxt < 0) break;
    }
    // once every read of the staged rows has returned, the next unit's copies
    // run behind the rest of this unit's work (fp32 reads the columns only
    // where it uses them: two transposed operands would not fit the registers)
    frag qa[kLateColumns<T> ? 1 : NDH * NC], ha[kLateColumns<T> ? 1 : NDH * NC];
    auto copy_next = [&]() {
      wave_lds_sync();
      if (nxt >= 0) {
        qsrc.issue(qt_at, nxt);
        hsrc.issue(ht_at, nxt);
        iqv = iq0[(int64_t)nxt * kUnit + l32];
      }
    };
    if constexpr (!kLateColumns<T>) {
#pragma unroll
      for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
          ha[dblk * NC + c] = U::col_frag(ht, cb, dblk, c);
          qa[dblk * NC + c] = U::col_frag(qt, cb, dblk, c);
        }
      copy_next();
    } else {
      wave_lds_sync();
    }
    // scaled in place: s = (q . k)/|q|; dp = dh . v, in fp16 with kfac
    float qsc[16];
    read_row_scales(sq, half, qsc);
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      scale_pair<T>(s, slo, r, qsc[r]);
      if constexpr (kPow2Rows<T>) dp[r] *= kfac;
    }
    __builtin_amdgcn_sched_barrier(0);
    // every lane forms its pair's weight and ds branch-free (the mask, 0
    // outside the window, from the unit's table: entry 16(r/8) + r%8 + 8half
    // - l32 + 31 for register r), for every register; with dropout, only for
    // the registers where some lane may pass a conservative gate on the
    // products (s > thr |k|), so the pair hash runs there only
    {
      const float* mrow = mt + (8 * half - l32 + 31);
      auto body = [&](int r) {
        const int off = 16 * (r >> 3) + (r & 7);
        const float av = pair_root<T>(s[r], slo[r], ikl, hp.r);
        float mk = mrow[off];
        if constexpr (DROP) mk *= dropout_factor(a.drop, bh, q0 + 8 * half + off, j);
        const float am = av * mk;
        s[r] = av * am;
        dp[r] = am * dp[r];
      };
      if constexpr (DROP) {  // the pair's hash only where some lane may pass
        const uint32_t pm0 = pass_mask(s, thk);
        for_each_set(pm0, body);
#pragma unroll
        for (int r = 0; r < 16; ++r)
          if (((pm0 >> r) & 1u) == 0u) { s[r] = 0.0f; dp[r] = 0.0f; }
      } else {  // every register: a = 0 gives no term, and no mask or branches
#pragma unroll
        for (int r = 0; r < 16; ++r) body(r);
      }
    }
    __builtin_amdgcn_sched_barrier(0);
    // ds/|q| (fp16: 1/|q|'s power of two goes to the Q columns, the rest here)
    if constexpr (kPow2Rows<T>) read_row_scales(sw_w[wave], half, qsc);
#pragma unroll
    for (int r = 0; r < 16; ++r) dp[r] *= qsc[r];
    if constexpr (kPow2Rows<T>) {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int dblk = 0; dblk < NDH; ++dblk) {
          scale_slots(qa[dblk * NC + c], sc_w[wave][0], c, half);
          if (two) scale_slots(qa[dblk * NC + c], sc_w[wave][1], c, half);
        }
    }
    // dv^T[d][j] += sum_i dH^T[d][i] P[i][j];  dk^T[d][j] += sum_i Q^T[d][i] (ds/|q|)[i][j]
    frag pb[NC], db[NC];
#pragma unroll
    for (int c = 0; c < NC; ++c) {
      pb[c] = M::pack(s, c * PER);
      db[c] = M::pack(dp, c * PER);
    }
    if constexpr (kLateColumns<T>) {
#pragma unroll
      for (int op = 0; op < 2; ++op) {
#pragma unroll
        for (int dblk = 0; dblk < NDH; ++dblk) {
          frag f[NC];
#pragma unroll
          for (int c = 0; c < NC; ++c) f[c] = U::col_frag(op == 0 ? ht : qt, cb, dblk, c);
          f32x16& acc = op == 0 ? acc_v[dblk] : acc_k[dblk];
#pragma unroll
          for (int c = 0; c < NC; ++c) acc = M::mma_ng(f[c], op == 0 ? pb[c] : db[c], acc);
          guard_run(f, acc);
        }
      }
      guard_keep(pb);
      guard_keep(db);
      copy_next();
    } else {
#pragma unroll
      for (int c = 0; c < NC; ++c)
#pragma unroll
        for (int dblk = 0; dblk < NDH; ++dblk) {
          acc_v[dblk] = M::mma_ng(ha[dblk * NC + c], pb[c], acc_v[dblk]);
          acc_k[dblk] = M::mma_ng(qa[dblk * NC + c], db[c], acc_k[dblk]);
        }
      guard_run(qa, acc_k[NDH - 1]);
      guard_keep(ha);
      guard_keep(pb);
      guard_keep(db);
    }
    cur = nxt;
  }

  if (S > 1 && !alone) {
    auto part = [&](int w) { return reinterpret_cast<float(*)[kWave]>(stage[w]); };
    auto add_up = [&](f32x16 (&acc)[NDH]) {
      if (wave > 0)
#pragma unroll
        for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
          for (int r = 0; r < 16; ++r) part(wave)[dblk * 16 + r][lane] = acc[dblk][r];
      __syncthreads();
      if (wave == 0)
        for (int w = 1; w < S; ++w)
#pragma unroll
          for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
            for (int r = 0; r < 16; ++r) acc[dblk][r] += part(w)[dblk * 16 + r][lane];
      __syncthreads();
    };
    add_up(acc_k);
    add_up(acc_v);
    if (wave > 0) return;
  }
#pragma unroll
  for (int dblk = 0; dblk < NDH; ++dblk)
#pragma unroll
    for (int r = 0; r < 16; ++r) acc_k[dblk][r] *= kPow2Rows<T> ? 1.0f : kfac;
  zero_past_d<T, DP>(acc_k, a.D);
  zero_past_d<T, DP>(acc_v, a.D);
  write_norm_bwd<T, DP>(acc_k, kr.k.f, jvalid, a.D, a.eps, half, (T*)a.dk + orow);
  write_norm_bwd<T, DP>(acc_v, kr.v.f, jvalid, a.D, a.eps, half, (T*)a.dv + orow);
}

// Workspace: [dr/dw partials][dh][1/|q|], each 256-byte aligned.
static int64_t bwd_part_bytes(const Geometry& g) { return round_up((int64_t)2 * g.B * g.H * 2 * g.nqt * 4, 256); }
static int64_t bwd_dh_bytes(const Geometry& g) {
  return round_up((int64_t)g.B * g.H * g.Tq_pad * g.DP * (int64_t)g.esize, 256);
}
size_t bwd_ws_bytes(const Geometry& g) {
  return bwd_part_bytes(g) + bwd_dh_bytes(g) + round_up((int64_t)g.B * g.H * g.Tq_pad * 4, 256);
}

template <typename T, int DP>
static hipError_t launch_bwd_t(const BwdCall& c) {
  const Geometry& g = c.g;
  BwdKArgs ka;
  ka.q = c.q; ka.qs = c.qs; ka.k = c.k; ka.ks = c.ks; ka.v = c.v; ka.vs = c.vs; ka.kpm = c.kpm;
  ka.y = c.y; ka.dy = c.dy; ka.hnorm = c.hnorm;
  ka.r = c.r; ka.w = c.w; ka.bits = c.bits;
  ka.dq = c.dq; ka.dk = c.dk; ka.dv = c.dv; ka.dr = c.dr; ka.dw = c.dw;
  char* ws = (char*)c.workspace;
  ka.part = (float*)ws;
  ka.dh = ws + bwd_part_bytes(g);
  ka.iqs = (float*)(ws + bwd_part_bytes(g) + bwd_dh_bytes(g));
  ka.B = g.B; ka.H = g.H; ka.Tq = g.Tq; ka.Tk = g.Tk; ka.D = g.D;
  ka.nqt = g.nqt; ka.nkt = g.nkt; ka.nku_words = g.nku_words; ka.causal = g.causal;
  ka.Tq_pad = g.Tq_pad;
  ka.eps = c.eps;
  ka.drop = c.drop;
  // launches with few rows split each row's live units over S waves
  auto split = [&](int tiles) {
    const int64_t rows = (int64_t)2 * tiles * g.B * g.H;
    return split_waves<T>(rows);
  };
  auto launch_split = [&](int S, auto&& fn) {
    auto with = [&](auto drop) {
      if (S == 4) fn(std::integral_constant<int, 4>{}, drop);
      else if (S == 2) fn(std::integral_constant<int, 2>{}, drop);
      else fn(std::integral_constant<int, 1>{}, drop);
    };
    if (c.drop.on) with(std::true_type{});
    else with(std::false_type{});
  };
  const dim3 qgrid((unsigned)(2 * g.nqt), (unsigned)(g.B * g.H)), kgrid((unsigned)(2 * g.nkt), (unsigned)(g.B * g.H));
  timer_begin(5, c.stream);
  launch_split(split(g.nqt), [&](auto waves, auto drop) {
    constexpr int S = decltype(waves)::value;
    hipLaunchKernelGGL((dq_kernel<T, DP, S, decltype(drop)::value>), qgrid, dim3(64 * S), 0, c.stream, ka);
  });
  timer_end(5, c.stream);
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  timer_begin(4, c.stream);
  launch_split(split(g.nkt), [&](auto waves, auto drop) {
    constexpr int S = decltype(waves)::value;
    hipLaunchKernelGGL((dkdv_kernel<T, DP, S, decltype(drop)::value>), kgrid, dim3(64 * S), 0, c.stream, ka);
  });
  timer_end(4, c.stream);
  return hipGetLastError();
}

hipError_t launch_bwd(const BwdCall& c) {
  const int DP = c.g.DP;
  if (c.g.dtype == 1) {
    if (DP == 32) return launch_bwd_t<bf16, 32>(c);
    if (DP == 64) return launch_bwd_t<bf16, 64>(c);
    return launch_bwd_t<bf16, 128>(c);
  }
  if (c.g.dtype == 2) {
    if (DP == 32) return launch_bwd_t<f16, 32>(c);
    if (DP == 64) return launch_bwd_t<f16, 64>(c);
    return launch_bwd_t<f16, 128>(c);
  }
  if (DP == 32) return launch_bwd_t<float, 32>(c);
  if (DP == 64) return launch_bwd_t<float, 64>(c);
  return launch_bwd_t<float, 128>(c);
}

}  // namespace msa
