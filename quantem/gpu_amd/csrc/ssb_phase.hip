// Exact per-BF phase path for Hermitian stacks and even aberration phases
// (every reconstruction's stack; C10, C12, C30 and the other even terms):
// phi_b = angle(IFFT2(C_b)), C_b(Q) = G_b(Q) conj(Gamma^_b(Q)) with its DC bin
// replaced by dc, and the moments sum_b phi_b, sum_b phi_b^2 per scan position.
// The general path (full-plane stacks, odd aberrations, unequal detector
// sampling) is in ssb_loss.hip, whose finishing kernels both share.
//
// For an even chi, Gamma^_b(-Q) = -conj(Gamma^_b(Q)), so C_b is antihermitian
// wherever -Q is on the scan's frequency grid and G_b is Hermitian: all of it
// but the Nyquist row and column and, for an imported stack, columns 0 and
// N/2 themselves.  Split C_b = i Y + H, Y = -i (C(Q) - conj C(-Q)) / 2 and
// H = (C(Q) + conj C(-Q)) / 2, both Hermitian: IFFT2(C_b) = h + i r with the
// real images r = IFFT2(Y) and h = IFFT2(H), and H lives on columns 0 and N/2
// and the Nyquist row only, so
//   h(x, y) = e(x) + (-1)^y g(x) + (-1)^x f(y)
// (e holds dc).  r needs a real transform: half the columns, half the rows,
// half the bytes between the two passes.
//
//   k_phase_cols  a wave per (BF pixel, S slot columns): the corrected columns
//                 of the half plane, Y's inverse FFT along q in registers and
//                 the wave's own LDS, T[b][slot][x]; slot 0 packs the real
//                 columns 0 and N/2; e and g from one more transform; the
//                 Nyquist row of H for the BF pixels that reach it
//   k_phase_rows  a wave per S pairs of rows, two rows a complex transform;
//                 phi = atan2(r, h), compensated moments in registers
//
// 16 trials of C10, C30 and rotation at 256 x 256, 800 BF pixels: 8.70 ms on
// the general path (complex planes, chi at Q - k and Q + k, workgroup
// barriers in every FFT stage), 3.35 ms here; 64 quadratic trials at
// 128 x 128: 9.70 and 4.05 ms.  A trial at 256 x 256 takes k_phase_cols 88 us
// (420 MB, the rate of a large copy) and k_phase_rows 109 us (210 MB; its LDS
// exchanges and the arctangents bound it, at 4 waves a SIMD).
#include "ssb_internal.h"
#include "ssb_overlap.h"

namespace qssb {

namespace {

__device__ __forceinline__ void wave_fence() { asm volatile("" ::: "memory"); }

// Inverse N-point FFT of S sequences by one wave.  In: x[s][m] = element
// lane + 64 m.  Out: o[p][r] = element fft_index(lane, p, r) of sequence
// fft_seq(lane, p).  An R-point DFT over m in registers, twiddles, then
// 64-point Stockham radix-4 stages over the S R sub-sequences through the
// wave's LDS (a wave's LDS operations keep their order: compiler fences
// only); every twiddle stays in registers.
template <int N, int S>
struct WaveIfft {
  static constexpr int R = N / 64;
  static constexpr int P = S * R / 4;     // radix-4 butterflies a lane and stage
  static constexpr int SP = 65;           // padded sub-sequence stride
  static constexpr int LDS = S * R * SP;  // float2 of LDS a wave
  static_assert(R >= 2 && P >= 1 && S * R % 4 == 0, "whole butterflies");

  float2 w1[R];   // e^{2 pi i lane k / N}
  float2 w2[3], w3[3];

  __device__ __forceinline__ void init(const float2* __restrict__ tw, int lane) {
#pragma unroll
    for (int k = 1; k < R; ++k) w1[k] = cconj(tw[(k * lane) & (N - 1)]);
    const int jj = lane & 15;
#pragma unroll
    for (int r = 1; r < 4; ++r) {
      w2[r - 1] = cconj(tw[(R * 4 * r * (jj & 3)) & (N - 1)]);
      w3[r - 1] = cconj(tw[(R * r * jj) & (N - 1)]);
    }
    // arrived here, or the loops' first uses would wait for their prefetches too, every time
#pragma unroll
    for (int k = 1; k < R; ++k) asm volatile("" : "+v"(w1[k].x), "+v"(w1[k].y));
#pragma unroll
    for (int r = 0; r < 3; ++r)
      asm volatile("" : "+v"(w2[r].x), "+v"(w2[r].y), "+v"(w3[r].x), "+v"(w3[r].y));
  }

  // sequence and element of output (p, r) of a lane
  __device__ static __forceinline__ int seq(int lane, int p) { return ((lane >> 4) + 4 * p) / R; }
  __device__ static __forceinline__ int index(int lane, int p, int r) {
    return ((lane >> 4) + 4 * p) % R + R * (lane & 15) + 16 * R * r;
  }

  __device__ __forceinline__ void run(float2 (&x)[S][R], float2* __restrict__ xb, int lane, float2 (&o)[P][4]) const {
    wave_fence();
#pragma unroll
    for (int s = 0; s < S; ++s) {
      dft_regs<R, true>(x[s]);
      xb[(s * R) * SP + lane] = x[s][0];
#pragma unroll
      for (int k = 1; k < R; ++k) xb[(s * R + k) * SP + lane] = cmul(x[s][k], w1[k]);
    }
#pragma unroll
    for (int ns = 1; ns < 64; ns *= 4) {
      wave_fence();
      const int jj = lane & 15, k = jj & (ns - 1);
      float2 v[P][4];
#pragma unroll
      for (int p = 0; p < P; ++p) {
        const int sq = (lane >> 4) + 4 * p;
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          float2 y = xb[sq * SP + jj + 16 * r];
          if (ns > 1 && r > 0) y = cmul(y, ns == 4 ? w2[r - 1] : w3[r - 1]);
          v[p][r] = y;
        }
      }
      wave_fence();
#pragma unroll
      for (int p = 0; p < P; ++p) {
        dft4<true>(v[p][0], v[p][1], v[p][2], v[p][3], o[p]);
        if (ns < 16) {
          const int base = ((lane >> 4) + 4 * p) * SP + (jj / ns) * ns * 4 + k;
#pragma unroll
          for (int r = 0; r < 4; ++r) xb[base + r * ns] = o[p][r];
        }
      }
    }
    wave_fence();
  }
};

// (a + b) / 2 rounded once, whatever a + b is.
__device__ __forceinline__ float mean2(float a, float b) { return fmaf(0.5f, a, 0.5f * b); }

// Whether a BF pixel's apertures can reach the Nyquist row: |Q -/+ k| >=
// |q_N/2| - |kx| there.
__device__ __forceinline__ bool reaches_nyquist(float qn, float kx, const ApIso& ap) {
  return fabsf(qn) - fabsf(kx) < ap.rout * 1.0001f;
}

// atan(q) for |q| <= 1: minimax polynomial in q^2 (fitted for it by
// iteratively reweighted least squares, 1.5e-8; 1.3e-7 relative evaluated in
// float32, as the library's).
__device__ __forceinline__ float atan_unit(float q) {
  const float u = q * q;
  float p = fmaf(0.0028497937601059675f, u, -0.016068270429968834f);
  p = fmaf(p, u, 0.042690981179475784f);
  p = fmaf(p, u, -0.07504252344369888f);
  p = fmaf(p, u, 0.10640916228294373f);
  p = fmaf(p, u, -0.14203640818595886f);
  p = fmaf(p, u, 0.19992618262767792f);
  p = fmaf(p, u, -0.3333307206630707f);
  return fmaf(p * u, q, q);
}

// a / b to the last place or two, for kQuotientLo <= b <= kQuotientHi (the hardware's
// reciprocal knows no denormals, neither given nor returned).
constexpr float kQuotientLo = 0x1p-125f, kQuotientHi = 0x1p125f;
__device__ __forceinline__ float quotient(float a, float b) {
  const float inv = __builtin_amdgcn_rcpf(b);
  const float q = a * inv;
  return fmaf(fmaf(-q, b, a), inv, q);
}

// atan2 by the octants, for arguments of any size; where x > |y| it is
// atan_unit(quotient(y, x)), to which it then reduces bit for bit (both operands
// come to the exponent of the larger first: the same mantissas).
__device__ __forceinline__ float phase_of(float y, float x) {
  const float ay = fabsf(y), ax = fabsf(x);
  const bool steep = ay > ax;                                   // (fmaxf and fminf would lose a NaN)
  const float mx = steep ? ay : ax, mn = steep ? ax : ay;
  const int ex = __builtin_amdgcn_frexp_expf(mx);
  float q = quotient(ldexpf(mn, -ex), ldexpf(mx, -ex));
  q = mx > 0.0f || mn != mn ? q : mx;   // 0 / 0 -> 0
  q = mx == INFINITY ? (mn < mx ? 0.0f : (mn == mx ? 1.0f : mn)) : q;
  float a = atan_unit(q);
  a = steep ? 1.5707963267948966f - a : a;
  a = x < 0.0f ? 3.1415926535897931f - a : a;
  return copysignf(a, y);
}

}  // namespace

// Waves of k_phase_cols: `groups` ranges of the chunk's BF pixels, slot group
// by slot group: the low columns hold most of the points inside the apertures
// and start first, so that the waves end together (with the slot groups dealt
// out evenly in 4096 waves the CUs held 1.4 waves a SIMD on average).
template <int N, int S, bool GENERAL>
__global__ void __launch_bounds__(256)
k_phase_cols(const float2* __restrict__ Gt, const BfInfo* __restrict__ info, GeomPtrs gp, EvenChi ch_arg,
             const EvenChi* __restrict__ ch_dev, ApIso ap, df rout2, const float2* __restrict__ tw, int b_begin,
             int b_count, int groups, float2* __restrict__ T, float2* __restrict__ EG, float2* __restrict__ Hrow) {
  typedef WaveIfft<N, S> Fft;
  constexpr int R = Fft::R, HALF = N / 2, GCOLS = HALF + 1, NSG = HALF / S;
  __shared__ float2 xbuf[4][Fft::LDS];
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  float2* xb = xbuf[w];
  const int wave = blockIdx.x * 4 + w;
  const int sg = wave / groups, grp = wave - sg * groups;
  if (sg >= NSG) return;
  int cnt = info->nbf - b_begin;
  cnt = cnt > b_count ? b_count : cnt;
  const int i0 = (int)((long long)grp * cnt / groups), i1 = (int)((long long)(grp + 1) * cnt / groups);
  if (i0 >= i1) return;
  const EvenChi& ch = ch_dev ? *ch_dev : ch_arg;
  Fft fft;
  fft.init(tw, lane);
  float qx[R];
#pragma unroll
  for (int m = 0; m < R; ++m) qx[m] = gp.qx[lane + 64 * m];
#pragma unroll
  for (int m = 0; m < R; ++m) asm volatile("" : "+v"(qx[m]));   // arrived here
  const float qn = as_const(gp.qx)[HALF];
  const float k0 = ch.k0, k4 = ch.k4, m12c = ch.m12c, m12s = ch.m12s, m12s2 = 2.0f * m12s;

  // the low words of qx where registers are left for them
  constexpr int LOWS = R <= 4 ? R : 0;
  float qxl[LOWS ? LOWS : 1];
#pragma unroll
  for (int m = 0; m < LOWS; ++m) qxl[m] = gp.qxl[lane + 64 * m];
  auto low_of = [&](int m) { return LOWS ? qxl[LOWS ? m : 0] : gp.qxl[lane + 64 * m]; };

  // what a point needs of its BF pixel
  struct Pixel {
    float kx2, ky2, cb, u, vx, vy, margin, ak, chik, kxl, kyl, cbl;
  } px;
  auto term = [&](float2 G, int m, float qxv, int col, float qyv) {   // row lane + 64 m
    const float B = fmaf(qxv, px.kx2, qyv * px.ky2) + 0.0f;   // no negative zero
    const float q2 = fmaf(qxv, qxv, qyv * qyv);
    const float base = px.cb - q2;
    const float near = base + fabsf(B), far = base - fabsf(B);
    float2 z = make_float2(0.0f * G.x, 0.0f * G.y);   // a NaN or infinity stays
    if (near > -px.margin) {
      float s, t;
      if constexpr (GENERAL) {
        const float kxh = 0.5f * px.kx2, kyh = 0.5f * px.ky2;
        float cm, cp, odd;
        chi_parts(ch.cp, qxv - kxh, qyv - kyh, cm, odd);
        chi_parts(ch.cp, qxv + kxh, qyv + kyh, cp, odd);
        cm -= px.chik;
        cp -= px.chik;
        constexpr float kTurn = 0.15915494309189535f;   // 1 / 2pi
        t = (cp - cm) * kTurn;
        s = (cp + cm) * kTurn;
      } else {
        const float w4 = fmaf(k4, q2, px.u);
        t = fmaf(qxv, px.vx, fmaf(qyv, px.vy, B * fmaf(k4, q2, w4)));
        s = fmaf(q2, w4, k4 * (B * B));
        s = add_cancelling((qxv - qyv) * (qxv + qyv) * m12c, fmaf(qxv * qyv, m12s2, s));
      }
      t = B < 0.0f ? -t : t;
      z = overlap_term(G, near, far, B, s, t, near_whole(s), px.margin, px.ak, ap, [&](float& dm, float& dp) {
        const df x = df_in_branch(df{qxv, low_of(m)}), y = df_in_branch(df{qyv, as_const(gp.qyl)[col]});
        exact_d(x, y, square_of(x, y), df{px.kx2, 2.0f * px.kxl}, df{px.ky2, 2.0f * px.kyl}, df{px.cb, px.cbl}, dm, dp);
      });
    }
    return z;
  };

  float2 nxt[S][R];
  auto fetch = [&](int i) {
    const float2* g = Gt + (long long)(b_begin + i) * GCOLS * N + (long long)sg * S * N;
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int m = 0; m < R; ++m) nxt[s][m] = g[s * N + lane + 64 * m];
  };
  fetch(i0);
  for (int i = i0; i < i1; ++i) {
    const int b = b_begin + i;
    const float kx = as_const(gp.kx)[b], ky = as_const(gp.ky)[b];   // scalar loads
    const float kxl = as_const(gp.kxl)[b], kyl = as_const(gp.kyl)[b];
    px.kx2 = 2.0f * kx;
    px.ky2 = 2.0f * ky;
    px.kxl = kxl;
    px.kyl = kyl;
    {
      const df kxd{kx, kxl}, kyd{ky, kyl};
      const df cb = df_sub(rout2, df_add(df_mul(kxd, kxd), df_mul(kyd, kyd)));
      px.cb = cb.hi;
      px.cbl = cb.lo;
    }
    px.u = fmaf(2.0f * k4, fmaf(kx, kx, ky * ky), k0);
    px.vx = 2.0f * fmaf(m12c, kx, m12s * ky);
    px.vy = 2.0f * fmaf(m12s, kx, -(m12c * ky));
    px.ak = as_const(gp.ak)[b];
    px.margin = edge_margin(px.ak, ap);
    if (px.ak == 0.0f) px.cb = -1e30f;   // no overlap at all (ak takes part in no other form)
    if (px.ak == 0.0f) px.margin = ap.edge;
    px.chik = 0.0f;
    if constexpr (GENERAL) {
      float odd;
      chi_parts(ch.cp, kx, ky, px.chik, odd);
    }
    const bool nyq = reaches_nyquist(qn, kx, ap);   // wave-uniform
    float2 g[S][R];
#pragma unroll
    for (int s = 0; s < S; ++s)
#pragma unroll
      for (int m = 0; m < R; ++m) g[s][m] = nxt[s][m];
    fetch(min(i + 1, i1 - 1));   // unconditional: a load behind a branch is waited for at its end
    float2 c[S][R];
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const int j = sg * S + s;
      const float qy = as_const(gp.qy)[j];
#pragma unroll
      for (int m = 0; m < R; ++m) {
        c[s][m] = term(g[s][m], m, qx[m], j, qy);
        __builtin_amdgcn_sched_barrier(0);   // one point at a time
      }
      if (j != 0) {
        if (nyq) {
          // the Nyquist row (lane 0, m = R / 2): its partner, column N - j, is
          // evaluated at its own grid frequency (q_N/2, -qy)
          const float2 cb = term(cconj(g[s][R / 2]), R / 2, qx[R / 2], N - j, -qy);
          if (lane == 0) {
            const float2 ca = c[s][R / 2];
            Hrow[(long long)i * HALF + j] = make_float2(mean2(ca.x, cb.x), mean2(ca.y, -cb.y));
            c[s][R / 2] = make_float2(mean2(ca.x, -cb.x), mean2(ca.y, cb.y));
          }
        }
        // Y = -i C
#pragma unroll
        for (int m = 0; m < R; ++m) c[s][m] = make_float2(c[s][m].y, -c[s][m].x);
      }
    }
    float2 eg[S][R];
    if (sg == 0) {
      // slot 0: columns 0 and N/2, each with its own rows -q as partners
      float2 h[R];
      const float2* gh = Gt + ((long long)b * GCOLS + HALF) * N;
      const float qy = as_const(gp.qy)[HALF];
#pragma unroll
      for (int m = 0; m < R; ++m) h[m] = term(gh[lane + 64 * m], m, qx[m], HALF, qy);
      if (lane == 0) c[0][0] = make_float2(info->dc_re, info->dc_im);
      wave_fence();
      float2 pc[R], ph[R];
#pragma unroll
      for (int m = 0; m < R; ++m) xb[lane + 64 * m] = c[0][m];
      wave_fence();
#pragma unroll
      for (int m = 0; m < R; ++m) pc[m] = xb[(N - lane - 64 * m) & (N - 1)];
      wave_fence();
#pragma unroll
      for (int m = 0; m < R; ++m) xb[lane + 64 * m] = h[m];
      wave_fence();
#pragma unroll
      for (int m = 0; m < R; ++m) ph[m] = xb[(N - lane - 64 * m) & (N - 1)];
#pragma unroll
      for (int s = 0; s < S; ++s)
#pragma unroll
        for (int m = 0; m < R; ++m) eg[s][m] = make_float2(0.0f, 0.0f);
#pragma unroll
      for (int m = 0; m < R; ++m) {
        // D = (C - conj C(-Q)) / 2 and H = (C + conj C(-Q)) / 2 of both columns
        const float2 d0 = make_float2(mean2(c[0][m].x, -pc[m].x), mean2(c[0][m].y, pc[m].y));
        const float2 dh = make_float2(mean2(h[m].x, -ph[m].x), mean2(h[m].y, ph[m].y));
        const float2 h0 = make_float2(mean2(c[0][m].x, pc[m].x), mean2(c[0][m].y, -pc[m].y));
        const float2 hh = make_float2(mean2(h[m].x, ph[m].x), mean2(h[m].y, -ph[m].y));
        // Y0 + i Yh = -i D0 + Dh, and H0 + i Hh
        c[0][m] = make_float2(d0.y + dh.x, dh.y - d0.x);
        eg[0][m] = make_float2(h0.x - hh.y, h0.y + hh.x);
      }
    }
    float2 o[Fft::P][4];
    fft.run(c, xb, lane, o);
    float2* tb = T + ((long long)i * HALF + sg * S) * N;
#pragma unroll
    for (int p = 0; p < Fft::P; ++p)
#pragma unroll
      for (int r = 0; r < 4; ++r) tb[Fft::seq(lane, p) * N + Fft::index(lane, p, r)] = o[p][r];
    if (sg == 0) {
      fft.run(eg, xb, lane, o);
#pragma unroll
      for (int p = 0; p < Fft::P; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r)
          if (Fft::seq(lane, p) == 0) EG[(long long)i * N + Fft::index(lane, p, r)] = o[p][r];
    }
  }
}

// Block = ROWS rows x0.., split of the chunk's BF pixels: the block's W waves
// stage each BF pixel's ROWS x (N/2) values of T (whole 128-byte pieces) in
// LDS, the next pixel's on the way, and each transforms S pairs of rows.
// Moments are carried in M1/M2[split][x][y] as (Kahan sum, compensation);
// `first` starts them at 0.
template <int N, int S, int ROWS>
__global__ void __launch_bounds__(64 * (ROWS / (2 * S)))
k_phase_rows(const float2* __restrict__ T, const float2* __restrict__ EG, const float2* __restrict__ Hrow,
             const BfInfo* __restrict__ info, const float* __restrict__ kxp, const float* __restrict__ qxp, ApIso ap,
             int b_begin, int b_count, int nsplit, const float2* __restrict__ tw, float2* __restrict__ M1,
             float2* __restrict__ M2, int first) {
  typedef WaveIfft<N, S> Fft;
  constexpr int R = Fft::R, P = Fft::P, HALF = N / 2, W = ROWS / (2 * S), THREADS = 64 * W;
  constexpr int LD = ROWS + 2;                       // padded slot stride (float2): rows of 16-byte words spread over the banks
  constexpr int VEC = HALF * ROWS / 2 / THREADS;     // 16-byte loads a thread
  static_assert(VEC >= 1 && HALF * ROWS % (2 * THREADS) == 0, "whole loads");
  __shared__ __attribute__((aligned(16))) float2 tile[2][HALF * LD];
  __shared__ float2 xbuf[W][Fft::LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  float2* xb = xbuf[w];
  const int x0 = blockIdx.x * ROWS, split = blockIdx.y;
  int cnt = info->nbf - b_begin;
  cnt = cnt > b_count ? b_count : (cnt < 0 ? 0 : cnt);
  const int i0 = (int)((long long)split * cnt / nsplit), i1 = (int)((long long)(split + 1) * cnt / nsplit);
  Fft fft;
  fft.init(tw, lane);
  const float qn = as_const(qxp)[HALF];
  const long long plane = (long long)split * N * N;
  const int xw = x0 + 2 * S * w;                     // the wave's first row
  // position of output (p, r): rows xa, xa + 1 of the sequence, column y
  auto offset = [&](int p, int r) {
    return plane + (long long)(xw + 2 * Fft::seq(lane, p)) * N + Fft::index(lane, p, r);
  };
  Kahan k1[P][4][2], k2[P][4][2];
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        float2 u = make_float2(0.f, 0.f), v = u;
        if (!first) {
          u = M1[offset(p, r) + a * N];
          v = M2[offset(p, r) + a * N];
        }
        k1[p][r][a].s = u.x;
        k1[p][r][a].c = u.y;
        k2[p][r][a].s = v.x;
        k2[p][r][a].c = v.y;
      }
  float4 nxt[VEC];
  auto fetch = [&](int i) {
    const float2* tb = T + (long long)i * HALF * N + x0;
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      const int e = tid + v * THREADS, slot = e / (ROWS / 2), x = (e % (ROWS / 2)) * 2;
      nxt[v] = *reinterpret_cast<const float4*>(tb + (long long)slot * N + x);
    }
  };
  auto stage = [&](int buf) {
#pragma unroll
    for (int v = 0; v < VEC; ++v) {
      const int e = tid + v * THREADS, slot = e / (ROWS / 2), x = (e % (ROWS / 2)) * 2;
      *reinterpret_cast<float4*>(&tile[buf][slot * LD + x]) = nxt[v];
    }
  };
  if (i0 < i1) {
    fetch(i0);
    stage(0);
    fetch(min(i0 + 1, i1 - 1));
  }
  __syncthreads();
  for (int i = i0; i < i1; ++i) {
    const int cur = (i - i0) & 1;
    // e and g of the wave's rows (scalar loads: they wait for no prefetch)
    const Const<float> egp = as_const(reinterpret_cast<const float*>(EG + (long long)i * N + xw));
    float2 egv[2 * S];
#pragma unroll
    for (int a = 0; a < 2 * S; ++a) egv[a] = make_float2(egp[2 * a], egp[2 * a + 1]);
    const bool nyq = reaches_nyquist(qn, as_const(kxp)[b_begin + i], ap);
    float2 o[P][4];
    {
      float2 z[S][R];
#pragma unroll
      for (int s = 0; s < S; ++s) {
        const float2* t = tile[cur] + 2 * S * w + 2 * s;
        // Ya + i Yb of the rows' Hermitian spectra: elements c and N - c
#pragma unroll
        for (int m = 0; m < R; ++m) {
          const int c = lane + 64 * m;
          const int cs = c < HALF ? c : N - c;       // 0 and N/2 come from slot 0
          const float4 v = *reinterpret_cast<const float4*>(t + (c == HALF ? 0 : cs) * LD);
          float2 y;
          if (m < R / 2) {
            y = make_float2(v.x - v.w, v.y + v.z);
            if (m == 0 && lane == 0) y = make_float2(v.x, v.z);
          } else {
            y = make_float2(v.x + v.w, v.z - v.y);
            if (m == R / 2 && lane == 0) y = make_float2(v.y, v.w);
          }
          z[s][m] = y;
        }
      }
      fft.run(z, xb, lane, o);
    }
    float f[P][4];
#pragma unroll
    for (int p = 0; p < P; ++p)
#pragma unroll
      for (int r = 0; r < 4; ++r) f[p][r] = 0.0f;
    if (nyq) {
      // f(y): the Nyquist row of H, for every sequence (each lane needs its own y)
      float2 z[S][R], fo[P][4];
#pragma unroll
      for (int m = 0; m < R; ++m) {
        const int c = lane + 64 * m;
        float2 y = Hrow[(long long)i * HALF + (c < HALF ? c : (c == HALF ? 1 : N - c))];
        if (m >= R / 2) y.y = -y.y;
        if ((m == 0 || m == R / 2) && lane == 0) y = make_float2(0.f, 0.f);
#pragma unroll
        for (int s = 0; s < S; ++s) z[s][m] = y;
      }
      fft.run(z, xb, lane, fo);
#pragma unroll
      for (int p = 0; p < P; ++p)
#pragma unroll
        for (int r = 0; r < 4; ++r) f[p][r] = fo[p][r].x;
    }
#pragma unroll
    for (int p = 0; p < P; ++p) {
      const int s = Fft::seq(lane, p);
      float2 ea = egv[0], eb = egv[1];
#pragma unroll
      for (int a = 1; a < S; ++a) {
        if (s == a) {
          ea = egv[2 * a];
          eb = egv[2 * a + 1];
        }
      }
      float h[4][2], lo = INFINITY, hi = 0.0f;
      bool easy = true;
#pragma unroll
      for (int r = 0; r < 4; ++r) {
        const bool odd = Fft::index(lane, p, r) & 1;
        h[r][0] = ea.x + (odd ? -ea.y : ea.y) + f[p][r];
        h[r][1] = eb.x + (odd ? -eb.y : eb.y) - f[p][r];
        easy &= (h[r][0] > fabsf(o[p][r].x)) & (h[r][1] > fabsf(o[p][r].y));
        lo = fminf(lo, fminf(h[r][0], h[r][1]));
        hi = fmaxf(hi, fmaxf(h[r][0], h[r][1]));
      }
      easy &= (lo >= kQuotientLo) & (hi <= kQuotientHi);
      // a bright field brighter than its modulation leaves the first octants only
      float ph[4][2];
      if (__all(easy)) {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          ph[r][0] = atan_unit(quotient(o[p][r].x, h[r][0]));
          ph[r][1] = atan_unit(quotient(o[p][r].y, h[r][1]));
        }
      } else {
#pragma unroll
        for (int r = 0; r < 4; ++r) {
          ph[r][0] = phase_of(o[p][r].x, h[r][0]);
          ph[r][1] = phase_of(o[p][r].y, h[r][1]);
        }
      }
#pragma unroll
      for (int r = 0; r < 4; ++r)
#pragma unroll
        for (int a = 0; a < 2; ++a) {
          k1[p][r][a].add(ph[r][a]);
          k2[p][r][a].add(ph[r][a] * ph[r][a]);
        }
    }
    stage(cur ^ 1);              // (the last two rounds move a pixel that is not used)
    fetch(min(i + 2, i1 - 1));   // unconditional: a load behind a branch is waited for at its end
    __syncthreads();
  }
#pragma unroll
  for (int p = 0; p < P; ++p)
#pragma unroll
    for (int r = 0; r < 4; ++r)
#pragma unroll
      for (int a = 0; a < 2; ++a) {
        M1[offset(p, r) + a * N] = make_float2(k1[p][r][a].s, k1[p][r][a].c);
        M2[offset(p, r) + a * N] = make_float2(k2[p][r][a].s, k2[p][r][a].c);
      }
}

// ------------------------------------------------------------------------
// Launch
// ------------------------------------------------------------------------
bool phase_even_path(int N, int gcols, const Optics& o, bool odd) {
  return gcols == N / 2 + 1 && optics_isotropic(o) && !odd;
}

// BF pixels whose T (4 N^2 bytes each) is written before the row pass reads
// it: 67 MB, well inside the 256 MB last-level cache, but 268 MB at N = 256,
// where one launch a pass for 800 BF pixels (210 MB) is faster than four.
int phase_chunk_bf(int N) { return N == 128 ? 1024 : (N == 256 ? 1024 : (N == 512 ? 64 : 16)); }
int phase_splits(int N) { return N == 128 ? 128 : (N == 256 ? 32 : (N == 512 ? 8 : 4)); }

size_t phase_workspace_floats2(int N) {
  return (size_t)phase_chunk_bf(N) * (N / 2) * (N + 2 + 1) + 64;   // T, EG (N), Hrow (N/2)
}

hipError_t launch_phase_even(int N, const float2* Gt, const BfInfo* info, int nbf, const GeomPtrs& gp,
                             const EvenChi& ch, const EvenChi* ch_dev, const Optics& o, const float2* tw, float2* ws,
                             float2* M1, float2* M2, float* var_part, float* phase, float* loss, hipStream_t s) {
  df rout2;
  const ApIso ap = iso_aperture(o, rout2);
  const int chunk = phase_chunk_bf(N);
  const int nb = nbf > 0 ? nbf : 1;
  // Small selections.  A split costs the finishing kernel two planes: at least two BF
  // pixels each (a loss of 13 pixels at 128 x 128 takes 47 us in 128 splits, 22 in 7, 27
  // in 4; of 81 at 256 x 256 49 us in 32 and 51 in 21).  And waves enough for a few
  // rounds, whose first loads hide behind each other (81 pixels at 256 x 256: 57 us with
  // 2048 waves of two pixels, 46 with one pixel a wave; at 1024, one wave a SIMD, more
  // rounds cost 193 -> 199).
  const int nsplit = phase_splits(N) < (nb + 1) / 2 ? phase_splits(N) : (nb + 1) / 2;
  const int fill = N == 1024 ? 2048 : 8192;
  const int half = N / 2;
  float2* T = ws;
  float2* EG = T + (size_t)chunk * half * N;
  float2* Hrow = EG + (size_t)chunk * N;
#define QSSB_PHASE(NN, SC, SR, ROWS)                                                                              \
  do {                                                                                                            \
    int groups = cnt / 4; /* four BF pixels a wave, fewer to have `fill` waves */                                 \
    if (groups < fill / (half / SC)) groups = fill / (half / SC);                                                 \
    if (groups > cnt) groups = cnt;                                                                               \
    const unsigned g1 = (unsigned)(((long long)groups * (half / SC) + 3) / 4);                                    \
    if (ch.general)                                                                                               \
      hipLaunchKernelGGL((k_phase_cols<NN, SC, true>), dim3(g1), dim3(256), 0, s, Gt, info, gp, ch, ch_dev, ap, rout2, \
                         tw, b0, cnt, groups, T, EG, Hrow);                                                       \
    else                                                                                                          \
      hipLaunchKernelGGL((k_phase_cols<NN, SC, false>), dim3(g1), dim3(256), 0, s, Gt, info, gp, ch, ch_dev, ap,    \
                         rout2, tw, b0, cnt, groups, T, EG, Hrow);                                                \
    hipLaunchKernelGGL((k_phase_rows<NN, SR, ROWS>), dim3(NN / ROWS, nsplit), dim3(64 * (ROWS / (2 * SR))), 0, s, T, EG, \
                       Hrow, info, gp.kx, gp.qx, ap, b0, cnt, nsplit, tw, M1, M2, b0 == 0 ? 1 : 0);               \
  } while (0)
  for (int b0 = 0; b0 < nb; b0 += chunk) {
    const int cnt = nb - b0 < chunk ? nb - b0 : chunk;
    switch (N) {
      case 128: QSSB_PHASE(128, 2, 2, 16); break;
      case 256: QSSB_PHASE(256, 2, 1, 16); break;
      case 512: QSSB_PHASE(512, 1, 1, 8); break;
      case 1024: QSSB_PHASE(1024, 1, 1, 8); break;
      default: return hipErrorInvalidValue;
    }
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
  }
#undef QSSB_PHASE
  return launch_moments_finish(N, nsplit, info, M1, M2, var_part, phase, loss, s);
}

}  // namespace qssb
