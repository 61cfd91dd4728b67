// Object path of Hermitian stacks with equal detector sampling (every
// reconstruction, and sessions' object previews): S(Q) = sum_b G_b(Q)
// conj(Gamma^_b(Q)) over the columns c <= N/2 of the scan frequencies, with one
// phasor a term (overlap_term), and the scan-column FFT of a session's stack.
// The other columns follow: for an even chi the term at -Q is -conj of the term
// at Q, but for the Nyquist row, whose grid has no -Q, and for columns 0 and
// N/2, which are summed themselves.  Full-plane stacks and unequal detector
// sampling are in ssb_object.hip, the reduction of the partial planes too.
#include "ssb_internal.h"
#include "ssb_overlap.h"

namespace qssb {

namespace {

__device__ __forceinline__ float lane_value(float v, int lane) {
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), lane));
}

// The wave's BF pixel `lane` of 64 held one a lane: wave-uniform values.
__device__ __forceinline__ QuadPixel pixel_of_lane(const QuadPixel& p, int lane) {
  QuadPixel o;
  o.kx2 = lane_value(p.kx2, lane);
  o.ky2 = lane_value(p.ky2, lane);
  o.cb = lane_value(p.cb, lane);
  o.tx = lane_value(p.tx, lane);
  o.ty = lane_value(p.ty, lane);
  o.margin = lane_value(p.margin, lane);
  o.ak = lane_value(p.ak, lane);
  return o;
}

// BF pixels of group g of `groups`: g, g + groups, ...  Neighbours in the list
// are neighbours on the detector; dealt out in ranges, the groups at the edge
// of the disk would hold the pixels that need the general form most.
__device__ __forceinline__ int group_count(int g, int groups, int nbf) {
  return nbf > g ? (nbf - g + groups - 1) / groups : 0;
}

// Smallest and largest of a value over the wave (the scan frequencies may be
// set in any order).
__device__ __forceinline__ void wave_range(float v, float& lo, float& hi) {
  lo = hi = v;
#pragma unroll
  for (int off = 1; off < 64; off *= 2) {
    lo = fminf(lo, __shfl_xor(lo, off, 64));
    hi = fmaxf(hi, __shfl_xor(hi, off, 64));
  }
  lo = lane_value(lo, 0);
  hi = lane_value(hi, 0);
}

struct Kahan2 {
  Kahan r, i;
  __device__ __forceinline__ void init() {
    r.init();
    i.init();
  }
  __device__ __forceinline__ void add(float2 v) {
    r.add(v.x);
    i.add(v.y);
  }
  __device__ __forceinline__ float2 sum() const { return make_float2(r.s - r.c, i.s - i.c); }
};

// The term of one point, row q + dq and column col + dcol (sign -1: of -qy),
// given B = 2 q.k and base = Rout^2 - |k|^2 - |q|^2.
__device__ __forceinline__ float2 quad_term(float2 G, float B, float base, float s, float t, const QuadPixel& p,
                                            const ApIso& ap, const GeomPtrs& gp, df rout2, int b, int q, int dq, int col,
                                            int dcol, float sign) {
  const float near = base + fabsf(B), far = base - fabsf(B);
  t = B < 0.0f ? -t : t;
  return overlap_term(G, near, far, B, s, t, p.margin, p.ak, ap, [&](df& dm, df& dp) {
    asm volatile("" : "+v"(q), "+v"(col));   // no addresses kept ahead of the branch
    q += dq;
    col += dcol;
    const df kx{0.5f * p.kx2, as_const(gp.kxl)[b]}, ky{0.5f * p.ky2, as_const(gp.kyl)[b]};
    exact_d(df{gp.qx[q], gp.qxl[q]}, df{sign * gp.qy[col], sign * gp.qyl[col]}, kx, ky,
            df_sub(rout2, df_add(df_mul(kx, kx), df_mul(ky, ky))), dm, dp);
  });
}

__device__ __forceinline__ float half_sum(const QuadTurns& ev, float qx, float qy) {
  return fmaf(qx, fmaf(qx, ev.k0 + ev.m12c, 2.0f * qy * ev.m12s), qy * qy * (ev.k0 - ev.m12c));
}

}  // namespace

// ------------------------------------------------------------------------
// From a resident stack Gt[b][c][q].  A wave sums four tiles of 16 x 4
// frequencies (a point a lane: 128-byte pieces of G, and few tiles meet an
// aperture's edge, where the general form costs the wave three times the
// phasor) over one group of BF pixels.  The tiles lie in different quarters of
// the rows and of the columns, so that every wave has its share of the low
// frequencies, which are inside the apertures for every BF pixel; pixels whose
// apertures miss all four are passed over, and lanes outside both apertures
// load their tile's first value instead of their own.  Column N/2 is
// summed by waves of its own, 4 x 64 rows.
// ------------------------------------------------------------------------
template <int N>
__global__ void __launch_bounds__(256, 4)
k_object_tiles(const float2* __restrict__ Gt, const BfInfo* __restrict__ info, GeomPtrs gp, QuadTurns ev, ApIso ap,
               df rout2, int groups, float2* __restrict__ S_part) {
  constexpr int HALF = N / 2, GCOLS = HALF + 1;
  constexpr int RQ = N / 64, CQ = N / 32;            // tiles in a quarter of the rows, of the columns
  constexpr int SETS = RQ * CQ * 4, LAST = (N + 255) / 256;
  const int lane = threadIdx.x & 63;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int wave = blockIdx.x * 4 + w;
  const int g = wave % groups, t = wave / groups;
  if (t >= SETS + LAST) return;
  const bool last = t >= SETS;                       // column N/2
  const int turn = t & 3, rt = (t >> 2) % RQ, ct = (t >> 2) / RQ;
  const int n = group_count(g, groups, info->nbf);   // BF pixels g + i groups
  float2* sp = S_part + (long long)g * N * N;

  int row0[4], col0[4];                              // the tiles' first row and column (wave-uniform)
  float qx[4], qy[4], q2[4], s[4], x0[4], x1[4], y0[4], y1[4];
  const int lr = last ? lane : lane & 15, lc = last ? 0 : lane >> 4;
  const unsigned loff = lc * N + lr;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    row0[i] = last ? ((t - SETS) * 256 + 64 * i) & (N - 1) : (((i + turn) & 3) * RQ + rt) * 16;
    col0[i] = last ? HALF : (i * CQ + ct) * 4;
    qx[i] = gp.qx[row0[i] + lr];
    qy[i] = gp.qy[col0[i] + lc];
    wave_range(qx[i], x0[i], x1[i]);
    wave_range(qy[i], y0[i], y1[i]);
    // (at N = 128 the rows of column N/2 fill two of the four)
    q2[i] = last && (t - SETS) * 256 + 64 * i >= N ? INFINITY : fmaf(qx[i], qx[i], qy[i] * qy[i]);
    s[i] = half_sum(ev, qx[i], qy[i]);
  }
  // the tile of the rows from N/2, whose first row has partners of its own
  const int ny = last || rt != 0 ? -1 : (2 - turn) & 3;
  float nqx = 0.f, nqy = 0.f, nq2 = 0.f, ny0 = 0.f, ny1 = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i == ny) {
      nqx = qx[i];
      nqy = -qy[i];
      nq2 = q2[i];
      ny0 = -y1[i];
      ny1 = -y0[i];
    }
  }
  const float qn = as_const(gp.qx)[HALF];
  Kahan2 acc[4], nyq;
#pragma unroll
  for (int i = 0; i < 4; ++i) acc[i].init();
  nyq.init();

  struct Ahead {
    float2 G[4];
  };
  auto B_of = [&](int i, const QuadPixel& p) { return fmaf(qx[i], p.kx2, qy[i] * p.ky2) + 0.0f; };   // no negative zero
  for (int c0 = 0; c0 < n; c0 += 64) {
    const QuadPixel pl = quad_pixel(gp, g + min(c0 + lane, n - 1) * groups, ev, rout2);
    bool reach = ny >= 0 && apertures_reach(pl, rout2.hi, qn, qn, ny0, ny1);
    unsigned long long nmask = __ballot(reach);
#pragma unroll
    for (int i = 0; i < 4; ++i) reach |= apertures_reach(pl, rout2.hi, x0[i], x1[i], y0[i], y1[i]);
    unsigned long long mask = __ballot(reach && c0 + lane < n);
    if (!mask) continue;
    auto ahead = [&](int l, const QuadPixel& p) {
      Ahead a;
      const float2* gb = Gt + (long long)(g + (c0 + l) * groups) * GCOLS * N;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const bool in = p.cb - q2[i] + fabsf(B_of(i, p)) > -p.margin || (i == ny && lr == 0);
        const float2* gt = gb + (col0[i] * N + row0[i]);
        asm volatile("" : "+s"(gt));
        a.G[i] = gt[in ? loff : 0u];
      }
      return a;
    };
    int l = __builtin_ctzll(mask);
    QuadPixel p = pixel_of_lane(pl, l);
    Ahead cur = ahead(l, p);
    while (true) {
      mask &= mask - 1;
      const int ln = mask ? __builtin_ctzll(mask) : l;
      const QuadPixel pn = pixel_of_lane(pl, ln);
      const Ahead nxt = ahead(ln, pn);
      const int b = g + (c0 + l) * groups;
#pragma unroll
      for (int i = 0; i < 4; ++i) {
        const float B = B_of(i, p), base = p.cb - q2[i];
        if (base + fabsf(B) > -p.margin)
          acc[i].add(quad_term(cur.G[i], B, base, s[i], fmaf(qx[i], p.tx, qy[i] * p.ty), p, ap, gp, rout2, b, lr, row0[i],
                               lc, col0[i], 1.0f));
        __builtin_amdgcn_sched_barrier(0);
      }
      if (nmask >> l & 1) {
        // the Nyquist row's partners, columns N - j: their own frequencies (q_N/2, -qy)
        const float B = fmaf(nqx, p.kx2, nqy * p.ky2) + 0.0f, base = p.cb - nq2;
        float2 G = cur.G[0];
        int c = col0[0];
#pragma unroll
        for (int i = 1; i < 4; ++i) {
          if (i == ny) {
            G = cur.G[i];
            c = col0[i];
          }
        }
        if (lr == 0 && base + fabsf(B) > -p.margin)
          nyq.add(quad_term(cconj(G), B, base, half_sum(ev, nqx, nqy), fmaf(nqx, p.tx, nqy * p.ty), p, ap, gp, rout2, b, HALF,
                            0, lc, c, -1.0f));
      }
      if (!mask) break;
      cur = nxt;
      p = pn;
      l = ln;
    }
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int row = row0[i] + lr, col = col0[i] + lc;
    if (last && (t - SETS) * 256 + 64 * i >= N) continue;
    const float2 v = acc[i].sum();
    sp[(long long)col * N + row] = v;
    if (!last && col != 0)
      sp[(long long)(N - col) * N + ((N - row) & (N - 1))] = i == ny && lr == 0 ? nyq.sum() : make_float2(-v.x, v.y);
  }
}

// ------------------------------------------------------------------------
// From the row-transformed stack H[b][r][slot] (slot 0 packs the real columns 0
// and N/2).  A wave takes S = 1024 / N slot columns of every BF pixel of its
// group, 16 points a lane: N = K * 16, element jj + 16 m, the K-point DFTs over
// m in registers (over Q = K / 16 neighbouring lanes where K > 16), twiddles,
// one exchange through the wave's own LDS, then 16-point DFTs over jj, so that
// lane col * K + k1 ends with the rows k1 + K r of its column and every r of
// the wave is a tile of K rows and S columns.  A workgroup takes the 16 columns
// of one 128-byte line of H and keeps step over it with a barrier a BF pixel
// (without: the lines are fetched again).  BF pixels whose apertures miss the
// line's columns are passed over.  STORE: no sums, the stack is written.
// ------------------------------------------------------------------------
template <int N>
struct ColumnFft {
  static constexpr int S = 1024 / N, K = N / 16, HALF = N / 2;
  static constexpr int Q = K > 16 ? K / 16 : 1;
  static constexpr int SP = 17;                 // padded sequence stride
  static constexpr int LDS = 64 * SP;           // float2 of LDS a wave

  // load e (0..15) of a lane, from H's column base: row jj + 16 h + 16 Q e of
  // column lane / 16 Q, or (K = 8) row jj + 16 (e & 7) of column lane / 16 + 4 (e >> 3)
  __device__ static __forceinline__ unsigned load_lane(int lane, bool one) {
    const int row = (lane / Q & 15) + 16 * (lane % Q);
    return row * HALF + (one ? 0 : lane / (16 * Q));
  }
  __device__ static constexpr int load_step(int e, bool one) {
    return K == 8 ? 16 * (e & 7) * HALF + (one ? 0 : 4 * (e >> 3)) : 16 * Q * e * HALF;
  }

  __device__ static __forceinline__ float2 dpp(float2 v, bool far) {
    auto mv = [&](float x) {
      return __int_as_float(far ? __builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, true)
                                : __builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, true));
    };
    return make_float2(mv(v.x), mv(v.y));
  }

  // The lanes' twiddles, 64 a row (one address, no bank conflicts): rows 0..15
  // w_N^(jj k1) of output ka, rows 16.. w_K^(h ka) where lanes share a DFT.
  static constexpr int TW = 64 * (Q > 1 ? 32 : (K == 8 ? 8 : 16));
  __device__ static __forceinline__ int base_k1(int lane) {
    const int h = lane % Q;
    return Q == 4 ? 16 * (((h & 1) << 1) | (h >> 1)) : 16 * h;
  }
  __device__ static __forceinline__ void twiddles(float2* __restrict__ twl, const float2* __restrict__ tw, int tid,
                                                  int threads) {
    for (int i = tid; i < TW; i += threads) {
      const int lane = i & 63, k = i >> 6;
      const int jj = K == 8 ? lane & 15 : (lane / Q) & 15;
      twl[i] = k < 16 ? tw[((k + (K == 8 ? 0 : base_k1(lane))) * jj) & (N - 1)] : tw[(16 * (k - 16) * (lane % Q)) & (N - 1)];
    }
  }

  // x: the loads; on return x[r] = element lane % K + K r of column lane / K
  __device__ static __forceinline__ void run(float2 (&x)[16], const float2* __restrict__ twl, float2* __restrict__ ex,
                                             int lane) {
    const float2* tw = twl + lane;
    asm volatile("" ::: "memory");
    if constexpr (K == 8) {
      const int jj = lane & 15;
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float2 y[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) y[m] = x[8 * u + m];
        dft_regs<8, false>(y);
        float2* e = ex + ((lane >> 4) + 4 * u) * 8 * SP + jj;
        e[0] = y[0];
#pragma unroll
        for (int k = 1; k < 8; ++k) e[k * SP] = cmul(y[k], tw[64 * k]);
      }
    } else {
      const int h = lane % Q, jj = (lane / Q) & 15, col = lane / (16 * Q);
      dft_regs<16, false>(x);
      if constexpr (Q > 1) {
#pragma unroll
        for (int k = 1; k < 16; ++k) x[k] = cmul(x[k], tw[64 * (16 + k)]);
        if constexpr (Q == 4) {
#pragma unroll
          for (int k = 0; k < 16; ++k) {
            const float2 o = dpp(x[k], true);
            float2 v = (h & 2) ? csub(o, x[k]) : cadd(x[k], o);
            if (h == 3) v = cmul_mi<false>(v);
            x[k] = v;
          }
        }
#pragma unroll
        for (int k = 0; k < 16; ++k) {
          const float2 o = dpp(x[k], false);
          x[k] = (h & 1) ? csub(o, x[k]) : cadd(x[k], o);
        }
      }
      float2* e = ex + (col * K + (Q > 1 ? base_k1(lane) : 0)) * SP + jj;   // k1 = ka + base_k1
#pragma unroll
      for (int k = 0; k < 16; ++k) e[k * SP] = cmul(x[k], tw[64 * k]);
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = ex[lane * SP + j];
    asm volatile("" ::: "memory");
    dft_regs<16, false>(x);
  }

  // Columns 0 and N/2 come packed in slot 0's transform z: with zm = z of row
  // -q, (z + conj zm) / 2 and (z - conj zm) / 2i.  put: the lanes of column 0
  // leave their rows in LDS for mirror(r), the value of row -(k1 + K r).
  __device__ static __forceinline__ void put(const float2 (&x)[16], float2* __restrict__ ex, int lane) {
    asm volatile("" ::: "memory");
    if (lane < K) {
#pragma unroll
      for (int r = 0; r < 16; ++r) ex[lane * SP + r] = x[r];
      ex[lane * SP + 16] = x[0];
    }
    asm volatile("" ::: "memory");
  }
  __device__ static __forceinline__ float2 mirror(int r, const float2* __restrict__ ex, int lane) {
    const int k1 = lane % K;
    return ex[((K - k1) % K) * SP + (k1 == 0 ? 1 : 0) + 15 - r];
  }
};

__device__ __forceinline__ float2 unpack_first(float2 z, float2 zm) {
  return make_float2(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y));
}
__device__ __forceinline__ float2 unpack_half(float2 z, float2 zm) {
  return make_float2(0.5f * (z.y + zm.y), -0.5f * (z.x - zm.x));
}

constexpr int column_waves(int N) { return N == 128 ? 2 : 4; }

template <int N, bool STORE>
__global__ void __launch_bounds__(64 * column_waves(N), STORE ? 2 : 3)
k_columns(const float2* __restrict__ H, const BfInfo* __restrict__ info, GeomPtrs gp, QuadTurns ev, ApIso ap,
          df rout2, const float2* __restrict__ tw_g, int groups, float2* __restrict__ out) {
  typedef ColumnFft<N> Fft;
  constexpr int S = Fft::S, K = Fft::K, HALF = N / 2, GCOLS = HALF + 1;
  constexpr int NW = column_waves(N), CG = S * NW;   // columns a workgroup
  constexpr int NCG = HALF / CG, LG = 16 / CG;       // workgroups that share a line of H
  __shared__ float2 twl[Fft::TW];
  __shared__ float qxS[N];
  __shared__ float2 exS[NW][Fft::LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  for (int i = tid; i < N; i += 64 * NW) qxS[i] = gp.qx[i];
  Fft::twiddles(twl, tw_g, tid, 64 * NW);
  __syncthreads();
  float2* ex = exS[w];
  // workgroups go round the 8 XCDs: XCD x takes the groups x, x + 8, ..., the
  // low columns (the long items) first; the items of column N/2 come last, a
  // group a wave
  const int items = groups * NCG;
  int cg = NCG, gl = ((int)blockIdx.x - items) * NW + w;
  if ((int)blockIdx.x < items) {
    const int per = groups / 8 * LG, k8 = blockIdx.x >> 3;
    const int line = k8 / per, rem = k8 - line * per;
    cg = line * LG + rem % LG;
    gl = rem / LG * 8 + (blockIdx.x & 7);
  }
  const bool last = cg == NCG;
  if (gl >= groups) return;                             // (only waves of column N/2, which meet no barrier)
  const int n = group_count(gl, groups, info->nbf);  // BF pixels gl + i groups
  const int jbase = last ? 0 : cg * CG + S * w;
  const int col = lane / K, k1 = lane % K;
  const int j = last ? HALF : jbase + col;           // the lane's column after the transform
  const bool first_col = jbase == 0;                 // wave-uniform: it holds slot 0
  const bool live = !last || col == 0;

  const unsigned loff = Fft::load_lane(lane, last);
  float2 h[16];
  auto fetch = [&](int b) {
    const float2* hb = H + (long long)b * N * HALF + jbase;
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      const float2* he = hb + Fft::load_step(e, last);
      asm volatile("" : "+s"(he));   // a scalar address and one lane offset for all
      h[e] = he[loff];
    }
  };

  if constexpr (STORE) {
    if (n == 0) return;
    fetch(gl);
    for (int i = 0; i < n; ++i) {
      const int b = gl + i * groups;
      float2 x[16];
#pragma unroll
      for (int e = 0; e < 16; ++e) x[e] = h[e];
      __builtin_amdgcn_s_barrier();
      fetch(min(b + groups, gl + (n - 1) * groups));
      Fft::run(x, twl, ex, lane);
      float2* gb = out + (long long)b * GCOLS * N;
      if (first_col) {
        Fft::put(x, ex, lane);
        if (col == 0) {
#pragma unroll
          for (int r = 0; r < 16; ++r) {
            const float2 m = Fft::mirror(r, ex, lane);
            gb[(long long)HALF * N + k1 + K * r] = unpack_half(x[r], m);
            x[r] = unpack_first(x[r], m);
          }
        }
      }
#pragma unroll
      for (int r = 0; r < 16; ++r) gb[(long long)j * N + k1 + K * r] = x[r];
    }
  } else {
    const float qy = gp.qy[j];
    float y0, y1;
    wave_range(gp.qy[last ? HALF : cg * CG + lane % CG], y0, y1);
    const float qn = as_const(gp.qx)[HALF];
    const float sxx = ev.k0 + ev.m12c, sxy = 2.0f * qy * ev.m12s, syy = qy * qy * (ev.k0 - ev.m12c);
    Kahan2 acc[16], nyq;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r].init();
    nyq.init();
    for (int c0 = 0; c0 < n; c0 += 64) {
      const QuadPixel pl = quad_pixel(gp, gl + min(c0 + lane, n - 1) * groups, ev, rout2);
      // the same for every wave of the workgroup
      unsigned long long mask =
          __ballot(c0 + lane < n && apertures_reach(pl, rout2.hi, -INFINITY, INFINITY, y0, y1));
      if (!mask) continue;
      int l = __builtin_ctzll(mask);
      fetch(gl + (c0 + l) * groups);
      while (true) {
        const QuadPixel p = pixel_of_lane(pl, l);
        const int b = gl + (c0 + l) * groups;
        mask &= mask - 1;
        l = mask ? __builtin_ctzll(mask) : l;
        float2 x[16];
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] = h[e];
        Fft::run(x, twl, ex, lane);
        if (!last) __builtin_amdgcn_s_barrier();
        fetch(gl + (c0 + l) * groups);
        if (first_col) Fft::put(x, ex, lane);
        const float Bq = qy * p.ky2, tq = qy * p.ty;
        const float cq = live ? p.cb - qy * qy : -INFINITY;
#pragma unroll
        for (int r = 0; r < 16; ++r) {
          const float qx = qxS[k1 + K * r];
          const float B = fmaf(qx, p.kx2, Bq) + 0.0f;      // no negative zero
          const float base = fmaf(-qx, qx, cq);
          if (first_col && col == 0) {
            const float2 m = Fft::mirror(r, ex, lane);
            x[r] = last ? unpack_half(x[r], m) : unpack_first(x[r], m);
          }
          if (base + fabsf(B) > -p.margin)
            acc[r].add(quad_term(x[r], B, base, fmaf(qx, fmaf(qx, sxx, sxy), syy), fmaf(qx, p.tx, tq), p, ap, gp, rout2,
                                 b, k1, K * r, j, 0, 1.0f));
          __builtin_amdgcn_sched_barrier(0);               // one point at a time
        }
        if (!last && apertures_reach(p, rout2.hi, qn, qn, -y1, -y0)) {
          // the Nyquist row's partners, columns N - j: their own frequencies (q_N/2, -qy)
          const float B = fmaf(qn, p.kx2, -Bq) + 0.0f, base = fmaf(-qn, qn, cq);
          if (k1 == 0 && base + fabsf(B) > -p.margin)
            nyq.add(quad_term(cconj(x[8]), B, base, fmaf(qn, fmaf(qn, sxx, -sxy), syy), fmaf(qn, p.tx, -tq), p, ap, gp,
                              rout2, b, HALF, 0, j, 0, -1.0f));
        }
        if (!mask) break;
      }
    }
    if (!live) return;
    float2* sp = out + (long long)gl * N * N;
#pragma unroll
    for (int r = 0; r < 16; ++r) {
      const int q = k1 + K * r;
      const float2 v = acc[r].sum();
      sp[(long long)j * N + q] = v;
      if (!last && j != 0)
        sp[(long long)(N - j) * N + ((N - q) & (N - 1))] = q == HALF ? nyq.sum() : make_float2(-v.x, v.y);
    }
  }
}

// ------------------------------------------------------------------------
// Launch
// ------------------------------------------------------------------------
// From H: N = 512 and 1024.  A wave's loads take 32 bytes of every 128-byte
// line of H at N <= 256 and keep few waves busy there (16 points a lane are
// 8 waves a CU at 256): 151 us against k_trotter_wave's 119 at N = 256 and 114
// against k_trotter_slots' 53 at 128, but NEW_512 us against 867 at 512.
bool columns_path(int N, const Optics& o) { return N >= 512 && optics_isotropic(o); }

// BF groups (partial planes): the tuner's candidates, the default first.
int columns_variants(int N) { return N == 512 ? 3 : 1; }
int columns_groups(int N, int variant) {
  return N == 512 ? 32 >> (variant > 0 && variant < 3 ? variant : 0) : 8;
}
// 4096 waves where the partial planes are few: four a SIMD, all in flight at once
// (with three a SIMD a third of them made a second round: 60 us for 53 at N = 256)
int object_tile_groups(int N) { return N == 128 ? 64 : (N == 256 ? 32 : (N == 512 ? 8 : 2)); }

#define QSSB_BY_SIZE(CALL) \
  switch (N) {             \
    case 128: CALL(128); break; \
    case 256: CALL(256); break; \
    case 512: CALL(512); break; \
    case 1024: CALL(1024); break; \
    default: return hipErrorInvalidValue; \
  }

hipError_t launch_object_tiles(int N, const float2* Gt, const BfInfo* info, const GeomPtrs& gp, const QuadTurns& ev,
                               const Optics& o, float2* S_part, hipStream_t s, int* groups_used) {
  df rout2;
  const ApIso ap = iso_aperture(o, rout2);
  const int groups = object_tile_groups(N);
  const unsigned grid = (unsigned)(groups * ((N / 64) * (N / 32) + (N + 1023) / 1024));
#define QSSB_CALL(NN) \
  hipLaunchKernelGGL((k_object_tiles<NN>), dim3(grid), dim3(256), 0, s, Gt, info, gp, ev, ap, rout2, groups, S_part)
  QSSB_BY_SIZE(QSSB_CALL)
#undef QSSB_CALL
  *groups_used = groups;
  return hipGetLastError();
}

hipError_t launch_columns_trotter(int N, const float2* H, const BfInfo* info, const GeomPtrs& gp, const QuadTurns& ev,
                                  const Optics& o, const float2* tw, float2* S_part, int variant, hipStream_t s,
                                  int* groups_used) {
  df rout2;
  const ApIso ap = iso_aperture(o, rout2);
  const int groups = columns_groups(N, variant), nw = column_waves(N);   // groups: whole rounds of the 8 XCDs
  const unsigned grid = (unsigned)(groups * (N / 2 / (1024 / N * nw)) + (groups + nw - 1) / nw);
#define QSSB_CALL(NN)                                                                                               \
  hipLaunchKernelGGL((k_columns<NN, false>), dim3(grid), dim3(64 * column_waves(NN)), 0, s, H, info, gp, ev, ap, rout2, \
                     tw, groups, S_part)
  switch (N) {
    case 512: QSSB_CALL(512); break;
    case 1024: QSSB_CALL(1024); break;
    default: return hipErrorInvalidValue;
  }
#undef QSSB_CALL
  *groups_used = groups;
  return hipGetLastError();
}

// H to the resident stack Gt[b][c][q], c <= N/2.
hipError_t launch_columns_store(int N, const float2* H, const BfInfo* info, const GeomPtrs& gp, const float2* tw,
                                float2* Gt, hipStream_t s) {
  const int groups = N <= 256 ? 128 : 64;
  const unsigned grid = (unsigned)(groups * (N / 2 / (1024 / N * column_waves(N))));
#define QSSB_CALL(NN)                                                                                                \
  hipLaunchKernelGGL((k_columns<NN, true>), dim3(grid), dim3(64 * column_waves(NN)), 0, s, H, info, gp, QuadTurns{}, ApIso{}, df{0.f, 0.f}, \
                     tw, groups, Gt)
  QSSB_BY_SIZE(QSSB_CALL)
#undef QSSB_CALL
  return hipGetLastError();
}
#undef QSSB_BY_SIZE

}  // namespace qssb
