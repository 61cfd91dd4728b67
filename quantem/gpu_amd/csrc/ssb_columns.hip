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
  o.kx2l = lane_value(p.kx2l, lane);
  o.ky2l = lane_value(p.ky2l, lane);
  o.cbl = lane_value(p.cbl, lane);
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

// The term of one point, given B = 2 q.k and base = Rout^2 - |k|^2 - |q|^2; point
// gives its frequency in double-float, in the branch that needs it.
template <typename Point>
__device__ __forceinline__ float2 quad_term(float2 G, float B, float base, float s, float t, bool whole,
                                            const QuadPixel& p, const ApIso& ap, Point point) {
  const float near = base + fabsf(B), far = base - fabsf(B);
  t = B < 0.0f ? -t : t;
  return overlap_term(G, near, far, B, s, t, whole, p.margin, p.ak, ap, [&](float& dm, float& dp) {
    df x, y;
    point(x, y);
    exact_d(x, y, square_of(x, y), df{p.kx2, p.kx2l}, df{p.ky2, p.ky2l}, df{p.cb, p.cbl}, dm, dp);
  });
}

// k q^2 less its whole turns (2: the period of e^{i pi s}), for s of overlap_unit: s =
// turn_part(sxx, qx) + turn_part(syy, qy) + qx cross_part(sxy, qy).  Each part is rounded at its
// remainder, not at its tens of turns.  Odd in k: where C10 and C12 cancel (on the
// diagonals without C10, on an axis with |C10| = |C12|) s is zero, not what rounding
// leaves, whose sign the term would take.
__device__ __forceinline__ float turn_part(df k, df q) {
#pragma clang fp contract(off)
  const df v = df_mul(k, df_mul(q, q));
  const float n = rintf(0.5f * v.hi);
  return (v.hi - 2.0f * n) + v.lo;
}
__device__ __forceinline__ float cross_part(df k, df q) { return 2.0f * df_mul(k, q).hi; }

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

  // a lane's four frequencies in double-float, for the points at an edge (from LDS: the
  // wave waits less than for the tables)
  __shared__ float4 own[4 * 256];
  auto own_point = [&](int i, float sign, df& x, df& y) {
    int at = i * 256 + threadIdx.x;
    asm volatile("" : "+v"(at));                     // in the branch, not ahead of it
    const float4 v = own[at];
    x = df{v.x, v.y};
    y = df{sign * v.z, sign * v.w};
  };
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
    const df x{qx[i], gp.qxl[row0[i] + lr]}, y{qy[i], gp.qyl[col0[i] + lc]};
    s[i] = fmaf(qx[i], cross_part(ev.sxy, y), turn_part(ev.sxx, x) + turn_part(ev.syy, y));
    own[i * 256 + threadIdx.x] = make_float4(x.hi, x.lo, y.hi, y.lo);
  }
  // the tile of the rows from N/2, whose first row has partners of its own
  const int ny = last || rt != 0 ? -1 : (2 - turn) & 3;
  float nqx = 0.f, nqy = 0.f, nq2 = 0.f, ns = 0.f, ny0 = 0.f, ny1 = 0.f;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    if (i == ny) {
      nqx = qx[i];
      nqy = -qy[i];
      nq2 = q2[i];
      ns = fmaf(nqx, 4.0f * nqy * ev.sxy.hi, s[i]);   // its term in qx qy the other way round
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
    const QuadPixel pl = quad_pixel(gp, g + min(c0 + lane, n - 1) * groups, ev, rout2, ap);
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
          acc[i].add(quad_term(cur.G[i], B, base, s[i], fmaf(qx[i], p.tx, qy[i] * p.ty), near_whole(s[i]), p, ap,
                               [&](df& x, df& y) { own_point(i, 1.0f, x, y); }));
        __builtin_amdgcn_sched_barrier(0);
      }
      if (nmask >> l & 1) {
        // the Nyquist row's partners, columns N - j: their own frequencies (q_N/2, -qy)
        const float B = fmaf(nqx, p.kx2, nqy * p.ky2) + 0.0f, base = p.cb - nq2;
        float2 G = cur.G[0];
#pragma unroll
        for (int i = 1; i < 4; ++i) {
          if (i == ny) {
            G = cur.G[i];
          }
        }
        if (lr == 0 && base + fabsf(B) > -p.margin)
          nyq.add(quad_term(cconj(G), B, base, ns, fmaf(nqx, p.tx, nqy * p.ty), near_whole(ns), p, ap,
                            [&](df& x, df& y) { own_point(ny, -1.0f, x, y); }));
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
// the wave is a tile of K rows and S columns.  A workgroup loads its waves'
// columns together (a 128-byte line of every row of H; half a line at 512),
// one BF pixel ahead, and deals them out through LDS: with a wave's own loads,
// 32 or 16 bytes of every line, the lines went through the caches eight times
// (N = 256: 151 us a reconstruction for 112, 512: 412 for 263; the workgroup
// kernels before: 119 and 867).  BF pixels whose apertures miss the workgroup's
// columns are passed over.  STORE: no sums, the stack is written.
// Two to three waves a SIMD (64 registers of sums) and the exchanges bound it:
// 800 BF pixels at 256 move 150 MB in 96 us, at 512 take 303 (93 and 263 with
// the lens' soft band from float32 estimates, wrong by up to 1e-5 of a term).
// ------------------------------------------------------------------------
// Workgroup barrier for LDS only: this wave's LDS operations complete, then
// s_barrier; its global loads stay in flight.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

template <int N>
struct ColumnFft {
  static constexpr int S = 1024 / N, K = N / 16, HALF = N / 2;
  static constexpr int Q = K > 16 ? K / 16 : 1;
  static constexpr int SP = 17;                 // padded stride of the 16-value sequences
  // padded column stride: the 32 lanes of a staging write (whole rows of the
  // workgroup's columns) meet every bank once
  static constexpr int CS = K * SP + (K == 64 ? 8 : (K == 32 ? 4 : (K == 16 ? 2 : 10)));
  static constexpr int LDS = S * CS;            // float2 of LDS a wave

  // where row and column (of the wave's S) of the staged values lie
  __device__ static __forceinline__ int place(int row, int col) { return col * CS + (row >> 4) * SP + (row & 15); }

  __device__ static __forceinline__ float2 dpp(float2 v, bool far) {
    auto mv = [&](float x) {
      return __int_as_float(far ? __builtin_amdgcn_mov_dpp(__float_as_int(x), 0x4E, 0xF, 0xF, true)
                                : __builtin_amdgcn_mov_dpp(__float_as_int(x), 0xB1, 0xF, 0xF, true));
    };
    return make_float2(mv(v.x), mv(v.y));
  }

  // The lanes' twiddles, 64 a row (one address, no bank conflicts): w_N^(jj k1) of
  // output ka; after them w_K^(h ka) where lanes share a DFT, Q a row (lanes of one h
  // read one address).
  static constexpr int TW1 = 64 * (K == 8 ? 8 : 16), TW = TW1 + (Q > 1 ? 16 * Q : 0);
  __device__ static __forceinline__ int base_k1(int lane) {
    const int h = lane % Q;
    return Q == 4 ? 16 * (((h & 1) << 1) | (h >> 1)) : 16 * h;
  }
  __device__ static __forceinline__ void twiddles(float2* __restrict__ twl, const float2* __restrict__ tw, int tid,
                                                  int threads) {
    for (int i = tid; i < TW; i += threads) {
      const int lane = i & 63, k = i >> 6, u = i - TW1;
      const int jj = K == 8 ? lane & 15 : (lane / Q) & 15;
      twl[i] = tw[(i < TW1 ? (k + (K == 8 ? 0 : base_k1(lane))) * jj : 16 * (u / Q) * (u % Q)) & (N - 1)];
    }
  }

  // From the staged values; x[r] = element lane % K + K r of column lane / K.
  __device__ static __forceinline__ void run(float2 (&x)[16], const float2* __restrict__ twl, float2* __restrict__ ex,
                                             int lane) {
    const float2* tw = twl + lane;
    if constexpr (K == 8) {
      const int jj = lane & 15;
      float2* e = ex + (lane >> 4) * CS + jj;
#pragma unroll
      for (int m = 0; m < 16; ++m) x[m] = e[(m >> 3) * 4 * CS + (m & 7) * SP];
      asm volatile("" ::: "memory");
#pragma unroll
      for (int u = 0; u < 2; ++u) {
        float2 y[8];
#pragma unroll
        for (int m = 0; m < 8; ++m) y[m] = x[8 * u + m];
        dft_regs<8, false>(y);
        float2* eu = e + 4 * u * CS;
        eu[0] = y[0];
#pragma unroll
        for (int k = 1; k < 8; ++k) eu[k * SP] = cmul(y[k], tw[64 * k]);
      }
    } else {
      const int h = lane % Q, jj = (lane / Q) & 15, col = lane / (16 * Q);
#pragma unroll
      for (int m = 0; m < 16; ++m) x[m] = ex[col * CS + (Q * m + h) * SP + jj];
      asm volatile("" ::: "memory");
      dft_regs<16, false>(x);
      if constexpr (Q > 1) {
#pragma unroll
        for (int k = 1; k < 16; ++k) x[k] = cmul(x[k], twl[TW1 + k * Q + h]);
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
      float2* e = ex + col * CS + (Q > 1 ? base_k1(lane) : 0) * SP + jj;   // k1 = ka + base_k1
#pragma unroll
      for (int k = 0; k < 16; ++k) e[k * SP] = cmul(x[k], tw[64 * k]);
    }
    asm volatile("" ::: "memory");
#pragma unroll
    for (int j = 0; j < 16; ++j) x[j] = ex[(lane / K) * CS + (lane % K) * SP + j];
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
          df rout2, const float2* __restrict__ tw_g, int groups, int part, int parts, float2* __restrict__ out) {
  typedef ColumnFft<N> Fft;
  constexpr int S = Fft::S, K = Fft::K, HALF = N / 2, GCOLS = HALF + 1;
  constexpr int NW = column_waves(N), CG = S * NW;   // columns a workgroup
  constexpr int NCG = HALF / CG, LG = 16 / CG;       // workgroups that share a line of H
  __shared__ float2 twl[Fft::TW];
  // the rows' frequencies (high and low words) and parts of s, the columns' frequencies
  __shared__ float qxS[STORE ? 1 : N], qxlS[STORE ? 1 : N], sxS[STORE ? 1 : N];
  __shared__ float2 qyS[CG];
  __shared__ float2 exS[NW][Fft::LDS];
  const int tid = threadIdx.x, lane = tid & 63;
  const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
  if constexpr (!STORE) {
    for (int i = tid; i < N; i += 64 * NW) {
      const df x{gp.qx[i], gp.qxl[i]};
      qxS[i] = x.hi;
      qxlS[i] = x.lo;
      sxS[i] = turn_part(ev.sxx, x);
    }
  }
  Fft::twiddles(twl, tw_g, tid, 64 * NW);
  __syncthreads();
  float2* ex = exS[w];
  // part `part` of `parts`: BF pixels [lo, hi) into its share of the groups
  const int nbf = info->nbf;
  const int lo = (int)((long long)nbf * part / parts), hi = (int)((long long)nbf * (part + 1) / parts);
  const int gpp = groups / parts;
  // workgroups go round the 8 XCDs: XCD x takes the groups x, x + 8, ..., the
  // low columns (the long items) first, column N/2 last
  const int per = gpp / 8 * LG, k8 = blockIdx.x >> 3;
  const int line = k8 / per, rem = k8 - line * per;
  const bool last = line * LG >= NCG;                // one item a group, of the columns that hold slot 0
  const int cg = last ? 0 : line * LG + rem % LG;
  const int gl = (last ? k8 - NCG / LG * per : rem / LG) * 8 + (blockIdx.x & 7);
  const int n = group_count(gl, gpp, hi - lo);
  const int bg = lo + gl;                            // BF pixels bg + i gpp
  const int jbase = cg * CG + S * w;
  const int col = lane / K, k1 = lane % K;
  const int j = last ? HALF : jbase + col;           // the lane's column after the transform
  const bool first_col = jbase == 0;                 // wave-uniform: it holds slot 0
  const bool live = !last || (w == 0 && col == 0);

  // the workgroup's rows of CG columns, 16 bytes a lane and load, whole pieces
  // of H's lines, to the waves' columns through LDS
  constexpr int ROWS = 64 * NW / (CG / 2), VEC = N / ROWS;
  static_assert(VEC == 8, "8 loads a lane");
  const int lrow = tid / (CG / 2), lcol = tid % (CG / 2) * 2;
  const unsigned loff = lrow * (HALF / 2) + lcol / 2;
  float4 h[VEC];
  auto fetch = [&](int b) {
    const float4* hb = reinterpret_cast<const float4*>(H + (long long)b * N * HALF + cg * CG);
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      const float4* he = hb + e * ROWS * (HALF / 2);
      asm volatile("" : "+s"(he));   // a scalar address and one lane offset for all
      h[e] = he[loff];
    }
  };
  float2* const st0 = exS[lcol / S] + Fft::place(lrow, lcol % S);
  float2* const st1 = exS[(lcol + 1) / S] + Fft::place(lrow, (lcol + 1) % S);
  auto stage = [&]() {
    lds_barrier();                                   // every wave is done with the pixel before
#pragma unroll
    for (int e = 0; e < VEC; ++e) {
      constexpr int step = ROWS / 16 * Fft::SP;
      static_assert(ROWS % 16 == 0, "a load moves whole sequences on");
      st0[e * step] = make_float2(h[e].x, h[e].y);
      st1[e * step] = make_float2(h[e].z, h[e].w);
    }
  };

  if constexpr (STORE) {
    if (n == 0) return;
    fetch(bg);
    for (int i = 0; i < n; ++i) {
      const int b = bg + i * gpp;
      stage();
      fetch(min(b + gpp, bg + (n - 1) * gpp));
      lds_barrier();
      float2 x[16];
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
    if (tid < CG) qyS[tid] = make_float2(gp.qy[last ? HALF : cg * CG + tid], gp.qyl[last ? HALF : cg * CG + tid]);
    __syncthreads();
    auto point = [&](int q, int dq, float sign, df& x, df& y) {
      int c = last ? 0 : S * w + col;
      asm volatile("" : "+v"(q), "+v"(c));           // no addresses kept ahead of the branch
      x = df{qxS[q + dq], qxlS[q + dq]};
      const float2 v = qyS[c];
      y = df{sign * v.x, sign * v.y};
    };
    float y0, y1;
    wave_range(gp.qy[last ? HALF : cg * CG + lane % CG], y0, y1);
    const float qn = as_const(gp.qx)[HALF];
    const df yd{qy, gp.qyl[j]};
    const float sxy = cross_part(ev.sxy, yd), sy = turn_part(ev.syy, yd);
    // whether a point of the wave, the mean's apart, has s near a whole number: s is
    // the point's alone, and without one its terms need not ask (a scalar branch)
    bool whole = false;
    for (int r = 0; r < 16; ++r)
      whole |= near_whole(fmaf(qxS[k1 + K * r], sxy, sxS[k1 + K * r] + sy)) && (j != 0 || k1 + K * r != 0);
    const bool ask = __any(whole);
    Kahan2 acc[16], nyq;
#pragma unroll
    for (int r = 0; r < 16; ++r) acc[r].init();
    nyq.init();
    for (int c0 = 0; c0 < n; c0 += 64) {
      const QuadPixel pl = quad_pixel(gp, bg + min(c0 + lane, n - 1) * gpp, ev, rout2, ap);
      // the same for every wave of the workgroup
      unsigned long long mask =
          __ballot(c0 + lane < n && apertures_reach(pl, rout2.hi, -INFINITY, INFINITY, y0, y1));
      if (!mask) continue;
      int l = __builtin_ctzll(mask);
      fetch(bg + (c0 + l) * gpp);
      while (true) {
        const QuadPixel p = pixel_of_lane(pl, l);
        const int b = bg + (c0 + l) * gpp;
        mask &= mask - 1;
        l = mask ? __builtin_ctzll(mask) : l;
        stage();
        fetch(bg + (c0 + l) * gpp);               // the next pixel's, while this one's are summed
        lds_barrier();
        if (last && w != 0) {
          if (!mask) break;
          continue;
        }
        float2 x[16];
        Fft::run(x, twl, ex, lane);
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
          const float s = fmaf(qx, sxy, sxS[k1 + K * r] + sy);
          whole = false;
          if (ask) {
            float at = s;
            asm volatile("" : "+v"(at));             // not ahead of the branch
            whole = near_whole(at);
          }
          if (base + fabsf(B) > -p.margin)
            acc[r].add(quad_term(x[r], B, base, s, fmaf(qx, p.tx, tq), whole, p, ap,
                                 [&](df& x, df& y) { point(k1, K * r, 1.0f, x, y); }));
          __builtin_amdgcn_sched_barrier(0);               // one point at a time
        }
        if (!last && apertures_reach(p, rout2.hi, qn, qn, -y1, -y0)) {
          // the Nyquist row's partners, columns N - j: their own frequencies (q_N/2, -qy)
          const float B = fmaf(qn, p.kx2, -Bq) + 0.0f, base = fmaf(-qn, qn, cq);
          const float ns = fmaf(qn, -sxy, sxS[HALF] + sy);
          if (k1 == 0 && base + fabsf(B) > -p.margin)
            nyq.add(quad_term(cconj(x[8]), B, base, ns, fmaf(qn, p.tx, -tq), near_whole(ns), p, ap,
                              [&](df& x, df& y) { point(HALF, 0, -1.0f, x, y); }));
        }
        if (!mask) break;
      }
    }
    if (!live) return;
    float2* sp = out + (long long)(part * gpp + gl) * N * N;
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
// From H: N >= 256.  At 128 a wave's 16 points a lane keep few waves busy: 94 us
// in 64 groups and 49 in 192, with 9 and 22 us to sum the planes, against
// k_trotter_slots' 53 and 9.
bool columns_path(int N, const Optics& o) { return N >= 256 && optics_isotropic(o); }

// BF groups (partial planes): the tuner's candidates, the default first.  Whole
// rounds of the 8 XCDs in each of two parts.  At N = 256 (800 BF pixels) 64, 96
// and 128 take 112, 93 and 91 us, their sums 8, 10 and 13; at 512 32, 64 and
// 128 take 263, 277 and 305, their sums 14, 24 and 54.  Fewer groups keep fewer
// waves in flight and are there for small selections: whole reconstructions of 48 x 48
// frames with 800 BF pixels take 290, 313, 336, 401 and 589 us with the candidates at
// 256 and 996, 1185 and 1565 us at 512.
int columns_variants(int N) { return N == 512 ? 3 : (N == 256 ? 5 : 1); }
int columns_groups(int N, int variant) {
  static const int g256[5] = {96, 64, 48, 32, 16};
  if (variant < 0 || variant >= columns_variants(N)) variant = 0;
  return N == 512 ? 32 >> variant : (N == 256 ? g256[variant] : 8);
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
                                  int* groups_used, int part, int parts) {
  df rout2;
  const ApIso ap = iso_aperture(o, rout2);
  const int groups = columns_groups(N, variant), nw = column_waves(N);
  if (parts < 1 || part < 0 || part >= parts || groups % (8 * parts)) return hipErrorInvalidValue;
  const unsigned grid = (unsigned)(groups / parts * (N / 2 / (1024 / N * nw) + 1));
#define QSSB_CALL(NN)                                                                                               \
  hipLaunchKernelGGL((k_columns<NN, false>), dim3(grid), dim3(64 * column_waves(NN)), 0, s, H, info, gp, ev, ap, rout2, \
                     tw, groups, part, parts, S_part)
  switch (N) {
    case 256: QSSB_CALL(256); break;
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
                     tw, groups, 0, 1, Gt)
  QSSB_BY_SIZE(QSSB_CALL)
#undef QSSB_CALL
  return hipGetLastError();
}
#undef QSSB_BY_SIZE

}  // namespace qssb
