// Object-path kernels of the MI355X SSB engine: the trotter reduction over
// bright-field pixels (fused with the scan-column FFT when it starts from the
// row-transformed stack H, or reading a resident Fourier stack), and the
// final inverse FFT to the object and its phase.
//
// Reference behaviour (paths relative to bobleesj/quantem.gpu):
//   Fourier-sum trotter   src/quantem/gpu/ssb/compute/cuda/kernels/fft256.py:967-1030
//   overlap / guard       src/quantem/gpu/ssb/compute/cuda/kernels/common.py:115-236
//   object + IFFT         src/quantem/gpu/ssb/compute/cuda/engine.py:1047-1107
//   phase = angle(object) src/quantem/gpu/ssb/results.py:117-122
#include "ssb_internal.h"
#include "ssb_overlap.h"

namespace qssb {

int object_groups(int N) { return N == 128 ? 64 : (N == 256 ? 16 : (N == 512 ? 8 : 4)); }

// The phasor tables (PhasorJob) on their own launch; m_dev, when given,
// holds the quadratic chi instead of m_arg.
__global__ void __launch_bounds__(256)
k_phasors(const BfInfo* __restrict__ info, GeomPtrs gp, QuadChi m_arg, int N, float2* __restrict__ rowph,
          float2* __restrict__ colph, float2* __restrict__ echi, const QuadChi* __restrict__ m_dev) {
  const PhasorJob j{info, gp, m_dev ? *m_dev : m_arg, N, rowph, colph, echi};
  phasor_work(j, (long long)blockIdx.x * 256 + threadIdx.x, (long long)gridDim.x * 256);
}

// ------------------------------------------------------------------------
// Trotter over Hermitian slot columns.  Work item = (BF group g, slot group
// sg of SG slots).  Per BF pixel the slot columns G_b(:, j) are staged in
// LDS -- from H through the scan-column FFT (FROM_H) or copied from the
// resident stack Gt[b][c][q] -- and each G_b(q, j) contributes to
//   output A = S(q, j)          with G_b(q, j), and
//   output B = S(-q, N-j)       with conj(G_b(q, j))        (j >= 1),
// or, for slot 0, A = S(q, 0) with G_b(q, 0) and B = S(q, N/2) with
// G_b(q, N/2) (slot 0 of H packs the two real columns 0 and N/2).
// For j >= 1 and q != N/2, Q_B = -Q_A, so chi(Q_B) = chi(Q_A),
// theta_B = -theta_A, A(Q_B -/+ k) = A(Q_A +/- k): one aperture pair and one
// phasor serve both outputs.  Points whose two apertures vanish contribute
// exactly zero and are skipped.
// BLOCK is a multiple of N: each thread keeps one scan-frequency row q.
// ------------------------------------------------------------------------
template <int N, int SG, int BLOCK, bool FROM_H, bool ISO>
__global__ void __launch_bounds__(BLOCK)
k_trotter_slots(const float2* __restrict__ src, const BfInfo* __restrict__ info, GeomPtrs gp,
                const float2* __restrict__ rowph_g, const float2* __restrict__ colph_g,
                const float2* __restrict__ echi_g, ApIso ap, df rout2, Optics o,
                const float2* __restrict__ tw_g, int groups, float2* __restrict__ S_part) {
  constexpr int HALF = N / 2;
  constexpr int NSG = HALF / SG;
  constexpr int P = SG * N / BLOCK;      // points per thread
  constexpr int SSTEP = BLOCK / N;       // slot step between a thread's points
  constexpr int GCOLS = HALF + 1;
  constexpr int TILE = N * SG;           // complex values per BF tile
  constexpr int COPIES = (TILE + 2 * BLOCK - 1) / (2 * BLOCK);
  constexpr int TSTRIDE = N + 1;
  // slot groups sharing one 128-byte line of H
  constexpr int LG = (FROM_H && SG * 8 < 128) ? 128 / (SG * 8) : 1;
  static_assert(TILE % 128 == 0, "tile must split into whole waves of 16-byte copies");
  // a lane's 16-byte copy takes two adjacent slots of one row of H
  static_assert(!FROM_H || SG % 2 == 0, "row-transformed stacks need an even slot count");
  // Async landing buffers (double-buffered).  FROM_H: interleaved rows of H,
  // element (s, r) at [r * SG + s]; otherwise Gt columns, (s, q) at [s * N + q].
  __shared__ __attribute__((aligned(16))) float2 abuf[2][TILE];
  // FROM_H: transformed columns, (s, q) at [s * TSTRIDE + q]
  __shared__ float2 tileT[FROM_H ? SG * TSTRIDE : 1];
  __shared__ float2 tw[FROM_H ? N : 1];
  __shared__ float qyS[SG + 1], qySl[SG + 1];
  // output-B constants where Q_B != -Q_A: column N/2 (slot 0) per row, and
  // the Nyquist row q = N/2 per slot
  __shared__ float2 ehalfc[N];
  __shared__ df q2halfc[N];
  __shared__ float2 enyqr[SG];
  // ISO: column terms of d(Q -/+ k) for the SG slot columns and column N/2,
  // double-buffered over BF pixels:
  //   colA = (Rout^2 - |k|^2) - qy^2 + 2 qy ky,  colB = (Rout^2 - |k|^2) - qy^2 - 2 qy ky
  __shared__ df colA_s[2][SG + 1], colB_s[2][SG + 1];

  const int tid = threadIdx.x;
  if (FROM_H)
    for (int i = tid; i < N; i += BLOCK) tw[i] = tw_g[i];
  const int nbf = info->nbf;
  const long long items = (long long)groups * NSG;
  const int q = tid % N;
  const int s0 = tid / N;
  const int qm = (N - q) & (N - 1);
  const df qxA{gp.qx[q], gp.qxl[q]};
  const df qxB0{gp.qx[qm], gp.qxl[qm]};   // row of output B when j >= 1
  const df q2x = df_mul(qxA, qxA);
  const int wave_base = tid & ~63;

  for (long long item = blockIdx.x; item < items; item += gridDim.x) {
    // XCD-aware order: workgroups are dispatched round-robin over the 8 XCDs,
    // so items i, i+8, ..., i+8(LG-1) run together on one XCD; give them the
    // LG slot groups that share each 128-byte line of H (read once per L2).
    // From a resident stack, slot groups in increasing order over the BF
    // groups: the low slot columns (more points inside the apertures, the
    // long items) start first (measured faster there; from H the BF-group
    // order is kept: the other order measured slower at scan 128).
    const long long sl = (item >> 3) % LG;
    const long long t = (item / (8 * LG)) * 8 + (item & 7);
    const int g = FROM_H ? (int)(t / (NSG / LG)) : (int)(t % groups);
    const int sg = FROM_H ? (int)((t % (NSG / LG)) * LG + sl) : (int)((t / groups) * LG + sl);
    int b0, b1;
    group_range(g, groups, nbf, b0, b1);
    // copy the source tile of BF pixel b into landing buffer `slot`
    auto issue = [&](int b, int slot) {
#pragma unroll
      for (int c = 0; c < COPIES; ++c) {
        const int e0 = (c * BLOCK + wave_base) * 2;         // wave's first element
        if (e0 >= TILE) continue;                           // wave-uniform
        const int el = e0 + (tid & 63) * 2;                 // this lane's first element
        const float2* gsrc;
        if (FROM_H) {
          const int r = el / SG, sl = el % SG;
          gsrc = src + ((long long)b * N + r) * HALF + sg * SG + sl;
        } else {
          gsrc = src + ((long long)b * GCOLS + sg * SG) * N + el;
        }
        copy_async16(gsrc, &abuf[slot][e0]);
      }
    };
    // column terms of BF pixel b into buffer `slot` (threads 0..SG)
    auto colterms = [&](int b, int slot) {
      if (ISO && tid <= SG) {
        const int col = (tid < SG) ? sg * SG + tid : HALF;
        const df qy{gp.qy[col], gp.qyl[col]};
        const df kx{gp.kx[b], gp.kxl[b]}, ky{gp.ky[b], gp.kyl[b]};
        const df cbv = df_sub(rout2, df_add(df_mul(kx, kx), df_mul(ky, ky)));
        const df base = df_sub(cbv, df_mul(qy, qy));
        const df qk = df_mul(qy, df{2.0f * ky.hi, 2.0f * ky.lo});
        colA_s[slot][tid] = df_add(base, qk);
        colB_s[slot][tid] = df_sub(base, qk);
      }
    };
    __syncthreads();
    if (b0 < b1) issue(b0, 0);
    if (b0 < b1) colterms(b0, 0);
    if (tid <= SG) {
      const int col = (tid < SG) ? sg * SG + tid : HALF;
      qyS[tid] = gp.qy[col];
      qySl[tid] = gp.qyl[col];
    }
    if (sg == 0 && tid < N) {
      const df qx{gp.qx[tid], gp.qxl[tid]};
      const df qh{gp.qy[HALF], gp.qyl[HALF]};   // not qyS: written in this same phase
      if (!ISO) q2halfc[tid] = df_add(df_mul(qx, qx), df_mul(qh, qh));
      ehalfc[tid] = echi_g[(long long)HALF * N + tid];
    }
    if (tid < SG) {
      const int j = sg * SG + tid;
      enyqr[tid] = echi_g[(long long)((N - j) & (N - 1)) * N + HALF];
    }
    __syncthreads();
    // per-point constants
    float2 echiA[P];
    df q2A[P];
    Kahan arA[P], aiA[P], arB[P], aiB[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int s = s0 + i * SSTEP;
      const df qy{qyS[s], qySl[s]};
      q2A[i] = ISO ? df{0.f, 0.f} : df_add(df_mul(qxA, qxA), df_mul(qy, qy));
      echiA[i] = echi_g[(long long)(sg * SG + s) * N + q];
      arA[i].init();
      aiA[i].init();
      arB[i].init();
      aiB[i].init();
    }

    for (int b = b0; b < b1; ++b) {
      const int cur = (b - b0) & 1;
      wait_async_copies();
      __syncthreads();
      // per-BF operands are loaded before the next tile's copies are queued,
      // so waiting on them never waits on the prefetch
      const float kxh = gp.kx[b], kyh = gp.ky[b];
      const df kx{kxh, gp.kxl[b]}, ky{kyh, gp.kyl[b]};
      const float ak = gp.ak[b];
      const float2 rowA = rowph_g[(long long)b * N + q];
      float2 colp[P];
#pragma unroll
      for (int i = 0; i < P; ++i) colp[i] = colph_g[(long long)b * GCOLS + sg * SG + s0 + i * SSTEP];
      const float2 colHalf = colph_g[(long long)b * GCOLS + HALF];
      float2 gHalf = make_float2(0.f, 0.f);
      if (!FROM_H && sg == 0) gHalf = src[((long long)b * GCOLS + HALF) * N + q];
      asm volatile("" ::: "memory");
      if (b + 1 < b1) issue(b + 1, cur ^ 1);
      if (b + 1 < b1) colterms(b + 1, cur ^ 1);
      if (FROM_H) fft_lds_il<N, SG, BLOCK, TSTRIDE, false>(abuf[cur], tileT, tw);
      const float2* tile = FROM_H ? tileT : abuf[cur];
      constexpr int TS = FROM_H ? TSTRIDE : N;
      // ISO row terms of d(Q -/+ k), -qx^2 +/- 2 qx kx, as float32 estimates
      // (the double-float terms are formed only for points near the soft edge)
      const df kx2{2.0f * kx.hi, 2.0f * kx.lo};
      float uq = 0.0f, vq = 0.0f;
      df cb{0.f, 0.f};
      if constexpr (ISO) {
        uq = row_estimate_minus(qxA, kx2, q2x);
        vq = row_estimate_plus(qxA, kx2, q2x);
      } else {
        cb = df_sub(rout2, df_add(df_mul(kx, kx), df_mul(ky, ky)));
      }
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const int s = s0 + i * SSTEP;
        const int j = sg * SG + s;
        const float2 z = tile[s * TS + q];
        float2 GA, GB;
        if (j == 0) {
          if (FROM_H) {
            const float2 zm = tile[s * TS + qm];
            GA = make_float2(0.5f * (z.x + zm.x), 0.5f * (z.y - zm.y));
            GB = make_float2(0.5f * (z.y + zm.y), -0.5f * (z.x - zm.x));
          } else {
            GA = z;
            GB = gHalf;
          }
        } else {
          GA = z;
          GB = cconj(z);
        }
        const df qy{qyS[s], qySl[s]};
        float am, app;
        if constexpr (ISO) {
          iso_aperture_pair(uq, vq, qxA, kx2, q2x, colA_s[cur][s], colB_s[cur][s], ap, am, app);
        } else {
          aperture_pair<ISO>(qxA, qy, kx, ky, cb, q2A[i], ap, o, am, app);
        }
        const float2 eA = cmul(rowA, colp[i]);
        // Mirror points (j >= 1, q != N/2): output B sees the apertures
        // swapped, conj(e^{i theta}), the same e^{i chi} and conj(G), so its
        // Gamma is -conj(Gamma_A) with the same norm and its term is exactly
        // -conj(term_A) (every operation is sign-symmetric, Kahan included):
        // B is not accumulated and is written as -conj(A) at the end.
        const bool mirror = (j != 0) && (q != HALF);
        if (am != 0.0f || app != 0.0f) {
          const float wr = (am - app) * echiA[i].x;
          const float wi = -(am + app) * echiA[i].y;
          float gr = ak * (eA.x * wr - eA.y * wi);
          float gi = ak * (eA.x * wi + eA.y * wr);
          const float mag2 = gr * gr + gi * gi;
          const float sc = (mag2 > 1e-16f) ? rsqrtf(mag2) : 1e8f;
          gr *= sc;
          gi *= sc;
          arA[i].add(GA.x * gr + GA.y * gi);
          aiA[i].add(GA.y * gr - GA.x * gi);
        }
        // wave-uniform test first: most waves hold only mirror points and
        // branch over the B path
        const bool wave_b = __ballot(!mirror) != 0ull;
        if (wave_b) if (!mirror) {
          // j == 0: row q, column N/2; q == N/2: row N/2, column N-j
          const float2 echiB = (j == 0) ? ehalfc[q] : enyqr[s];
          float bm, bp;
          if constexpr (ISO) {
            // j == 0: row q, column N/2; q == N/2: row N/2 (this row), column -qy
            iso_aperture_pair(uq, vq, qxA, kx2, q2x, (j == 0) ? colA_s[cur][SG] : colB_s[cur][s],
                              (j == 0) ? colB_s[cur][SG] : colA_s[cur][s], ap, bm, bp);
          } else {
            const df qyB = (j == 0) ? df{qyS[SG], qySl[SG]} : df{-qy.hi, -qy.lo};
            const df qxB = (j == 0) ? qxA : qxB0;
            const df q2B = (j == 0) ? q2halfc[q] : q2A[i];
            aperture_pair<ISO>(qxB, qyB, kx, ky, cb, q2B, ap, o, bm, bp);
          }
          // rows q and -q coincide at q == N/2, so the row phasor is rowA
          const float2 eB = cmul(rowA, (j == 0) ? colHalf : cconj(colp[i]));
          if (bm != 0.0f || bp != 0.0f) {
            const float wr = (bm - bp) * echiB.x;
            const float wi = -(bm + bp) * echiB.y;
            float gr = ak * (eB.x * wr - eB.y * wi);
            float gi = ak * (eB.x * wi + eB.y * wr);
            const float mag2 = gr * gr + gi * gi;
            const float sc = (mag2 > 1e-16f) ? rsqrtf(mag2) : 1e8f;
            gr *= sc;
            gi *= sc;
            arB[i].add(GB.x * gr + GB.y * gi);
            aiB[i].add(GB.y * gr - GB.x * gi);
          }
        }
        // one point at a time: keeps the scheduler from overlapping the
        // points' temporaries, which would spill the accumulators
        __builtin_amdgcn_sched_barrier(0);
      }
    }
    float2* sp = S_part + (long long)g * N * N;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int s = s0 + i * SSTEP;
      const int j = sg * SG + s;
      const int colB = (j == 0) ? HALF : N - j;
      const int rowB = (j == 0) ? q : qm;
      const float2 outA = make_float2(arA[i].s - arA[i].c, aiA[i].s - aiA[i].c);
      const bool mirror = (j != 0) && (q != HALF);
      sp[(long long)j * N + q] = outA;
      sp[(long long)colB * N + rowB] =
          mirror ? make_float2(-outA.x, outA.y) : make_float2(arB[i].s - arB[i].c, aiB[i].s - aiB[i].c);
    }
  }
}

// ------------------------------------------------------------------------
// Trotter from a full (non-Hermitian) stack Gt[b][c][q], c < N: each full
// column is its own output (test seam for imported full-plane stacks).
// ------------------------------------------------------------------------
template <int N, int CG, int BLOCK>
__global__ void __launch_bounds__(BLOCK)
k_trotter_full(const float2* __restrict__ Gt, const BfInfo* __restrict__ info, GeomPtrs gp,
               const float2* __restrict__ rowph_g, QuadChi m, Optics o, int groups, float2* __restrict__ S_part) {
  constexpr int NCG = N / CG;
  constexpr int P = CG * N / BLOCK;
  __shared__ float2 colph[CG];
  __shared__ float qyS[CG], qySl[CG];
  const int tid = threadIdx.x;
  const int nbf = info->nbf;
  const long long items = (long long)groups * NCG;
  for (long long item = blockIdx.x; item < items; item += gridDim.x) {
    const int g = (int)(item / NCG);
    const int cg = (int)(item - (long long)g * NCG);
    int b0, b1;
    group_range(g, groups, nbf, b0, b1);
    __syncthreads();
    if (tid < CG) {
      qyS[tid] = gp.qy[cg * CG + tid];
      qySl[tid] = gp.qyl[cg * CG + tid];
    }
    __syncthreads();
    float2 echi[P];
    Kahan ar[P], ai[P];
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int pidx = tid + i * BLOCK;
      const int row = pidx % N, cl = pidx / N;
      float sn, cs;
      sincosf(chi_quad(m, gp.qx[row], qyS[cl]), &sn, &cs);
      echi[i] = make_float2(cs, sn);
      ar[i].init();
      ai[i].init();
    }
    for (int b = b0; b < b1; ++b) {
      const Coord kc{gp.kx[b], gp.kxl[b], gp.ky[b], gp.kyl[b]};
      const float tb = 2.0f * (m.mxy * kc.x + m.myy * kc.y);
      __syncthreads();
      if (tid < CG) {
        float sn, cs;
        sincosf(qyS[tid] * tb, &sn, &cs);
        colph[tid] = make_float2(cs, sn);
      }
      __syncthreads();
      const float2* gb = Gt + (long long)b * N * N;
#pragma unroll
      for (int i = 0; i < P; ++i) {
        const int pidx = tid + i * BLOCK;
        const int row = pidx % N, cl = pidx / N;
        const int col = cg * CG + cl;
        const float2 G = gb[(long long)col * N + row];
        const Coord qc{gp.qx[row], gp.qxl[row], qyS[cl], qySl[cl]};
        const float2 eth = cmul(rowph_g[(long long)b * N + row], colph[cl]);
        const float2 t = trotter_term(G, qc, kc, gp.ak[b], eth, echi[i], o);
        ar[i].add(t.x);
        ai[i].add(t.y);
      }
    }
    float2* sp = S_part + (long long)g * N * N;
#pragma unroll
    for (int i = 0; i < P; ++i) {
      const int pidx = tid + i * BLOCK;
      const int row = pidx % N, cl = pidx / N;
      sp[(long long)(cg * CG + cl) * N + row] = make_float2(ar[i].s - ar[i].c, ai[i].s - ai[i].c);
    }
  }
}

// ------------------------------------------------------------------------
// Finish: reduce partial planes, inverse FFT, angle.
// ------------------------------------------------------------------------
// Sum of the groups' partial planes (Kahan, in group order), /N_bf, DC :=
// dc, then the inverse FFT along q of COUNT columns of column-major S[c][q]
template <int N, int COUNT>
__global__ void __launch_bounds__(256)
k_reduce_ifft_cols(const float2* __restrict__ S_part, const BfInfo* __restrict__ info, int groups,
                   const float2* __restrict__ tw_g, float2* __restrict__ S) {
  constexpr int STRIDE = N + 1;
  constexpr long long NN = (long long)N * N;
  __shared__ float2 buf[COUNT * STRIDE];
  __shared__ float2 tw[N];
  const int tid = threadIdx.x;
  for (int i = tid; i < N; i += 256) tw[i] = tw_g[i];
  const int c0 = blockIdx.x * COUNT;
  const int nbf = info->nbf;
  const float inv = 1.0f / (float)(nbf > 0 ? nbf : 1);
  for (int idx = tid; idx < COUNT * N; idx += 256) {
    const int ci = idx / N, r = idx % N;
    const long long e = (long long)(c0 + ci) * N + r;
    Kahan kr, ki;
    kr.init();
    ki.init();
    int g = 0;
    for (; g + 16 <= groups; g += 16) {    // sixteen loads in flight, then the adds in group order
      float2 v[16];
#pragma unroll
      for (int u = 0; u < 16; ++u) v[u] = S_part[(long long)(g + u) * NN + e];
#pragma unroll
      for (int u = 0; u < 16; ++u) {
        kr.add(v[u].x);
        ki.add(v[u].y);
      }
    }
    for (; g < groups; ++g) {
      const float2 v = S_part[(long long)g * NN + e];
      kr.add(v.x);
      ki.add(v.y);
    }
    buf[ci * STRIDE + r] = (e == 0) ? make_float2(info->dc_re, info->dc_im)
                                    : make_float2((kr.s - kr.c) * inv, (ki.s - ki.c) * inv);
  }
  __syncthreads();
  fft_lds<N, COUNT, 256, STRIDE, true>(buf, tw);
  for (int idx = tid; idx < COUNT * N; idx += 256) {
    const int ci = idx / N, r = idx % N;
    S[(long long)(c0 + ci) * N + r] = buf[ci * STRIDE + r];
  }
}

// inverse FFT along c for COUNT rows, scale 1/N^2, object + phase (row-major)
template <int N, int COUNT>
__global__ void __launch_bounds__(256)
k_ifft_rows_phase(const float2* __restrict__ S, const float2* __restrict__ tw_g, float2* __restrict__ obj,
                  float* __restrict__ phase) {
  constexpr int STRIDE = N + 1;
  __shared__ float2 buf[COUNT * STRIDE];
  __shared__ float2 tw[N];
  const int tid = threadIdx.x;
  for (int i = tid; i < N; i += 256) tw[i] = tw_g[i];
  const int r0 = blockIdx.x * COUNT;
  for (int idx = tid; idx < COUNT * N; idx += 256) {
    const int c = idx / COUNT, ri = idx % COUNT;
    buf[ri * STRIDE + c] = S[(long long)c * N + r0 + ri];
  }
  __syncthreads();
  fft_lds<N, COUNT, 256, STRIDE, true>(buf, tw);
  const float scale = 1.0f / ((float)N * (float)N);
  for (int idx = tid; idx < COUNT * N; idx += 256) {
    const int ri = idx / N, c = idx % N;
    const float2 v = cscale(buf[ri * STRIDE + c], scale);
    const long long o = (long long)(r0 + ri) * N + c;
    if (obj) obj[o] = v;
    if (phase) phase[o] = atan2f(v.y, v.x);
  }
}

// ------------------------------------------------------------------------
// Launch wrappers
// ------------------------------------------------------------------------
static unsigned grid_items(long long items, long long cap) {
  if (items < 1) items = 1;
  if (items > cap) items = cap;
  return (unsigned)items;
}

ApIso iso_aperture(const Optics& o, df& rout2_df) {
  // Rout = (semi + ang/2) / lambda; the isotropic form needs ang_y == ang_x
  const double lam = (double)o.lam.hi + (double)o.lam.lo;
  const double semi = (double)o.semi.hi + (double)o.semi.lo;
  const double ang = (double)o.angy.hi + (double)o.angy.lo;
  const double rout = (semi + 0.5 * ang) / lam;
  const double rin = (semi - 0.5 * ang) / lam;
  const double r2 = rout * rout;
  const float hi = (float)r2;
  rout2_df = df{hi, (float)(r2 - (double)hi)};
  ApIso a;
  a.rout2 = hi;
  a.rout = (float)rout;
  a.scale = (float)(lam / ang);
  // exact 0/1 outside the band, with a relative margin above FP32 noise
  a.d_in = (rin > 0.0) ? (float)((r2 - rin * rin) * (1.0 + 1e-5)) : INFINITY;
  a.d_out = (float)(-r2 * 1e-5);
  a.edge = (float)(r2 > 25.0 ? 4e-6 * r2 : 1e-4);
  return a;
}

bool optics_isotropic(const Optics& o) { return o.angy.hi == o.angx.hi && o.angy.lo == o.angx.lo; }

hipError_t launch_phasors(int N, const BfInfo* info, int nbf_hint, const GeomPtrs& gp, QuadChi m, float2* rowph,
                          float2* colph, float2* echi, hipStream_t s,
                          const QuadChi* m_dev) {
  long long total = (long long)(nbf_hint > 0 ? nbf_hint : 1) * (N + N / 2 + 1);
  if (total < (long long)N * N) total = (long long)N * N;
  hipLaunchKernelGGL(k_phasors, dim3(grid_items((total + 255) / 256, 4096)), dim3(256), 0, s, info, gp, m, N, rowph,
                     colph, echi, m_dev);
  return hipGetLastError();
}

// Tile shapes (SG slot columns, BLOCK threads) of the fused column FFT +
// trotter on the row-transformed stack (the reconstruction path); at N = 128
// with equal sampling variant 0 is the default, the others are the tuner's
// candidates.  SG is even there: each lane's 16-byte staging copy moves two
// adjacent slots of a row of H.  From N = 256 on equal sampling goes through
// ssb_columns.hip (columns_path), whose variants are numbers of BF groups.
int trotter_variants(int N) { return N >= 256 ? columns_variants(N) : 3; }

int trotter_groups_max(int N) {
  int g = object_groups(N);
  g = object_tile_groups(N) > g ? object_tile_groups(N) : g;
  for (int v = 0; N >= 256 && v < columns_variants(N); ++v) g = columns_groups(N, v) > g ? columns_groups(N, v) : g;
  return g;
}

hipError_t launch_trotter_slots(int N, bool from_h, const float2* src, const BfInfo* info, const GeomPtrs& gp,
                                const float2* rowph, const float2* colph, const float2* echi, const Optics& o,
                                const float2* tw, float2* S_part, int variant, hipStream_t s, int* groups_used) {
  df rout2;
  const ApIso ap = iso_aperture(o, rout2);
  const bool iso = optics_isotropic(o);
  if (iso && (!from_h || N != 128)) return hipErrorInvalidValue;   // ssb_columns.hip's
  // a resident stack at N = 256: 32 BF groups (2048 items, two rounds of four
  // workgroups a CU, so that the heavy-first order can even out the CUs: an object
  // of 800 BF pixels takes 181 us, in 16 groups 193)
  const int groups = (!from_h && N == 256) ? 2 * object_groups(N) : object_groups(N);
  if (groups_used) *groups_used = groups;
#define QSSB_SLOTS_ONE(NN, SGV, BL, FH, IS)                                                                 \
  hipLaunchKernelGGL((k_trotter_slots<NN, SGV, BL, FH, IS>), dim3(grid), dim3(BL), 0, s, src, info, gp, rowph, \
                     colph, echi, ap, rout2, o, tw, groups, S_part)
#define QSSB_SLOTS(NN, SGV, BL)                                                                \
  do {                                                                                        \
    const unsigned grid = grid_items((long long)groups * ((NN / 2) / SGV), 65536);            \
    if (from_h) QSSB_SLOTS_ONE(NN, SGV, BL, true, false);                                     \
    else QSSB_SLOTS_ONE(NN, SGV, BL, false, false);                                           \
  } while (0)
#define QSSB_SLOTS_ISO(NN, SGV, BL)                                                            \
  do {                                                                                        \
    const unsigned grid = grid_items((long long)groups * ((NN / 2) / SGV), 65536);            \
    QSSB_SLOTS_ONE(NN, SGV, BL, true, true);                                                  \
  } while (0)
  switch (N) {
    case 128:
      if (iso && variant == 1) QSSB_SLOTS_ISO(128, 2, 256);
      else if (iso && variant == 2) QSSB_SLOTS_ISO(128, 8, 256);
      else if (iso) QSSB_SLOTS_ISO(128, 4, 256);
      else QSSB_SLOTS(128, 4, 256);
      break;
    case 256:
      QSSB_SLOTS(256, 2, 256);
      break;
    case 512:
      QSSB_SLOTS(512, 2, 512);
      break;
    case 1024:
      if (from_h) {
        // one slot per tile would split the 16-byte staging copies across rows
        const unsigned grid = grid_items((long long)groups * ((1024 / 2) / 2), 65536);
        QSSB_SLOTS_ONE(1024, 2, 1024, true, false);
      } else {
        const unsigned grid = grid_items((long long)groups * ((1024 / 2) / 1), 65536);
        QSSB_SLOTS_ONE(1024, 1, 1024, false, false);
      }
      break;
    default:
      return hipErrorInvalidValue;
  }
#undef QSSB_SLOTS_ISO
#undef QSSB_SLOTS
#undef QSSB_SLOTS_ONE
  return hipGetLastError();
}

hipError_t launch_trotter_full(int N, const float2* Gt, const BfInfo* info, const GeomPtrs& gp, const float2* rowph,
                               QuadChi m, const Optics& o, float2* S_part, hipStream_t s) {
  const int groups = object_groups(N);
  switch (N) {
    case 128:
      hipLaunchKernelGGL((k_trotter_full<128, 16, 256>), dim3(grid_items(groups * 8LL, 65536)), dim3(256), 0, s, Gt,
                         info, gp, rowph, m, o, groups, S_part);
      break;
    case 256:
      hipLaunchKernelGGL((k_trotter_full<256, 8, 256>), dim3(grid_items(groups * 32LL, 65536)), dim3(256), 0, s, Gt,
                         info, gp, rowph, m, o, groups, S_part);
      break;
    case 512:
      hipLaunchKernelGGL((k_trotter_full<512, 4, 256>), dim3(grid_items(groups * 128LL, 65536)), dim3(256), 0, s,
                         Gt, info, gp, rowph, m, o, groups, S_part);
      break;
    case 1024:
      hipLaunchKernelGGL((k_trotter_full<1024, 1, 256>), dim3(grid_items(groups * 1024LL, 65536)), dim3(256), 0, s,
                         Gt, info, gp, rowph, m, o, groups, S_part);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

hipError_t launch_finish_object(int N, const float2* S_part, int groups, const BfInfo* info, const float2* tw,
                                float2* S, float2* obj, float* phase, hipStream_t s) {
  const int G = groups;
  switch (N) {
    case 128:
      hipLaunchKernelGGL((k_reduce_ifft_cols<128, 4>), dim3(128 / 4), dim3(256), 0, s, S_part, info, G, tw, S);
      hipLaunchKernelGGL((k_ifft_rows_phase<128, 8>), dim3(128 / 8), dim3(256), 0, s, S, tw, obj, phase);
      break;
    case 256:
      hipLaunchKernelGGL((k_reduce_ifft_cols<256, 1>), dim3(256), dim3(256), 0, s, S_part, info, G, tw, S);
      hipLaunchKernelGGL((k_ifft_rows_phase<256, 4>), dim3(256 / 4), dim3(256), 0, s, S, tw, obj, phase);
      break;
    case 512:
      hipLaunchKernelGGL((k_reduce_ifft_cols<512, 1>), dim3(512), dim3(256), 0, s, S_part, info, G, tw, S);
      hipLaunchKernelGGL((k_ifft_rows_phase<512, 2>), dim3(512 / 2), dim3(256), 0, s, S, tw, obj, phase);
      break;
    case 1024:
      hipLaunchKernelGGL((k_reduce_ifft_cols<1024, 1>), dim3(1024), dim3(256), 0, s, S_part, info, G, tw, S);
      hipLaunchKernelGGL((k_ifft_rows_phase<1024, 1>), dim3(1024), dim3(256), 0, s, S, tw, obj, phase);
      break;
    default:
      return hipErrorInvalidValue;
  }
  return hipGetLastError();
}

}  // namespace qssb
