// Row kernel (layout in pasif_rows.hpp): one workgroup per instance, one
// thread per unit and slot, stage state and set points in LDS, terms streamed
// from the caches in wave-blocked order, one LDS-only barrier per stage.
//
// What bounds it: a stage is one pass over the instance's terms by one
// compute unit (a value and 2 bytes an index from L2, one LDS read a factor) and a
// barrier, four times a step, and steps are sequential.  Measured on
// energy gradients of chains (forward and adjoint step together): 5.0 us for
// 70 to 250 DOF (one unit per thread, terms in registers: LDS latency and
// the barriers), 60 us for 2,001 DOF (eight units per thread, terms from L2);
// the tile kernel took 52 us at 150 DOF, the kernel with every vector in
// device memory 694 us at 2,001.
#include <hip/hip_runtime.h>

#include "pasif_rows.hpp"
#include "pasif_tiles.hpp"

namespace pasif {
namespace {

__device__ __forceinline__ double rfma(double a, double b, double c) { return __builtin_fma(a, b, c); }
__device__ __forceinline__ float rfma(float a, float b, float c) { return __builtin_fmaf(a, b, c); }
__device__ __forceinline__ double rabs(double a) { return __builtin_fabs(a); }
__device__ __forceinline__ float rabs(float a) { return __builtin_fabsf(a); }

__device__ __forceinline__ uint32_t runi(uint32_t v) {
  return static_cast<uint32_t>(__builtin_amdgcn_readfirstlane(static_cast<int>(v)));
}
__device__ __forceinline__ uint64_t runi64(uint64_t v) {
  return (uint64_t(runi(uint32_t(v >> 32))) << 32) | runi(uint32_t(v));
}

// Workgroup barrier ordering LDS only (global data is read back by the
// thread that wrote it).
__device__ __forceinline__ void row_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
  __builtin_amdgcn_s_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

template <typename R>
__device__ __forceinline__ R at(const unsigned char* b, uint32_t off) {
  return *reinterpret_cast<const R*>(b + off);
}

// A block header: first value and index word (in blocks of 64), trip counts
// of the four kinds (7 bits each) and these flags.
enum : uint32_t { kBlkForced = 1u << 28, kBlkSplit = 1u << 29 };

// Sum of the lane's terms of one block: kinds summed in order, each from
// zero in the unit's order.  Kind 1 packs two terms' offsets in a word.
// Padding terms have value 0 and point at slots that hold 0.  `v` and `w` are
// uniform (scalar base, lane offset), and four linear or quadratic terms are
// requested together: a block's terms come from L2, and a wave waits for
// each batch.
template <typename R>
__device__ __forceinline__ R row_terms(const R* v, const uint32_t* w, uint32_t cnt, uint32_t ln,
                                       const unsigned char* Y, const unsigned char* X) {
  const uint32_t c1 = cnt & 127u, c2 = (cnt >> 7) & 127u, c3 = (cnt >> 14) & 127u,
                 c4 = (cnt >> 21) & 127u;
  R t1 = R(0), t2 = R(0), t3 = R(0), t4 = R(0);
  uint32_t i = c1;
#pragma unroll 1
  for (; i >= 4u; i -= 4u, v += 256, w += 128) {
    const uint32_t p = w[ln], q = w[ln + 64u];
    const R a = v[ln], b = v[ln + 64u], c = v[ln + 128u], d = v[ln + 192u];
    t1 = rfma(a, at<R>(Y, p & 0xFFFFu), t1);
    t1 = rfma(b, at<R>(Y, p >> 16), t1);
    t1 = rfma(c, at<R>(Y, q & 0xFFFFu), t1);
    t1 = rfma(d, at<R>(Y, q >> 16), t1);
  }
  if (i) {  // two left (counts are even)
    const uint32_t p = w[ln];
    const R a = v[ln], b = v[ln + 64u];
    t1 = rfma(a, at<R>(Y, p & 0xFFFFu), t1);
    t1 = rfma(b, at<R>(Y, p >> 16), t1);
    v += 128;
    w += 64;
  }
#pragma unroll 1
  for (i = c2; i >= 4u; i -= 4u, v += 256, w += 256) {
    const uint32_t p = w[ln], q = w[ln + 64u], r = w[ln + 128u], s = w[ln + 192u];
    const R a = v[ln], b = v[ln + 64u], c = v[ln + 128u], d = v[ln + 192u];
    t2 = rfma(a * at<R>(Y, p & 0xFFFFu), at<R>(X, p >> 16), t2);
    t2 = rfma(b * at<R>(Y, q & 0xFFFFu), at<R>(X, q >> 16), t2);
    t2 = rfma(c * at<R>(Y, r & 0xFFFFu), at<R>(X, r >> 16), t2);
    t2 = rfma(d * at<R>(Y, s & 0xFFFFu), at<R>(X, s >> 16), t2);
  }
  if (i) {
    const uint32_t p = w[ln], q = w[ln + 64u];
    const R a = v[ln], b = v[ln + 64u];
    t2 = rfma(a * at<R>(Y, p & 0xFFFFu), at<R>(X, p >> 16), t2);
    t2 = rfma(b * at<R>(Y, q & 0xFFFFu), at<R>(X, q >> 16), t2);
    v += 128;
    w += 128;
  }
#pragma unroll 1
  for (i = c3; i > 0u; --i, v += 64, w += 128) {
    const uint32_t p = w[ln], q = w[ln + 64u];
    R t = v[ln] * at<R>(Y, p & 0xFFFFu);
    t = t * at<R>(X, p >> 16);
    t3 = rfma(t, at<R>(X, q & 0xFFFFu), t3);
  }
#pragma unroll 1
  for (i = c4; i > 0u; --i, v += 64, w += 128) {
    const uint32_t p = w[ln], q = w[ln + 64u];
    R t = v[ln] * at<R>(Y, p & 0xFFFFu);
    t = t * at<R>(X, p >> 16);
    t = t * at<R>(X, q & 0xFFFFu);
    t4 = rfma(t, at<R>(X, q >> 16), t4);
  }
  return ((t1 + t2) + t3) + t4;
}

// The lane's terms of one block in registers, up to kRowRes* of each kind.
// With one unit per thread (and every block within these) they stay there
// for a whole phase and a stage reads nothing but LDS.
template <typename R>
struct RowRes {
  R v1[kRowRes1], v2[kRowRes2], v3[kRowRes3], v4[kRowRes4];
  uint32_t w1[kRowRes1 / 2], w2[kRowRes2], w3[2 * kRowRes3], w4[2 * kRowRes4];

  __device__ __forceinline__ void load(const R* v, const uint32_t* w, uint32_t cnt, uint32_t ln) {
    const uint32_t c1 = cnt & 127u, c2 = (cnt >> 7) & 127u, c3 = (cnt >> 14) & 127u,
                   c4 = (cnt >> 21) & 127u;
#pragma unroll
    for (uint32_t i = 0; i < kRowRes1; i += 2u) {
      v1[i] = v1[i + 1u] = R(0);
      w1[i / 2u] = 0u;
      if (i < c1) {
        v1[i] = v[i * 64u + ln];
        v1[i + 1u] = v[(i + 1u) * 64u + ln];
        w1[i / 2u] = w[i * 32u + ln];
      }
    }
    v += c1 * 64u;
    w += c1 * 32u;
#pragma unroll
    for (uint32_t i = 0; i < kRowRes2; i += 2u) {
      v2[i] = v2[i + 1u] = R(0);
      w2[i] = w2[i + 1u] = 0u;
      if (i < c2) {
        v2[i] = v[i * 64u + ln];
        v2[i + 1u] = v[(i + 1u) * 64u + ln];
        w2[i] = w[i * 64u + ln];
        w2[i + 1u] = w[(i + 1u) * 64u + ln];
      }
    }
    v += c2 * 64u;
    w += c2 * 64u;
#pragma unroll
    for (uint32_t i = 0; i < kRowRes3; ++i) {
      v3[i] = R(0);
      w3[2u * i] = w3[2u * i + 1u] = 0u;
      if (i < c3) {
        v3[i] = v[i * 64u + ln];
        w3[2u * i] = w[2u * i * 64u + ln];
        w3[2u * i + 1u] = w[(2u * i + 1u) * 64u + ln];
      }
    }
    v += c3 * 64u;
    w += c3 * 128u;
#pragma unroll
    for (uint32_t i = 0; i < kRowRes4; ++i) {
      v4[i] = R(0);
      w4[2u * i] = w4[2u * i + 1u] = 0u;
      if (i < c4) {
        v4[i] = v[i * 64u + ln];
        w4[2u * i] = w[2u * i * 64u + ln];
        w4[2u * i + 1u] = w[(2u * i + 1u) * 64u + ln];
      }
    }
  }

  // as row_terms; the trip counts are a wave's, so the groups are skipped by
  // scalar branches and the LDS reads of a group are in flight together
  __device__ __forceinline__ R sum(uint32_t cnt, const unsigned char* Y,
                                   const unsigned char* X) const {
    const uint32_t c1 = cnt & 127u, c2 = (cnt >> 7) & 127u, c3 = (cnt >> 14) & 127u,
                   c4 = (cnt >> 21) & 127u;
    R t1 = R(0), t2 = R(0), t3 = R(0), t4 = R(0);
#pragma unroll
    for (uint32_t b = 0; b < kRowRes1; b += 4u)
      if (c1 > b) {
        R y[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
          const uint32_t x = w1[(b + i) / 2u];
          y[i] = at<R>(Y, (i & 1u) ? x >> 16 : x & 0xFFFFu);
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
          if (i < 2u || c1 > b + 2u) t1 = rfma(v1[b + i], y[i], t1);
      }
#pragma unroll
    for (uint32_t b = 0; b < kRowRes2; b += 4u)
      if (c2 > b) {
        R y[4], x[4];
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i) {
          y[i] = at<R>(Y, w2[b + i] & 0xFFFFu);
          x[i] = at<R>(X, w2[b + i] >> 16);
        }
#pragma unroll
        for (uint32_t i = 0; i < 4u; ++i)
          if (i < 2u || c2 > b + 2u) t2 = rfma(v2[b + i] * y[i], x[i], t2);
      }
#pragma unroll
    for (uint32_t b = 0; b < kRowRes3; b += 2u)
      if (c3 > b) {
        R f[2][3];
#pragma unroll
        for (uint32_t i = 0; i < 2u; ++i) {
          f[i][0] = at<R>(Y, w3[2u * (b + i)] & 0xFFFFu);
          f[i][1] = at<R>(X, w3[2u * (b + i)] >> 16);
          f[i][2] = at<R>(X, w3[2u * (b + i) + 1u] & 0xFFFFu);
        }
        t3 = rfma((v3[b] * f[0][0]) * f[0][1], f[0][2], t3);
        if (c3 > b + 1u) t3 = rfma((v3[b + 1u] * f[1][0]) * f[1][1], f[1][2], t3);
      }
#pragma unroll
    for (uint32_t i = 0; i < kRowRes4; ++i)
      if (c4 > i) {
        const R f0 = at<R>(Y, w4[2u * i] & 0xFFFFu), f1 = at<R>(X, w4[2u * i] >> 16);
        const R f2 = at<R>(X, w4[2u * i + 1u] & 0xFFFFu), f3 = at<R>(X, w4[2u * i + 1u] >> 16);
        t4 = rfma(((v4[i] * f0) * f1) * f2, f3, t4);
      }
    return ((t1 + t2) + t3) + t4;
  }
};

// forcing at (step n, stage): the rules of the other kernels (zero-order
// hold e[n], e[n + 1] when 0 < s < L; interpolation on the half-step grid
// when 0 < i < L, e[L] read as 0)
template <typename R>
__device__ __forceinline__ R row_force(const RowArgs<R>& a, int32_t exc, uint32_t n, uint32_t part) {
  if (exc < 0) return R(0);
  const R* E = a.excit + static_cast<size_t>(exc) * a.exc_len;
  const uint32_t L = a.exc_len;
  const uint32_t n1 = n + (part == 2u ? 1u : 0u);
  if (a.interp_w == 0u) return (n1 > 0u && n1 < L) ? E[n1] : R(0);
  const uint32_t W = a.interp_w;
  const uint32_t hs = 2u * n1 + (part == 1u ? 1u : 0u);
  const uint32_t i = hs / W, j = hs - i * W;
  if (!(i > 0u && i < L)) return R(0);
  const R e1 = (i + 1u < L) ? E[i + 1u] : R(0);
  return rfma(a.interp[W + j], E[i], a.interp[j] * e1);
}

// One side of the instance for one wave: its program and the headers of the
// wave's blocks, in scalar registers.
template <typename R, int RS>
struct Side {
  const R* val;
  const uint32_t* word;
  uint32_t vb[RS], wb[RS], cnt[RS];
  uint32_t units, pub, aux, nsink;
  size_t unit;
  const uint4* blk;
  const uint32_t* sink;
  uint32_t nblk;

  __device__ __forceinline__ void load(const RowArgs<R>& a, const RowProg& p, uint32_t wave,
                                       uint32_t nw) {
    units = runi(p.units);
    pub = runi(p.pub);
    aux = runi(p.aux);
    nsink = runi(p.nsink);
    unit = runi64(p.unit);
    blk = a.blk + runi64(p.blk);
    sink = a.sink + runi64(p.sink);
    val = a.val + runi64(p.val);
    word = a.word + runi64(p.word);
    nblk = (units + 63u) >> 6;
#pragma unroll
    for (int j = 0; j < RS; ++j) {
      const uint32_t b = uint32_t(j) * nw + wave;
      uint4 h = make_uint4(0, 0, 0, 0);
      if (b < nblk) h = blk[b];
      vb[j] = runi(h.x);
      wb[j] = runi(h.y);
      cnt[j] = runi(h.z);
    }
  }
};

template <typename R, bool ADJ, int RS, bool RES>
__global__ void __launch_bounds__(kRowThreads) row_kernel(RowArgs<R> a) {
  extern __shared__ __align__(16) unsigned char row_smem[];
  constexpr int kStageUnroll = RES ? 4 : 1;
  const RowInst& I = a.inst[blockIdx.x];
  const uint32_t NW = runi(I.waves);
  const uint32_t wave = runi(threadIdx.x >> 6), lane = threadIdx.x & 63u;
  // waves beyond the instance's own (the launch is as wide as its widest
  // instance) end here; barriers wait for the remaining waves only
  if (wave >= NW) return;
  const uint32_t NT = NW * 64u, tid = threadIdx.x;
  constexpr uint32_t EL = sizeof(R);
  unsigned char* const Yb = row_smem;
  const uint32_t ys = runi(I.ys) * EL, xs = runi(I.xs) * EL;
  unsigned char* const Xb = Yb + 2u * ys;
  R* const part = reinterpret_cast<R*>(Xb + 2u * xs);
  R* const ft = part + runi(I.ps);

  // unit of slot j, computed where it is used: the slots are unrolled, and
  // addresses derived from it ahead of the step loop would be held (or
  // spilled) through it
  auto unit_of = [&](int j) -> uint32_t {
    uint32_t t = tid;
    asm volatile("" : "+v"(t));
    return uint32_t(j) * NT + t;
  };

  const uint32_t T = runi(I.steps), nf = runi(I.n_f);
  const int32_t exc = static_cast<int32_t>(runi(static_cast<uint32_t>(I.exc)));
  const bool adjoint = ADJ && a.adjoint != 0u;
  const bool exact = adjoint && a.exact != 0u;
  const bool store = adjoint && a.store != 0u;
  const uint32_t K = adjoint ? (store ? (T > 0u ? T : 1u) : a.ck_every) : 1u;
  const uint32_t out_f = runi(I.out_f), out_a = runi(I.out_a);
  const uint32_t pubf = runi(I.f.pub), unitsf = runi(I.f.units);
  const uint32_t puba = ADJ ? runi(I.a.pub) : 0u, unitsa = ADJ ? runi(I.a.units) : 0u;
  R* const vecf = a.vec_f + runi64(I.vec_f);
  R* const veca = ADJ ? a.vec_a + runi64(I.vec_a) : nullptr;
  R* const ck = ADJ ? a.ckpt + runi64(I.ck) : nullptr;
  R* const seg = ADJ ? a.segbuf + runi64(store ? I.path : I.seg) : nullptr;
  const R h = a.h, h2 = a.h2, h6 = a.h6;
  const uint32_t SE = a.save_every;

  uint32_t* pst = a.progress + 4u * blockIdx.x;
  uint32_t n = runi(pst[0]), phase = runi(pst[1]), sg = runi(pst[2]);
  uint32_t budget = a.budget;

  // slots that padding terms read
  if (tid < 2u) {
    const uint32_t z = pubf > puba ? pubf : puba;
    *reinterpret_cast<R*>(Yb + tid * ys + z * EL) = R(0);
    if (adjoint) *reinterpret_cast<R*>(Xb + tid * xs + pubf * EL) = R(0);
  }

  R q[RS], l[ADJ ? RS : 1];
#pragma unroll
  for (int j = 0; j < RS; ++j) {
    const uint32_t u = unit_of(j);
    q[j] = R(0);
    if (u < unitsf)
      q[j] = (n == 0u && phase == kPhaseForward) ? a.init[runi64(I.f.unit) + u] : vecf[u];
  }
  if constexpr (ADJ) {
#pragma unroll
    for (int j = 0; j < RS; ++j) {
      const uint32_t u = unit_of(j);
      l[j] = R(0);
      if (adjoint && phase != kPhaseForward && u < unitsa) l[j] = veca[u];
    }
  }

  Side<R, RS> S;
  RowRes<R> P;  // RES (one unit per thread): the unit's terms
  auto load_side = [&](const RowProg& p) {
    S.load(a, p, wave, NW);
    if constexpr (RES)
      P.load(S.val + size_t(S.vb[0]) * 64u, S.word + size_t(S.wb[0]) * 64u, S.cnt[0], lane);
  };
  // what a phase loads lands before its step loop: inside it the in-order
  // counter would also hold a stage for the path's stores and prefetches
  auto landed = [] { __builtin_amdgcn_s_waitcnt(0); };
  // sum of each multi-piece sink (its units start at `pub`) handed to
  // put(sink, row, sum) on one lane; st[] are the side's unit states
  auto sinks = [&](const R* st, auto put) {
    if (S.nsink == 0u) return;
    const uint32_t np = runi(S.sink[3u * (S.nsink - 1u) + 2u]);  // pieces in all
#pragma unroll
    for (int j = 0; j < RS; ++j) {
      const uint32_t u = unit_of(j);
      if (u >= S.pub && u < S.pub + np) part[u - S.pub] = st[j];
    }
    row_sync();
    for (uint32_t i = wave; i < S.nsink; i += NW) {
      const uint32_t b = runi(S.sink[3u * i + 1u]), e = runi(S.sink[3u * i + 2u]);
      R t = R(0);
      for (uint32_t k = b + lane; k < e; k += 64u) t = t + part[k];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) t = t + __shfl_xor(t, o);
      if (lane == 0u) put(i, S.sink[3u * i], t);
    }
    row_sync();
  };
  // final states (and running maxima) of every forward row
  auto put_rows = [&](R* out, uint32_t base) {
#pragma unroll
    for (int j = 0; j < RS; ++j) {
      const uint32_t u = unit_of(j);
      if (u < unitsf) {
        const uint32_t r = a.row[S.unit + u];
        if (r != kRowNone) out[base + r] = q[j];
      }
    }
    sinks(q, [&](uint32_t, uint32_t r, R t) { out[base + r] = t; });
  };
  // sums of the pieces of split rows for this stage
  auto pieces = [&](const unsigned char* Y, const unsigned char* X) {
    if (S.aux == 0u) return;
    const uint32_t na = (S.aux + 63u) >> 6;
    for (uint32_t b = wave; b < na; b += NW) {
      const uint4 hd = S.blk[S.nblk + b];
      const R t = row_terms(S.val + size_t(runi(hd.x)) * 64u, S.word + size_t(runi(hd.y)) * 64u,
                            runi(hd.z), lane, Y, X);
      if (b * 64u + lane < S.aux) part[b * 64u + lane] = t;
    }
    row_sync();
  };
  auto slope = [&](int j, uint32_t u, const unsigned char* Y, const unsigned char* X) -> R {
    uint32_t vb = S.vb[j], wb = S.wb[j], cnt = S.cnt[j], ln = lane;
    asm volatile("" : "+s"(vb), "+s"(wb), "+s"(cnt), "+v"(ln));
    R k;
    if constexpr (RES) {
      k = P.sum(cnt, Y, X);
    } else {
      k = row_terms(S.val + size_t(vb) * 64u, S.word + size_t(wb) * 64u, cnt, ln, Y, X);
    }
    if (cnt & kBlkSplit) {
      const uint32_t pr = a.piece[S.unit + u];
      for (uint32_t g = pr & 0xFFFFu; g < (pr >> 16); ++g) k = k + part[g];
    }
    return k;
  };

  if (n == 0u && phase == kPhaseForward && T == 0u) {
    load_side(I.f);
    put_rows(a.out_q, out_f);
  }

  while (budget > 0u && phase != kPhaseDone) {
    if (phase != kPhaseBackward) {
      // ---------------- forward / recompute ----------------
      const bool recompute = phase == kPhaseRecompute;
      load_side(I.f);
      const uint32_t s0 = recompute ? sg * K : 0u;
      const bool keep = recompute || store;  // set points of every step to seg
#pragma unroll
      for (int j = 0; j < RS; ++j) {
        const uint32_t u = unit_of(j);
        if (u < pubf) {
          if (recompute && n == s0) q[j] = ck[size_t(sg) * nf + u];
          if (keep && !exact && n == s0) seg[u] = q[j];
          *reinterpret_cast<R*>(Yb + u * EL) = q[j];
        }
      }
      const R force0 = RES && tid < unitsf ? a.force[S.unit + tid] : R(0);
      landed();
      row_sync();
      const uint32_t e = recompute ? min(T, s0 + K) : T;
      const uint32_t nend = (e - n < budget) ? e : n + budget;
      budget -= nend - n;
      uint32_t fb = n, left = 0;
      for (; n < nend; ++n) {
        if (left == 0u) {
          left = min(kRowChunk, nend - n);
          fb = n;
          for (uint32_t k = tid; k < 3u * left; k += NT) {
            const uint32_t m = k / 3u;
            ft[k] = row_force(a, exc, n + m, k - 3u * m);
          }
          row_sync();
        }
        --left;
        if (adjoint && !keep && (n % K) == 0u) {
#pragma unroll
          for (int j = 0; j < RS; ++j) {
            const uint32_t u = unit_of(j);
            if (u < pubf) ck[size_t(n / K) * nf + u] = q[j];
          }
        }
        R* rec = (exact && keep) ? seg + size_t(4u * (n - s0)) * pubf : nullptr;
        R acc[RS];
#pragma unroll kStageUnroll
        for (uint32_t s = 0; s < 4u; ++s) {
          const unsigned char* Y = Yb + (s & 1u) * ys;
          unsigned char* Yn = Yb + ((s + 1u) & 1u) * ys;
          const R us = ft[3u * (n - fb) + (s == 0u ? 0u : (s == 3u ? 2u : 1u))];
          const R cs = s < 2u ? h2 : h;
          const R wa = (s == 1u || s == 2u) ? R(2) : R(1);
          pieces(Y, Y);
#pragma unroll
          for (int j = 0; j < RS; ++j) {
            const uint32_t u0 = uint32_t(j) * NT + wave * 64u, u = unit_of(j);
            if (u0 >= (recompute ? pubf : unitsf)) continue;
            R fv = R(0);
            if constexpr (RES)
              fv = force0;
            else if (S.cnt[j] & kBlkForced)
              fv = a.force[S.unit + u];
            R k = slope(j, u, Y, Y);
            if (S.cnt[j] & kBlkForced) k = rfma(fv, us, k);
            acc[j] = s == 0u ? k : rfma(wa, k, acc[j]);
            R y;
            if (s < 3u) {
              y = rfma(cs, k, q[j]);
            } else {
              y = rfma(h6, acc[j], q[j]);
            }
            if (u < pubf) {
              if (rec) {
                if (s == 0u) rec[u] = q[j];
                if (s < 3u) rec[size_t(s + 1u) * pubf + u] = y;
              }
              *reinterpret_cast<R*>(Yn + u * EL) = y;
            }
            if (s == 3u) q[j] = y;
          }
          row_sync();
        }
        if (keep && !exact) {
          R* o = seg + size_t(n + 1u - s0) * pubf;
#pragma unroll
          for (int j = 0; j < RS; ++j) {
            const uint32_t u = unit_of(j);
            if (u < pubf) o[u] = q[j];
          }
        }
        if (!recompute) {
          if (SE && n % SE == 0u && n / SE < a.nslots)
            put_rows(a.traj + size_t(n / SE) * a.out_len, out_f);
          if (a.window && n + 1u + a.window > T) {
            R* mx = vecf + unitsf;
#pragma unroll
            for (int j = 0; j < RS; ++j) {
              const uint32_t u = unit_of(j);
              if (u < unitsf) mx[u] = max(mx[u], rabs(q[j]));
            }
            sinks(q, [&](uint32_t i, uint32_t, R t) {
              R* m = vecf + 2u * unitsf + i;
              *m = max(*m, rabs(t));
            });
          }
          if (n + 1u == T) {
            put_rows(a.out_q, out_f);
            if (a.window) {
#pragma unroll
              for (int j = 0; j < RS; ++j) {
                const uint32_t u = unit_of(j);
                if (u < unitsf && a.row[S.unit + u] != kRowNone)
                  a.out_max[out_f + a.row[S.unit + u]] = vecf[unitsf + u];
              }
              for (uint32_t i = wave; i < S.nsink; i += NW)
                if (lane == 0u) a.out_max[out_f + S.sink[3u * i]] = vecf[2u * unitsf + i];
            }
          }
        }
      }
      if (n == e && !recompute && SE)
        // trajectory slots after the last step hold the final state
        for (uint32_t slot = (T + SE - 1u) / SE; slot < a.nslots; ++slot)
          put_rows(a.traj + size_t(slot) * a.out_len, out_f);
      if (n == e) {
        if (recompute) {
          phase = kPhaseBackward;
        } else if (adjoint && T > 0u) {
          sg = store ? 0u : (T - 1u) / K;
          n = store ? T : sg * K;
          phase = store ? kPhaseBackward : kPhaseRecompute;
          if constexpr (ADJ) {
#pragma unroll
            for (int j = 0; j < RS; ++j) {
              const uint32_t u = unit_of(j);
              if (u < unitsa) l[j] = a.init[runi64(I.a.unit) + u];
            }
          }
        } else {
          phase = kPhaseDone;
          if constexpr (ADJ) {
            if (adjoint) {  // no steps: the terminal state is the gradient
              load_side(I.a);
#pragma unroll
              for (int j = 0; j < RS; ++j) {
                const uint32_t u = unit_of(j);
                l[j] = u < unitsa ? a.init[S.unit + u] : R(0);
                if (u < unitsa && a.row[S.unit + u] != kRowNone)
                  a.out_grad[out_a + a.row[S.unit + u]] = l[j];
              }
              sinks(l, [&](uint32_t, uint32_t r, R t) { a.out_grad[out_a + r] = t; });
            }
          }
        }
      }
      row_sync();
    } else if constexpr (ADJ) {
      // ---------------- adjoint (reverse) ----------------
      load_side(I.a);
      const uint32_t s0 = sg * K;
      // set points: the buffer a stage reads is written a stage ahead from
      // registers that were requested a stage (exact) or a step before.
      //   reference: x_n in buffer 0 (stage 1), the midpoint in buffer 1
      //   (stages 2, 3), x_{n-1} in buffer 0 (stage 4 and the next stage 1)
      //   exact: y4, y3, y2, y1 alternately, positions m descending
      R xn[RS];
      uint32_t m = exact ? 4u * (n - s0) - 1u : n - s0;
#pragma unroll
      for (int j = 0; j < RS; ++j) {
        const uint32_t u = unit_of(j);
        xn[j] = R(0);
        if (u < pubf) {
          *reinterpret_cast<R*>(Xb + u * EL) = seg[size_t(m) * pubf + u];
          if (m > 0u) xn[j] = seg[size_t(m - 1u) * pubf + u];
        }
        if (u < puba) *reinterpret_cast<R*>(Yb + u * EL) = exact ? h6 * l[j] : l[j];
      }
      landed();
      row_sync();
      const uint32_t nend = (n - s0 < budget) ? s0 : n - budget;
      budget -= n - nend;
      const R h3 = R(2) * h6;
      for (; n > nend; --n) {
        R acc[RS];
#pragma unroll kStageUnroll
        for (uint32_t s = 0; s < 4u; ++s) {
          const unsigned char* Y = Yb + (s & 1u) * ys;
          unsigned char* Yn = Yb + ((s + 1u) & 1u) * ys;
          const uint32_t xb = exact ? (s & 1u) : ((s == 1u || s == 2u) ? 1u : 0u);
          const unsigned char* X = Xb + xb * xs;
          // next value: y = cs k + cl l, and the slopes' weights
          const R cs = exact ? (s == 0u ? h : h2) : (s < 2u ? h2 : h);
          const R cl = exact ? (s < 2u ? h3 : h6) : R(1);
          const R wa = (!exact && (s == 1u || s == 2u)) ? R(2) : R(1);
          pieces(Y, X);
#pragma unroll
          for (int j = 0; j < RS; ++j) {
            const uint32_t u0 = uint32_t(j) * NT + wave * 64u, u = unit_of(j);
            if (u0 >= unitsa) continue;
            const R k = slope(j, u, Y, X);
            acc[j] = s == 0u ? k : rfma(wa, k, acc[j]);
            R y;
            if (s < 3u) {
              y = rfma(cs, k, exact ? cl * l[j] : l[j]);
            } else {
              l[j] = exact ? l[j] + acc[j] : rfma(h6, acc[j], l[j]);
              y = exact ? h6 * l[j] : l[j];
            }
            if (u < puba) *reinterpret_cast<R*>(Yn + u * EL) = y;
          }
          if (exact) {
            unsigned char* Xn = Xb + (xb ^ 1u) * xs;
#pragma unroll
            for (int j = 0; j < RS; ++j) {
              const uint32_t u = unit_of(j);
              if (u < pubf) {
                if (m > 0u) *reinterpret_cast<R*>(Xn + u * EL) = xn[j];
                if (m > 1u) xn[j] = seg[size_t(m - 2u) * pubf + u];
              }
            }
            --m;
          } else if (s == 0u) {
#pragma unroll
            for (int j = 0; j < RS; ++j) {
              const uint32_t u = unit_of(j);
              if (u < pubf)
                *reinterpret_cast<R*>(Xb + xs + u * EL) = R(0.5) * (at<R>(Xb, u * EL) + xn[j]);
            }
          } else if (s == 1u) {
#pragma unroll
            for (int j = 0; j < RS; ++j) {
              const uint32_t u = unit_of(j);
              if (u < pubf) {
                *reinterpret_cast<R*>(Xb + u * EL) = xn[j];
                if (m > 1u) xn[j] = seg[size_t(m - 2u) * pubf + u];
              }
            }
            --m;
          }
          row_sync();
        }
      }
      if (n == s0) {
        if (sg == 0u) {
          phase = kPhaseDone;
#pragma unroll
          for (int j = 0; j < RS; ++j) {
            const uint32_t u = unit_of(j);
            if (u < unitsa) {
              const uint32_t r = a.row[S.unit + u];
              if (r != kRowNone) a.out_grad[out_a + r] = l[j];
            }
          }
          sinks(l, [&](uint32_t, uint32_t r, R t) { a.out_grad[out_a + r] = t; });
        } else {
          sg -= 1u;
          n = sg * K;
          phase = kPhaseRecompute;
        }
      }
      row_sync();
    } else {
      phase = kPhaseDone;
    }
  }
#pragma unroll
  for (int j = 0; j < RS; ++j) {
    const uint32_t u = unit_of(j);
    if (u < unitsf) vecf[u] = q[j];
    if constexpr (ADJ) {
      if (adjoint && u < unitsa) veca[u] = l[j];
    }
  }
  if (tid == 0u) {
    pst[0] = n;
    pst[1] = phase;
    pst[2] = sg;
  }
}

template <typename R, bool ADJ, int RS, bool RES>
hipError_t launch_rows_cfg(const RowArgs<R>& a, uint32_t ninst, uint32_t waves, size_t lds,
                           hipStream_t s) {
  auto kern = row_kernel<R, ADJ, RS, RES>;
  if (lds > 65536) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, int(lds));
    if (e != hipSuccess) return e;
  }
  hipLaunchKernelGGL(kern, dim3(ninst), dim3(waves * 64u), lds, s, a);
  return hipGetLastError();
}

template <typename R, bool ADJ>
hipError_t launch_rows_adj(const RowArgs<R>& a, uint32_t ninst, uint32_t waves, uint32_t slots,
                           size_t lds, hipStream_t s) {
  if (slots <= 1u && a.resident)
    return launch_rows_cfg<R, ADJ, 1, true>(a, ninst, waves, lds, s);
  if (slots <= 1u) return launch_rows_cfg<R, ADJ, 1, false>(a, ninst, waves, lds, s);
  if (slots <= 2u) return launch_rows_cfg<R, ADJ, 2, false>(a, ninst, waves, lds, s);
  if (slots <= 4u) return launch_rows_cfg<R, ADJ, 4, false>(a, ninst, waves, lds, s);
  return launch_rows_cfg<R, ADJ, int(kRowSlots), false>(a, ninst, waves, lds, s);
}

template <typename R>
hipError_t launch_rows_impl(const RowArgs<R>& a, uint32_t ninst, uint32_t waves, uint32_t slots,
                            hipStream_t s) {
  if (ninst == 0u) return hipSuccess;
  const size_t lds = size_t(a.lds_slots) * sizeof(R);
  if (waves == 0u || waves * 64u > kRowThreads || slots > kRowSlots || lds > kMaxLdsBytes)
    return hipErrorInvalidValue;
  return a.adjoint ? launch_rows_adj<R, true>(a, ninst, waves, slots, lds, s)
                   : launch_rows_adj<R, false>(a, ninst, waves, slots, lds, s);
}

}  // namespace

hipError_t launch_rows(const RowArgs<double>& a, uint32_t ninst, uint32_t waves, uint32_t slots,
                       hipStream_t s) {
  return launch_rows_impl(a, ninst, waves, slots, s);
}
hipError_t launch_rows(const RowArgs<float>& a, uint32_t ninst, uint32_t waves, uint32_t slots,
                       hipStream_t s) {
  return launch_rows_impl(a, ninst, waves, slots, s);
}

}  // namespace pasif
