// Mixed-radix Stockham FFT over pencils staged in LDS.
//
// A pencil of length N is transformed by G threads.  Stage s with radix R
// and Ns = product of the radices before it performs N/R butterflies; the
// butterfly b reads elements b + r*N/R (r < R), twiddles them by
// w^(k*r) with w = exp(-+2 pi i / (Ns*R)) and k = b mod Ns, applies a radix-R
// DFT and writes element (b - k)*R + k + r*Ns.  After the last stage the
// pencil is in natural order (self-sorting, no bit reversal).  Each stage
// reads all of its inputs, synchronises the block, then writes its outputs,
// so a single LDS buffer per pencil is transformed in place.
//
// A thread works on NP pencils at once (for example the x, y and z
// components of a field): their loads are issued together, the twiddles and
// barriers are shared, so NP independent transforms cost one transform's
// latency.
//
// The first stage takes its inputs from a caller functor `src(j, n)` (pencil
// j, element n) and the last stage hands its outputs to
// `dst(j, n, value, slot)`, which is how loads from HBM (with any fused
// pre-processing) and stores to HBM (with any fused epilogue) are folded into
// the FFT.  `slot` is a compile-time-constant index of the output within the
// calling thread, identical for every transform with the same plan, so
// epilogues can keep per-output values in registers across transforms.
//
// Two engines share the stage code: `fft_rt` takes a runtime plan (any
// length that factors into 2 .. 13; one code path per radix) and
// `fft_ct<N>` a length fixed at compile time, for which every index is a
// constant and the stages unroll into straight-line code.
//
// Twiddles come from a per-length table of the N roots of unity
// exp(-2 pi i j / N) computed in double precision on the host and rounded
// once to float.  No normalisation is applied in either direction.
#pragma once

#include <type_traits>

#include "kw_common.h"

namespace kw {

// A transform of length N.  For N = 2^a 3^b 5^c 7^d 11^e 13^f the stages run
// at length L = N.  Any other N runs as Bluestein's chirp-z transform: with the
// chirp w_n = exp(-i pi n^2 / N), X_k = w_k sum_n (x_n w_n) conj(w_(k-n)),
// a circular convolution of length L >= 2N - 1 (L = 2^a 3^b 5^c) computed
// with two length-L transforms in LDS; `chirp` (N entries) and `bspec`
// (L entries: 1/L times the length-L transform of the chirp filter conj(w_m),
// m = -(N-1) .. N-1, wrapped) are set, and the inverse uses their conjugates.
struct FftPlan {
  int32_t N;   // length of the transform
  int32_t L;   // length the stages run at (N, or the chirp-z length)
  int32_t nst;
  int32_t radix[KW_MAX_STAGES];
  const cf* tw;     // L twiddles exp(-2 pi i j / L)
  const cf* chirp;  // Bluestein only (else NULL): w_n, n < N
  const cf* bspec;  // Bluestein only: transform of the chirp filter, L entries
};

// ---- compile-time plans -----------------------------------------------------
// The stages of a fixed length.  A stage costs a thread its elements and, in
// LDS round trip, barrier and index arithmetic, about kStageCost more; the plan
// has the least of that over all radix sequences (486: 9 9 6 for six stages of
// radix 2 and 3).
struct CtPlan {
  int nst = 0;
  int r[KW_MAX_STAGES] = {};
  int cost = 1 << 30;
};
constexpr int kStageCost = 3;

// elements of one stage of radix R per thread
KW_HOSTDEV constexpr int ct_stage_work(int N, int R, int G) { return (N / R + G - 1) / G * R; }

// `slots`: some stage leaves a thread at most that many elements
KW_HOSTDEV constexpr void ct_search(int N, int rest, int G, int emax, CtPlan cur, int cost, int top,
                         CtPlan& best, int slots = 1 << 20, int least = 1 << 20) {
  if (rest == 1) {
    if (cur.nst > 0 && cost < best.cost && least <= slots) {
      best = cur;
      best.cost = cost;
    }
    return;
  }
  if (cost >= best.cost || cur.nst >= 8) return;
  const int radices[9] = {12, 10, 9, 8, 6, 5, 4, 3, 2};
  for (int i = 0; i < 9; ++i) {
    const int R = radices[i];
    if (R > top || rest % R != 0) continue;
    const int w = ct_stage_work(N, R, G);
    if (w > emax) continue;
    CtPlan nx = cur;
    nx.r[nx.nst++] = R;
    ct_search(N, rest / R, G, emax, nx, cost + w + kStageCost, R, best, slots,
              w < least ? w : least);
  }
}

// strided plan of length N with G threads, at most 12 elements per thread,
// largest radix first (the first stage has no twiddles)
KW_HOSTDEV constexpr CtPlan ct_strided(int N, int G, int most = 12) {
  CtPlan best;
  ct_search(N, N, G, most, CtPlan{}, 0, 12, best);
  return best;
}
// threads per pencil of the strided plan: the least work over all lanes,
// then the most threads (half the elements per thread and five stages instead
// of four took the last axis of 1024 x 1024 from 21 to 23 us)
KW_HOSTDEV constexpr int strided_threads(int N, int most = 12) {
  int g = 0, work = 1 << 30;
  for (int G = (N + most - 1) / most; G <= (N + 5) / 6; ++G) {
    if (G > (N + 7) / 8 && g > 0) break;
    const CtPlan p = ct_strided(N, G, most);
    if (p.nst > 0 && p.cost * G <= work) {
      g = G;
      work = p.cost * G;
    }
  }
  return g;
}
// The y passes of an axis above 256 (384 is the only such length with a fixed y
// pass): at most eight elements per thread.  Their blocks have 768 threads and more, of which a CU holds two only while a
// thread's registers are few (384 = 12 8 4 on 48 threads: 224 us a forward
// launch of 384^3, 167 as 8 8 6 on 64).
KW_HOSTDEV constexpr int y_most(int N) { return N > 256 && strided_threads(N, 8) > 0 ? 8 : 12; }
KW_HOSTDEV constexpr int y_threads(int N) { return strided_threads(N, y_most(N)); }
// x plan: the stage that leaves a thread the fewest elements last, at most
// kXSlots, the largest of the others first.  The x passes keep several values
// per element in registers; with the plan of least work alone 72, 80 and 648
// left eight elements and 81, 90, 729 and 810 nine: x_div of 80 x 240 x 240
// 75 us as 10 8, 42 as 8 5 2, a step 281 -> 234; 648 x 96 x 96 396 -> 325.  The
// stages more cost small grids of 81 and 90 points (90 x 90 35 -> 38 us a step).
constexpr int kXSlots = 6;
KW_HOSTDEV constexpr CtPlan ct_xplan(int N, int G) {
  CtPlan p;
  ct_search(N, N, G, 12, CtPlan{}, 0, 10, p, kXSlots);
  int last = 0;
  for (int s = 1; s < p.nst; ++s)
    if (ct_stage_work(N, p.r[s], G) <= ct_stage_work(N, p.r[last], G)) last = s;
  const int R = p.r[last];
  for (int s = last; s + 1 < p.nst; ++s) p.r[s] = p.r[s + 1];
  if (p.nst > 0) p.r[p.nst - 1] = R;
  return p;
}

// upper bound of butterflies per thread for the runtime engine
template <int R>
struct MaxB {
  static constexpr int v = (KW_E + R - 1) / R;
};
// lengths with a factor 7 run with G = ceil(N/7) threads (see kw_sim.h), so
// a radix-7 stage has one butterfly per thread, as the larger radices have
// with any G >= N / 8
template <>
struct MaxB<7> {
  static constexpr int v = 1;
};
// largest number of last-stage outputs one thread can own with G = ceil(N/KW_E)
constexpr int kMaxSlots = 10;
static_assert(MaxB<2>::v * 2 <= kMaxSlots && MaxB<3>::v * 3 <= kMaxSlots &&
                  MaxB<4>::v * 4 <= kMaxSlots && MaxB<5>::v * 5 <= kMaxSlots &&
                  MaxB<8>::v * 8 <= kMaxSlots,
              "slot bound");

// Twiddle table of a plan as the stages read it: in HBM (each read a vector
// memory load through the same address path as the data streams), or
// copied once per block into LDS (put_twiddles).
struct TwG {
  const cf* p;
};
struct TwL {
  const cf* p;
};

template <bool INV>
KW_BODY cf twiddle(const TwG& tw, int idx) {
  cf w = KW_LD32(tw.p, (uint32_t)idx);
  if (INV) w.y = -w.y;
  return w;
}
template <bool INV>
KW_BODY cf twiddle(const TwL& tw, int idx) {
  cf w = lds_ld(tw.p + idx);
  if (INV) w.y = -w.y;
  return w;
}

// the L twiddles of a plan copied into the block's LDS at `dst` by all
// threads of the block (the caller synchronises), four loads in flight per
// thread: a small tile has fewer threads than twiddles, and one load at a
// time would cost it a memory latency per round
template <class Ctx>
KW_BODY TwL put_twiddles(Ctx& c, const FftPlan& pl, cf* dst) {
  const int L = pl.L, nt = c.nthreads();
  for (int i = c.tid(); i < L; i += 4 * nt) {
    cf w[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const int n = i + k * nt;
      w[k] = KW_LD32(pl.tw, (uint32_t)(n < L ? n : i));
    }
#pragma unroll
    for (int k = 0; k < 4; ++k)
      if (i + k * nt < L) lds_st(dst + i + k * nt, w[k]);
  }
  return TwL{dst};
}

// value of input n (slot: its place among the calling thread's inputs of
// the first stage), from a source that takes the slot or one that does not
template <class Src>
KW_BODY cf fetch(Src& src, int j, int n, int slot) {
  if constexpr (std::is_invocable_v<Src&, int, int, int>)
    return src(j, n, slot);
  else
    return src(j, n);
}

// x times a constant held as a rounded float and its remainder.  A radix's
// rounded sine is wrong by up to 3e-8 in every transform of a simulation, the
// same way each step: over 400 steps of 600 points the radix-3 and radix-5
// constants made most of the error against double precision.
struct Const2 {
  float hi, lo;
  constexpr Const2(double v) : hi((float)v), lo((float)(v - (double)(float)v)) {}
};
KW_BODY float mulc(float x, const Const2& k) { return x * k.hi + x * k.lo; }
KW_BODY cf mulc(cf a, const Const2& k) { return cf{mulc(a.x, k), mulc(a.y, k)}; }

// radix-R DFT in place; forward uses exp(-2 pi i rs/R), inverse exp(+...)
template <int R, bool INV>
KW_BODY void dft(cf* v);

template <>
KW_BODY void dft<2, false>(cf* v) {
  cf a = v[0], b = v[1];
  v[0] = cadd(a, b);
  v[1] = csub(a, b);
}
template <>
KW_BODY void dft<2, true>(cf* v) {
  dft<2, false>(v);
}

template <bool INV>
KW_BODY void dft3(cf* v) {
  constexpr Const2 s3(0.866025403784438646763723170752936183);  // sin(2 pi/3)
  cf t = cadd(v[1], v[2]);
  cf d = csub(v[1], v[2]);
  cf m = cf{v[0].x - 0.5f * t.x, v[0].y - 0.5f * t.y};
  cf sd = mulc(d, s3);
  // forward: X1 = m - i sd, X2 = m + i sd
  cf isd = INV ? cmul_pi(sd) : cmul_mi(sd);
  v[0] = cadd(v[0], t);
  v[1] = cadd(m, isd);
  v[2] = csub(m, isd);
}
template <>
KW_BODY void dft<3, false>(cf* v) { dft3<false>(v); }
template <>
KW_BODY void dft<3, true>(cf* v) { dft3<true>(v); }

template <bool INV>
KW_BODY void dft4(cf* v) {
  cf t0 = cadd(v[0], v[2]);
  cf t1 = csub(v[0], v[2]);
  cf t2 = cadd(v[1], v[3]);
  cf t3 = csub(v[1], v[3]);
  // forward: X1 = t1 - i t3, X3 = t1 + i t3
  cf it3 = INV ? cmul_pi(t3) : cmul_mi(t3);
  v[0] = cadd(t0, t2);
  v[2] = csub(t0, t2);
  v[1] = cadd(t1, it3);
  v[3] = csub(t1, it3);
}
template <>
KW_BODY void dft<4, false>(cf* v) { dft4<false>(v); }
template <>
KW_BODY void dft<4, true>(cf* v) { dft4<true>(v); }

template <bool INV>
KW_BODY void dft5(cf* v) {
  constexpr Const2 c1(0.309016994374947424102293417182819059);   // cos(2 pi/5)
  constexpr Const2 c2(-0.809016994374947424102293417182819059);  // cos(4 pi/5)
  constexpr Const2 s1(0.951056516295153572116439333379382143);   // sin(2 pi/5)
  constexpr Const2 s2(0.587785252292473129168705954639072769);   // sin(4 pi/5)
  cf a1 = cadd(v[1], v[4]), b1 = csub(v[1], v[4]);
  cf a2 = cadd(v[2], v[3]), b2 = csub(v[2], v[3]);
  cf x0 = v[0];
  // z + p a + q b, the remainders of the constants first
  auto lin = [](float z, const Const2& p, float a, const Const2& q, float b) {
    return ((z + (p.lo * a + q.lo * b)) + p.hi * a) + q.hi * b;
  };
  auto dif = [](const Const2& p, float a, const Const2& q, float b) {
    return ((p.lo * a - q.lo * b) + p.hi * a) - q.hi * b;
  };
  cf m1 = cf{lin(x0.x, c1, a1.x, c2, a2.x), lin(x0.y, c1, a1.y, c2, a2.y)};
  cf m2 = cf{lin(x0.x, c2, a1.x, c1, a2.x), lin(x0.y, c2, a1.y, c1, a2.y)};
  cf n1 = cf{lin(0.f, s1, b1.x, s2, b2.x), lin(0.f, s1, b1.y, s2, b2.y)};
  cf n2 = cf{dif(s2, b1.x, s1, b2.x), dif(s2, b1.y, s1, b2.y)};
  // forward: X1 = m1 - i n1, X4 = m1 + i n1, X2 = m2 - i n2, X3 = m2 + i n2
  cf in1 = INV ? cmul_pi(n1) : cmul_mi(n1);
  cf in2 = INV ? cmul_pi(n2) : cmul_mi(n2);
  v[0] = cf{x0.x + a1.x + a2.x, x0.y + a1.y + a2.y};
  v[1] = cadd(m1, in1);
  v[4] = csub(m1, in1);
  v[2] = cadd(m2, in2);
  v[3] = csub(m2, in2);
}
template <>
KW_BODY void dft<5, false>(cf* v) { dft5<false>(v); }
template <>
KW_BODY void dft<5, true>(cf* v) { dft5<true>(v); }

// odd prime radix from the pairs a_k = v_k + v_(R-k), b_k = v_k - v_(R-k):
// X_j = v_0 + sum_k cos(2 pi jk/R) a_k -+ i sum_k sin(2 pi jk/R) b_k
// (Rounded to single, without remainders: a stage of radix 13 holds 12 constants
// already, the runtime engine has no registers for twice as many.)
template <int R>
struct PrimeTrig;  // cos and sin of 2 pi m / R, m = 1 .. (R - 1) / 2
template <>
struct PrimeTrig<7> {
  static constexpr float c[3] = {0.6234898018587335f, -0.2225209339563144f, -0.9009688679024191f};
  static constexpr float s[3] = {0.7818314824680298f, 0.9749279121818236f, 0.4338837391175581f};
};
template <>
struct PrimeTrig<11> {
  static constexpr float c[5] = {0.8412535328311812f, 0.4154150130018864f, -0.142314838273285f,
                                 -0.654860733945285f, -0.9594929736144974f};
  static constexpr float s[5] = {0.5406408174555976f, 0.9096319953545184f, 0.9898214418809327f,
                                 0.7557495743542583f, 0.2817325568414297f};
};
template <>
struct PrimeTrig<13> {
  static constexpr float c[6] = {0.8854560256532099f, 0.5680647467311558f, 0.1205366802553230f,
                                 -0.3546048870425356f, -0.7485107481711011f, -0.9709418174260521f};
  static constexpr float s[6] = {0.4647231720437685f, 0.8229838658936564f, 0.9927088740980540f,
                                 0.9350162426854148f, 0.6631226582407952f, 0.2393156642875578f};
};
template <int R, bool INV>
KW_BODY void dft_prime(cf* v) {
  constexpr int H = (R - 1) / 2;
  cf a[H], b[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    a[k] = cadd(v[k + 1], v[R - 1 - k]);
    b[k] = csub(v[k + 1], v[R - 1 - k]);
  }
  float co_[H], si_[H];
#pragma unroll
  for (int k = 0; k < H; ++k) {
    co_[k] = kw_fresh_s(PrimeTrig<R>::c[k]);
    si_[k] = kw_fresh_s(PrimeTrig<R>::s[k]);
  }
  const cf x0 = v[0];
  cf sum = x0;
#pragma unroll
  for (int k = 0; k < H; ++k) sum = cadd(sum, a[k]);
  v[0] = sum;
#pragma unroll
  for (int j = 1; j <= H; ++j) {
    cf m = x0, n = cf{0.f, 0.f};
#pragma unroll
    for (int k = 1; k <= H; ++k) {
      const int q = j * k % R;
      const float co = co_[(q <= H ? q : R - q) - 1];
      const float si = q <= H ? si_[q - 1] : -si_[R - q - 1];
      m = cf{m.x + co * a[k - 1].x, m.y + co * a[k - 1].y};
      n = cf{n.x + si * b[k - 1].x, n.y + si * b[k - 1].y};
    }
    // forward: X_j = m - i n, X_(R-j) = m + i n
    const cf in = INV ? cmul_pi(n) : cmul_mi(n);
    v[j] = cadd(m, in);
    v[R - j] = csub(m, in);
  }
}
template <> KW_BODY void dft<7, false>(cf* v) { dft_prime<7, false>(v); }
template <> KW_BODY void dft<7, true>(cf* v) { dft_prime<7, true>(v); }
template <> KW_BODY void dft<11, false>(cf* v) { dft_prime<11, false>(v); }
template <> KW_BODY void dft<11, true>(cf* v) { dft_prime<11, true>(v); }
template <> KW_BODY void dft<13, false>(cf* v) { dft_prime<13, false>(v); }
template <> KW_BODY void dft<13, true>(cf* v) { dft_prime<13, true>(v); }

template <bool INV>
KW_BODY void dft8(cf* v) {
  constexpr Const2 h(0.707106781186547524400844362104849039);
  cf e[4] = {v[0], v[2], v[4], v[6]};
  cf o[4] = {v[1], v[3], v[5], v[7]};
  dft4<INV>(e);
  dft4<INV>(o);
  // o[k] *= w8^k, w8 = exp(-+ 2 pi i/8)
  const cf a = mulc(cf{o[1].x - o[1].y, o[1].x + o[1].y}, h);  // o[1] exp(+i pi/4)
  const cf b = mulc(cf{o[3].x - o[3].y, o[3].x + o[3].y}, h);  // o[3] exp(+i pi/4)
  o[1] = INV ? a : cf{a.y, -a.x};
  o[2] = INV ? cmul_pi(o[2]) : cmul_mi(o[2]);
  o[3] = INV ? cmul_pi(b) : cf{-b.x, -b.y};
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    v[k] = cadd(e[k], o[k]);
    v[k + 4] = csub(e[k], o[k]);
  }
}
template <>
KW_BODY void dft<8, false>(cf* v) { dft8<false>(v); }
template <>
KW_BODY void dft<8, true>(cf* v) { dft8<true>(v); }

// radix A B with A and B coprime by the prime-factor map (no twiddles):
// input (B i + A j) mod AB, output k with k = i' mod A and k = j' mod B
template <int A, int B, bool INV>
KW_BODY void dft_pfa(cf* v) {
  constexpr int R = A * B;
  cf t[B][A];
#pragma unroll
  for (int j = 0; j < B; ++j) {
#pragma unroll
    for (int i = 0; i < A; ++i) t[j][i] = v[(B * i + A * j) % R];
    dft<A, INV>(t[j]);
  }
  // after the A transforms column i holds B values per output i
#pragma unroll
  for (int i = 0; i < A; ++i) {
    cf w[B];
#pragma unroll
    for (int j = 0; j < B; ++j) w[j] = t[j][i];
    dft<B, INV>(w);
#pragma unroll
    for (int k = 0; k < R; ++k)
      if (k % A == i) v[k] = w[k % B];
  }
}
template <> KW_BODY void dft<6, false>(cf* v) { dft_pfa<3, 2, false>(v); }
template <> KW_BODY void dft<6, true>(cf* v) { dft_pfa<3, 2, true>(v); }
template <> KW_BODY void dft<10, false>(cf* v) { dft_pfa<5, 2, false>(v); }
template <> KW_BODY void dft<10, true>(cf* v) { dft_pfa<5, 2, true>(v); }
template <> KW_BODY void dft<12, false>(cf* v) { dft_pfa<3, 4, false>(v); }
template <> KW_BODY void dft<12, true>(cf* v) { dft_pfa<3, 4, true>(v); }

// multiply by exp(-+ i angle) given its cosine and sine
template <bool INV>
KW_BODY cf cturn(cf a, const Const2& co, const Const2& si) {
  const cf p = mulc(a, co), q = mulc(a, si);
  return INV ? cf{p.x - q.y, p.y + q.x} : cf{p.x + q.y, p.y - q.x};
}

// radix 9 as 3 x 3: input 3 n1 + n2, output k1 + 3 k2, constant twiddles
// between
template <bool INV>
KW_BODY void dft9(cf* v) {
  // cos and sin of 2 pi j / 9, j = 1, 2, 4
  constexpr Const2 c1(0.766044443118978035202392650555416673), s1(0.642787609686539326322643409907263432);
  constexpr Const2 c2(0.173648177666930348851716626769314796), s2(0.984807753012208059366743024589523013);
  constexpr Const2 c4(-0.939692620785908384054109277324731469), s4(0.342020143325668733044099614682259580);
  cf t[3][3];
#pragma unroll
  for (int i = 0; i < 3; ++i) {
#pragma unroll
    for (int j = 0; j < 3; ++j) t[i][j] = v[3 * j + i];
    dft<3, INV>(t[i]);
  }
  t[1][1] = cturn<INV>(t[1][1], c1, s1);
  t[1][2] = cturn<INV>(t[1][2], c2, s2);
  t[2][1] = cturn<INV>(t[2][1], c2, s2);
  t[2][2] = cturn<INV>(t[2][2], c4, s4);
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    cf w[3] = {t[0][k], t[1][k], t[2][k]};
    dft<3, INV>(w);
#pragma unroll
    for (int m = 0; m < 3; ++m) v[k + 3 * m] = w[m];
  }
}
template <> KW_BODY void dft<9, false>(cf* v) { dft9<false>(v); }
template <> KW_BODY void dft<9, true>(cf* v) { dft9<true>(v); }

KW_BODY int mod_ns(int b, int Ns) {
  // b mod Ns; Ns is a compile-time constant in the fixed-length engine and
  // a power of two for every stage before the first radix-3/5 stage
  return (Ns & (Ns - 1)) == 0 ? (b & (Ns - 1)) : b % Ns;
}

// One Stockham stage over NP pencils (see the file comment).  MB is the
// number of butterflies per thread (exact for the fixed-length engine, an
// upper bound for the runtime engine).  `src` must be safe to call for
// every thread, including threads with active == false.
// `rns` is 1 / Ns for a runtime Ns (b mod Ns by an integer division would be
// some forty instructions per butterfly; in float it is exact for b + 0.5
// below 2^20) and 0 for a compile-time one.
template <int R, int NP, bool INV, int MB, class Ctx, class TW, class Src, class Dst>
KW_BODY void stage(Ctx& c, int N, int Ns, int G, int g, bool active, const TW& tw, Src& src,
                   Dst& dst, float rns = 0.f) {
  auto mod = [&](int b) {
    return rns != 0.f ? b - Ns * (int)(((float)b + 0.5f) * rns) : mod_ns(b, Ns);
  };
  const int nb = N / R;
  const int twstep = N / (Ns * R);
  cf v[NP][MB][R];
  // loads and arithmetic run for every thread (callers make src safe for
  // threads without a pencil) so that they are not split into conditional
  // regions; only the stores are guarded by `active`
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int b = g + m * G;
    if (MB * G == nb || b < nb) {
      cf w[R];
      if (Ns > 1) {
        const int k = mod(b);
#pragma unroll
        for (int r = 1; r < R; ++r) w[r] = twiddle<INV>(tw, k * r * twstep);
      }
#pragma unroll
      for (int j = 0; j < NP; ++j) {
#pragma unroll
        for (int r = 0; r < R; ++r) v[j][m][r] = fetch(src, j, b + r * nb, m * R + r);
      }
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        if (Ns > 1) {
#pragma unroll
          for (int r = 1; r < R; ++r) v[j][m][r] = cmul(v[j][m][r], w[r]);
        }
        dft<R, INV>(v[j][m]);
      }
    }
  }
  c.sync();
#pragma unroll
  for (int j = 0; j < NP; ++j) {
#pragma unroll
    for (int m = 0; m < MB; ++m) {
      const int b = g + m * G;
      if (active && (MB * G == nb || b < nb)) {
        const int k = mod(b);
        const int j0 = (b - k) * R + k;
#pragma unroll
        for (int r = 0; r < R; ++r) dst(j, j0 + r * Ns, v[j][m][r], m * R + r);
      }
    }
  }
  c.sync();
}

// LDS view of NP pencils: element n of pencil j at base[j*sj + n*sn + pad]
// with pad = (n >> 3) when `padded` (breaks the power-of-two strides of the
// Stockham writes across LDS banks)
struct LdsPencils {
  cf* base;
  int sj, sn;
  bool padded;
  KW_BODY int at(int j, int n) const { return j * sj + n * sn + (padded ? (n >> 3) : 0); }
  KW_BODY cf get(int j, int n) const { return lds_ld(base + at(j, n)); }
  KW_BODY void set(int j, int n, cf v) const { lds_st(base + at(j, n), v); }
};

// ---- runtime-length engine --------------------------------------------------
// Any N = 2^a 3^b 5^c 7^d 11^e 13^f.  The transform is staged entirely in LDS: a strided,
// coalesced pass loads the pencil into LDS through the caller's functor, the
// Stockham stages run from LDS to LDS, and a strided pass hands element
// n = g + i*G to the caller as slot i.  The caller's functors are
// instantiated once per call site instead of once per radix and stage
// position, which would multiply the code size past the instruction cache.

constexpr int kRtSlots = 10;  // ceil(N / G) for G = ceil(N / KW_E)
static_assert(kRtSlots <= kMaxSlots, "slot bound");

// Threads without a pencil (active == false) may share another pencil's LDS
// to keep their loads in bounds, so they never store, here as in the
// fixed-length engine.
template <int NP, bool INV, class Ctx, class TW>
KW_BODY void fft_stages_rt(Ctx& c, const FftPlan& pl, const TW& tw, int g, int G, bool active,
                           const LdsPencils& lds) {
  auto lsrc = [&](int j, int n) -> cf { return lds.get(j, n); };
  auto ldst = [&](int j, int n, cf v, int) { lds.set(j, n, v); };
  int Ns = 1;
  const int L = pl.L;
  for (int s = 0; s < pl.nst; ++s) {
    const int R = pl.radix[s];
    const float rns = 1.0f / (float)Ns;
    // a fresh thread index per stage, or every radix's element indices are
    // hoisted out of this loop and spill
    const int gs = kw_fresh(g);
#define KW_RT_STAGE(RR)                                                                           \
  case RR: stage<RR, NP, INV, MaxB<RR>::v>(c, L, Ns, G, gs, active, tw, lsrc, ldst, rns); break;
    switch (R) {
      KW_RT_STAGE(2)
      KW_RT_STAGE(3)
      KW_RT_STAGE(4)
      KW_RT_STAGE(5)
      KW_RT_STAGE(7)
      KW_RT_STAGE(8)
      KW_RT_STAGE(9)
      KW_RT_STAGE(10)
      KW_RT_STAGE(11)
      KW_RT_STAGE(13)
    }
#undef KW_RT_STAGE
    Ns *= R;
  }
}

// Bluestein's transform of length N (see FftPlan) over the length-L stages:
// the chirped input zero-padded to L, a forward transform, the product with
// the filter's transform (which holds the 1/L), an inverse transform, and the
// chirped outputs; the inverse transform conjugates the chirp and the filter.
// Each thread reads and writes only its own elements n = g + i G between
// barriers, as the plain runtime engine does.
template <int NP, bool INV, class Ctx, class TW, class Src, class Dst>
KW_BODY void fft_bluestein(Ctx& c, const FftPlan& pl, const TW& tw, int g, int G, bool active,
                           Src& src, Dst& dst, const LdsPencils& lds) {
  const int N = pl.N, L = pl.L;
  auto chirp = [&](int n) -> cf {
    cf w = KW_LD32(pl.chirp, (uint32_t)n);
    if (INV) w.y = -w.y;
    return w;
  };
#pragma unroll
  for (int i = 0; i < kRtSlots; ++i) {
    const int n = g + i * G;
    if (n < L) {
      const cf w = n < N ? chirp(n) : cf{0.f, 0.f};
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        const cf v = n < N ? cmul(src(j, n), w) : cf{0.f, 0.f};
        if (active) lds.set(j, n, v);
      }
    }
  }
  c.sync();
  fft_stages_rt<NP, false>(c, pl, tw, g, G, active, lds);
#pragma unroll
  for (int i = 0; i < kRtSlots; ++i) {
    const int n = g + i * G;
    if (active && n < L) {
      cf b = KW_LD32(pl.bspec, (uint32_t)n);
      if (INV) b.y = -b.y;
#pragma unroll
      for (int j = 0; j < NP; ++j) lds.set(j, n, cmul(lds.get(j, n), b));
    }
  }
  c.sync();
  fft_stages_rt<NP, true>(c, pl, tw, g, G, active, lds);
#pragma unroll
  for (int i = 0; i < kRtSlots; ++i) {
    const int n = g + i * G;
    if (active && n < N) {
      const cf w = chirp(n);
#pragma unroll
      for (int j = 0; j < NP; ++j) dst(j, n, cmul(lds.get(j, n), w), i);
    }
  }
  c.sync();
}

template <int NP, bool INV, class Ctx, class TW, class Src, class Dst>
KW_BODY void fft_rt(Ctx& c, const FftPlan& pl, const TW& tw, int g, int G, bool active, Src& src,
                    Dst& dst, const LdsPencils& lds) {
  const int N = pl.N;
  g = kw_fresh(g);
  if (pl.chirp) {
    fft_bluestein<NP, INV>(c, pl, tw, g, G, active, src, dst, lds);
    return;
  }
#pragma unroll
  for (int i = 0; i < kRtSlots; ++i) {
    const int n = g + i * G;
    if (n < N) {
#pragma unroll
      for (int j = 0; j < NP; ++j) {
        const cf v = src(j, n);
        if (active) lds.set(j, n, v);
      }
    }
  }
  c.sync();
  fft_stages_rt<NP, INV>(c, pl, tw, g, G, active, lds);
#pragma unroll
  for (int i = 0; i < kRtSlots; ++i) {
    const int n = g + i * G;
    if (active && n < N) {
#pragma unroll
      for (int j = 0; j < NP; ++j) dst(j, n, lds.get(j, n), i);
    }
  }
  c.sync();
}

// the (slot, n) pairs this thread owns after a runtime-length transform
template <class F>
KW_BODY void last_slots_rt(const FftPlan& pl, int g, int G, bool, F& f) {
  g = kw_fresh(g);
#pragma unroll
  for (int i = 0; i < kRtSlots; ++i) {
    const int n = g + i * G;
    if (n < pl.N) f(i, n);
  }
}

// ---- fixed-length engine ------------------------------------------------------

// N, threads per pencil G and the plan family (X: x passes) as constants
template <int N_, int G_, bool X, int MOST = 12>
struct CtShape {
  static constexpr int N = N_;
  static constexpr int G = G_;
  static constexpr CtPlan plan = X ? ct_xplan(N, G) : ct_strided(N, G, MOST);
  static constexpr int nst = plan.nst;
  static_assert(nst > 0, "length must factor into 2, 3 and 5");
  static constexpr int radix(int s) { return plan.r[s]; }
  static constexpr int ns(int s) {
    int p = 1;
    for (int i = 0; i < s; ++i) p *= plan.r[i];
    return p;
  }
  static constexpr int mb(int s) { return (N / plan.r[s] + G - 1) / G; }
  // inputs of the first and outputs of the last stage per thread
  static constexpr int first_slots = mb(0) * plan.r[0];
  static constexpr int last_slots = mb(nst - 1) * plan.r[nst - 1];
};

template <class Sh, int S, int NP, bool INV>
struct CtStages {
  static constexpr int R = Sh::radix(S);
  static constexpr int Ns = Sh::ns(S);
  static constexpr int MB = Sh::mb(S);
  template <class Ctx, class TW, class Src, class Dst, class LSrc, class LDst>
  KW_BODY static void run(Ctx& c, int g, bool active, const TW& tw, Src& src0, Dst& dstN,
                          LSrc& lsrc, LDst& ldst) {
    if constexpr (S == 0 && Sh::nst == 1) {
      stage<R, NP, INV, MB>(c, Sh::N, Ns, Sh::G, g, active, tw, src0, dstN);
    } else if constexpr (S == 0) {
      stage<R, NP, INV, MB>(c, Sh::N, Ns, Sh::G, g, active, tw, src0, ldst);
    } else if constexpr (S == Sh::nst - 1) {
      stage<R, NP, INV, MB>(c, Sh::N, Ns, Sh::G, g, active, tw, lsrc, dstN);
    } else {
      stage<R, NP, INV, MB>(c, Sh::N, Ns, Sh::G, g, active, tw, lsrc, ldst);
    }
    if constexpr (S + 1 < Sh::nst)
      CtStages<Sh, S + 1, NP, INV>::run(c, g, active, tw, src0, dstN, lsrc, ldst);
  }
};

template <class Sh, int NP, bool INV, class Ctx, class TW, class Src, class Dst>
KW_BODY void fft_ct(Ctx& c, const TW& tw, int g, bool active, Src& src0, Dst& dstN,
                    const LdsPencils& lds) {
  g = kw_fresh(g);
  auto lsrc = [&](int j, int n) -> cf { return lds.get(j, n); };
  auto ldst = [&](int j, int n, cf v, int) { lds.set(j, n, v); };
  CtStages<Sh, 0, NP, INV>::run(c, g, active, tw, src0, dstN, lsrc, ldst);
}

// f(slot, n) for this thread's inputs of the first stage, in the order the
// stage reads them
template <class Sh, class F>
KW_BODY void first_slots_ct(int g, F& f) {
  constexpr int R = Sh::radix(0), nb = Sh::N / R, MB = Sh::mb(0);
  g = kw_fresh(g);
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int b = g + m * Sh::G;
    if (MB * Sh::G == nb || b < nb) {
#pragma unroll
      for (int r = 0; r < R; ++r) f(m * R + r, b + r * nb);
    }
  }
}

template <class Sh, class F>
KW_BODY void last_slots_ct(int g, bool, F& f) {
  constexpr int S = Sh::nst - 1;
  constexpr int R = Sh::radix(S), Ns = Sh::ns(S), nb = Sh::N / R, MB = Sh::mb(S);
  g = kw_fresh(g);
#pragma unroll
  for (int m = 0; m < MB; ++m) {
    const int b = g + m * Sh::G;
    if (MB * Sh::G == nb || b < nb) {
      const int k = mod_ns(b, Ns);
      const int j0 = (b - k) * R + k;
#pragma unroll
      for (int r = 0; r < R; ++r) f(m * R + r, j0 + r * Ns);
    }
  }
}

// ---- plan selectors -----------------------------------------------------------
// A kernel body templated on a selector runs the runtime engine (PlanRt) or
// the fixed-length engine (PlanCt<N>) for one axis.

// Start of a block: `load_first` issues the loads of a transform's first
// stage before the block has its twiddles, which that stage does not use, so
// the two memory latencies overlap; `fft_pre` runs the transform from them.

struct PlanRt {
  static constexpr int fixed = 0;
  static constexpr int G = 0;  // threads per pencil: chosen at run time
  template <class Src>
  struct Pre {};
  template <class Src>
  KW_BODY static void load_first(int, Src&, Pre<Src>&) {}
  // the runtime stages start from LDS, so the block's twiddles are waited
  // for before anything else
  static constexpr bool twiddles_first = true;
  template <int NP, bool INV, class Ctx, class TW, class Src, class Dst>
  KW_BODY static void fft_pre(Ctx& c, const FftPlan& pl, const TW& tw, int g, int G, bool active,
                              Src& src, Pre<Src>&, Dst& dst, const LdsPencils& lds) {
    fft_rt<NP, INV>(c, pl, tw, g, G, active, src, dst, lds);
  }
  template <int NP, bool INV, class Ctx, class TW, class Src, class Dst>
  KW_BODY static void fft_tw(Ctx& c, const FftPlan& pl, const TW& tw, int g, int G, bool active,
                             Src& src, Dst& dst, const LdsPencils& lds) {
    fft_rt<NP, INV>(c, pl, tw, g, G, active, src, dst, lds);
  }
  template <class F>
  KW_BODY static void last_slots(const FftPlan& pl, int g, int G, bool active, F& f) {
    last_slots_rt(pl, g, G, active, f);
  }
};

// threads per pencil of the fixed-length x passes: the smallest power of two
// with at most six elements of the pencil each, so that every pencil lies in
// one wavefront and the stages synchronise with wavefront barriers instead of
// block barriers (the extra lanes idle in stages with fewer butterflies than
// lanes); lengths above 384 take a wavefront per 256 elements (one step of 600
// points 37 -> 29 us against N / 8 threads)
KW_HOSTDEV constexpr int x_threads(int N) {
  for (int p = 1; p <= 64; p <<= 1)
    if (6 * p >= N) return p;
  return (N + 255) / 256 * 64;
}

// elements a thread owns after an x transform, and whether the 3-D x_div
// kernel of that length also writes the p time series: it holds a dozen
// registers per element, and from six elements on the record's few more cost
// it a wavefront per SIMD (192: 128 -> 129 VGPRs, 74 -> 90 us at 192^3; at
// 128^3 and 144 x 160 x 192 no difference).  2-D grids always record.
KW_HOSTDEV constexpr int x_slots(int N) {
  const int G = x_threads(N);
  const CtPlan p = ct_xplan(N, G);
  return ct_stage_work(N, p.r[p.nst - 1], G);
}
KW_HOSTDEV constexpr bool x_div_records(int dim, int fixed) {
  return dim == 2 || fixed == 0 || x_slots(fixed) < 6;
}

template <class Sh>
struct PlanFixed {
  static constexpr int fixed = Sh::N;
  // threads per pencil; when N is not a multiple of G some threads get
  // fewer butterflies (the stages guard them)
  static constexpr int G = Sh::G;
  // with one stage there is no block barrier between the twiddles and their
  // first use (and no twiddle is used)
  static constexpr bool twiddles_first = false;
  template <class Src>
  struct Pre {
    cf v[Sh::first_slots];
  };
  template <class Src>
  KW_BODY static void load_first(int g, Src& src, Pre<Src>& pre) {
    auto f = [&](int slot, int n) { pre.v[slot] = src(0, n); };
    first_slots_ct<Sh>(g, f);
  }
  template <int NP, bool INV, class Ctx, class TW, class Src, class Dst>
  KW_BODY static void fft_pre(Ctx& c, const FftPlan&, const TW& tw, int g, int, bool active,
                              Src&, Pre<Src>& pre, Dst& dst, const LdsPencils& lds) {
    static_assert(NP == 1, "one pencil");
    auto held = [&](int, int, int slot) -> cf { return pre.v[slot]; };
    fft_ct<Sh, 1, INV>(c, tw, g, active, held, dst, lds);
  }
  template <int NP, bool INV, class Ctx, class TW, class Src, class Dst>
  KW_BODY static void fft_tw(Ctx& c, const FftPlan&, const TW& tw, int g, int, bool active,
                             Src& src, Dst& dst, const LdsPencils& lds) {
    fft_ct<Sh, NP, INV>(c, tw, g, active, src, dst, lds);
  }
  template <class F>
  KW_BODY static void last_slots(const FftPlan&, int g, int, bool active, F& f) {
    last_slots_ct<Sh>(g, active, f);
  }
};

// the plans of the last-axis and the strided y passes for a fixed length
template <int N>
using PlanCt = PlanFixed<CtShape<N, strided_threads(N), false>>;
template <int N>
using PlanCtY = PlanFixed<CtShape<N, y_threads(N), false, y_most(N)>>;

// the plan of the x passes for a fixed length
template <int N>
struct PlanCtX : PlanFixed<CtShape<N, x_threads(N), true>> {
  static_assert(CtShape<N, x_threads(N), true>::last_slots <= kXSlots, "slot bound");
};

}  // namespace kw
