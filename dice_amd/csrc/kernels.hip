// SHCI variational-step kernels for CDNA4 (gfx950, wave64).
//
//   energy / Hij batches      SHCI/Determinants.cpp:252-300,406-505,564-631
//   heat-bath screening       SHCI/SHCIgetdeterminants.cpp:586-739
//   connected-pair CSR        SHCI/SHCImakeHamiltonian.cpp:486-715 (row content)
//   sigma = H x               SHCI/Hmult.h:52-150
//   Davidson vector algebra   SHCI/Davidson.cpp:85-348
#include <algorithm>
#include <type_traits>
#include <cfloat>
#include <cmath>
#include <cstdlib>
#include <mutex>
#include <string>

#include "kernels.h"

namespace shci {

namespace {

constexpr int kBlock = 256;
constexpr int kWaves = kBlock / 64;

inline unsigned gridFor(int64_t n, int per = kBlock, int64_t cap = 1 << 20) {
  int64_t g = (n + per - 1) / per;
  if (g < 1) g = 1;
  if (g > cap) g = cap;
  return (unsigned)g;
}

// orders a wave's LDS accesses: what its lanes wrote is seen by their reads
__device__ __forceinline__ void waveSync() {
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  __builtin_amdgcn_wave_barrier();
}

// ---------------------------------------------------------------------------
// determinant primitives

template <int W>
__global__ void kEnergy(DevSystem S, const uint64_t* dets, int64_t n, double* out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) d[w] = dets[i * W + w];
    out[i] = detEnergy<W>(S, d);
  }
}

template <int W>
__global__ void kHijPairs(DevSystem S, const uint64_t* bra, const uint64_t* ket, int64_t n, double* out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    uint64_t b[W], k[W];
#pragma unroll
    for (int w = 0; w < W; w++) {
      b[w] = bra[i * W + w];
      k[w] = ket[i * W + w];
    }
    out[i] = hijElement<W>(S, b, k);
  }
}

// ---------------------------------------------------------------------------
// membership table

__global__ void kFillNeg(int32_t* t, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x)
    t[i] = -1;
}

template <int W>
__device__ __forceinline__ bool detEqual(const uint64_t* a, const uint64_t* b) {
  bool e = true;
#pragma unroll
  for (int w = 0; w < W; w++) e &= (a[w] == b[w]);
  return e;
}

template <int W>
__global__ void kHashInsert(const uint64_t* dets, int64_t begin, int64_t end, int32_t* table, uint64_t mask) {
  for (int64_t i = begin + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < end;
       i += (int64_t)gridDim.x * blockDim.x) {
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) d[w] = dets[i * W + w];
    uint64_t h = detHash<W>(d) & mask;
    while (true) {
      int32_t prev = atomicCAS(&table[h], -1, (int32_t)i);
      if (prev == -1) break;
      if (detEqual<W>(dets + (int64_t)prev * W, d)) break;
      h = (h + 1) & mask;
    }
  }
}

template <int W>
__device__ __forceinline__ bool hashContains(const int32_t* table, uint64_t mask, const uint64_t* dets,
                                             const uint64_t* key) {
  uint64_t h = detHash<W>(key) & mask;
  while (true) {
    int32_t v = table[h];
    if (v < 0) return false;
    if (detEqual<W>(dets + (int64_t)v * W, key)) return true;
    h = (h + 1) & mask;
  }
}

// ---------------------------------------------------------------------------
// screening

__global__ void kCmax(const double* ci, int nroots, int64_t ld, int64_t n, double* cmax) {
  for (int64_t j = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; j < n; j += (int64_t)gridDim.x * blockDim.x) {
    double s = 0.0;
    for (int r = 0; r < nroots; r++) {
      double c = fabs(ci[r * ld + j]);
      s = __dadd_rn(s, __dmul_rn(c, c));
    }
    cmax[j] = sqrt(s);
  }
}

// emit one candidate per lane with `want`, skipping determinants already in
// the variational space; wave-aggregated append
template <int W>
__device__ __forceinline__ void emitCandidate(bool want, const uint64_t* cand, const int32_t* table, uint64_t mask,
                                              const uint64_t* dets, uint64_t* out, unsigned long long* counter,
                                              int64_t cap) {
  bool keep = want && !hashContains<W>(table, mask, dets, cand);
  uint64_t m = __ballot(keep);
  if (m == 0) return;
  const int lane = __lane_id();
  unsigned long long base = 0;
  int leader = __ffsll((unsigned long long)m) - 1;
  if (lane == leader) base = atomicAdd(counter, (unsigned long long)__popcll(m));
  base = __shfl(base, leader, 64);
  if (keep) {
    unsigned long long pos = base + __popcll(m & lanemaskLt());
    if ((int64_t)pos < cap) {
#pragma unroll
      for (int w = 0; w < W; w++) out[pos * W + w] = cand[w];
    }
  }
}

// The screening's candidates of one wave: as emitCandidate, but queued in LDS
// (128 determinants) and appended 64 at a time, so that the one counter, on
// which atomics are serialised, takes an atomic per 64 candidates and not one
// per step that finds any.  With it kScreen of 400,009 sources in 24 orbitals
// (and, few sources, the cut by pairs) took 2.86 -> 2.10 ms.
template <int W>
struct CandidateQueue {
  uint64_t* queue;  // 128 x W
  int queued;       // wave-uniform
  const int32_t* table;
  uint64_t mask;
  const uint64_t* dets;
  uint64_t* out;
  unsigned long long* counter;
  int64_t cap;
  bool trev;
  __device__ __forceinline__ void append(int count) {
    const int lane = __lane_id();
    unsigned long long base = 0;
    if (lane == 0) base = atomicAdd(counter, (unsigned long long)count);
    base = __shfl(base, 0, 64);
    if (lane < count && (int64_t)(base + lane) < cap) {
#pragma unroll
      for (int w = 0; w < W; w++) out[(base + lane) * W + w] = queue[lane * W + w];
    }
  }
  __device__ __forceinline__ void put(bool want, const uint64_t* candIn) {
    uint64_t cand[W];
#pragma unroll
    for (int w = 0; w < W; w++) cand[w] = candIn[w];
    // with time reversal the space holds standard forms (SHCI/SHCIbasics.cpp:984-996)
    if (trev) makeStandardForm<W>(cand);
    const bool keep = want && !hashContains<W>(table, mask, dets, cand);
    const uint64_t m = __ballot(keep);
    if (m == 0ull) return;
    if (keep) {
      const int q = queued + __popcll(m & lanemaskLt());
#pragma unroll
      for (int w = 0; w < W; w++) queue[q * W + w] = cand[w];
    }
    queued += __popcll(m);
    if (queued < 64) return;
    waveSync();
    append(64);
    const int lane = __lane_id();
    queued -= 64;
    uint64_t t[W];
#pragma unroll
    for (int w = 0; w < W; w++) t[w] = queue[(64 + lane) * W + w];
    waveSync();
    if (lane < queued) {
#pragma unroll
      for (int w = 0; w < W; w++) queue[lane * W + w] = t[w];
    }
    waveSync();
  }
  __device__ __forceinline__ void finish() {
    waveSync();
    if (queued) append(queued);
    queued = 0;
    waveSync();
  }
};

__device__ __forceinline__ void emitRecord(bool want, const CandRecord& r, CandRecord* out,
                                           unsigned long long* counter, int64_t cap) {
  uint64_t m = __ballot(want);
  if (m == 0) return;
  const int lane = __lane_id();
  unsigned long long base = 0;
  int leader = __ffsll((unsigned long long)m) - 1;
  if (lane == leader) base = atomicAdd(counter, (unsigned long long)__popcll(m));
  base = __shfl(base, leader, 64);
  if (want) {
    unsigned long long pos = base + __popcll(m & lanemaskLt());
    if ((int64_t)pos < cap) out[pos] = r;
  }
}

// MODE 0: singles and doubles emitted as determinants (the reference's
// screening).  MODE 1: singles only.  MODE 2: no singles; every double
// excitation whose heat-bath value passes eps / loosen (a superset of the
// accepted ones) is emitted as a CandRecord for the learned ranking.
// A source's pairs of electrons are cut into `slices` parts, a wave each (with
// more than one, part 0 is the singles): a run's first iteration screens one
// determinant, whose lists one wave walked in 22 ms on 40 orbitals.  What bounds
// it then are the lists' lengths, a search for each pair, and the few
// candidates that a source has left.
template <int W, int MODE>
__global__ void __launch_bounds__(kBlock) kScreen(DevSystem S, const uint64_t* dets, int64_t srcBegin,
                                                  int64_t ndets, const double* cmax, double eps1, int ncore,
                                                  int nact, const int32_t* table, uint64_t mask, uint64_t* out,
                                                  unsigned long long* counter, int64_t cap, double loosen,
                                                  CandRecord* rec, int slices) {
  __shared__ uint8_t sClosed[kWaves][128];
  __shared__ uint8_t sOpen[kWaves][128];
  __shared__ int sExcl[kWaves][65];
  __shared__ int64_t sStart[kWaves][64];
  __shared__ int sPair[kWaves][64];
  __shared__ uint64_t sQueue[MODE == 2 ? 1 : kWaves][MODE == 2 ? 1 : 128 * W];
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  const int nso = S.nso;
  CandidateQueue<W> queue{&sQueue[MODE == 2 ? 0 : wave][0], 0, table, mask, dets, out, counter, cap, S.trev != 0};
  for (int64_t wi = (int64_t)blockIdx.x * kWaves + wave; wi < (ndets - srcBegin) * slices;
       wi += (int64_t)gridDim.x * kWaves) {
    const int64_t di = srcBegin + wi / slices;
    const int slice = (int)(wi - (wi / slices) * slices);
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) d[w] = dets[di * W + w];
    const double eps = eps1 / fabs(cmax[di]);
    // ascending closed / open spin-orbital lists
    int nclosed = 0, nopen = 0;
    for (int base = 0; base < nso; base += 64) {
      int k = base + lane;
      bool valid = k < nso;
      bool o = valid && occ<W>(d, k);
      uint64_t mc = __ballot(o), mo = __ballot(valid && !o);
      if (o) sClosed[wave][nclosed + __popcll(mc & lanemaskLt())] = (uint8_t)k;
      if (valid && !o) sOpen[wave][nopen + __popcll(mo & lanemaskLt())] = (uint8_t)k;
      nclosed += __popcll(mc);
      nopen += __popcll(mo);
    }
    __syncwarp();
    int cur[SHCI_MAX_RESTRICT];
    for (int r = 0; r < S.nrestrict; r++) {
      int c = 0;
      for (int k = 0; k < nclosed; k++) c += S.rmult[r * nso + sClosed[wave][k]];
      cur[r] = c;
    }
    // ---- single excitations
    const int nsingle = MODE == 2 || slice != 0 ? 0 : nclosed * nopen;
    for (int t0 = 0; t0 < nsingle; t0 += 64) {
      int t = t0 + lane;
      bool want = false;
      uint64_t cand[W];
#pragma unroll
      for (int w = 0; w < W; w++) cand[w] = d[w];
      if (t < nsingle) {
        int i = t / nopen, a = t - (t / nopen) * nopen;
        int ci = sClosed[wave][i], oa = sOpen[wave][a];
        bool ok = !((ci >> 1) < ncore || (oa >> 1) >= ncore + nact);
        for (int r = 0; r < S.nrestrict && ok; r++) {
          int e = cur[r] - S.rmult[r * nso + ci] + S.rmult[r * nso + oa];
          if (e < S.rmin[r] || e > S.rmax[r]) ok = false;
        }
        if (ok) {
          double integral = S.singles[oa * nso + ci];
          if (fabs(integral) > eps)
            if (((ci ^ oa) & 1) == 0) integral = hijSingle<W>(S, d, oa, ci);
          if (fabs(integral) > eps) {
            want = true;
            cand[oa >> 6] |= (1ull << (oa & 63));
            cand[ci >> 6] &= ~(1ull << (ci & 63));
          }
        }
      }
      queue.put(want, cand);
    }
    // ---- double excitations
    if (MODE == 1) continue;
    const double epsD = MODE == 2 ? eps / loosen : eps;
    if (S.maxEntryAbs < epsD) continue;
    const int npairs = nclosed * (nclosed - 1) / 2;
    const int perSlice = slices > 1 ? (npairs + slices - 2) / (slices - 1) : npairs;
    const int pBegin = slices > 1 ? (slice == 0 ? npairs : (slice - 1) * perSlice) : 0;
    const int pEnd = pBegin + perSlice < npairs ? pBegin + perSlice : npairs;
    for (int p0 = pBegin; p0 < pEnd; p0 += 64) {
      int p = p0 + lane;
      int len = 0;
      int64_t st = 0;
      if (p < pEnd) {
        // p = i*(i-1)/2 + j with i > j
        int i = (int)((1.0 + sqrt(1.0 + 8.0 * (double)p)) * 0.5);
        while (i * (i - 1) / 2 > p) i--;
        while ((i + 1) * i / 2 <= p) i++;
        int j = p - i * (i - 1) / 2;
        int ci = sClosed[wave][i], cj = sClosed[wave][j];
        if (!((ci >> 1) < ncore || (cj >> 1) < ncore)) {
          int I = ci >> 1, J = cj >> 1;
          int X = I > J ? I : J, Y = I > J ? J : I;
          int pairIndex = X * (X + 1) / 2 + Y;
          int sameSpin = ((ci ^ cj) & 1) == 0 ? 1 : 0;
          int64_t s0 = S.hbStart[sameSpin][pairIndex], s1 = S.hbStart[sameSpin][pairIndex + 1];
          const float* v = S.hbVal[sameSpin];
          // number of leading entries with |v| >= eps (list is |v|-descending)
          int64_t lo = s0, hi = s1;
          while (lo < hi) {
            int64_t mid = (lo + hi) >> 1;
            if ((double)fabsf(v[mid]) < epsD)
              hi = mid;
            else
              lo = mid + 1;
          }
          len = (int)(lo - s0);
          st = s0;
        }
        sPair[wave][lane] = i | (j << 8) | ((((sClosed[wave][i] ^ sClosed[wave][j]) & 1) == 0 ? 1 : 0) << 16);
      }
      // exclusive prefix of len over lanes
      int inc = len;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
      }
      sExcl[wave][lane] = inc - len;
      sStart[wave][lane] = st;
      int total = __shfl(inc, 63, 64);
      __syncwarp();
      for (int k0 = 0; k0 < total; k0 += 64) {
        int k = k0 + lane;
        bool want = false;
        uint64_t cand[W];
        CandRecord recTmp{};
#pragma unroll
        for (int w = 0; w < W; w++) cand[w] = d[w];
        if (k < total) {
          // owner lane q: last q with sExcl[q] <= k
          int lo = 0, hi = 63;
          while (lo < hi) {
            int mid = (lo + hi + 1) >> 1;
            if (sExcl[wave][mid] <= k)
              lo = mid;
            else
              hi = mid - 1;
          }
          int q = lo;
          int pk = sPair[wave][q];
          int i = pk & 0xFF, j = (pk >> 8) & 0xFF, same = (pk >> 16) & 1;
          int ci = sClosed[wave][i], cj = sClosed[wave][j];
          int64_t idx = sStart[wave][q] + (k - sExcl[wave][q]);
          uint32_t ab = S.hbPair[same][idx];
          int a = 2 * (int)(ab & 0xFFFF) + (ci & 1), b = 2 * (int)(ab >> 16) + (cj & 1);
          bool ok = !((a >> 1) >= ncore + nact || (b >> 1) >= ncore + nact);
          for (int r = 0; r < S.nrestrict && ok; r++) {
            const int8_t* m = S.rmult + r * nso;
            int e = cur[r] - m[ci] - m[cj] + m[a] + m[b];
            if (e < S.rmin[r] || e > S.rmax[r]) ok = false;
          }
          if (ok && !(occ<W>(d, a) || occ<W>(d, b))) {
            want = true;
            if (MODE == 2) {
              recTmp.src = (uint32_t)di;
              recTmp.ci = (uint8_t)ci;
              recTmp.cj = (uint8_t)cj;
              recTmp.a = (uint8_t)a;
              recTmp.b = (uint8_t)b;
              recTmp.v = S.hbVal[same][idx];
            }
            cand[a >> 6] |= (1ull << (a & 63));
            cand[b >> 6] |= (1ull << (b & 63));
            cand[ci >> 6] &= ~(1ull << (ci & 63));
            cand[cj >> 6] &= ~(1ull << (cj & 63));
          }
        }
        if (MODE == 2)
          emitRecord(want, recTmp, rec, counter, cap);
        else
          queue.put(want, cand);
      }
      __syncwarp();
    }
  }
  if (MODE != 2) queue.finish();
}

// ---------------------------------------------------------------------------
// deterministic EN-PT2 (SHCI/SHCIbasics.cpp:453-728 with the candidate rules of
// SHCI/SHCIgetdeterminants.cpp:40-171)

// partition of a candidate among nparts passes (hash bits above the ones the
// membership table uses)
template <int W>
__device__ __forceinline__ uint32_t ptPart(const uint64_t* d, uint32_t nparts) {
  return nparts == 1 ? 0u : (uint32_t)((detHash<W>(d) >> 40) % nparts);
}

// Count pass: per-lane counters.  Fill pass: wave-uniform cursor with ballot
// positions, so a source's candidates land in the reference's generation
// order (singles by (closed i, open a), then doubles by (i > j) pair and
// heat-bath order).
template <int W, bool FILL>
struct PtSink {
  int64_t pos;
  int cnt;
  uint64_t* outD;
  double* outN;
  double* outN2;     // semistochastic: second-moment numerator
  uint8_t* outP;     // semistochastic: term passes epsilon2Large
  __device__ __forceinline__ void put(bool keep, const uint64_t* cand, double num, double num2 = 0.0,
                                      bool present = false) {
    if (!FILL) {
      cnt += keep ? 1 : 0;
      return;
    }
    const uint64_t m = __ballot(keep);
    if (keep) {
      const int64_t p = pos + __popcll(m & lanemaskLt());
#pragma unroll
      for (int w = 0; w < W; w++) outD[p * W + w] = cand[w];
      outN[p] = num;
      if (outN2) {
        outN2[p] = num2;
        outP[p] = present ? 1 : 0;
      }
    }
    pos += __popcll(m);
  }
};

// Semistochastic mode (SHCI/SHCIgetdeterminants.cpp:889-1046): source k is
// determinant src[k] with sample weight w[k]; num = H_ai w, num2 = H_ai^2 w
// (w Nmc / (Nmc - 1) - c) with a double's H_ai^2 formed in float as there,
// present = |H_ai| > epsilon2Large / |c|.
struct PtStoch {
  const uint32_t* src;
  const double* w;
  double eps2Large;
  double nmc;
  double* outN2;
  uint8_t* outP;
};

// a dense copy of one spin case's heat-bath lists (cleared to NaN first)
__global__ void kFillNan(float* v, int64_t m) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = NAN;
}
__global__ void kDenseHeatBath(const float* val, const uint32_t* pair, const int64_t* start, int64_t npair, int norb,
                               float* dense) {
  for (int64_t p = blockIdx.x; p < npair; p += gridDim.x)
    for (int64_t k = start[p] + threadIdx.x; k < start[p + 1]; k += blockDim.x)
      dense[p * norb * norb + (int64_t)(pair[k] & 0xFFFF) * norb + (pair[k] >> 16)] = val[k];
}

// Candidates D_a of sources [0, ndets) with numerator H_ai c_i: singles with
// |Hij_1Excite| > eps, doubles while the float heat-bath value passes eps
// (numerator = value x parity of the excitation x c_i), eps = |eps2 / c_i|,
// no active-space limits, the PT restrictions in S; kept when D_a is not a
// variational determinant and falls in partition `part`.
//
// Work: a source's pairs of electrons are cut into `slices` parts (with more
// than one, part 0 is the singles), a wave each, so that a few sources fill
// the chip too.  A pair's doubles are found in one of two ways, whichever
// looks at fewer places: the prefix of the pair's |v|-sorted list that passes
// eps, most of whose entries excite into occupied orbitals, or every pair of
// open orbitals, whose values a dense copy of the lists gives (dense[same
// spin][pair][a n + b], NaN where the list has no entry).
// Measured: 200 sampled sources of 57,963 determinants of 40 orbitals (eps2
// 3e-4), count and fill 33 + 41 -> 0.71 + 0.89 ms with the parts; 27,685
// sources of 24 orbitals (eps2 3e-4, 33 million determinants found), one part
// each, 12.6 + 14.8 -> 7.5 + 8.8 ms with the open pairs: there the membership
// probes bound it.
template <int W, bool FILL, bool STOCH>
__global__ void __launch_bounds__(kBlock) kPtGen(DevSystem S, const uint64_t* dets, int64_t ndets, const double* ci,
                                                 double eps2, const int32_t* table, uint64_t mask, uint32_t nparts,
                                                 uint32_t part, int64_t* counts, const int64_t* fillStart,
                                                 uint64_t* outD, double* outN, PtStoch st, int slices,
                                                 const float* __restrict__ dense0, const float* __restrict__ dense1) {
  __shared__ uint8_t sClosed[kWaves][128];
  __shared__ uint8_t sOpen[kWaves][128];
  __shared__ uint8_t sSpin[kWaves][2][64];  // open spatial orbitals of each spin
  __shared__ int sExcl[kWaves][65];
  __shared__ int64_t sStart[kWaves][64];
  __shared__ int sPair[kWaves][64];
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  const int nso = S.nso, norb = S.norb;
  for (int64_t wi = (int64_t)blockIdx.x * kWaves + wave; wi < ndets * slices; wi += (int64_t)gridDim.x * kWaves) {
    const int64_t di = wi / slices;
    const int slice = (int)(wi - di * slices);
    const int64_t src = STOCH ? (int64_t)st.src[di] : di;
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) d[w] = dets[src * W + w];
    const double c = ci[src];
    const double wt = STOCH ? st.w[di] : c;
    const double eps = STOCH ? __ddiv_rn(eps2, fabs(c)) : fabs(eps2 / c);
    const double epsL = STOCH ? __ddiv_rn(st.eps2Large, fabs(c)) : 0.0;
    const double wfac = STOCH ? __dsub_rn(__ddiv_rn(__dmul_rn(wt, st.nmc), st.nmc - 1.0), c) : 0.0;
    PtSink<W, FILL> sink;
    sink.pos = FILL ? fillStart[wi] : 0;
    sink.cnt = 0;
    sink.outD = outD;
    sink.outN = outN;
    sink.outN2 = STOCH ? st.outN2 : nullptr;
    sink.outP = STOCH ? st.outP : nullptr;
    int nclosed = 0, nopen = 0;
    for (int base = 0; base < nso; base += 64) {
      int k = base + lane;
      bool valid = k < nso;
      bool o = valid && occ<W>(d, k);
      uint64_t mc = __ballot(o), mo = __ballot(valid && !o);
      if (o) sClosed[wave][nclosed + __popcll(mc & lanemaskLt())] = (uint8_t)k;
      if (valid && !o) sOpen[wave][nopen + __popcll(mo & lanemaskLt())] = (uint8_t)k;
      nclosed += __popcll(mc);
      nopen += __popcll(mo);
    }
    int nSpin[2];
#pragma unroll
    for (int sp = 0; sp < 2; sp++) {  // (at most 63 spatial orbitals)
      const bool o = lane < norb && !occ<W>(d, 2 * lane + sp);
      const uint64_t mo = __ballot(o);
      if (o) sSpin[wave][sp][__popcll(mo & lanemaskLt())] = (uint8_t)lane;
      nSpin[sp] = __popcll(mo);
    }
    __syncwarp();
    int cur[SHCI_MAX_RESTRICT];
    for (int r = 0; r < S.nrestrict; r++) {
      int cc = 0;
      for (int k = 0; k < nclosed; k++) cc += S.rmult[r * nso + sClosed[wave][k]];
      cur[r] = cc;
    }
    // ---- single excitations
    const int nsingle = slice == 0 ? nclosed * nopen : 0;
    for (int t0 = 0; t0 < nsingle; t0 += 64) {
      int t = t0 + lane;
      bool keep = false, pres = false;
      double num = 0.0, num2 = 0.0;
      uint64_t cand[W];
#pragma unroll
      for (int w = 0; w < W; w++) cand[w] = d[w];
      if (t < nsingle) {
        int i = t / nopen, a = t - (t / nopen) * nopen;
        int cI = sClosed[wave][i], oa = sOpen[wave][a];
        bool ok = true;
        for (int r = 0; r < S.nrestrict && ok; r++) {
          int e = cur[r] - S.rmult[r * nso + cI] + S.rmult[r * nso + oa];
          if (e < S.rmin[r] || e > S.rmax[r]) ok = false;
        }
        // (a spin-changing single has only the one-electron term, which is 0)
        const double integral = (ok && ((cI ^ oa) & 1) == 0) ? hijSingle<W>(S, d, oa, cI) : 0.0;
        if (ok && fabs(integral) > eps) {
          cand[oa >> 6] |= (1ull << (oa & 63));
          cand[cI >> 6] &= ~(1ull << (cI & 63));
          num = __dmul_rn(integral, wt);
          if (STOCH) {
            num2 = __dmul_rn(__dmul_rn(__dmul_rn(integral, integral), wt), wfac);
            pres = fabs(integral) > epsL;
          }
          keep = ptPart<W>(cand, nparts) == part && !hashContains<W>(table, mask, dets, cand);
        }
      }
      sink.put(keep, cand, num, num2, pres);
    }
    // ---- double excitations
    if (!(S.maxEntryAbs < eps)) {
      const int npairs = nclosed * (nclosed - 1) / 2;
      const int perSlice = slices > 1 ? (npairs + slices - 2) / (slices - 1) : npairs;
      const int pBegin = slices > 1 ? (slice == 0 ? npairs : (slice - 1) * perSlice) : 0;
      const int pEnd = pBegin + perSlice < npairs ? pBegin + perSlice : npairs;
      for (int p0 = pBegin; p0 < pEnd; p0 += 64) {
        int p = p0 + lane;
        int len = 0;
        int64_t st = 0;
        if (p < pEnd) {
          int i = (int)((1.0 + sqrt(1.0 + 8.0 * (double)p)) * 0.5);
          while (i * (i - 1) / 2 > p) i--;
          while ((i + 1) * i / 2 <= p) i++;
          int j = p - i * (i - 1) / 2;
          int cI = sClosed[wave][i], cJ = sClosed[wave][j];
          int I = cI >> 1, J = cJ >> 1;
          int X = I > J ? I : J, Y = I > J ? J : I;
          int pairIndex = X * (X + 1) / 2 + Y;
          int sameSpin = ((cI ^ cJ) & 1) == 0 ? 1 : 0;
          int64_t s0 = S.hbStart[sameSpin][pairIndex], s1 = S.hbStart[sameSpin][pairIndex + 1];
          const float* v = S.hbVal[sameSpin];
          int64_t lo = s0, hi = s1;
          while (lo < hi) {
            int64_t mid = (lo + hi) >> 1;
            if ((double)fabsf(v[mid]) < eps)
              hi = mid;
            else
              lo = mid + 1;
          }
          len = (int)(lo - s0);
          st = s0;
          const int na = nSpin[cI & 1], all = sameSpin ? na * (na - 1) / 2 : na * nSpin[cJ & 1];
          const bool direct = all < len;
          if (direct) {
            len = all;
            st = (int64_t)pairIndex * norb * norb;
          }
          sPair[wave][lane] = i | (j << 8) | (sameSpin << 16) | (direct ? 1 << 17 : 0);
        }
        int inc = len;
#pragma unroll
        for (int o = 1; o < 64; o <<= 1) {
          int tt = __shfl_up(inc, o, 64);
          if (lane >= o) inc += tt;
        }
        sExcl[wave][lane] = inc - len;
        sStart[wave][lane] = st;
        int total = __shfl(inc, 63, 64);
        __syncwarp();
        for (int k0 = 0; k0 < total; k0 += 64) {
          int k = k0 + lane;
          bool keep = false, pres = false;
          double num = 0.0, num2 = 0.0;
          uint64_t cand[W];
#pragma unroll
          for (int w = 0; w < W; w++) cand[w] = d[w];
          if (k < total) {
            int lo = 0, hi = 63;
            while (lo < hi) {
              int mid = (lo + hi + 1) >> 1;
              if (sExcl[wave][mid] <= k)
                lo = mid;
              else
                hi = mid - 1;
            }
            int q = lo;
            int pk = sPair[wave][q];
            int i = pk & 0xFF, j = (pk >> 8) & 0xFF, same = (pk >> 16) & 1;
            int cI = sClosed[wave][i], cJ = sClosed[wave][j];
            const int kk = k - sExcl[wave][q];
            int a, b;
            float hv;
            bool ok = true;
            if ((pk >> 17) & 1) {
              int x, y;  // places in the lists of open orbitals: x > y for one spin
              if (same) {
                x = (int)((1.0f + sqrtf(1.0f + 8.0f * (float)kk)) * 0.5f);
                while (x * (x - 1) / 2 > kk) x--;
                while ((x + 1) * x / 2 <= kk) x++;
                y = kk - x * (x - 1) / 2;
              } else {
                const int nb = nSpin[cJ & 1];
                x = kk / nb;
                y = kk - x * nb;
              }
              const int A = sSpin[wave][cI & 1][x], B = sSpin[wave][cJ & 1][y];
              hv = (same ? dense1 : dense0)[sStart[wave][q] + A * norb + B];
              // (as the walk: an eps that is NaN, 0 / 0, cuts nothing off)
              ok = !isnan(hv) && !((double)fabsf(hv) < eps);
              a = 2 * A + (cI & 1);
              b = 2 * B + (cJ & 1);
            } else {
              const int64_t idx = sStart[wave][q] + kk;
              const uint32_t ab = S.hbPair[same][idx];
              a = 2 * (int)(ab & 0xFFFF) + (cI & 1);
              b = 2 * (int)(ab >> 16) + (cJ & 1);
              ok = !(occ<W>(d, a) || occ<W>(d, b));
              hv = ok ? S.hbVal[same][idx] : 0.0f;
            }
            for (int r = 0; r < S.nrestrict && ok; r++) {
              const int8_t* m = S.rmult + r * nso;
              int e = cur[r] - m[cI] - m[cJ] + m[a] + m[b];
              if (e < S.rmin[r] || e > S.rmax[r]) ok = false;
            }
            if (ok) {
              cand[a >> 6] |= (1ull << (a & 63));
              cand[b >> 6] |= (1ull << (b & 63));
              cand[cI >> 6] &= ~(1ull << (cI & 63));
              cand[cJ >> 6] &= ~(1ull << (cJ & 63));
              // Determinant::parity(a, b, cI, cJ) on the new determinant
              // (SHCI/Determinants.cpp:332-357): a -> cI, then b -> cJ
              int nb = countBetween<W>(cand, a < cI ? a : cI, a < cI ? cI : a);
              uint64_t mid2[W];
#pragma unroll
              for (int w = 0; w < W; w++) mid2[w] = cand[w];
              mid2[a >> 6] &= ~(1ull << (a & 63));
              mid2[cI >> 6] |= (1ull << (cI & 63));
              nb += countBetween<W>(mid2, b < cJ ? b : cJ, b < cJ ? cJ : b);
              const double sgn = (nb & 1) ? -1.0 : 1.0;
              num = __dmul_rn(__dmul_rn((double)hv, sgn), wt);
              if (STOCH) {
                num2 = __dmul_rn(__dmul_rn((double)__fmul_rn(hv, hv), wt), wfac);
                pres = (double)fabsf(hv) > epsL;
              }
              keep = ptPart<W>(cand, nparts) == part && !hashContains<W>(table, mask, dets, cand);
            }
          }
          sink.put(keep, cand, num, num2, pres);
        }
        __syncwarp();
      }
    }
    if (!FILL) {
      int cc = sink.cnt;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) cc += __shfl_xor(cc, o, 64);
      if (lane == 0) counts[wi] = cc;
    }
  }
}

// ---------------------------------------------------------------------------
// RDMs of <bra| ... |ket> (the quantities of SHCI/SHCIrdm.cpp:863-1100):
//   g1[P*n + R]                 = sum_s   <a+_{P s} a_{R s}>
//   g2[((P*n + Q)*n + R)*n + S] = sum_s,t <a+_{P s} a+_{Q t} a_{S t} a_{R s}>
// and optionally the spin-orbital ones
//   s1[p*nso + r]               = <a+_p a_r>
//   s2[pair(p,q)*npair + pair(r,s)] = <a+_p a+_q a_s a_r>, p > q, r > s,
//   pair(p,q) = p(p+1)/2 + q, npair = nso(nso+1)/2
// Off-diagonal pairs come from the J < I entries of the full symmetric CSR
// (an element with bra[I] ket[J] and its transpose with bra[J] ket[I]); the
// diagonal is a rank-n product of the occupation matrix.
//
// g2 is assembled from three accumulators, so that each connection costs
// few FP64 atomics:
//   A[P,Q,R,S]  one element of every exchange pair G[PQRS] = G[QPSR] (and,
//               when bra = ket, of every hermitian pair G[PQRS] = G[RSPQ]);
//               G = A + A[QPSR] (+ the hermitian images)
//   Z[X,Y,K]    single excitations X <- Y times the number of common
//               occupied spin-orbitals of spatial orbital K; it adds to
//               G[X,K,Y,K] and G[K,X,K,Y]
//   Zs[X,Y,K]   the same over the common spin-orbitals with the spin of the
//               excitation; it subtracts from G[X,K,K,Y] and G[K,X,Y,K]

// parity of the occupied spin-orbitals of d below k
template <int W>
__device__ __forceinline__ int belowParity(const uint64_t* d, int k) {
  int c = 0;
#pragma unroll
  for (int w = 0; w < W; w++) {
    const int lo = 64 * w;
    if (k >= lo + 64)
      c += __popcll(d[w]);
    else if (k > lo)
      c += __popcll(d[w] & ((1ull << (k - lo)) - 1ull));
  }
  return c & 1;
}

struct RdmOut {
  double *g1, *g2, *s1, *s2;  // s1 / s2 may be null
  double *A, *Z, *Zs;         // accumulators of g2
  int n, nso;
  int64_t npair;
  bool herm;  // bra == ket: only one element of each hermitian pair is accumulated
  __device__ __forceinline__ void acc(int P, int Q, int R, int S, double v) const {
    atomicAdd(A + (((int64_t)P * n + Q) * n + R) * n + S, v);
  }
  __device__ __forceinline__ void add2(int P, int Q, int R, int S, double v) const {
    atomicAdd(g2 + (((int64_t)P * n + Q) * n + R) * n + S, v);
  }
  __device__ __forceinline__ void spin2(int p, int q, int r, int s, double v) const {
    // p > q, r > s
    atomicAdd(s2 + ((int64_t)p * (p + 1) / 2 + q) * npair + ((int64_t)r * (r + 1) / 2 + s), v);
  }
};

// diagonal part: M[p*nso + q] = sum_I bra[I] ket[I] occ_p(I) occ_q(I), a
// rank-n product of the occupation matrix; thread t of a workgroup owns row
// p = t / TPR and QPT consecutive columns of it in registers over the
// workgroup's slice of determinants, then adds them to M
template <int W>
__global__ void __launch_bounds__(kBlock) kRdmOcc(const uint64_t* dets, const double* bra, const double* ket, int64_t n,
                                                  double* M) {
  constexpr int QPT = W == 2 ? 64 : 16, TPR = 64 * W / QPT, NSO = 64 * W;
  const int p = threadIdx.x / TPR, h = threadIdx.x % TPR;
  const int qw = (h * QPT) >> 6, qs = (h * QPT) & 63;
  double acc[QPT];
#pragma unroll
  for (int j = 0; j < QPT; j++) acc[j] = 0.0;
  const int64_t per = (n + gridDim.x - 1) / gridDim.x;
  const int64_t b = (int64_t)blockIdx.x * per, e = b + per < n ? b + per : n;
  for (int64_t I = b; I < e; I++) {
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) d[w] = dets[I * W + w];
    if (!((d[p >> 6] >> (p & 63)) & 1ull)) continue;
    const double c2 = bra[I] * ket[I];
    const uint64_t row = d[qw] >> qs;
#pragma unroll
    for (int j = 0; j < QPT; j++)
      if ((row >> j) & 1ull) acc[j] += c2;
  }
#pragma unroll
  for (int j = 0; j < QPT; j++)
    if (acc[j] != 0.0) atomicAdd(M + (int64_t)p * NSO + h * QPT + j, acc[j]);
}

// scatters M (NSO x NSO) into the RDMs: <a+_p a_p> = n_p,
// <a+_p a+_q a_q a_p> = n_p n_q and <a+_p a+_q a_p a_q> = -n_p n_q (p != q)
__global__ void kRdmOccScatter(RdmOut o, const double* M, int NSO) {
  const int nso = o.nso;
  for (int t = blockIdx.x * blockDim.x + threadIdx.x; t < nso * nso; t += gridDim.x * blockDim.x) {
    const int p = t / nso, q = t % nso;
    const double v = M[(int64_t)p * NSO + q];
    if (v == 0.0) continue;
    if (p == q) {
      atomicAdd(o.g1 + (int64_t)(p >> 1) * o.n + (p >> 1), v);
      if (o.s1) atomicAdd(o.s1 + (int64_t)p * nso + p, v);
      continue;
    }
    o.add2(p >> 1, q >> 1, p >> 1, q >> 1, v);
    if (((p ^ q) & 1) == 0) o.add2(p >> 1, q >> 1, q >> 1, p >> 1, -v);
    if (o.s2 && p > q) o.spin2(p, q, p, q, v);
  }
}

template <int W>
__global__ void __launch_bounds__(kBlock) kRdm(RdmOut o, const uint64_t* dets, const int64_t* rp, const int32_t* cols,
                                               const double* bra, const double* ket, int64_t ndets) {
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  const int nso = o.nso, norb = o.n;
  for (int64_t I = (int64_t)blockIdx.x * kWaves + wave; I < ndets; I += (int64_t)gridDim.x * kWaves) {
    uint64_t dI[W];
#pragma unroll
    for (int w = 0; w < W; w++) dI[w] = dets[I * W + w];
    const double bI = bra[I], kI = ket[I];
    const int64_t b = rp[I], e = rp[I + 1];
    for (int64_t p = b + lane; p < e; p += 64) {
      const int64_t J = cols[p];
      if (J >= I) continue;
      uint64_t dJ[W];
#pragma unroll
      for (int w = 0; w < W; w++) dJ[w] = dets[J * W + w];
      int cre[2] = {0, 0}, des[2] = {0, 0}, nc = 0, nd = 0;
#pragma unroll
      for (int w = 0; w < W; w++) {
        uint64_t x = dI[w] & ~dJ[w], y = dJ[w] & ~dI[w];
        while (x) {
          const int q = 64 * w + __ffsll((unsigned long long)x) - 1;
          x &= x - 1;
          if (nc < 2) cre[nc] = q;
          nc++;
        }
        while (y) {
          const int q = 64 * w + __ffsll((unsigned long long)y) - 1;
          y &= y - 1;
          if (nd < 2) des[nd] = q;
          nd++;
        }
      }
      if (nc == 1 && nd == 1) {
        // I = a+_a a_i J: sign = parity of the occupied of J strictly between
        const int a = cre[0], i = des[0];
        const int lo = a < i ? a : i, hi = a < i ? i : a;
        const double sg = (countBetween<W>(dJ, lo, hi) & 1) ? -1.0 : 1.0;
        const double vE = sg * bI * ket[J], vT = sg * bra[J] * kI;
        const int A = a >> 1, Ii = i >> 1;
        atomicAdd(o.g1 + (int64_t)A * norb + Ii, vE);
        atomicAdd(o.g1 + (int64_t)Ii * norb + A, vT);
        if (o.s1) {
          atomicAdd(o.s1 + (int64_t)a * nso + i, vE);
          atomicAdd(o.s1 + (int64_t)i * nso + a, vT);
        }
        // common occupied spin-orbitals, per spatial orbital: count and
        // count with the excitation's spin
        const int64_t zE = ((int64_t)A * norb + Ii) * norb, zT = ((int64_t)Ii * norb + A) * norb;
        const int sa = a & 1;
#pragma unroll
        for (int w = 0; w < W; w++) {
          const uint64_t common = dJ[w] & dI[w];
          uint64_t sp = (common | (common >> 1)) & 0x5555555555555555ull;
          while (sp) {
            const int bit = __ffsll((unsigned long long)sp) - 1;
            sp &= sp - 1;
            const int K = (64 * w + bit) >> 1;
            const uint64_t pairBits = (common >> bit) & 3ull;
            const double cnt = (double)__popcll(pairBits);
            atomicAdd(o.Z + zE + K, cnt * vE);
            if (!o.herm) atomicAdd(o.Z + zT + K, cnt * vT);
            if ((pairBits >> sa) & 1ull) {
              atomicAdd(o.Zs + zE + K, vE);
              if (!o.herm) atomicAdd(o.Zs + zT + K, vT);
            }
          }
        }
        if (o.s2) {
#pragma unroll
          for (int w = 0; w < W; w++) {
            uint64_t common = dJ[w] & dI[w];
            while (common) {
              const int k = 64 * w + __ffsll((unsigned long long)common) - 1;
              common &= common - 1;
              // <a+_max(k,a) a+_min(k,a) a_min(k,i) a_max(k,i)>: one swap
              // when k lies between a and i
              const double f = (k > lo && k < hi) ? -1.0 : 1.0;
              const int ah = k > a ? k : a, al = k > a ? a : k, ih = k > i ? k : i, il = k > i ? i : k;
              o.spin2(ah, al, ih, il, f * vE);
              o.spin2(ih, il, ah, al, f * vT);
            }
          }
        }
      } else if (nc == 2 && nd == 2) {
        // I = a+_a a+_b a_j a_i J (a < b, i < j): sign from applying the
        // operators one by one
        const int a = cre[0], bb = cre[1], i = des[0], j = des[1];
        uint64_t d[W];
#pragma unroll
        for (int w = 0; w < W; w++) d[w] = dJ[w];
        int par = belowParity<W>(d, i);
        d[i >> 6] ^= 1ull << (i & 63);
        par += belowParity<W>(d, j);
        d[j >> 6] ^= 1ull << (j & 63);
        par += belowParity<W>(d, bb);
        d[bb >> 6] ^= 1ull << (bb & 63);
        par += belowParity<W>(d, a);
        const double sg = (par & 1) ? -1.0 : 1.0;
        const double vE = sg * bI * ket[J], vT = sg * bra[J] * kI;
        const int A = a >> 1, B = bb >> 1, Ii = i >> 1, Jj = j >> 1;
        // G[A,B,I,J] += vE (exchange image G[B,A,J,I]), G[I,J,A,B] += vT;
        // G[A,B,J,I] -= vE (image G[B,A,I,J]), G[J,I,A,B] -= vT
        if (((a ^ i) & 1) == 0 && ((bb ^ j) & 1) == 0) {
          o.acc(A, B, Ii, Jj, vE);
          if (!o.herm) o.acc(Ii, Jj, A, B, vT);
        }
        if (((a ^ j) & 1) == 0 && ((bb ^ i) & 1) == 0) {
          o.acc(A, B, Jj, Ii, -vE);
          if (!o.herm) o.acc(Jj, Ii, A, B, -vT);
        }
        if (o.s2) {  // <a+_b a+_a a_i a_j> = <a+_a a+_b a_j a_i>
          o.spin2(bb, a, j, i, vE);
          o.spin2(j, i, bb, a, vT);
        }
      }
    }
  }
}

// g2 from the accumulators (one thread per element; overwrites g2)
__global__ void kRdmFinish(RdmOut o) {
  const int n = o.n;
  const int64_t n2 = (int64_t)n * n, n4 = n2 * n2;
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n4; t += (int64_t)gridDim.x * blockDim.x) {
    const int S = (int)(t % n), R = (int)((t / n) % n), Q = (int)((t / n2) % n), P = (int)(t / (n2 * n));
    auto at = [&](int p, int q, int r, int s) { return o.A[(((int64_t)p * n + q) * n + r) * n + s]; };
    auto z = [&](const double* Z, int x, int y, int k) {
      const double v = Z[((int64_t)x * n + y) * n + k];
      return o.herm ? v + Z[((int64_t)y * n + x) * n + k] : v;
    };
    double g = at(P, Q, R, S) + at(Q, P, S, R);
    if (o.herm) g += at(R, S, P, Q) + at(S, R, Q, P);
    if (Q == S) g += z(o.Z, P, R, Q);
    if (P == R) g += z(o.Z, Q, S, P);
    if (Q == R) g -= z(o.Zs, P, S, Q);
    if (P == S) g -= z(o.Zs, Q, R, P);
    o.g2[t] = g;
  }
}

// ---------------------------------------------------------------------------
// time reversal: the adapted basis of the standard determinants S and the
// plain basis E = S followed by the flipped copies of the open-shell ones
// (in determinant order).  Basis function of I: |I> when I is closed-shell,
// else (|I> + p_I |flip I>) / sqrt 2, p_I = the flip parity (the Hamiltonian
// of SHCI/Determinants.cpp:32-121 and SHCI/SHCImakeHamiltonian.cpp:411-483,
// which leaves out the Treversal sign).

template <int W>
__global__ void kTrevMark(const uint64_t* dets, int64_t i0, int64_t i1, int64_t* flag) {
  for (int64_t i = i0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < i1; i += (int64_t)gridDim.x * blockDim.x) {
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) d[w] = dets[i * W + w];
    flag[i - i0] = hasUnpaired<W>(d) ? 1 : 0;
  }
}

// After an exclusive scan of the flags of [i0, i1): the block of E for these
// determinants (the cnt = i1 - i0 determinants, then the flipped copies of
// the open-shell ones), placed at E index base; each determinant's index in
// E, its partner's (-1 when closed-shell) and its flip parity
template <int W>
__global__ void kTrevBlock(const uint64_t* dets, int64_t i0, int64_t i1, const int64_t* pos, int64_t base,
                           uint64_t* block, int64_t* eIdx, int64_t* partner, double* parity) {
  const int64_t cnt = i1 - i0;
  for (int64_t i = i0 + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < i1; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t k = i - i0;
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) {
      d[w] = dets[i * W + w];
      block[k * W + w] = d[w];
    }
    const bool u = pos[k + 1] != pos[k];
    eIdx[i] = base + k;
    parity[i] = flipParity<W>(d);
    partner[i] = u ? base + cnt + pos[k] : -1;
    if (u) {
#pragma unroll
      for (int w = 0; w < W; w++) block[(cnt + pos[k]) * W + w] = flipWord(d[w]);
    }
  }
}

// xE = U x (k columns, ld / ldE)
__global__ void kTrevExpand(const double* x, int64_t n, int k, int64_t ld, const int64_t* eIdx,
                            const int64_t* partner, const double* parity, double* xE, int64_t ldE) {
  const double r2 = 1.0 / sqrt(2.0);
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n * k; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = t % n, c = t / n;
    const double v = x[c * ld + i];
    const int64_t q = partner[i], e = eIdx[i];
    if (q < 0) {
      xE[c * ldE + e] = v;
    } else {
      xE[c * ldE + e] = v * r2;
      xE[c * ldE + q] = parity[i] * v * r2;
    }
  }
}

// y = U^T yE
__global__ void kTrevContract(const double* yE, int64_t ldE, int64_t n, int k, const int64_t* eIdx,
                              const int64_t* partner, const double* parity, double* y, int64_t ld) {
  const double r2 = 1.0 / sqrt(2.0);
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n * k; t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = t % n, c = t / n;
    const int64_t q = partner[i], e = eIdx[i];
    y[c * ld + i] = q < 0 ? yE[c * ldE + e] : (yE[c * ldE + e] + parity[i] * yE[c * ldE + q]) * r2;
  }
}

// unpackTrevState (SHCI/SHCIbasics.cpp:730-776): c_I / sqrt 2 and
// Treversal p_I c_I / sqrt 2 for the partner, per root (ld n -> ldE)
__global__ void kTrevUnpack(const double* ci, int64_t n, int nroots, int64_t ld, const int64_t* partner,
                            const double* parity, int trev, double* out, int64_t ldE) {
  const double s2 = sqrt(2.0);
  for (int64_t t = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; t < n * nroots;
       t += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = t % n, c = t / n;
    const double v = ci[c * ld + i];
    const int64_t q = partner[i];
    if (q < 0) {
      out[c * ldE + i] = v;
    } else {
      out[c * ldE + i] = v / s2;
      out[c * ldE + q] = trev * parity[i] * v / s2;
    }
  }
}

// ---------------------------------------------------------------------------
// learned screening: features, targets and the exact test of ranked records

// X[r * din + f]: f < nso occupation bit f of the source determinant; then
// one-hot blocks (nso each) of ci, cj, a, b; then log10 |cmax[src]|; zero
// padding up to din
template <int W>
__global__ void kCandFeatures(const CandRecord* rec, int64_t n, const uint64_t* dets, int nso, const double* cmax,
                              float* X, int din) {
  const int64_t total = n * din;
  for (int64_t q = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; q < total; q += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = q / din;
    const int f = (int)(q - r * din);
    const CandRecord c = rec[r];
    float v = 0.f;
    if (f < nso) {
      v = (float)((dets[(int64_t)c.src * W + (f >> 6)] >> (f & 63)) & 1ull);
    } else if (f < 5 * nso) {
      const int blk = (f - nso) / nso, o = (f - nso) - blk * nso;
      const int which = blk == 0 ? c.ci : blk == 1 ? c.cj : blk == 2 ? c.a : c.b;
      v = which == o ? 1.f : 0.f;
    } else if (f == 5 * nso) {
      v = (float)log10(fabs(cmax[c.src]) + 1e-300);
    }
    X[q] = v;
  }
}

// t[r] = log10(|cmax[src]| * |v|): the screening value of the record
__global__ void kCandTargets(const CandRecord* rec, int64_t n, const double* cmax, float* t) {
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x)
    t[r] = (float)log10(fabs(cmax[rec[r].src]) * (double)fabsf(rec[r].v) + 1e-300);
}

// records whose score >= tau are evaluated with the reference's double test
// (|v| >= eps1 / |cmax|) and, when accepted, emitted as determinants not yet
// held; counts[0] += evaluated, counts[1] += accepted
template <int W>
__global__ void __launch_bounds__(kBlock) kCandExact(const CandRecord* rec, int64_t n, const float* score, float tau,
                                                     const uint64_t* dets, const double* cmax, double eps1,
                                                     const int32_t* table, uint64_t mask, uint64_t* out,
                                                     unsigned long long* counter, int64_t cap,
                                                     unsigned long long* counts) {
  for (int64_t r0 = (int64_t)blockIdx.x * blockDim.x; r0 < n; r0 += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = r0 + threadIdx.x;
    bool sel = false, pass = false;
    uint64_t cand[W];
#pragma unroll
    for (int w = 0; w < W; w++) cand[w] = 0;
    if (r < n && score[r] >= tau) {
      sel = true;
      const CandRecord c = rec[r];
      const double eps = eps1 / fabs(cmax[c.src]);
      pass = (double)fabsf(c.v) >= eps;
      if (pass) {
#pragma unroll
        for (int w = 0; w < W; w++) cand[w] = dets[(int64_t)c.src * W + w];
        cand[c.a >> 6] |= (1ull << (c.a & 63));
        cand[c.b >> 6] |= (1ull << (c.b & 63));
        cand[c.ci >> 6] &= ~(1ull << (c.ci & 63));
        cand[c.cj >> 6] &= ~(1ull << (c.cj & 63));
      }
    }
    const uint64_t ms = __ballot(sel), mp = __ballot(pass);
    if (__lane_id() == 0 && ms) {
      atomicAdd(&counts[0], (unsigned long long)__popcll(ms));
      atomicAdd(&counts[1], (unsigned long long)__popcll(mp));
    }
    emitCandidate<W>(pass, cand, table, mask, dets, out, counter, cap);  // (no time reversal in this form)
  }
}

__global__ void kGatherRecords(const CandRecord* rec, const int64_t* idx, int64_t m, CandRecord* out) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = rec[idx[i]];
}

// sampled records: flags[i] = (pass ? 1 : 0) | (score >= tau ? 2 : 0) for
// record idx[i]; vals[i] = its score
__global__ void kCandSample(const CandRecord* rec, const float* score, const int64_t* idx, int m, const double* cmax,
                            double eps1, float tau, int* flags, float* vals) {
  for (int i = blockIdx.x * blockDim.x + threadIdx.x; i < m; i += gridDim.x * blockDim.x) {
    const CandRecord c = rec[idx[i]];
    const float sc = score[idx[i]];
    const double eps = eps1 / fabs(cmax[c.src]);
    flags[i] = ((double)fabsf(c.v) >= eps ? 1 : 0) | (sc >= tau ? 2 : 0);
    vals[i] = sc;
  }
}

// ---------------------------------------------------------------------------
// string tables

__device__ __forceinline__ uint64_t compressEven(uint64_t x) {
  x &= 0x5555555555555555ull;
  x = (x | (x >> 1)) & 0x3333333333333333ull;
  x = (x | (x >> 2)) & 0x0F0F0F0F0F0F0F0Full;
  x = (x | (x >> 4)) & 0x00FF00FF00FF00FFull;
  x = (x | (x >> 8)) & 0x0000FFFF0000FFFFull;
  x = (x | (x >> 16)) & 0x00000000FFFFFFFFull;
  return x;
}

template <int W>
__global__ void kExtractStrings(const uint64_t* dets, int64_t n, uint64_t* alpha, uint64_t* beta) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    uint64_t a = 0, b = 0;
#pragma unroll
    for (int w = 0; w < W; w++) {
      uint64_t x = dets[i * W + w];
      a |= compressEven(x) << (32 * w);
      b |= compressEven(x >> 1) << (32 * w);
    }
    alpha[i] = a;
    beta[i] = b;
  }
}

__device__ __forceinline__ int64_t lowerBound(const uint64_t* arr, int64_t n, uint64_t x) {
  int64_t lo = 0, hi = n;
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (arr[mid] < x)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

__global__ void kIndexOf(const uint64_t* str, int64_t n, const uint64_t* sorted, int64_t ns, uint32_t* idx) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    idx[i] = (uint32_t)lowerBound(sorted, ns, str[i]);
}

__global__ void kGroupKeys(const uint32_t* major, int64_t n, uint64_t* key, uint32_t* val) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    key[i] = (uint64_t)major[i] * (uint64_t)n + (uint64_t)i;
    val[i] = (uint32_t)i;
  }
}

// key = major * nminor + minor (members of a group ordered by minor)
__global__ void kGroupKeys2(const uint32_t* major, const uint32_t* minor, int64_t n, uint64_t nminor, uint64_t* key,
                            uint32_t* val) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    key[i] = (uint64_t)major[i] * nminor + (uint64_t)minor[i];
    val[i] = (uint32_t)i;
  }
}

__global__ void kGroupStarts(const uint64_t* key, int64_t n, uint64_t nminor, int64_t ngroups, int64_t* start,
                             const uint32_t* val, const uint64_t* partnerStr, uint64_t* memberPartner) {
  for (int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; m <= n; m += (int64_t)gridDim.x * blockDim.x) {
    if (m == n) {
      start[ngroups] = n;
      continue;
    }
    uint64_t g = key[m] / nminor;
    if (m == 0 || key[m - 1] / nminor != g) start[g] = m;
    memberPartner[m] = partnerStr[val[m]];
  }
}

// Bitmaps of the large alpha groups over the beta strings: per 64 strings a
// word, and the members of the group before it.  flag: 1 for a group with
// one; scanned, its slot.
__global__ void kBitmapFlags(const int64_t* aStart, int64_t nA, int64_t thr, int64_t* flag) {
  for (int64_t g = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; g <= nA; g += (int64_t)gridDim.x * blockDim.x)
    flag[g] = g < nA && aStart[g + 1] - aStart[g] >= thr ? 1 : 0;
}
__global__ void kBitmapSet(const uint32_t* aIdx, const uint32_t* bIdx, int64_t n, const int64_t* slot, int64_t words,
                           uint4* bm) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t a = aIdx[i], b = bIdx[i];
    if (slot[a + 1] == slot[a]) continue;
    uint32_t* w = reinterpret_cast<uint32_t*>(bm + slot[a] * words + (b >> 6));
    atomicOr(w + ((b >> 5) & 1), 1u << (b & 31));
  }
}
// one wave per group: its slot (or -1) and the counts before each word
__global__ void kBitmapCounts(const int64_t* slot, int64_t nA, int64_t words, int32_t* bmSlot, uint4* bm) {
  const int lane = __lane_id();
  for (int64_t g = ((int64_t)blockIdx.x * blockDim.x + threadIdx.x) / 64; g < nA;
       g += (int64_t)gridDim.x * blockDim.x / 64) {
    const int64_t s = slot[g];
    const bool has = slot[g + 1] != s;
    if (lane == 0) bmSlot[g] = has ? (int32_t)s : -1;
    if (!has) continue;
    uint32_t before = 0;
    for (int64_t w0 = 0; w0 < words; w0 += 64) {
      const int64_t w = w0 + lane;
      uint32_t c = 0;
      if (w < words) {
        const uint4 e = bm[s * words + w];
        c = (uint32_t)(__popc(e.x) + __popc(e.y));
      }
      uint32_t inc = c;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        const uint32_t t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
      }
      if (w < words) bm[s * words + w].z = before + inc - c;
      before += __shfl(inc, 63, 64);
    }
  }
}

// alpha strings one excitation away from each unique alpha string
template <bool FILL>
__global__ void kStringSingles(const uint64_t* sorted, int64_t ns, int norb, const int64_t* start, int64_t* count,
                               uint32_t* out) {
  for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < ns; s += (int64_t)gridDim.x * blockDim.x) {
    uint64_t str = sorted[s];
    int64_t c = 0, pos = FILL ? start[s] : 0;
    uint64_t occd = str;
    while (occd) {
      int j = __ffsll((unsigned long long)occd) - 1;
      occd &= occd - 1;
      uint64_t emp = ~str & ((norb >= 64) ? ~0ull : ((1ull << norb) - 1ull));
      while (emp) {
        int k = __ffsll((unsigned long long)emp) - 1;
        emp &= emp - 1;
        uint64_t t = (str & ~(1ull << j)) | (1ull << k);
        int64_t f = lowerBound(sorted, ns, t);
        if (f < ns && sorted[f] == t) {
          if (FILL) out[pos++] = (uint32_t)f;
          c++;
        }
      }
    }
    if (!FILL) count[s] = c;
  }
}

// ---------------------------------------------------------------------------
// connected-pair rows: one wavefront per row

struct RowTables {
  const uint64_t* alpha;
  const uint64_t* beta;
  const uint32_t* aIdx;
  const uint32_t* bIdx;
  const int64_t* aStart;
  const int64_t* bStart;
  const uint32_t* aMajorDet;
  const uint32_t* bMajorDet;
  const uint64_t* aMajorB;
  const uint64_t* bMajorA;
  const int64_t* aSinglesStart;
  const uint32_t* aSingles;
  const int64_t* bSinglesStart;
  const uint32_t* bSingles;
  const uint64_t* sortedB;
  const uint64_t* aSortB;
  const uint32_t* aSortDet;
  const int32_t* bmSlot;
  const uint4* bm;
  int64_t bmWords;
  int64_t n;
};

// Collects the connections of row I.  Count pass: per-lane counters; fill
// pass: in the order they come.  A few of 64 candidates are connections, so
// the fill pass queues them in LDS and evaluates 64 elements at a time, with
// all lanes, into consecutive places of the row (the fill pass of 400,009
// determinants of 24 orbitals, 1.4e8 connections, 23.8 -> 8.9 ms, the count
// pass 14.2 -> 6.0 ms, by this and the shorter enumeration below).
// SPLIT stores each FP64 value as FP32 hi = fp32(v) and lo = fp32(v - hi).
template <int W, bool FILL, bool SPLIT, bool LOWER>
struct RowSink {
  const DevSystem* S;
  const uint64_t* dets;
  const uint64_t* dI;
  int64_t I;
  int32_t* cols;
  double* vals;
  float* hi;
  float* lo;
  uint32_t* queue;  // 128 entries of the wave (fill)
  int queued;       // of them in use, wave-uniform
  int64_t pos;      // the row's next place, wave-uniform (fill)
  int cnt;          // per-lane count (count)
  __device__ __forceinline__ void evaluate(int count) {
    const int lane = __lane_id();
    if (lane < count) {
      const uint32_t J = queue[lane];
      const int64_t p = pos + lane;
      uint64_t dJ[W];
#pragma unroll
      for (int w = 0; w < W; w++) dJ[w] = dets[(int64_t)J * W + w];
      const double v = ((int64_t)J < I) ? hijElement<W>(*S, dJ, dI) : hijElement<W>(*S, dI, dJ);
      cols[p] = (int32_t)J;
      if (SPLIT) {
        const float h = (float)v;
        hi[p] = h;
        lo[p] = (float)(v - (double)h);
      } else {
        vals[p] = v;
      }
    }
    pos += count;
  }
  __device__ __forceinline__ void hit(bool h, uint32_t J) {
    if (LOWER) h = h && (int64_t)J < I;  // half storage: row max(I, J) only
    if (!FILL) {
      cnt += h ? 1 : 0;
      return;
    }
    const uint64_t m = __ballot(h);
    if (m == 0ull) return;
    if (h) queue[queued + __popcll(m & lanemaskLt())] = J;
    queued += __popcll(m);
    if (queued >= 64) {
      waveSync();
      evaluate(64);
      const int lane = __lane_id(), rest = queued - 64;
      const uint32_t t = queue[64 + lane];  // (past the last entry: not used)
      waveSync();
      if (lane < rest) queue[lane] = t;
      waveSync();
      queued = rest;
    }
  }
  __device__ __forceinline__ void finish() {
    waveSync();
    evaluate(queued);
    waveSync();
    queued = 0;
  }
};

// first position in [lo, hi) whose determinant index is >= x (members of a
// group are stored in increasing determinant index)
__device__ __forceinline__ int64_t firstDetAtLeast(const uint32_t* a, int64_t lo, int64_t hi, uint32_t x) {
  while (lo < hi) {
    int64_t mid = (lo + hi) >> 1;
    if (a[mid] < x)
      lo = mid + 1;
    else
      hi = mid;
  }
  return lo;
}

// running maximum over the wave's lanes (values >= 0)
__device__ __forceinline__ int waveMaxScan(int v) {
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x111, 0xf, 0xf, true));   // row_shr:1
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x112, 0xf, 0xf, true));   // row_shr:2
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x114, 0xf, 0xf, true));   // row_shr:4
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x118, 0xf, 0xf, true));   // row_shr:8
  v = max(v, __builtin_amdgcn_update_dpp(0, v, 0x142, 0xa, 0xf, false));  // row_bcast:15 into rows 1 and 3
  return max(v, __builtin_amdgcn_update_dpp(0, v, 0x143, 0xc, 0xf, false));  // row_bcast:31 into rows 2 and 3
}

// Visits every connection of row I (all J != I one or two excitations
// apart, restricted to J >= jmin, and to J < jmax where a group's members are
// scanned): sink.hit(bool, J) is called by all 64 lanes together, once per
// candidate slot.  (a) the same-beta group: alpha
// singles and alpha-alpha doubles; (b) the same-alpha group: beta singles
// and beta-beta doubles; (c) alpha single x beta single: members of the
// groups of alpha strings one excitation away whose beta string is one
// excitation away.  Group members are in increasing determinant index, so
// jmin and jmax leave a prefix and a suffix of each group out (binary search).
// Bound by the vector memory path (TD 95% busy, the L1 waiting for misses 61%
// of the time, VALU 44 and 52% busy in the count and the fill pass): each
// group member's string, the bitmap words, and the elements' integrals.
template <class Sink>
__device__ __forceinline__ void enumerateRow(const RowTables& T, int64_t I, uint32_t jmin, uint32_t jmax,
                                             int wave, int lane,
                                             int (*sExcl)[64], int64_t (*sBeg)[64], int (*sLook)[64], int (*sMark)[64],
                                             Sink& sink) {
  const uint64_t astr = T.alpha[I], bstr = T.beta[I];
  const uint32_t ai = T.aIdx[I], bi = T.bIdx[I];
  {
    int64_t b0 = T.bStart[bi], b1 = T.bStart[bi + 1];
    if (jmin) b0 = firstDetAtLeast(T.bMajorDet, b0, b1, jmin);
    if (jmax < T.n) b1 = firstDetAtLeast(T.bMajorDet, b0, b1, jmax);
    for (int64_t m0 = b0; m0 < b1; m0 += 64) {
      int64_t m = m0 + lane;
      bool h = false;
      uint32_t J = 0;
      if (m < b1) {
        int dd = __popcll(T.bMajorA[m] ^ astr);
        h = (dd == 2 || dd == 4);
        if (h) J = T.bMajorDet[m];
      }
      sink.hit(h, J);
    }
  }
  {
    int64_t a0 = T.aStart[ai], a1 = T.aStart[ai + 1];
    if (jmin) a0 = firstDetAtLeast(T.aMajorDet, a0, a1, jmin);
    if (jmax < T.n) a1 = firstDetAtLeast(T.aMajorDet, a0, a1, jmax);
    for (int64_t m0 = a0; m0 < a1; m0 += 64) {
      int64_t m = m0 + lane;
      bool h = false;
      uint32_t J = 0;
      if (m < a1) {
        int dd = __popcll(T.aMajorB[m] ^ bstr);
        h = (dd == 2 || dd == 4);
        if (h) J = T.aMajorDet[m];
      }
      sink.hit(h, J);
    }
  }
  {
    // alpha single x beta single: per alpha single group either scan its
    // members for a beta one excitation from the row's (the members in
    // determinant order, from the first at or after jmin), or, when the
    // group is large, look up each of the row's beta singles in the group: in
    // its bitmap over the beta strings (a word and the members before it, one
    // load), or, without one, by binary search of its beta-ordered members.
    // (Which of the two ways a group takes sets the order of the row's
    // entries, and so does not depend on jmax.)
    int64_t s0 = T.aSinglesStart[ai], s1 = T.aSinglesStart[ai + 1];
    const int64_t bs0 = T.bSinglesStart[bi];
    const int nbs = (int)(T.bSinglesStart[bi + 1] - bs0);
    for (int64_t c0 = s0; c0 < s1; c0 += 64) {
      int64_t c = c0 + lane;
      int len = 0, look = -1;
      int64_t beg = 0;
      if (c < s1) {
        uint32_t sa = T.aSingles[c];
        const int64_t g0 = T.aStart[sa], g1 = T.aStart[sa + 1];
        beg = g0;
        if (jmin) beg = firstDetAtLeast(T.aMajorDet, beg, g1, jmin);
        len = (int)(g1 - beg);
        const int gsz = (int)(g1 - g0);
        const int steps = 66 - __clzll((unsigned long long)gsz);  // binary-search depth + 2
        if ((int64_t)nbs * steps < len) {
          const int slot = T.bmSlot[sa];
          look = slot >= 0 ? -2 - slot : gsz;
          len = nbs;
          beg = g0;
        } else if (jmax < T.n) {
          len = (int)(firstDetAtLeast(T.aMajorDet, beg, g1, jmax) - beg);
        }
      }
      int inc = len;
#pragma unroll
      for (int o = 1; o < 64; o <<= 1) {
        int t = __shfl_up(inc, o, 64);
        if (lane >= o) inc += t;
      }
      const int start = inc - len;
      sExcl[wave][lane] = start;
      sBeg[wave][lane] = beg;
      sLook[wave][lane] = look;
      const int total = __shfl(inc, 63, 64);
      int carry = 0;  // 1 + the group the chunk begins in
      for (int k0 = 0; k0 < total; k0 += 64) {
        int k = k0 + lane;
        bool h = false;
        uint32_t J = 0;
        // the group of each of 64 candidates: the groups that begin among them
        // leave their numbers at their first ones, a running maximum spreads
        // them (an LDS write and read instead of a binary search's six reads)
        sMark[wave][lane] = 0;
        waveSync();
        if (len > 0 && start >= k0 && start < k0 + 64) sMark[wave][start - k0] = lane + 1;
        waveSync();
        const int own = max(waveMaxScan(sMark[wave][lane]), carry);
        carry = __builtin_amdgcn_readlane(own, 63);
        if (k < total) {
          const int lo = own - 1;
          const int o = k - sExcl[wave][lo];
          const int g = sLook[wave][lo];
          if (g == -1) {
            int64_t m = sBeg[wave][lo] + o;
            h = __popcll(T.aMajorB[m] ^ bstr) == 2;
            if (h) J = T.aMajorDet[m];
          } else if (g < -1) {
            const uint32_t want = T.bSingles[bs0 + o];
            const uint4 e = T.bm[(int64_t)(-2 - g) * T.bmWords + (want >> 6)];
            const uint64_t bits = ((uint64_t)e.y << 32) | e.x;
            if ((bits >> (want & 63)) & 1ull) {
              J = T.aSortDet[sBeg[wave][lo] + e.z + __popcll(bits & ((1ull << (want & 63)) - 1ull))];
              h = J >= jmin;
            }
          } else {
            const uint64_t want = T.sortedB[T.bSingles[bs0 + o]];
            int64_t a = sBeg[wave][lo], b = a + g;  // [a, b)
            while (a < b) {
              const int64_t mid = (a + b) >> 1;
              if (T.aSortB[mid] < want)
                a = mid + 1;
              else
                b = mid;
            }
            if (a < sBeg[wave][lo] + g && T.aSortB[a] == want) {
              J = T.aSortDet[a];
              h = J >= jmin;
            }
          }
        }
        sink.hit(h, J);
      }
      waveSync();
    }
  }
}

// Rows I < nOld enumerate only connections to J >= nOld (the columns the
// previous Hamiltonian lacks); rows I >= nOld enumerate all connections.
// LOWER (half storage) keeps only J < I, so rows I < nOld gain nothing and
// are skipped.
template <int W, bool FILL, bool SPLIT, bool LOWER>
__global__ void __launch_bounds__(kBlock) kCsrRows(DevSystem S, const uint64_t* dets, RowTables T, int64_t nOld,
                                                   int64_t* rowCount, const int64_t* fillStart, int32_t* cols,
                                                   double* vals, float* hi, float* lo) {
  __shared__ int sExcl[kWaves][64], sMark[kWaves][64];
  __shared__ int64_t sBeg[kWaves][64];
  __shared__ int sLook[kWaves][64];
  __shared__ uint32_t sQueue[FILL ? kWaves : 1][128];
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  for (int64_t I = (int64_t)blockIdx.x * kWaves + wave; I < T.n; I += (int64_t)gridDim.x * kWaves) {
    uint64_t dI[W];
#pragma unroll
    for (int w = 0; w < W; w++) dI[w] = dets[I * W + w];
    if (LOWER && I < nOld) {
      if (!FILL && lane == 0) rowCount[I] = 0;
      continue;
    }
    const uint32_t jmin = I >= nOld ? 0u : (uint32_t)nOld;
    RowSink<W, FILL, SPLIT, LOWER> sink;
    sink.S = &S;
    sink.dets = dets;
    sink.dI = dI;
    sink.I = I;
    sink.cols = cols;
    sink.vals = vals;
    sink.hi = hi;
    sink.lo = lo;
    sink.queue = sQueue[FILL ? wave : 0];
    sink.queued = 0;
    sink.pos = FILL ? fillStart[I] : 0;
    sink.cnt = 0;
    enumerateRow(T, I, jmin, LOWER ? (uint32_t)I : 0xffffffffu, wave, lane, sExcl, sBeg, sLook, sMark, sink);
    if (FILL) sink.finish();
    if (!FILL) {
      int c = sink.cnt;
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o, 64);
      if (lane == 0) rowCount[I] = c;
    }
  }
}

// Direct sigma (no stored H): y[:, r] = diag .* x[:, r] + sum over the
// connections J of row I of Hij(bra = D_I, ket = D_J) x[J, r], the
// orientation of the reference's direct product; each element is evaluated
// once for all k <= 8 vectors.
template <int W>
struct DirectSink {
  const DevSystem* S;
  const uint64_t* dets;
  const uint64_t* dI;
  const double* x;
  int64_t ld;
  int k;
  double acc[8];
  __device__ __forceinline__ void hit(bool h, uint32_t J) {
    if (!h) return;
    uint64_t dJ[W];
#pragma unroll
    for (int w = 0; w < W; w++) dJ[w] = dets[(int64_t)J * W + w];
    const double v = hijElement<W>(*S, dI, dJ);
#pragma unroll
    for (int r = 0; r < 8; r++)
      if (r < k) acc[r] = fma(v, x[r * ld + J], acc[r]);
  }
};

template <int W>
__global__ void __launch_bounds__(kBlock) kSigmaDirect(DevSystem S, const uint64_t* dets, RowTables T,
                                                       const double* diag, const double* x, double* y, int k,
                                                       int64_t ld) {
  __shared__ int sExcl[kWaves][64], sMark[kWaves][64];
  __shared__ int64_t sBeg[kWaves][64];
  __shared__ int sLook[kWaves][64];
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  for (int64_t I = (int64_t)blockIdx.x * kWaves + wave; I < T.n; I += (int64_t)gridDim.x * kWaves) {
    uint64_t dI[W];
#pragma unroll
    for (int w = 0; w < W; w++) dI[w] = dets[I * W + w];
    DirectSink<W> sink;
    sink.S = &S;
    sink.dets = dets;
    sink.dI = dI;
    sink.x = x;
    sink.ld = ld;
    sink.k = k;
#pragma unroll
    for (int r = 0; r < 8; r++) sink.acc[r] = 0.0;
    enumerateRow(T, I, 0u, 0xffffffffu, wave, lane, sExcl, sBeg, sLook, sMark, sink);
#pragma unroll
    for (int r = 0; r < 8; r++) {
      if (r >= k) break;
      double v = sink.acc[r];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
      if (lane == 0) y[r * ld + I] = fma(diag[I], x[r * ld + I], v);
    }
  }
}

// new row length = kept old entries + new connections
__global__ void kNewRowLengths(const int64_t* oldRowPtr, int64_t nOld, int64_t n, int64_t* cnt) {
  for (int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; I < n; I += (int64_t)gridDim.x * blockDim.x)
    if (I < nOld) cnt[I] += oldRowPtr[I + 1] - oldRowPtr[I];
}

__global__ void kFillStart(const int64_t* oldRowPtr, int64_t nOld, int64_t n, const int64_t* rowPtr, int64_t* fs) {
  for (int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; I < n; I += (int64_t)gridDim.x * blockDim.x)
    fs[I] = rowPtr[I] + (I < nOld ? oldRowPtr[I + 1] - oldRowPtr[I] : 0);
}

// copy the old rows to the front of the new rows (one wavefront per row)
template <typename T1>
__global__ void __launch_bounds__(kBlock) kCopyOldRows(const int64_t* oldRowPtr, const int32_t* oldCols,
                                                       const T1* oldA, const T1* oldB, int64_t nOld,
                                                       const int64_t* rowPtr, int32_t* cols, T1* a, T1* b) {
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  for (int64_t I = (int64_t)blockIdx.x * kWaves + wave; I < nOld; I += (int64_t)gridDim.x * kWaves) {
    const int64_t s = oldRowPtr[I], e = oldRowPtr[I + 1], d = rowPtr[I];
    for (int64_t p = s + lane; p < e; p += 64) {
      cols[d + (p - s)] = __builtin_nontemporal_load(oldCols + p);
      a[d + (p - s)] = __builtin_nontemporal_load(oldA + p);
      if (oldB) b[d + (p - s)] = __builtin_nontemporal_load(oldB + p);
    }
  }
}

__global__ void kCast(const double* v, float* out, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    out[i] = (float)v[i];
}

// per-row insertion/shell sort of columns (rows are short relative to n)
__global__ void kSortRows(const int64_t* rowPtr, int64_t n, int32_t* cols, double* vals) {
  for (int64_t r = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; r < n; r += (int64_t)gridDim.x * blockDim.x) {
    int64_t b = rowPtr[r], e = rowPtr[r + 1];
    int64_t len = e - b;
    for (int64_t gap = len / 2; gap > 0; gap /= 2) {
      for (int64_t i = b + gap; i < e; i++) {
        int32_t c = cols[i];
        double v = vals[i];
        int64_t j = i;
        while (j - gap >= b && cols[j - gap] > c) {
          cols[j] = cols[j - gap];
          vals[j] = vals[j - gap];
          j -= gap;
        }
        cols[j] = c;
        vals[j] = v;
      }
    }
  }
}

// ---------------------------------------------------------------------------
// sigma = H x over the full symmetric CSR (gather only, no atomics): one
// wavefront per row, eight loads in flight per lane, FP64 accumulation, the
// diagonal term fused into the row's single store.  Values are VT,
// optionally plus an FP32 low part (hi + lo reproduces the FP64 value to
// ~2^-48 relative).  (Splitting the columns into per-XCD blocks, LDS-tiled
// gathers and 4-wide vector loads were all measured slower on a
// 1.2M-determinant matrix: the gathers of x are L2-request bound.)
template <typename VT, bool LO>
__global__ void __launch_bounds__(kBlock) kSigma(const int64_t* __restrict__ rowPtr, const int32_t* __restrict__ cols,
                                                 const VT* __restrict__ vals, const float* __restrict__ lo,
                                                 const double* __restrict__ diag, int64_t n,
                                                 const double* __restrict__ x, double* __restrict__ y, int k,
                                                 int64_t ld) {
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  constexpr int U = 8;  // loads in flight per lane
  for (int64_t I = (int64_t)blockIdx.x * kWaves + wave; I < n; I += (int64_t)gridDim.x * kWaves) {
    const int64_t b = rowPtr[I], e = rowPtr[I + 1];
    const double d = diag[I];
    for (int r = 0; r < k; r++) {
      const double* xr = x + r * ld;
      double acc[U];
#pragma unroll
      for (int u = 0; u < U; u++) acc[u] = 0.0;
      int64_t p = b + lane;
      for (; p + 64 * (U - 1) < e; p += 64 * U) {
        int32_t c[U];
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          c[u] = __builtin_nontemporal_load(cols + p + 64 * u);
          v[u] = (double)__builtin_nontemporal_load(vals + p + 64 * u);
          if (LO) v[u] += (double)__builtin_nontemporal_load(lo + p + 64 * u);
        }
#pragma unroll
        for (int u = 0; u < U; u++) acc[u] = fma(v[u], xr[c[u]], acc[u]);
      }
      for (; p < e; p += 64) acc[0] = fma((double)vals[p] + (LO ? (double)lo[p] : 0.0), xr[cols[p]], acc[0]);
      double sum = 0.0;
#pragma unroll
      for (int u = 0; u < U; u++) sum += acc[u];
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
      if (lane == 0) y[r * ld + I] = fma(d, xr[I], sum);
    }
  }
}

// ---------------------------------------------------------------------------
// sigma over the alpha-major relabelled copy of H.  Row m of the copy is
// determinant perm[m] (members of one alpha string are consecutive, in
// increasing determinant index) and its columns are alpha-major positions,
// so the x values a row gathers (same-alpha group members, members of the
// groups of alpha strings one excitation away) sit in a few contiguous
// ranges, and consecutive rows gather from the same ranges.  A work item is
// a chunk of consecutive rows, so that reuse stays within one CU.

__global__ void kInversePerm(const uint32_t* perm, int64_t n, uint32_t* pos) {
  for (int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; m < n; m += (int64_t)gridDim.x * blockDim.x)
    pos[perm[m]] = (uint32_t)m;
}

__global__ void kPermRowLengths(const int64_t* rowPtr, const uint32_t* perm, int64_t n, int64_t* len) {
  for (int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; m < n; m += (int64_t)gridDim.x * blockDim.x) {
    const int64_t I = perm[m];
    len[m] = rowPtr[I + 1] - rowPtr[I];
  }
}

// row m of the copy = row perm[m] of H with columns mapped through pos; with
// bIdx / bPos given, a column whose determinant has the row's beta string
// maps to n + bPos[J] instead (its place in a beta-major copy of x that
// follows the alpha-major one: a row's same-beta columns all lie in one beta
// group there, so their gathers share lines)
template <typename T1>
__global__ void __launch_bounds__(kBlock) kPermRows(const int64_t* rowPtr, const int32_t* cols, const T1* vals,
                                                    const uint32_t* perm, const uint32_t* pos,
                                                    const uint32_t* bIdx, const uint32_t* bPos, int64_t n,
                                                    const int64_t* rpP, int32_t* colsP, T1* valsP) {
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  for (int64_t m = (int64_t)blockIdx.x * kWaves + wave; m < n; m += (int64_t)gridDim.x * kWaves) {
    const int64_t I = perm[m];
    const int64_t b = rowPtr[I], e = rowPtr[I + 1], d = rpP[m];
    const uint32_t bi = bIdx ? bIdx[I] : 0u;
    for (int64_t p = b + lane; p < e; p += 64) {
      const int32_t J = __builtin_nontemporal_load(cols + p);
      colsP[d + (p - b)] = bIdx && bIdx[J] == bi ? (int32_t)(n + bPos[J]) : (int32_t)pos[J];
      valsP[d + (p - b)] = __builtin_nontemporal_load(vals + p);
    }
  }
}

// x in alpha-major order for the sigma kernels, followed (bPerm given) by
// x in beta-major order: row m < nx of the copy holds x[perm[m]] and row
// n + m' holds x[bPerm[m']], nx = 2n (n without bPerm); K == 1: xP[r * nx +
// m] for r < k; K > 1 (SpMM): interleaved, xP[m * K + r] (zero for k <= r <
// K).  Also zeroes the work counter of a persistent sigma launch that
// follows on the same stream.
// the persistent sigma's work counters: 8 words kSchedStride apart (the
// counter buffer holds 64 words)
constexpr int kSchedStride = 8;

template <typename XT, int K>
__global__ void kGatherPerm(const double* x, int k, int64_t ld, const uint32_t* perm, const uint32_t* bPerm, int64_t n,
                            XT* xP, unsigned* counter) {
  if (counter && blockIdx.x == 0 && threadIdx.x < 8) counter[kSchedStride * threadIdx.x] = 0u;
  const int64_t nx = bPerm ? 2 * n : n;
  for (int64_t m = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; m < nx; m += (int64_t)gridDim.x * blockDim.x) {
    const int64_t I = m < n ? perm[m] : bPerm[m - n];
    if (K == 1) {
      for (int r = 0; r < k; r++) xP[r * nx + m] = (XT)x[r * ld + I];
    } else {
#pragma unroll
      for (int r = 0; r < K; r++) xP[m * K + r] = r < k ? (XT)x[r * ld + I] : (XT)0;
    }
  }
}

// Row-chunk scheduler of the sigma kernels: CHUNK consecutive rows per work
// item; static (work item = workgroup) or persistent (workgroups take work
// items from an atomic counter until none is left, which evens out rows of
// very different lengths).
template <int CHUNK, bool PERSIST>
struct ChunkSched {
  int64_t nChunks;
  unsigned* counter;
  int64_t cur;
  __device__ __forceinline__ bool next() {
    if (!PERSIST) {
      if (cur < 0) {
        cur = blockIdx.x;
        return cur < nChunks;
      }
      return false;
    }
    // XCD-aware: workgroups are dispatched round-robin over the 8 XCDs, so
    // blockIdx mod 8 names the XCD.  Each XCD takes the chunks of its own
    // eighth of the rows first (consecutive alpha groups, whose x gathers
    // then share its L2), then helps the next XCDs; one counter per eighth
    // (kSchedCounters words apart, cleared by the gather kernel).  Results
    // do not depend on which workgroup takes a chunk.
    __shared__ int64_t sCur;
    const int x = blockIdx.x & 7;
    __syncthreads();
    if (threadIdx.x == 0) {
      sCur = -1;
      for (; off < 8; off++) {
        const int t = (x + off) & 7;
        const int64_t lo = nChunks * t / 8, hi = nChunks * (t + 1) / 8;
        const int64_t c = lo + (int64_t)atomicAdd(counter + kSchedStride * t, 1u);
        if (c < hi) {
          sCur = c;
          break;
        }
      }
    }
    __syncthreads();
    cur = sCur;
    return cur >= 0;
  }
  int off = 0;  // (thread 0) eighths already exhausted
};

// y[r*ld + perm[m]] = diag .* x + sum over row m of the copy (gathers from
// xP, one vector at a time, vectors nx apart)
template <typename VT, typename XT, int CHUNK, bool PERSIST>
__global__ void __launch_bounds__(kBlock) kSigmaPerm(const int64_t* __restrict__ rp, const int32_t* __restrict__ cols,
                                                     const VT* __restrict__ vals, const double* __restrict__ diag,
                                                     const uint32_t* __restrict__ perm, int64_t n,
                                                     const XT* __restrict__ xP, int64_t nx, const double* __restrict__ x,
                                                     double* __restrict__ y, int k, int64_t ld, unsigned* counter) {
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  constexpr int U = 8;
  ChunkSched<CHUNK, PERSIST> sched{(n + CHUNK - 1) / CHUNK, counter, -1};
  while (sched.next()) {
    const int64_t r0 = sched.cur * CHUNK;
    const int64_t r1 = r0 + CHUNK < n ? r0 + CHUNK : n;
    for (int64_t m = r0 + wave; m < r1; m += kWaves) {
      const int64_t b = rp[m], e = rp[m + 1];
      const int64_t I = perm[m];
      const double d = diag[I];
      for (int r = 0; r < k; r++) {
        const XT* xr = xP + r * nx;
        double acc[U];
#pragma unroll
        for (int u = 0; u < U; u++) acc[u] = 0.0;
        int64_t p = b + lane;
        for (; p + 64 * (U - 1) < e; p += 64 * U) {
          int32_t c[U];
          double v[U];
#pragma unroll
          for (int u = 0; u < U; u++) {
            c[u] = __builtin_nontemporal_load(cols + p + 64 * u);
            v[u] = (double)__builtin_nontemporal_load(vals + p + 64 * u);
          }
#pragma unroll
          for (int u = 0; u < U; u++) acc[u] = fma(v[u], (double)xr[c[u]], acc[u]);
        }
        for (; p < e; p += 64) acc[0] = fma((double)vals[p], (double)xr[cols[p]], acc[0]);
        double sum = 0.0;
#pragma unroll
        for (int u = 0; u < U; u++) sum += acc[u];
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, 64);
        if (lane == 0) y[r * ld + I] = fma(d, x[r * ld + I], sum);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Half storage: each unordered pair {I, J} stored once, in row max(I, J)
// (the reference's lower-triangular rows, SHCI/SHCImakeHamiltonian.cpp:549-711,
// without their diagonal), for spaces whose two-triangle Hamiltonian does not
// fit.  Sigma applies every stored element twice, as Hmult2 does
// (SHCI/Hmult.h:110-121): y[I] += h x[J] from a gather and y[J] += h x[I]
// by an FP64 atomic add at the L2, so its sums are not in a fixed order.

// rows [nOld, n] of a grown half-storage CSR: rowPtr[I] = rowPtr[nOld] +
// cnt[I], cnt the exclusive scan of new-row lengths (zero below nOld)
__global__ void kLowerRowPtr(const int64_t* cnt, int64_t nOld, int64_t n, int64_t* rowPtr) {
  const int64_t base = nOld ? rowPtr[nOld] : 0;
  for (int64_t I = nOld + (int64_t)blockIdx.x * blockDim.x + threadIdx.x; I <= n; I += (int64_t)gridDim.x * blockDim.x)
    if (I > nOld || nOld == 0) rowPtr[I] = base + cnt[I];
}

__global__ void kZeroVectors(double* y, int k, int64_t ld, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n * k; i += (int64_t)gridDim.x * blockDim.x) {
    const int64_t r = i / n;
    y[r * ld + (i - r * n)] = 0.0;
  }
}

template <typename VT, bool LO>
__global__ void __launch_bounds__(kBlock) kSigmaLower(const int64_t* __restrict__ rowPtr,
                                                      const int32_t* __restrict__ cols, const VT* __restrict__ vals,
                                                      const float* __restrict__ lo, const double* __restrict__ diag,
                                                      int64_t n, const double* __restrict__ x, double* __restrict__ y,
                                                      int k, int64_t ld) {
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  constexpr int U = 4;
  for (int64_t I = (int64_t)blockIdx.x * kWaves + wave; I < n; I += (int64_t)gridDim.x * kWaves) {
    const int64_t b = rowPtr[I], e = rowPtr[I + 1];
    for (int r = 0; r < k; r++) {
      const double* xr = x + r * ld;
      double* yr = y + r * ld;
      const double xi = xr[I];
      double acc = 0.0;
      int64_t p = b + lane;
      for (; p + 64 * (U - 1) < e; p += 64 * U) {
        int32_t c[U];
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          c[u] = __builtin_nontemporal_load(cols + p + 64 * u);
          v[u] = (double)__builtin_nontemporal_load(vals + p + 64 * u);
          if (LO) v[u] += (double)__builtin_nontemporal_load(lo + p + 64 * u);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          acc = fma(v[u], xr[c[u]], acc);
          unsafeAtomicAdd(yr + c[u], v[u] * xi);
        }
      }
      for (; p < e; p += 64) {
        const int32_t c = cols[p];
        const double v = (double)vals[p] + (LO ? (double)lo[p] : 0.0);
        acc = fma(v, xr[c], acc);
        unsafeAtomicAdd(yr + c, v * xi);
      }
#pragma unroll
      for (int o = 32; o > 0; o >>= 1) acc += __shfl_xor(acc, o, 64);
      if (lane == 0) unsafeAtomicAdd(yr + I, fma(diag[I], xi, acc));
    }
  }
}

// ---------------------------------------------------------------------------
// Tiled sigma.  The alpha-major rows are cut into blocks of kTileRows
// consecutive rows, and each block's entries are regrouped by column tile
// (kTileCols consecutive values of the permuted x).  One wave instruction
// takes up to 64 entries of one (block, tile) segment, so its gathers stay
// within one tile, and the tile's x lines, brought into L1 by the first
// instruction, serve the rest of the block's entries in that tile.  On the
// 1.18M-determinant benchmark space a row's entries touch 0.44 distinct
// 128-byte x lines per entry, a 256-row block's 0.038.  Within a segment
// the entries are ordered by the wave that placed them (row mod 4), then by
// row, then in the row's own order, so each row is one contiguous run; an
// instruction's products are summed per row by a segmented scan across
// lanes (each entry carries which of its steps add to it) and
// added into the executing wave's partial row sums in LDS, and the four
// partials are added in a fixed order at the end of the block.  Which wave
// takes which instructions is fixed by the layout, so the result does not
// depend on scheduling.  Segments of many instructions can gather from a
// copy of their x tile in LDS instead of from L1 (kSigmaTiled, STAGE).
constexpr int kTileRows = 256;
constexpr int kTileLog = 10;
constexpr int kTileCols = 1 << kTileLog;
constexpr int kTileMaxWords = 4096;  // bitmap of up to 131,072 tiles: x of up to 134M values
constexpr int kTileInstPad = 16;  // zero descriptors after the last one (the largest step of kSigmaTiled)
constexpr int kTileLdsSegs = 1024;  // blocks with at most this many segments count and fill in LDS
// an entry's 32-bit word: column in tile (bits 0-9), which of the six steps
// of the segmented scan of its instruction add to it (bits 10-15,
// segInclusiveScan), row in block (bits 16-23), last entry of its row run
// within the instruction (bit 31)
constexpr int kTileStepShift = 10;
// an instruction descriptor: its first entry (offset within the block),
// and a second word with the entry count (bits 0-6), the tile (bits 7-30),
// and bit 31 set when its segment has at least stageMin
// instructions (the staged kernel copies such a segment's x tile to LDS)
constexpr uint32_t kTileDescMask = 0xffffffu;

// the permuted-x column of H's column J in a row with beta string index bi
// (pos null: the input is the relabelled copy, whose columns are mapped)
__device__ __forceinline__ uint32_t tileMapCol(int32_t J, uint32_t bi, const uint32_t* __restrict__ pos,
                                               const uint32_t* __restrict__ bIdx,
                                               const uint32_t* __restrict__ bPos, int64_t n) {
  if (!pos) return (uint32_t)J;
  return (bIdx && bIdx[J] == bi) ? (uint32_t)(n + bPos[J]) : pos[J];
}

// inclusive scan over the block's threads (kBlock); returns the thread's
// inclusive value and the block total in *total
template <typename T>
__device__ __forceinline__ T blockInclusiveScan(T v, T* total) {
  __shared__ T waveSum[kWaves];
  const int lane = __lane_id(), wave = threadIdx.x >> 6;
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const T o = __shfl_up(v, d, 64);
    if (lane >= d) v += o;
  }
  if (lane == 63) waveSum[wave] = v;
  __syncthreads();
  T before = 0, all = 0;
#pragma unroll
  for (int w = 0; w < kWaves; w++) {
    if (w < wave) before += waveSum[w];
    all += waveSum[w];
  }
  __syncthreads();
  *total = all;
  return v + before;
}

// pre[k] = set bits before word k of bits[nwords]; returns the set bits
__device__ int tilePrefix(int nwords, const uint32_t* bits, uint32_t* pre) {
  const int per = (nwords + kBlock - 1) / kBlock;
  const int k0 = threadIdx.x * per, k1 = k0 + per < nwords ? k0 + per : nwords;
  int local = 0;
  for (int k = k0; k < k1; k++) local += __popc(bits[k]);
  int total = 0;
  int run = blockInclusiveScan(local, &total) - local;
  if (pre)
    for (int k = k0; k < k1; k++) {
      pre[k] = (uint32_t)run;
      run += __popc(bits[k]);
    }
  __syncthreads();
  return total;
}

__device__ __forceinline__ uint32_t tileRank(const uint32_t* bits, const uint32_t* pre, uint32_t t) {
  return pre[t >> 5] + __popc(bits[t >> 5] & ((1u << (t & 31)) - 1u));
}

// The build's passes wait for the row entries that they read: the tiles of a
// block are found once (kTileMark) and its bitmap kept, 4 nwords bytes a block,
// where each pass walked the block's entries for it; and the LDS follows the
// number of tiles (bits and pre, nwords words each), where room for the largest
// number allowed three workgroups per CU. 400,009 determinants, 24 orbitals:
// kTileCount 1.96 -> 1.08 ms, kTileFill 4.15 -> 3.23.

// pass 1: the tiles each block's entries touch (a bitmap per block, kept for
// the other passes) and their number (segCount[b])
__global__ void __launch_bounds__(kBlock) kTileMark(const int64_t* rowPtr, const int32_t* cols, const uint32_t* perm,
                                                    const uint32_t* pos, const uint32_t* bIdx, const uint32_t* bPos,
                                                    int64_t n, int nwords, int64_t* segCount, uint32_t* blockBits) {
  extern __shared__ uint32_t bits[];
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  for (int k = threadIdx.x; k < nwords; k += kBlock) bits[k] = 0u;
  __syncthreads();
  const int64_t m0 = (int64_t)blockIdx.x * kTileRows;
  const int rows = (int)(n - m0 < kTileRows ? n - m0 : kTileRows);
  for (int r = wave; r < rows; r += kWaves) {
    const int64_t I = perm ? (int64_t)perm[m0 + r] : m0 + r;
    const int64_t e0 = rowPtr[I], e1 = rowPtr[I + 1];
    const uint32_t bi = bIdx ? bIdx[I] : 0u;
    for (int64_t p = e0 + lane; p < e1; p += 64) {
      const uint32_t t = tileMapCol(cols[p], bi, pos, bIdx, bPos, n) >> kTileLog;
      const uint32_t bit = 1u << (t & 31);
      if (!(bits[t >> 5] & bit)) atomicOr(&bits[t >> 5], bit);
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < nwords; k += kBlock) blockBits[(int64_t)blockIdx.x * nwords + k] = bits[k];
  const int total = tilePrefix(nwords, bits, nullptr);
  if (threadIdx.x == 0) segCount[blockIdx.x] = total;
}

// pass 2: per (segment, wave) entry counts; segment tiles; per segment its
// entry and instruction offsets within the block; per (segment, wave) the
// fill cursor: the block-relative position of the wave's first entry in
// the segment; per block its entries and instructions
__global__ void __launch_bounds__(kBlock) kTileCount(const int64_t* rowPtr, const int32_t* cols, const uint32_t* perm,
                                                     const uint32_t* pos, const uint32_t* bIdx, const uint32_t* bPos,
                                                     int64_t n, int nwords, const uint32_t* blockBits,
                                                     const int64_t* segBase, uint32_t* segTile, uint32_t* segCnt,
                                                     uint32_t* segStart, uint32_t* segInst, uint32_t* segTotal,
                                                     uint32_t* fill, int64_t* blockE, int64_t* blockI) {
  extern __shared__ uint32_t bits[];
  uint32_t* pre = bits + nwords;
  __shared__ uint32_t cntL[kWaves][kTileLdsSegs];
  const int64_t b = blockIdx.x;
  for (int k = threadIdx.x; k < nwords; k += kBlock) bits[k] = blockBits[b * nwords + k];
  __syncthreads();
  tilePrefix(nwords, bits, pre);
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  const int64_t base = segBase[b];
  const bool inLds = segBase[b + 1] - base <= kTileLdsSegs;
  if (inLds)
    for (int k = threadIdx.x; k < kWaves * kTileLdsSegs; k += kBlock) (&cntL[0][0])[k] = 0u;
  __syncthreads();
  const int64_t m0 = b * kTileRows;
  const int rows = (int)(n - m0 < kTileRows ? n - m0 : kTileRows);
  for (int r = wave; r < rows; r += kWaves) {
    const int64_t I = perm ? (int64_t)perm[m0 + r] : m0 + r;
    const int64_t e0 = rowPtr[I], e1 = rowPtr[I + 1];
    const uint32_t bi = bIdx ? bIdx[I] : 0u;
    for (int64_t p = e0 + lane; p < e1; p += 64) {
      const uint32_t t = tileMapCol(cols[p], bi, pos, bIdx, bPos, n) >> kTileLog;
      const uint32_t sg = tileRank(bits, pre, t);
      if (inLds)
        atomicAdd(&cntL[wave][sg], 1u);
      else
        atomicAdd(&segCnt[(base + sg) * 4 + wave], 1u);
    }
  }
  if (inLds) {
    __syncthreads();
    const int64_t D = segBase[b + 1] - base;
    for (int64_t k = threadIdx.x; k < D * 4; k += kBlock) segCnt[base * 4 + k] = cntL[k & 3][k >> 2];
  }
  for (int k = threadIdx.x; k < nwords; k += kBlock) {
    uint32_t w = bits[k];
    uint32_t j = pre[k];
    while (w) {
      segTile[base + j] = ((uint32_t)k << 5) + (uint32_t)(__ffs(w) - 1);
      j++;
      w &= w - 1u;
    }
  }
  __threadfence();
  __syncthreads();
  const int64_t D = segBase[b + 1] - base;
  uint64_t carry = 0;  // entries (low 32 bits) and instructions (high 32 bits) so far
  for (int64_t s0 = 0; s0 < D; s0 += kBlock) {
    const int64_t s = s0 + threadIdx.x;
    uint64_t mine = 0;
    uint32_t c[4] = {0u, 0u, 0u, 0u};
    if (s < D) {
#pragma unroll
      for (int w = 0; w < 4; w++)
        c[w] = __hip_atomic_load(&segCnt[(base + s) * 4 + w], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const uint32_t tot = c[0] + c[1] + c[2] + c[3];
      segTotal[base + s] = tot;
      mine = (uint64_t)tot | ((uint64_t)((tot + 63u) / 64u) << 32);
    }
    uint64_t chunk = 0;
    const uint64_t incl = blockInclusiveScan(mine, &chunk);
    if (s < D) {
      const uint64_t ex = carry + incl - mine;
      const uint32_t st = (uint32_t)ex;
      segStart[base + s] = st;
      segInst[base + s] = (uint32_t)(ex >> 32);
      // the segment's entries are ordered by the wave that places them
      fill[(base + s) * 4 + 0] = st;
      fill[(base + s) * 4 + 1] = st + c[0];
      fill[(base + s) * 4 + 2] = st + c[0] + c[1];
      fill[(base + s) * 4 + 3] = st + c[0] + c[1] + c[2];
    }
    carry += chunk;
  }
  if (threadIdx.x == 0) {
    blockE[b] = (int64_t)(uint32_t)carry;
    blockI[b] = (int64_t)(carry >> 32);
  }
}

// pass 3: entries to their places, and the instruction descriptors
template <typename VT>
__global__ void __launch_bounds__(kBlock) kTileFill(const int64_t* rowPtr, const int32_t* cols, const VT* vals,
                                                    const uint32_t* perm, const uint32_t* pos, const uint32_t* bIdx,
                                                    const uint32_t* bPos, int64_t n, int nwords,
                                                    const uint32_t* blockBits,
                                                    const int64_t* segBase, const uint32_t* segTile,
                                                    const uint32_t* segStart, const uint32_t* segInst,
                                                    const uint32_t* segTotal, uint32_t* fill,
                                                    const int64_t* blockE, const int64_t* blockI, uint32_t* tIdx,
                                                    VT* tVal, uint2* inst, int stageMin, const float* lo,
                                                    float* tLo) {
  extern __shared__ uint32_t bits[];
  uint32_t* pre = bits + nwords;
  __shared__ uint32_t fillL[kWaves][kTileLdsSegs];
  const int64_t b = blockIdx.x;
  for (int k = threadIdx.x; k < nwords; k += kBlock) bits[k] = blockBits[b * nwords + k];
  __syncthreads();
  tilePrefix(nwords, bits, pre);
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  const int64_t base = segBase[b], eb = blockE[b];
  const bool inLds = segBase[b + 1] - base <= kTileLdsSegs;
  if (inLds)
    for (int64_t k = threadIdx.x; k < (segBase[b + 1] - base) * 4; k += kBlock) fillL[k & 3][k >> 2] = fill[base * 4 + k];
  __syncthreads();
  const int64_t m0 = b * kTileRows;
  const int rows = (int)(n - m0 < kTileRows ? n - m0 : kTileRows);
  for (int r = wave; r < rows; r += kWaves) {
    const int64_t I = perm ? (int64_t)perm[m0 + r] : m0 + r;
    const int64_t e0 = rowPtr[I], e1 = rowPtr[I + 1];
    const uint32_t bi = bIdx ? bIdx[I] : 0u;
    for (int64_t p0 = e0; p0 < e1; p0 += 64) {
      const int64_t p = p0 + lane;
      const bool valid = p < e1;
      uint32_t c = 0, s = 0;
      VT v = (VT)0;
      if (valid) {
        c = tileMapCol(cols[p], bi, pos, bIdx, bPos, n);
        s = tileRank(bits, pre, c >> kTileLog);
        v = vals[p];
      }
      // the entry's place in the block: the wave's fill cursor of the
      // segment, taken by an atomic add with return (lanes of one
      // instruction that share a cursor receive consecutive values in lane
      // order)
      uint32_t got = 0;
      if (valid) {
        if (inLds)
          got = atomicAdd(&fillL[wave][s], 1u);
        else
          got = atomicAdd(&fill[(base + s) * 4 + wave], 1u);
      }
      if (valid) {
        const int64_t q = eb + got;
        tIdx[q] = ((uint32_t)r << 16) | (c & (uint32_t)(kTileCols - 1));
        tVal[q] = v;
        if (lo) tLo[q] = lo[p];
      }
    }
  }
  const int64_t D = segBase[b + 1] - base, ib = blockI[b];
  for (int64_t s = threadIdx.x; s < D; s += kBlock) {
    const uint32_t tot = segTotal[base + s], st = segStart[base + s], tile = segTile[base + s];
    const int64_t i0 = ib + segInst[base + s];
    const uint32_t big = (tot + 63u) / 64u >= (uint32_t)stageMin ? 0x80000000u : 0u;
    for (uint32_t j = 0; 64u * j < tot; j++) {
      const uint32_t cnt = tot - 64u * j < 64u ? tot - 64u * j : 64u;
      inst[i0 + j] = make_uint2(st + 64u * j, big | (tile << 7) | cnt);
    }
  }
}

// The scan of an instruction's products: a segmented inclusive scan across
// the wave by DPP, whose steps are row_shr 1, 2, 4, 8 (within rows of 16
// lanes), row_bcast 15 (lane 15 into row 1, lane 47 into row 3) and row_bcast
// 31 (lane 31 into rows 2 and 3).  A lane adds a step's value when the lane it
// comes from lies in its run: by its distance `dist` to its run's first lane,
// counted within its row for the shifts.  Runs are contiguous, so every lane
// ends with the sum of its run up to itself.
__device__ __forceinline__ uint32_t segScanSteps(int lane, int dist) {
  const int col = lane & 15, inRow = dist < col ? dist : col;
  uint32_t m = 0;
  m |= inRow >= 1 ? 1u : 0u;
  m |= inRow >= 2 ? 2u : 0u;
  m |= inRow >= 4 ? 4u : 0u;
  m |= inRow >= 8 ? 8u : 0u;
  m |= ((lane >> 4) & 1) && dist > col ? 16u : 0u;
  m |= lane >= 32 && dist >= lane - 31 ? 32u : 0u;
  return m;
}

// pass 4: per entry, the scan steps that add to it and whether it is the last
// of its row run within its instruction (one wave per instruction)
__global__ void __launch_bounds__(kBlock) kTileRunBits(const uint2* __restrict__ inst,
                                                       const int64_t* __restrict__ blockI,
                                                       const int64_t* __restrict__ blockE, uint32_t* tIdx) {
  const int64_t b = blockIdx.x;
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  const int64_t i1 = blockI[b + 1], e0 = blockE[b];
  for (int64_t i = blockI[b] + wave; i < i1; i += kWaves) {
    const uint2 d = inst[i];
    const int cnt = (int)(d.y & 127u);
    const bool valid = lane < cnt;
    const int64_t p = e0 + d.x + lane;
    const uint32_t ix = valid ? tIdx[p] : 0u;
    const int key = valid ? (int)((ix >> 16) & (kTileRows - 1)) : -1 - lane;
    const int prev = __shfl_up(key, 1, 64), next = __shfl_down(key, 1, 64);
    const bool start = lane == 0 || prev != key;
    const bool last = lane == 63 || next != key;
    const unsigned long long starts = __ballot(start);
    // the highest run start at or below this lane
    const unsigned long long upTo = starts & (~0ull >> (63 - lane));
    const int first = 63 - __clzll(upTo);
    if (valid)
      tIdx[p] = (ix & ~((63u << kTileStepShift) | 0x80000000u)) | (segScanSteps(lane, lane - first) << kTileStepShift) |
                (last ? 0x80000000u : 0u);
  }
}

// One step: the value DPP control CTRL brings, masked to zero where the
// entry word's step bit is not set (an AND that takes the DPP operand itself;
// adding zero changes no bit of a sum but the sign of a zero).
template <int CTRL>
__device__ __forceinline__ void segScanStep(double& s, uint32_t ix, int bit) {
  const int m = (int)(ix << (31 - kTileStepShift - bit)) >> 31;
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(s), CTRL, 0xf, 0xf, true) & m;
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(s), CTRL, 0xf, 0xf, true) & m;
  s += __hiloint2double(hi, lo);
}

__device__ __forceinline__ double segInclusiveScan(double s, uint32_t ix) {
  segScanStep<0x111>(s, ix, 0);  // row_shr:1
  segScanStep<0x112>(s, ix, 1);  // row_shr:2
  segScanStep<0x114>(s, ix, 2);  // row_shr:4
  segScanStep<0x118>(s, ix, 3);  // row_shr:8
  segScanStep<0x142>(s, ix, 4);  // row_bcast:15
  segScanStep<0x143>(s, ix, 5);  // row_bcast:31
  return s;
}

// y[perm[m]] = diag .* x + (H x) over the tiled copy, one vector; xP holds x
// in the permuted order of the copy's columns
// One x tile (kTileCols values from xP at tile << kTileLog, nx values in all)
// into LDS by one wave, in 16-byte pieces; the last tile's values past nx
// read as 0 (no entry points at them)
template <typename XT>
__device__ __forceinline__ void stageTile(const XT* __restrict__ xP, int64_t nx, uint32_t tile, XT* xs) {
  constexpr int per = 16 / (int)sizeof(XT);  // values per 16-byte piece
  const int lane = __lane_id();
  const int64_t base = (int64_t)tile << kTileLog;
  if (base + kTileCols <= nx) {
    typedef XT V __attribute__((ext_vector_type(per)));
#pragma unroll
    for (int k = 0; k < kTileCols / (64 * per); k++) {
      const int j = (k * 64 + lane) * per;
      *(V*)(xs + j) = *(const V*)(xP + base + j);
    }
  } else {
    for (int j = lane; j < kTileCols; j += 64) xs[j] = base + j < nx ? xP[base + j] : (XT)0;
  }
}

// y[perm[m]] = diag .* x + (H x) over the tiled copy, one vector; xP holds x
// in the permuted order of the copy's columns (nx values).  STAGE: each wave
// takes a contiguous quarter of the block's instructions, and before an
// instruction of a large segment (descriptor bit 31) gathers, the wave
// copies that segment's x tile into its own LDS (once per tile) and gathers
// from there; otherwise the waves take turns of U instructions and gather
// from global memory.
template <typename VT, typename XT, bool PERSIST, int U, bool STAGE>
__global__ void __launch_bounds__(kBlock) kSigmaTiled(const uint2* __restrict__ inst, const int64_t* __restrict__ blockI,
                                                      const int64_t* __restrict__ blockE,
                                                      const uint32_t* __restrict__ tIdx, const VT* __restrict__ tVal,
                                                      const double* __restrict__ diag, const uint32_t* __restrict__ perm,
                                                      int64_t n, int64_t nblocks, const XT* __restrict__ xP, int64_t nx,
                                                      const double* __restrict__ x, double* __restrict__ y,
                                                      unsigned* counter) {
  __shared__ double yw[kWaves][kTileRows];
  __shared__ __align__(16) XT xs[STAGE ? kWaves : 1][STAGE ? kTileCols : 1];
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = __lane_id();
  static_assert(U <= kTileInstPad, "step larger than the descriptor padding");
  uint32_t staged = 0xffffffffu;  // the tile in this wave's LDS (x does not change within a launch)
  ChunkSched<1, PERSIST> sched{nblocks, counter, -1};
  while (sched.next()) {
    const int64_t b = sched.cur;
    for (int j = lane; j < kTileRows; j += 64) yw[wave][j] = 0.0;
    const int64_t i0 = blockI[b], i1 = blockI[b + 1], e0 = blockE[b];
    const int64_t len = i1 - i0;
    const int64_t w0 = STAGE ? i0 + len * wave / kWaves : i0 + (int64_t)wave * U;
    const int64_t wEnd = STAGE ? i0 + len * (wave + 1) / kWaves : i1;
    // the U instructions' loads are issued without branches, all matrix loads
    // before all gathers (vector loads return in order, so a gather issued
    // between them would make every later wait include it); absent
    // instructions and lanes past an instruction's count read the block's
    // first entry and their tile's first x value, and are dropped
    // each step takes U consecutive instructions (one scalar load of their
    // descriptors; the array has U zero descriptors of padding)
    for (int64_t i = w0; i < wEnd; i += STAGE ? (int64_t)U : (int64_t)kWaves * U) {
      uint32_t dx[U], dy[U];
      const uint2* dp = inst + i;
#pragma unroll
      for (int u = 0; u < U; u++) {
        const uint2 d = dp[u];
        dx[u] = d.x;
        dy[u] = i + u < wEnd ? d.y : (d.y & ~127u);  // count 0 past the range
      }
      uint32_t ix[U];
      double v[U];
#pragma unroll
      for (int u = 0; u < U; u++) {
        const bool valid = (uint32_t)lane < (dy[u] & 127u);
        const int64_t p = e0 + (valid ? (int64_t)dx[u] + lane : 0);
        ix[u] = __builtin_nontemporal_load(tIdx + p);
        v[u] = (double)__builtin_nontemporal_load(tVal + p);
      }
      double xv[U];
      if (STAGE) {
        // the tile of the step's first instruction from a large segment
        uint32_t want = 0xffffffffu;
#pragma unroll
        for (int u = 0; u < U; u++)
          if (want == 0xffffffffu && (dy[u] & 127u) && (dy[u] >> 31)) want = (dy[u] >> 7) & kTileDescMask;
        if (want != 0xffffffffu && want != staged) {
          stageTile<XT>(xP, nx, want, &xs[wave][0]);
          staged = want;
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          const bool valid = (uint32_t)lane < (dy[u] & 127u);
          const uint32_t col = valid ? (ix[u] & (uint32_t)(kTileCols - 1)) : 0u;
          const uint32_t tile = (dy[u] >> 7) & kTileDescMask;
          if (tile == staged)
            xv[u] = (double)xs[wave][col];
          else
            xv[u] = (double)xP[((size_t)tile << kTileLog) + col];
        }
      } else {
#pragma unroll
        for (int u = 0; u < U; u++) {
          const bool valid = (uint32_t)lane < (dy[u] & 127u);
          const size_t tb = (size_t)((dy[u] >> 7) & kTileDescMask) << kTileLog;
          xv[u] = (double)xP[tb + (valid ? (ix[u] & (uint32_t)(kTileCols - 1)) : 0u)];
        }
      }
      // products summed per row run by the segmented scan; the run's last
      // lane adds the sum into the wave's partial row (lanes past the count
      // sit above every valid lane, so no valid lane takes their values, and
      // are dropped)
#pragma unroll
      for (int u = 0; u < U; u++) {
        const bool valid = (uint32_t)lane < (dy[u] & 127u);
        const double sum = segInclusiveScan(v[u] * xv[u], ix[u]);
        if (valid && (int)ix[u] < 0) yw[wave][(ix[u] >> 16) & (kTileRows - 1)] += sum;
      }
    }
    __syncthreads();
    for (int t = threadIdx.x; t < kTileRows; t += kBlock) {
      const int64_t m = b * kTileRows + t;
      if (m < n) {
        const int64_t I = perm[m];
        y[I] = fma(diag[I], x[I], ((yw[0][t] + yw[1][t]) + yw[2][t]) + yw[3][t]);
      }
    }
    if (!PERSIST) break;
  }
}

// Half storage over the tiled copy: the copy holds each stored pair (I, J)
// once, in row I's block and J's column tile, and sigma needs each entry
// twice: v x[J] into row I and v x[I] into row J.  Both go into one
// accumulator per row, yT (the permuted order of x: row I's sum is split
// between its alpha-major and, with split columns, beta-major positions),
// kept in 64-bit fixed point so that the order of the sums does not matter
// and the result is the same on every run: a value t becomes the integer
// nearest t 2^-e, with 2^(e+61) above B max|x| (B: the largest off-diagonal
// row sum of |H_IJ|), so no row's sum of integers reaches 2^62 in
// magnitude, and each integer is off by at most 2^(e-1) (below
// 2^-61 B max|x|).  Row parts: each instruction's products are summed per
// row run in FP64 by the segmented scan, and each run's sum is one integer.
// Transposed parts: every product is one.  yT: nx sums (cleared first), then
// the bits of max|x|; bound: the bits of B.
//
// How the work is cut changes no bit, so the instructions are taken in an
// order of their own: kSymBlocks row blocks form a super block, whose
// instructions are sorted by tile (buildSymOrder).  A workgroup then keeps the x
// and the sums of the super block's rows and of the current tile's columns
// in LDS (32 KB, four workgroups of 512 threads per CU) for all the entries
// of that tile, so that nothing but the entries is read from memory per
// entry, and a tile's sums are added to yT once for 1,024 rows.  Bound by what
// it does per entry (VALU 59% busy, the LDS adds, the wait for the entries),
// not by bytes: with FP32 values it moves 8.6 GB a launch for 11.6 and takes as
// long.
//
// Measured, one product and the wait for it, against a workgroup per row block whose four waves
// each kept a tile's transposed sums of their own and gathered x through L1:
// 2,471 determinants of 16 orbitals 61 -> 15 us, 27,685 of 24 orbitals 423 ->
// 55, 57,963 of 40 orbitals 371 -> 89, 200,003 of 24 orbitals 569 -> 239,
// 1,000,003 of them (4.7e8 pairs) 2,569 -> 1,700 (3.3 TB/s over 12 bytes a
// pair), 300,007 of 40 orbitals with FP32 values 1,930 -> 980.  One after the
// other without a wait, where the old split's launches overlapped, the million
// 2,241 -> 1,598, two FP32 vectors of the 300,007 1,951 -> 1,702.  Super blocks
// of 2 and 8 blocks: 2,000 and 1,700 us on the million, 97 and 90 on the
// 57,963; 256 threads: 1,990 and 109; 2 and 8 instructions at a time: 1,730
// and 1,800.
constexpr int kSymBlocks = 4;
constexpr int kSymRows = kSymBlocks * kTileRows;
constexpr int kSymThreads = 512;
constexpr int kSymWaves = kSymThreads / 64;
constexpr int kSymStep = 4;  // instructions a wave loads together
// an instruction's second word in this order: entries (bits 0-6), row block in
// its super block (7-9), tile (10-31)
constexpr int kSymTileShift = 10;
constexpr uint32_t kSymSmall = 0x80000000u;

// a workgroup's work: `len` instructions of super block `sb` from `first` on,
// which lies in tile group `group`; with kSymSmall in sb, instructions of
// small groups.  len 0: unused.
struct __align__(16) SymUnit {
  uint32_t sb, first, len, group;
};

// place of every segment in the order (super block, tile, row block); per
// place its instructions as one of a large group (the instructions of one
// tile in one super block, at least bigMin) or of a small one, and whether
// it begins a large group
__global__ void kSymRank(const int64_t* __restrict__ segBase, int64_t blocks, int64_t segs,
                         const uint32_t* __restrict__ segTile, const uint32_t* __restrict__ segTotal, uint32_t bigMin,
                         uint32_t* order, uint32_t* blockOf, int64_t* bigI, int64_t* smallI, int64_t* lead) {
  for (int64_t s = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; s < segs; s += (int64_t)gridDim.x * blockDim.x) {
    int64_t lo = 0, hi = blocks - 1;  // the last block that begins at or before s
    while (lo < hi) {
      const int64_t mid = (lo + hi + 1) >> 1;
      if (segBase[mid] <= s)
        lo = mid;
      else
        hi = mid - 1;
    }
    const int64_t b = lo, q0 = b / kSymBlocks * kSymBlocks;
    const int64_t q1 = q0 + kSymBlocks < blocks ? q0 + kSymBlocks : blocks;
    const uint32_t tile = segTile[s];
    int64_t at = segBase[q0];
    uint32_t total = 0;
    bool first = true;
    for (int64_t c = q0; c < q1; c++) {
      int64_t i = segBase[c], j = segBase[c + 1];
      const int64_t c0 = i, c1 = j;
      while (i < j) {  // block c's first segment with a tile >= this one's
        const int64_t mid = (i + j) >> 1;
        if (segTile[mid] < tile)
          i = mid + 1;
        else
          j = mid;
      }
      at += i - c0;
      if (i < c1 && segTile[i] == tile) {
        total += (segTotal[i] + 63u) / 64u;
        if (c < b) {
          at++;
          first = false;
        }
      }
    }
    const int64_t mine = (segTotal[s] + 63u) / 64u;
    const bool big = total >= bigMin;
    order[at] = (uint32_t)s;
    blockOf[at] = (uint32_t)b;
    bigI[at] = big ? mine : 0;
    smallI[at] = big ? 0 : mine;
    lead[at] = big && first ? 1 : 0;
  }
}

// the instructions in that order, those of large groups first, and the large
// groups (bigI, smallI, lead: scanned)
__global__ void kSymEmit(int64_t segs, const uint32_t* __restrict__ order, const uint32_t* __restrict__ blockOf,
                         const int64_t* __restrict__ blockE, const uint32_t* __restrict__ segTile,
                         const uint32_t* __restrict__ segTotal, const uint32_t* __restrict__ segStart,
                         const int64_t* __restrict__ bigI, const int64_t* __restrict__ smallI,
                         const int64_t* __restrict__ lead, uint2* inst, uint2* groups) {
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
  const int64_t nBig = bigI[segs];
  for (int64_t p = tid; p < segs; p += (int64_t)gridDim.x * blockDim.x) {
    const uint32_t s = order[p], b = blockOf[p], tile = segTile[s], total = segTotal[s];
    const uint32_t rel = (uint32_t)(blockE[b] - blockE[b / kSymBlocks * kSymBlocks]) + segStart[s];
    const bool big = bigI[p + 1] != bigI[p];
    const int64_t at = big ? bigI[p] : nBig + smallI[p];
    for (uint32_t j = 0; 64u * j < total; j++)
      inst[at + j] = make_uint2(rel + 64u * j, (total - 64u * j < 64u ? total - 64u * j : 64u) |
                                                   ((b % kSymBlocks) << 7) | (tile << kSymTileShift));
    if (lead[p + 1] != lead[p]) groups[lead[p]] = make_uint2((uint32_t)bigI[p], tile);
  }
  if (tid == 0) groups[lead[segs]] = make_uint2((uint32_t)nBig, 0u);
}

// units per super block (units null), or the units themselves from the
// scanned counts; those past the last are marked unused
__global__ void kSymUnits(const int64_t* __restrict__ segBase, int64_t blocks, int64_t supers, int64_t segs,
                          const int64_t* __restrict__ bigI, const int64_t* __restrict__ smallI,
                          const int64_t* __restrict__ lead, const uint2* __restrict__ groups, int64_t per,
                          int64_t* unitStart, SymUnit* units, int64_t cap) {
  const int64_t tid = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, step = (int64_t)gridDim.x * blockDim.x;
  for (int64_t q = tid; q < supers; q += step) {
    const int64_t p0 = segBase[q * kSymBlocks];
    const int64_t p1 = segBase[(q + 1) * kSymBlocks < blocks ? (q + 1) * kSymBlocks : blocks];
    const int64_t b0 = bigI[p0], b1 = bigI[p1], s0 = bigI[segs] + smallI[p0], s1 = bigI[segs] + smallI[p1];
    if (!units) {
      unitStart[q] = (b1 - b0 + per - 1) / per + (s1 - s0 + per - 1) / per;
      continue;
    }
    SymUnit* u = units + unitStart[q];
    for (int64_t i = b0; i < b1; i += per) {
      int64_t a = lead[p0], b = lead[p1] - 1;  // the last group that begins at or before i
      while (a < b) {
        const int64_t mid = (a + b + 1) >> 1;
        if ((int64_t)groups[mid].x <= i)
          a = mid;
        else
          b = mid - 1;
      }
      *u++ = SymUnit{(uint32_t)q, (uint32_t)i, (uint32_t)(b1 - i < per ? b1 - i : per), (uint32_t)a};
    }
    for (int64_t i = s0; i < s1; i += per)
      *u++ = SymUnit{(uint32_t)q | kSymSmall, (uint32_t)i, (uint32_t)(s1 - i < per ? s1 - i : per), 0u};
  }
  if (!units) {
    if (tid == 0) unitStart[supers] = 0;
    return;
  }
  for (int64_t u = unitStart[supers] + tid; u < cap; u += step) units[u] = SymUnit{0u, 0u, 0u, 0u};
}

__device__ __forceinline__ double symFixRange(const unsigned long long* yT, int64_t nx,
                                              const unsigned long long* bound) {
  return __longlong_as_double((long long)yT[nx]) * __longlong_as_double((long long)*bound);
}
__device__ __forceinline__ int symFixExp(double range) {
  return range > 0.0 && range <= DBL_MAX ? ilogb(range) + 1 - 61 : 0;
}

// the integer nearest t (ties to even), |t| < 2^62, from four additions: t
// rounded to a multiple of 2^32 has that multiple in the low mantissa bits of
// t + 1.5 2^84, and the rest, exact and at most 2^31, its nearest integer in
// those of rest + 1.5 2^52.  (__double2ll_rn takes seven operations, most of
// them at a lower rate.)
__device__ __forceinline__ unsigned long long fixRound(double t) {
  const double a = t + 0x1.8p84;
  const double rest = t - (a - 0x1.8p84);
  const uint32_t hi = (uint32_t)__double2loint(a);
  const double b = rest + 0x1.8p52;
  return ((unsigned long long)((uint32_t)__double2hiint(b) - 0x43380000u + hi) << 32) | (uint32_t)__double2loint(b);
}

// ABS: the row sums of |H| for the bound B, every |v| rounded up to a multiple
// of 2^-32 and summed as an integer (x is not read)
template <typename VT, typename XT, bool LO, bool ABS>
__global__ void __launch_bounds__(kSymThreads) kSigmaTiledSym(const SymUnit* __restrict__ units,
                                                              const uint2* __restrict__ inst,
                                                              const uint2* __restrict__ groups,
                                                              const int64_t* __restrict__ blockE,
                                                              const uint32_t* __restrict__ tIdx,
                                                              const VT* __restrict__ tVal,
                                                              const float* __restrict__ tLo, int64_t n, int64_t nx,
                                                              const XT* __restrict__ xP, unsigned long long* yT,
                                                              const unsigned long long* __restrict__ bound) {
  __shared__ unsigned long long yr[kSymRows], yc[kTileCols];
  __shared__ double xr[kSymRows], xc[kTileCols];  // xr: times 2^-e
  const SymUnit unit = units[blockIdx.x];
  if (unit.len == 0u) return;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = __lane_id();
  const int e = ABS ? 0 : symFixExp(symFixRange(yT, nx, bound));
  const bool small = (unit.sb & kSymSmall) != 0u;
  const int64_t sb = unit.sb & ~kSymSmall, m0 = sb * kSymRows, e0 = blockE[sb * kSymBlocks];
  for (int j = threadIdx.x; j < kSymRows; j += kSymThreads) {
    yr[j] = 0ull;
    xr[j] = !ABS && m0 + j < n ? ldexp((double)xP[m0 + j], -e) : 0.0;
  }
  for (int j = threadIdx.x; j < kTileCols; j += kSymThreads) yc[j] = 0ull;
  // instructions [a, b) of one tile (staged) or of any (x and transposed sums
  // in memory), by one wave
  auto run = [&](uint32_t a, uint32_t b, bool staged) {
    for (uint32_t i = a; i < b; i += kSymStep) {
      uint32_t dx[kSymStep], dy[kSymStep], ix[kSymStep];
      double v[kSymStep];
#pragma unroll
      for (int u = 0; u < kSymStep; u++) {
        const uint2 d = inst[i + u < b ? i + u : a];
        dx[u] = d.x;
        dy[u] = i + u < b ? d.y : (d.y & ~127u);  // no entries past the range
      }
#pragma unroll
      for (int u = 0; u < kSymStep; u++) {
        ix[u] = 0u;
        v[u] = 0.0;
        if ((uint32_t)lane < (dy[u] & 127u)) {
          const int64_t p = e0 + dx[u] + lane;
          ix[u] = __builtin_nontemporal_load(tIdx + p);
          v[u] = (double)__builtin_nontemporal_load(tVal + p);
          if (LO) v[u] += (double)__builtin_nontemporal_load(tLo + p);
        }
      }
#pragma unroll
      for (int u = 0; u < kSymStep; u++) {
        const uint32_t cnt = dy[u] & 127u;
        if (cnt == 0u) continue;
        const bool valid = (uint32_t)lane < cnt;
        const uint32_t row = ((ix[u] >> 16) & (kTileRows - 1)) + (((dy[u] >> 7) & 7u) * kTileRows);
        const uint32_t col = ix[u] & (uint32_t)(kTileCols - 1);
        const size_t k0 = (size_t)(dy[u] >> kSymTileShift) << kTileLog;
        unsigned long long q;
        if (ABS) {
          q = (unsigned long long)ceil(ldexp(fabs(v[u]), 32));
          if (valid) atomicAdd(&yr[row], q);
        } else {
          const double xv = staged ? xc[col] : (double)xP[k0 + col];
          const double sum = segInclusiveScan(v[u] * xv, ix[u]);
          if (valid && (int)ix[u] < 0) atomicAdd(&yr[row], fixRound(ldexp(sum, -e)));
          q = fixRound(v[u] * xr[row]);
        }
        if (staged) {
          if (valid) atomicAdd(&yc[col], q);
        } else if (valid && q != 0ull) {
          atomicAdd(&yT[k0 + col], q);
        }
      }
    }
  };
  const uint32_t end = unit.first + unit.len;
  if (small) {
    __syncthreads();
    run(unit.first + unit.len * wave / kSymWaves, unit.first + unit.len * (wave + 1) / kSymWaves, false);
  } else {
    uint32_t at = unit.first;
    for (uint32_t g = unit.group; at < end; g++) {
      const uint32_t tile = groups[g].y, next = groups[g + 1].x, to = next < end ? next : end, len = to - at;
      const int64_t k0 = (int64_t)tile << kTileLog;
      if (!ABS)
        for (int j = threadIdx.x; j < kTileCols; j += kSymThreads) xc[j] = k0 + j < nx ? (double)xP[k0 + j] : 0.0;
      __syncthreads();
      run(at + len * wave / kSymWaves, at + len * (wave + 1) / kSymWaves, true);
      __syncthreads();
      for (int j = threadIdx.x; j < kTileCols; j += kSymThreads) {
        const unsigned long long a = yc[j];
        if (a != 0ull) {
          atomicAdd(&yT[k0 + j], a);
          yc[j] = 0ull;
        }
      }
      at = to;
    }
  }
  __syncthreads();
  for (int j = threadIdx.x; j < kSymRows; j += kSymThreads)
    if (yr[j] != 0ull) atomicAdd(&yT[m0 + j], yr[j]);
}

// y[I] = diag[I] x[I] + 2^e (yT[pos[I]] (+ yT[n + bPos[I]] with split
// columns))
__global__ void kSymFinish(const double* __restrict__ diag, const double* __restrict__ x, double* __restrict__ y,
                           const unsigned long long* __restrict__ yT, const unsigned long long* __restrict__ bound,
                           const uint32_t* __restrict__ pos, const uint32_t* __restrict__ bPos, int64_t n,
                           int64_t nx) {
  const double range = symFixRange(yT, nx, bound);
  const int e = symFixExp(range);
  const bool none = isinf(range);  // no fixed point holds the sums
  for (int64_t I = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; I < n; I += (int64_t)gridDim.x * blockDim.x) {
    long long t = (long long)yT[pos[I]];
    if (bPos) t += (long long)yT[n + bPos[I]];
    y[I] = none ? (double)NAN : fma(diag[I], x[I], ldexp((double)t, e));
  }
}

__global__ void kFillZeroU64(unsigned long long* v, int64_t m) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < m; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = 0ull;
}

// xP = x in the permuted order (as kGatherPerm for one vector), and the
// bits of max|x| into *mx (cleared first; the bits of non-negative doubles
// order as their values)
template <typename XT>
__global__ void kGatherPermMax(const double* __restrict__ x, const uint32_t* __restrict__ perm,
                               const uint32_t* __restrict__ bPerm, int64_t n, XT* __restrict__ xP,
                               unsigned long long* mx) {
  const int64_t nx = bPerm ? 2 * n : n;
  double m = 0.0;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < nx; i += (int64_t)gridDim.x * blockDim.x) {
    const double v = x[i < n ? perm[i] : bPerm[i - n]];
    // what has no place in a fixed point (NaN, infinite, beyond FP32 in its
    // form) stays out of the sums; with an infinite max|x| kSymFinish makes
    // every one of them NaN
    const XT t = (XT)v;
    const bool held = fabs((double)t) <= DBL_MAX;
    xP[i] = held ? t : (XT)0;
    m = fmax(m, held ? fabs(v) : (double)INFINITY);
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) m = fmax(m, __shfl_xor(m, o, 64));
  // one atomic per workgroup (the launch is capped at a few per CU):
  // atomics on one address are serialised
  __shared__ double wm[kWaves];
  if (__lane_id() == 0) wm[threadIdx.x >> 6] = m;
  __syncthreads();
  if (threadIdx.x == 0) {
    for (int w = 1; w < kWaves; w++) m = fmax(m, wm[w]);
    if (m > 0.0) atomicMax(mx, (unsigned long long)__double_as_longlong(m));
  }
}

// the largest sum of a row: a[pos[I]] (+ a[n + bPos[I]] with split columns)
__global__ void kMaxU64(const unsigned long long* __restrict__ a, const uint32_t* __restrict__ pos,
                        const uint32_t* __restrict__ bPos, int64_t n, unsigned long long* out) {
  unsigned long long m = 0ull;
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    unsigned long long t = a[pos[i]];
    if (bPos) t += a[n + bPos[i]];
    m = t > m ? t : m;
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    const unsigned long long t = __shfl_xor(m, o, 64);
    m = t > m ? t : m;
  }
  if (__lane_id() == 0 && m) atomicMax(out, m);
}

__global__ void kU64ScaledToDouble(unsigned long long* v) {
  if (blockIdx.x == 0 && threadIdx.x == 0) *v = (unsigned long long)__double_as_longlong(ldexp((double)*v, -32));
}

// SpMM: K interleaved vectors per gather (one K*sizeof(XT)-byte load per
// stored element serves all K products); rows read once.
template <typename XT, int K>
struct XVec {
  typedef XT T __attribute__((ext_vector_type(K)));
};

template <typename VT, typename XT, int K, int CHUNK, bool PERSIST>
__global__ void __launch_bounds__(kBlock) kSpmmPerm(const int64_t* __restrict__ rp, const int32_t* __restrict__ cols,
                                                    const VT* __restrict__ vals, const double* __restrict__ diag,
                                                    const uint32_t* __restrict__ perm, int64_t n,
                                                    const XT* __restrict__ xP, const double* __restrict__ x,
                                                    double* __restrict__ y, int k, int64_t ld, unsigned* counter) {
  typedef typename XVec<XT, K>::T XV;
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  constexpr int U = K >= 8 ? 1 : 8 / K;
  ChunkSched<CHUNK, PERSIST> sched{(n + CHUNK - 1) / CHUNK, counter, -1};
  while (sched.next()) {
    const int64_t r0 = sched.cur * CHUNK;
    const int64_t r1 = r0 + CHUNK < n ? r0 + CHUNK : n;
    for (int64_t m = r0 + wave; m < r1; m += kWaves) {
      const int64_t b = rp[m], e = rp[m + 1];
      const int64_t I = perm[m];
      double acc[K];
#pragma unroll
      for (int r = 0; r < K; r++) acc[r] = 0.0;
      int64_t p = b + lane;
      for (; p + 64 * (U - 1) < e; p += 64 * U) {
        int32_t c[U];
        double v[U];
#pragma unroll
        for (int u = 0; u < U; u++) {
          c[u] = __builtin_nontemporal_load(cols + p + 64 * u);
          v[u] = (double)__builtin_nontemporal_load(vals + p + 64 * u);
        }
#pragma unroll
        for (int u = 0; u < U; u++) {
          const XV xv = *reinterpret_cast<const XV*>(xP + (int64_t)c[u] * K);
#pragma unroll
          for (int r = 0; r < K; r++) acc[r] = fma(v[u], (double)xv[r], acc[r]);
        }
      }
      for (; p < e; p += 64) {
        const XV xv = *reinterpret_cast<const XV*>(xP + (int64_t)cols[p] * K);
        const double v = (double)vals[p];
#pragma unroll
        for (int r = 0; r < K; r++) acc[r] = fma(v, (double)xv[r], acc[r]);
      }
#pragma unroll
      for (int r = 0; r < K; r++) {
#pragma unroll
        for (int o = 32; o > 0; o >>= 1) acc[r] += __shfl_xor(acc[r], o, 64);
      }
      if (lane < k && lane < K) {
        double sum = acc[0];
#pragma unroll
        for (int r = 1; r < K; r++)
          if (lane == r) sum = acc[r];
        y[lane * ld + I] = fma(diag[I], x[lane * ld + I], sum);
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Davidson vector kernels

constexpr int kRedBlocks = 512;
// the PT reductions evaluate E_a of every unique external determinant: enough
// workgroups to keep every SIMD busy with latency-bound work
constexpr int kPtRedBlocks = 8192;

__device__ __forceinline__ double shflXor(double v, int o) { return __shfl_xor(v, o, 64); }

// acc[0 .. 2 O) over the wave: lanes with bit O keep the upper O sums.  Each
// step halves what is still summed, and adds the same pairs as a butterfly of
// every value does (so the same bits) with a sixth of its exchanges.
template <int O>
__device__ __forceinline__ double waveReduceScatter(double* acc) {
  const bool up = (__lane_id() & O) != 0;
#pragma unroll
  for (int q = 0; q < O; q++) {
    const double mine = up ? acc[q + O] : acc[q], other = up ? acc[q] : acc[q + O];
    acc[q] = mine + shflXor(other, O);
  }
  if constexpr (O > 1)
    return waveReduceScatter<O / 2>(acc);
  else
    return acc[0];
}

// Gram tiles: blockIdx.y = tile (ta, tb) of 8 x 8 entries (upper: tb >= ta
// only).  A thread has few rows to add and 64 sums to reduce, so what counts is
// that reduction: 63 exchanges a lane where a butterfly of each sum took 384.
// 4 roots of a 36-site lattice: 35.2 -> 14.7 us a product.
__global__ void __launch_bounds__(kBlock) kGramTile(const double* A, int ma, const double* B, int mb, int64_t n,
                                                    int64_t ld, bool upper, double* partial) {
  constexpr int T = 8;
  __shared__ double red[kWaves][T * T];
  const int tilesB = (mb + T - 1) / T;
  const int ta = blockIdx.y / tilesB, tb = blockIdx.y % tilesB;
  if (upper && tb < ta) return;
  const int na = min(T, ma - ta * T), nb = min(T, mb - tb * T);
  const double* A0 = A + (int64_t)ta * T * ld;
  const double* B0 = B + (int64_t)tb * T * ld;
  double acc[T * T];
#pragma unroll
  for (int q = 0; q < T * T; q++) acc[q] = 0.0;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
    double a[T], bb[T];
#pragma unroll
    for (int i = 0; i < T; i++) a[i] = i < na ? A0[i * ld + k] : 0.0;
#pragma unroll
    for (int j = 0; j < T; j++) bb[j] = j < nb ? B0[j * ld + k] : 0.0;
#pragma unroll
    for (int i = 0; i < T; i++)
#pragma unroll
      for (int j = 0; j < T; j++) acc[i * T + j] = fma(a[i], bb[j], acc[i * T + j]);
  }
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  red[wave][lane] = waveReduceScatter<32>(acc);
  __syncthreads();
  for (int q = threadIdx.x; q < T * T; q += blockDim.x) {
    double v = 0.0;
    for (int w = 0; w < kWaves; w++) v += red[w][q];
    partial[((int64_t)blockIdx.y * gridDim.x + blockIdx.x) * T * T + q] = v;
  }
}

// one block per output entry (i, j): fixed-order sum over the tile's partials;
// upper: entries i <= j, to both triangles
__global__ void __launch_bounds__(kBlock) kGramTileFinal(const double* partial, int nblocks, int ma, int mb,
                                                         bool upper, double* G) {
  constexpr int T = 8;
  __shared__ double red[kWaves];
  const int i = blockIdx.x / mb, j = blockIdx.x % mb;
  if (upper && j < i) return;
  const int tilesB = (mb + T - 1) / T;
  const int tile = (i / T) * tilesB + j / T;
  const int q = (i % T) * T + (j % T);
  double v = 0.0;
  for (int b = threadIdx.x; b < nblocks; b += blockDim.x) v += partial[((int64_t)tile * nblocks + b) * T * T + q];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (__lane_id() == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kWaves; w++) t += red[w];
    G[i * mb + j] = t;
    if (upper) G[j * mb + i] = t;
  }
}

// NJ columns of row k: out = alpha * A W + beta * out
template <int NJ>
__device__ __forceinline__ void gemmRow(const double* __restrict__ A, int ma, const double* sW, int mb, int64_t k,
                                        int64_t lda, double* __restrict__ out, int64_t ldo, double alpha,
                                        double beta) {
  double acc[NJ];
#pragma unroll
  for (int jj = 0; jj < NJ; jj++) acc[jj] = 0.0;
#pragma unroll 8
  for (int l = 0; l < ma; l++) {
    const double a = A[l * lda + k];
#pragma unroll
    for (int jj = 0; jj < NJ; jj++) acc[jj] = fma(a, sW[l * mb + jj], acc[jj]);
  }
#pragma unroll
  for (int jj = 0; jj < NJ; jj++) {
    double* o = out + (int64_t)jj * ldo + k;
    *o = beta == 0.0 ? alpha * acc[jj] : fma(beta, *o, alpha * acc[jj]);
  }
}

// out = alpha * A W + beta * out, one row per thread, 8 output columns per
// pass (blockIdx.y).  Few rows a thread: what counts is the chain of loads of a
// row, so eight are in flight (the number of columns is a constant of the inner
// loop for it).  14.8 -> 11.5 us on a 36-site lattice, 4 roots.
__global__ void __launch_bounds__(kBlock) kGemmTS(const double* __restrict__ A, int ma, const double* W, int mb,
                                                  int64_t n, int64_t lda, double* __restrict__ out, int64_t ldo,
                                                  double alpha, double beta) {
  __shared__ double sW[64 * 64];
  for (int q = threadIdx.x; q < ma * mb; q += blockDim.x) sW[q] = W[q];
  __syncthreads();
  const int j0 = blockIdx.y * 8;
  const double* w = sW + j0;
  double* o = out + (int64_t)j0 * ldo;
#define GEMM_CASE(NJ) \
  case NJ: gemmRow<NJ>(A, ma, w, mb, k, lda, o, ldo, alpha, beta); break
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
    switch (mb - j0) {
      GEMM_CASE(1);
      GEMM_CASE(2);
      GEMM_CASE(3);
      GEMM_CASE(4);
      GEMM_CASE(5);
      GEMM_CASE(6);
      GEMM_CASE(7);
      default: gemmRow<8>(A, ma, w, mb, k, lda, o, ldo, alpha, beta);
    }
  }
#undef GEMM_CASE
}

__device__ __forceinline__ double blockSum(double v) {
  __shared__ double red[kWaves];
  const int wave = threadIdx.x >> 6, lane = __lane_id();
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (lane == 0) red[wave] = v;
  __syncthreads();
  double t = 0.0;
  if (threadIdx.x == 0)
    for (int w = 0; w < kWaves; w++) t += red[w];
  __syncthreads();
  return t;
}

__global__ void __launch_bounds__(kBlock) kResidual(const double* sig, const double* b, const double* e, int64_t n,
                                                    double* r, double* partial) {
  const double ev = e[0];
  double acc = 0.0;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
    double v = sig[k] - ev * b[k];
    r[k] = v;
    acc = fma(v, v, acc);
  }
  double t = blockSum(acc);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

// one block per output value (blockIdx.x = q < nvals)
__global__ void __launch_bounds__(kBlock) kFinalSum(const double* partial, int nb, int stride, int nvals,
                                                    double* out) {
  __shared__ double red[kWaves];
  const int q = blockIdx.x;
  double v = 0.0;
  for (int b = threadIdx.x; b < nb; b += blockDim.x) v += partial[(int64_t)b * stride + q];
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, 64);
  if (__lane_id() == 0) red[threadIdx.x >> 6] = v;
  __syncthreads();
  if (threadIdx.x == 0) {
    double t = 0.0;
    for (int w = 0; w < kWaves; w++) t += red[w];
    out[q] = t;
  }
}

// Semistochastic reduction (SHCI/SHCIbasics.cpp:264-385): per run of equal
// determinants (sorted, generation order kept), a1/a2 = sums of num / num2,
// b1/b2 = the same over the terms present at epsilon2Large; per-block partial
// sums of (|a1|^2 Nmc/(Nmc-1) - a2) / (E_a - E0) and of the b version.
// The energy tables of E_a in LDS: hdiag (n), direct (n^2), exchange (n^2)
// when they fit (LDS_TAB), else read from global memory.
constexpr size_t kPtTabMaxBytes = 64 * 1024;
inline size_t ptTabBytes(int n) { return ((size_t)n + 2 * (size_t)n * n) * sizeof(double); }

template <int W, bool LDS_TAB>
__device__ __forceinline__ double ptEnergy(const DevSystem& S, const double* tab, const uint64_t* d) {
  // (the same additions in the same order as Energy(): E_a is bit-identical,
  // which matters for external determinants whose E0 - E_a is small; for the
  // others a sum from the source's energy would do)
  if (LDS_TAB) return detEnergyTab<W>(tab, tab + S.norb, tab + S.norb + S.norb * S.norb, S.norb, d);
  return detEnergy<W>(S, d);
}

template <bool LDS_TAB>
__device__ __forceinline__ double* ptStageTables(const DevSystem& S) {
  extern __shared__ double tab[];
  if (LDS_TAB) {
    const int n = S.norb, nn = n * n;
    for (int k = threadIdx.x; k < n + 2 * nn; k += blockDim.x)
      tab[k] = k < n ? S.h1[k * n + k] : (k < n + nn ? S.direct[k - n] : S.exch[k - n - nn]);
    __syncthreads();
  }
  return tab;
}

__global__ void kIota(uint32_t* v, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x)
    v[i] = (uint32_t)i;
}

// Over candidates sorted by determinant (stable, so equal determinants keep
// their generation order): the first entry of each run sums the run's
// numerators in that order (the reference's merge) and contributes
// num^2 / (E0 - E_a) and (num / (E0 - E_a))^2; per-block partial sums of
// (E_PT, psi1 norm, number of external determinants) in fixed order.

// This is evaluated over the run starts only (compacted in order first), so
// that every lane of the E_a evaluation works on a unique determinant
// instead of one lane in ~6 (runs average six candidates on the 1.18M-
// determinant space).
constexpr int kStartChunk = kBlock * 16;

template <int W>
__global__ void __launch_bounds__(kBlock) kPtCountStarts(const uint64_t* keys, int64_t m, int64_t* counts) {
  const int64_t b0 = (int64_t)blockIdx.x * kStartChunk;
  const int64_t b1 = b0 + kStartChunk < m ? b0 + kStartChunk : m;
  int c = 0;
  for (int64_t i = b0 + threadIdx.x; i < b1; i += blockDim.x)
    if (i == 0 || !detEqual<W>(keys + i * W, keys + (i - 1) * W)) c++;
  const double t = blockSum((double)c);
  if (threadIdx.x == 0) counts[blockIdx.x] = (int64_t)t;
}

template <int W>
__global__ void __launch_bounds__(kBlock) kPtWriteStarts(const uint64_t* keys, int64_t m, const int64_t* offs,
                                                         uint32_t* starts) {
  __shared__ int sWave[kWaves];
  __shared__ int64_t sBase;
  const int wave = threadIdx.x >> 6, lane = __lane_id();
  const int64_t b0 = (int64_t)blockIdx.x * kStartChunk;
  const int64_t b1 = b0 + kStartChunk < m ? b0 + kStartChunk : m;
  if (threadIdx.x == 0) sBase = offs[blockIdx.x];
  __syncthreads();
  for (int64_t t0 = b0; t0 < b1; t0 += blockDim.x) {
    const int64_t i = t0 + threadIdx.x;
    const bool f = i < b1 && (i == 0 || !detEqual<W>(keys + i * W, keys + (i - 1) * W));
    const uint64_t bal = __ballot(f);
    if (lane == 0) sWave[wave] = __popcll(bal);
    __syncthreads();
    int64_t base = sBase;
    for (int w = 0; w < wave; w++) base += sWave[w];
    if (f) starts[base + __popcll(bal & lanemaskLt())] = (uint32_t)i;
    __syncthreads();
    if (threadIdx.x == 0)
      for (int w = 0; w < kWaves; w++) sBase += sWave[w];
    __syncthreads();
  }
}

template <int W, bool LDS_TAB>
__global__ void __launch_bounds__(kBlock) kPtReduceStarts(DevSystem S, const uint64_t* keys, const uint32_t* idx,
                                                          const double* num, const uint32_t* starts, int64_t nu,
                                                          int64_t m, double e0, double* partial) {
  const double* tab = ptStageTables<LDS_TAB>(S);
  double sPt = 0.0, sPsi = 0.0, sCnt = 0.0;
  for (int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; u < nu; u += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = starts[u];
    double sum = num[idx[i]];
    for (int64_t j = i + 1; j < m && detEqual<W>(keys + j * W, keys + i * W); j++) sum = __dadd_rn(sum, num[idx[j]]);
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) d[w] = keys[i * W + w];
    const double den = __dsub_rn(e0, ptEnergy<W, LDS_TAB>(S, tab, d));
    sPt = __dadd_rn(sPt, __ddiv_rn(__dmul_rn(fabs(sum), fabs(sum)), den));
    const double r = __ddiv_rn(sum, den);
    sPsi = __dadd_rn(sPsi, __dmul_rn(fabs(r), fabs(r)));
    sCnt += 1.0;
  }
  const double t0 = blockSum(sPt), t1 = blockSum(sPsi), t2 = blockSum(sCnt);
  if (threadIdx.x == 0) {
    partial[3 * blockIdx.x] = t0;
    partial[3 * blockIdx.x + 1] = t1;
    partial[3 * blockIdx.x + 2] = t2;
  }
}


template <int W, bool LDS_TAB>
__global__ void __launch_bounds__(kBlock) kPtStochReduce(DevSystem S, const uint64_t* keys, const uint32_t* idx,
                                                         const double* num, const double* num2, const uint8_t* pres,
                                                         const uint32_t* starts, const int64_t* nStarts, int64_t m,
                                                         double e0, double nmc, double* partial) {
  const double* tab = ptStageTables<LDS_TAB>(S);
  double sA = 0.0, sB = 0.0;
  const int64_t nu = *nStarts;
  for (int64_t u = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; u < nu; u += (int64_t)gridDim.x * blockDim.x) {
    const int64_t i = starts[u];
    double a1 = 0.0, a2 = 0.0, b1 = 0.0, b2 = 0.0;
    for (int64_t j = i; j < m && detEqual<W>(keys + j * W, keys + i * W); j++) {
      const uint32_t q = idx[j];
      a1 = __dadd_rn(a1, num[q]);
      a2 = __dadd_rn(a2, num2[q]);
      if (pres[q]) {
        b1 = __dadd_rn(b1, num[q]);
        b2 = __dadd_rn(b2, num2[q]);
      }
    }
    uint64_t d[W];
#pragma unroll
    for (int w = 0; w < W; w++) d[w] = keys[i * W + w];
    const double den = __dsub_rn(ptEnergy<W, LDS_TAB>(S, tab, d), e0);
    sA = __dadd_rn(sA, __ddiv_rn(__dsub_rn(__ddiv_rn(__dmul_rn(__dmul_rn(fabs(a1), fabs(a1)), nmc), nmc - 1.0), a2),
                                 den));
    sB = __dadd_rn(sB, __ddiv_rn(__dsub_rn(__ddiv_rn(__dmul_rn(__dmul_rn(fabs(b1), fabs(b1)), nmc), nmc - 1.0), b2),
                                 den));
  }
  const double t0 = blockSum(sA), t1 = blockSum(sB);
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = t0;
    partial[2 * blockIdx.x + 1] = t1;
  }
}

__global__ void kPrecondition(double* r, const double* diag, const double* e, int64_t n) {
  const double ev = e[0];
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
    double den = ev - diag[k];
    if (fabs(den) > 1e-12)
      r[k] = r[k] / den;
    else
      r[k] = r[k] / (den - 1.e-12);
  }
}

__global__ void __launch_bounds__(kBlock) kDot2(const double* b, const double* r, int64_t n, double* partial) {
  double s0 = 0.0, s1 = 0.0;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x) {
    double bv = b[k];
    s0 = fma(bv, r[k], s0);
    s1 = fma(bv, bv, s1);
  }
  double t0 = blockSum(s0);
  double t1 = blockSum(s1);
  if (threadIdx.x == 0) {
    partial[2 * blockIdx.x] = t0;
    partial[2 * blockIdx.x + 1] = t1;
  }
}

__global__ void kOrthoStep(double* r, const double* b, const double* d, int64_t n) {
  const double ov = d[0], nn = d[1];
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    r[k] = r[k] - ov * b[k] / nn;
}

__global__ void __launch_bounds__(kBlock) kDot(const double* a, const double* b, int64_t n, double* partial) {
  double s = 0.0;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    s = fma(a[k], b[k], s);
  double t = blockSum(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

__global__ void __launch_bounds__(kBlock) kNorm2(const double* x, int64_t n, double* partial) {
  double s = 0.0;
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    s = fma(x[k], x[k], s);
  double t = blockSum(s);
  if (threadIdx.x == 0) partial[blockIdx.x] = t;
}

__global__ void kScaleInto(double* dst, const double* src, const double* nrm2, int64_t n) {
  const double nr = sqrt(nrm2[0]);
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    dst[k] = src[k] / nr;
}

__global__ void kAxpy(double* x, const double* y, double alpha, int64_t n) {
  for (int64_t k = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; k < n; k += (int64_t)gridDim.x * blockDim.x)
    x[k] = x[k] + alpha * y[k];
}

// Cyclic Jacobi for m <= kJacobiMax on one wavefront with the matrices in
// LDS: rotations are applied in the sequential (p, q) order, lane k updating
// element k of the two rows / columns, so every element sees the same
// operations in the same order as a one-thread sweep.  It is one chain of
// dependent operations (a rotation's angle, then its rows and columns), so
// what counts is the LDS round trips in it: two per rotation beside the read
// of the pivot.
constexpr int kJacobiMax = 32;

// a: the matrix (LDS, overwritten), v, order: LDS scratch; called by the 64
// lanes of one wave
__device__ void jacobiWave(double* a, double* v, int* order, int m, double* w, double* V) {
  const int lane = __lane_id();
  for (int q = lane; q < m * m; q += 64) v[q] = q / m == q % m ? 1.0 : 0.0;
  waveSync();
  for (int sweep = 0; sweep < 100; sweep++) {
    bool off = false;  // any element above the diagonal that is not zero
    for (int t = lane; t < m * m; t += 64) off |= t % m > t / m && a[t] != 0.0;
    if (__ballot(off) == 0ull) break;
    for (int p = 0; p < m; p++)
      for (int q = p + 1; q < m; q++) {
        const double apq = a[p * m + q], app = a[p * m + p], aqq = a[q * m + q];
        const double g = 100.0 * fabs(apq);
        if (sweep > 3 && fabs(app) + g == fabs(app) && fabs(aqq) + g == fabs(aqq)) {
          waveSync();
          if (lane == 0) {
            a[p * m + q] = 0.0;
            a[q * m + p] = 0.0;
          }
          waveSync();
          continue;
        }
        if (apq == 0.0) continue;
        double akp = 0.0, akq = 0.0, vkp = 0.0, vkq = 0.0;
        if (lane < m) {
          akp = a[lane * m + p];
          akq = a[lane * m + q];
          vkp = v[lane * m + p];
          vkq = v[lane * m + q];
        }
        const double theta = (aqq - app) / (2.0 * apq);
        const double t = (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
        const double c = 1.0 / sqrt(t * t + 1.0), sn = t * c;
        waveSync();
        if (lane < m) {
          a[lane * m + p] = c * akp - sn * akq;
          a[lane * m + q] = sn * akp + c * akq;
          v[lane * m + p] = c * vkp - sn * vkq;
          v[lane * m + q] = sn * vkp + c * vkq;
        }
        waveSync();
        if (lane < m) {
          const double apk = a[p * m + lane], aqk = a[q * m + lane];
          a[p * m + lane] = lane == q ? 0.0 : c * apk - sn * aqk;
          a[q * m + lane] = lane == p ? 0.0 : sn * apk + c * aqk;
        }
        waveSync();
      }
  }
  if (lane == 0) {
    for (int i = 0; i < m; i++) order[i] = i;
    for (int i = 1; i < m; i++) {  // stable insertion sort by eigenvalue
      const int o = order[i];
      int j = i;
      while (j > 0 && a[order[j - 1] * m + order[j - 1]] > a[o * m + o]) {
        order[j] = order[j - 1];
        j--;
      }
      order[j] = o;
    }
  }
  waveSync();
  if (lane < m) w[lane] = a[order[lane] * m + order[lane]];
  for (int q = lane; q < m * m; q += 64) {
    const int k = q / m, j = q % m;
    V[k * m + j] = v[k * m + order[j]];
  }
}

// ---- one step of the single-vector Davidson, in few launches --------------
//
// On small spaces its time was the launches: three for every dot product and
// step of the orthogonalisation, two for each norm, one for each rotation.
// Here a kernel that needs a sum over the vector ends the reduction of the
// previous kernel itself, every workgroup by itself and all in the same fixed
// order, and leaves its own partial sums for the next one.  Every element
// and every sum takes the operations of separate kernels for the Gram matrix,
// its eigenpairs, the rotation, the residual, the preconditioner, each dot
// product, each orthogonalisation step and the norms, in their order: the
// same bits.  With m columns m + 6 launches in place of 3 m + 12 and more, and
// the scalars the host decides on come through memory it can read.  The
// two-root solve on 57,963 determinants of 40 orbitals (184 iterations) 52 ->
// 30 ms, the whole step of an 8-orbital molecule (86 iterations) 20 -> 16.

// v summed over the wave as the xor tree 32, 16, 8, 4, 2, 1: the last four
// steps rotate within rows of 16 lanes (a step's value repeats with its
// distance, so the rotation brings what the xor would), without LDS
template <int CTRL>
__device__ __forceinline__ double dppAdd(double v) {
  const int lo = __builtin_amdgcn_update_dpp(0, __double2loint(v), CTRL, 0xf, 0xf, true);
  const int hi = __builtin_amdgcn_update_dpp(0, __double2hiint(v), CTRL, 0xf, 0xf, true);
  return v + __hiloint2double(hi, lo);
}
__device__ __forceinline__ double waveSumXor(double v) {
  v += __shfl_xor(v, 32, 64);
  v += __shfl_xor(v, 16, 64);
  v = dppAdd<0x128>(v);  // row_ror:8
  v = dppAdd<0x124>(v);
  v = dppAdd<0x122>(v);
  return dppAdd<0x121>(v);
}

// the workgroup's sums of v[NV], as blockSum; every thread gets them
template <int NV>
__device__ __forceinline__ void blockSums(double (&v)[NV], double* red) {
  const int wave = threadIdx.x >> 6, lane = __lane_id();
#pragma unroll
  for (int q = 0; q < NV; q++) {
    const double t = waveSumXor(v[q]);
    if (lane == 0) red[q * kWaves + wave] = t;
  }
  __syncthreads();
#pragma unroll
  for (int q = 0; q < NV; q++) {
    double t = 0.0;
    for (int w = 0; w < kWaves; w++) t += red[q * kWaves + w];
    v[q] = t;
  }
  __syncthreads();
}

// the sums kFinalSum forms of nb partials of NV values
template <int NV>
__device__ __forceinline__ void finalSums(const double* partial, int nb, double (&v)[NV], double* red) {
#pragma unroll
  for (int q = 0; q < NV; q++) {
    v[q] = 0.0;
    for (int b = threadIdx.x; b < nb; b += kBlock) v[q] += partial[(int64_t)b * NV + q];
  }
  blockSums<NV>(v, red);
}

// partial Gram entries B_i . S_j, i <= j, of exactly M columns
template <int M>
__global__ void __launch_bounds__(kBlock) kGramUpper(const double* __restrict__ B, const double* __restrict__ S,
                                                     int64_t n, int64_t ld, double* __restrict__ partial) {
  constexpr int Q = M * (M + 1) / 2;
  __shared__ double red[kWaves][Q];
  double acc[Q];
#pragma unroll
  for (int q = 0; q < Q; q++) acc[q] = 0.0;
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < n; k += (int64_t)gridDim.x * kBlock) {
    double a[M], b[M];
#pragma unroll
    for (int i = 0; i < M; i++) {
      a[i] = B[i * ld + k];
      b[i] = S[i * ld + k];
    }
    int q = 0;
#pragma unroll
    for (int i = 0; i < M; i++)
#pragma unroll
      for (int j = i; j < M; j++, q++) acc[q] = fma(a[i], b[j], acc[q]);
  }
  const int wave = threadIdx.x >> 6, lane = __lane_id();
#pragma unroll
  for (int q = 0; q < Q; q++) {
    const double t = waveSumXor(acc[q]);
    if (lane == 0) red[wave][q] = t;
  }
  __syncthreads();
  for (int q = threadIdx.x; q < Q; q += kBlock) {
    double v = 0.0;
    for (int w = 0; w < kWaves; w++) v += red[w][q];
    partial[(int64_t)blockIdx.x * Q + q] = v;
  }
}

// the Gram matrix from those partials (a wave per entry: the four wave sums
// of kFinalSum one after the other) and its eigenpairs; one workgroup
constexpr int kGramThreads = 1024;
__global__ void __launch_bounds__(kGramThreads) kGramJacobi(const double* __restrict__ partial, int nb, int m,
                                                            double* w, double* V) {
  __shared__ double a[kJacobiMax * kJacobiMax], v[kJacobiMax * kJacobiMax];
  __shared__ int order[kJacobiMax];
  const int wave = threadIdx.x >> 6, lane = __lane_id(), Q = m * (m + 1) / 2;
  for (int q = wave; q < Q; q += kGramThreads / 64) {
    double t = 0.0;
    for (int c = 0; c < kWaves; c++) {
      double u = 0.0;
      for (int b = c * 64 + lane; b < nb; b += kBlock) u += partial[(int64_t)b * Q + q];
      t += waveSumXor(u);
    }
    int i = 0, r = q;
    while (r >= m - i) {
      r -= m - i;
      i++;
    }
    if (lane == 0) {
      a[i * m + i + r] = t;
      a[(i + r) * m + i] = t;
    }
  }
  __syncthreads();
  if (wave == 0) jacobiWave(a, v, order, m, w, V);
}

// B and S rotated by V (m x m), the residuals S_i - w_i B_i of the columns
// i <= last (r: the last one), and the partial sums of their squares
constexpr int kResMax = 12;
__global__ void __launch_bounds__(kBlock) kRotateResidual(double* B, double* S, int m, int64_t n, int64_t ld,
                                                          const double* V, const double* w, int last, double* r,
                                                          double* partial) {
  __shared__ double sV[16 * 16];
  __shared__ double red[kWaves];
  for (int q = threadIdx.x; q < m * m; q += kBlock) sV[q] = V[q];
  __syncthreads();
  double acc[kResMax];
#pragma unroll
  for (int i = 0; i < kResMax; i++) acc[i] = 0.0;
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < n; k += (int64_t)gridDim.x * kBlock) {
    double bi[16], si[16];
#pragma unroll
    for (int l = 0; l < 16; l++)
      if (l < m) {
        bi[l] = B[l * ld + k];
        si[l] = S[l * ld + k];
      }
#pragma unroll
    for (int j = 0; j < 16; j++) {
      if (j >= m) break;
      double bo = 0.0, so = 0.0;
#pragma unroll
      for (int l = 0; l < 16; l++)
        if (l < m) {
          bo = fma(bi[l], sV[l * m + j], bo);
          so = fma(si[l], sV[l * m + j], so);
        }
      B[j * ld + k] = bo;
      S[j * ld + k] = so;
      if (j < kResMax && j <= last) {
        const double d = so - w[j] * bo;
        if (j == last) r[k] = d;
        acc[j] = fma(d, d, acc[j]);
      }
    }
  }
#pragma unroll
  for (int j = 0; j < kResMax; j++) {
    if (j > last) break;
    double t[1] = {acc[j]};
    blockSums<1>(t, red);
    if (threadIdx.x == 0) partial[(int64_t)blockIdx.x * (last + 1) + j] = t[0];
  }
}

// the residuals' sums, with the eigenvalues, to host memory: w (16), sums
__global__ void __launch_bounds__(kBlock) kResidualSums(const double* partial, int nb, int count, const double* w,
                                                        int m, double* host) {
  __shared__ double red[kWaves];
  for (int q = 0; q < count; q++) {
    double v[1] = {0.0};
    for (int b = threadIdx.x; b < nb; b += kBlock) v[0] += partial[(int64_t)b * count + q];
    blockSums<1>(v, red);
    if (threadIdx.x == 0) host[16 + q] = v[0];
  }
  if ((int)threadIdx.x < m) host[threadIdx.x] = w[threadIdx.x];
}

// r /= e - diag (kPrecondition) and the partials of b . r and b . b
__global__ void __launch_bounds__(kBlock) kPreconditionDot(double* r, const double* __restrict__ diag, const double* e,
                                                           const double* __restrict__ b, int64_t n, double* out) {
  __shared__ double red[2 * kWaves];
  const double ev = e[0];
  double v[2] = {0.0, 0.0};
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < n; k += (int64_t)gridDim.x * kBlock) {
    const double den = ev - diag[k];
    const double x = fabs(den) > 1e-12 ? r[k] / den : r[k] / (den - 1.e-12);
    r[k] = x;
    const double bv = b[k];
    v[0] = fma(bv, x, v[0]);
    v[1] = fma(bv, bv, v[1]);
  }
  blockSums<2>(v, red);
  if (threadIdx.x == 0) {
    out[2 * blockIdx.x] = v[0];
    out[2 * blockIdx.x + 1] = v[1];
  }
}

// r -= (b . r) b / (b . b) with the sums of `in`, then the partials of next . r
// and next . next, or (next null) of r . r
__global__ void __launch_bounds__(kBlock) kOrthoDot(double* r, const double* __restrict__ b,
                                                    const double* __restrict__ next, int64_t n, const double* in,
                                                    double* out) {
  __shared__ double red[2 * kWaves];
  double s[2];
  finalSums<2>(in, (int)gridDim.x, s, red);
  double v[2] = {0.0, 0.0};
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < n; k += (int64_t)gridDim.x * kBlock) {
    const double x = r[k] - s[0] * b[k] / s[1];
    r[k] = x;
    if (next) {
      const double bv = next[k];
      v[0] = fma(bv, x, v[0]);
      v[1] = fma(bv, bv, v[1]);
    } else {
      v[0] = fma(x, x, v[0]);
    }
  }
  blockSums<2>(v, red);
  if (threadIdx.x == 0) {
    if (next) {
      out[2 * blockIdx.x] = v[0];
      out[2 * blockIdx.x + 1] = v[1];
    } else {
      out[blockIdx.x] = v[0];
    }
  }
}

// dst = r / sqrt(sum of in)
__global__ void __launch_bounds__(kBlock) kScaleSum(double* dst, const double* __restrict__ r, int64_t n,
                                                    const double* in) {
  __shared__ double red[kWaves];
  double s[1];
  finalSums<1>(in, (int)gridDim.x, s, red);
  const double nr = sqrt(s[0]);
  for (int64_t k = (int64_t)blockIdx.x * kBlock + threadIdx.x; k < n; k += (int64_t)gridDim.x * kBlock)
    dst[k] = r[k] / nr;
}

// The same eigenproblem with the rotations of a sweep in round-robin
// (tournament) order: the m'/2 disjoint pairs of a step (m' = m rounded up
// to even) are rotated at once, m'-1 steps per sweep, so a sweep needs
// m'-1 rounds of barriers instead of m(m-1)/2.  Another rotation order than
// jacobiWave's, so the eigenpairs agree with it to rounding, not bit for bit;
// used by the block Davidson.  A chain of steps again: a step's rotations (two
// divisions and two roots), then all elements.  Thread (R, C) has the four
// elements of the row pair R and the column pair C, which no other pair mixes,
// and applies C's rotation and then R's to them in registers (16 x 16 threads
// cover the largest m), so a step is two barriers and one LDS round trip, not
// four passes of one wave over the matrix.  m = 8..24: 209 -> 102 us.
__global__ void __launch_bounds__(kBlock) kJacobiRR(const double* A, int m, double* w, double* V) {
  static_assert(kJacobiMax <= 32 && kBlock == 256, "a thread per pair of pairs");
  __shared__ double a[kJacobiMax * kJacobiMax], v[kJacobiMax * kJacobiMax];
  __shared__ double rc[16], rs[16];
  __shared__ int rp[16], rq[16];
  __shared__ int rk[16];  // 1: rotate, 0: leave, -1: zero the pivot only
  __shared__ int order[kJacobiMax];
  const int tid = threadIdx.x;
  const int mm = (m + 1) & ~1, half = mm / 2;
  for (int q = tid; q < m * m; q += kBlock) {
    a[q] = A[q];
    v[q] = q / m == q % m ? 1.0 : 0.0;
  }
  const int R = tid >> 4, C = tid & 15;
  const bool mine = R < half && C < half;
  const int k0 = 2 * R, k1 = 2 * R + 1;  // this thread's rows of v (pair C)
  __syncthreads();
  for (int sweep = 0; sweep < 100; sweep++) {
    int off = 0;
    for (int t = tid; t < m * m; t += kBlock)
      if (t % m > t / m && a[t] != 0.0) off = 1;
    if (!__syncthreads_or(off)) break;
    for (int step = 0; step < mm - 1; step++) {
      if (tid < half) {
        // round-robin: player 0 fixed, the others rotate by step
        int p = 0, q = mm - 2 - tid + step;
        if (tid > 0) {
          p = tid - 1 + step;
          p = (p >= mm - 1 ? p - (mm - 1) : p) + 1;
        }
        q = (q >= mm - 1 ? q - (mm - 1) : q) + 1;
        if (p > q) {
          const int t = p;
          p = q;
          q = t;
        }
        double c = 1.0, sn = 0.0;
        int kind = 0;
        if (q < m) {
          const double apq = a[p * m + q], app = a[p * m + p], aqq = a[q * m + q];
          const double g = 100.0 * fabs(apq);
          if (sweep > 3 && fabs(app) + g == fabs(app) && fabs(aqq) + g == fabs(aqq)) {
            kind = -1;  // negligible: zero it without a rotation
          } else if (apq != 0.0) {
            const double theta = (aqq - app) / (2.0 * apq);
            const double t = (theta >= 0 ? 1.0 : -1.0) / (fabs(theta) + sqrt(theta * theta + 1.0));
            c = 1.0 / sqrt(t * t + 1.0);
            sn = t * c;
            kind = 1;
          }
        }
        rp[tid] = p;
        rq[tid] = q;
        rk[tid] = kind;
        rc[tid] = c;
        rs[tid] = sn;
      }
      __syncthreads();
      if (mine) {
        const int p = rp[R], q = rq[R], kindR = rk[R];
        const int pc = rp[C], qc = rq[C], kindC = rk[C];
        if (kindR != 0 || kindC != 0) {
          // q or qc == m: the pair of the one left over (odd m), no such row
          const bool hasQ = q < m, hasQc = qc < m;
          double pp = a[p * m + pc], pq = 0.0, qp = 0.0, qq = 0.0;
          if (hasQc) pq = a[p * m + qc];
          if (hasQ) qp = a[q * m + pc];
          if (hasQ && hasQc) qq = a[q * m + qc];
          if (kindC > 0) {
            const double c = rc[C], sn = rs[C];
            const double x = c * pp - sn * pq, y = sn * pp + c * pq;
            pp = x;
            pq = y;
            const double z = c * qp - sn * qq, u = sn * qp + c * qq;
            qp = z;
            qq = u;
            if (k0 < m) {
              const double vp = v[k0 * m + pc], vq = v[k0 * m + qc];
              v[k0 * m + pc] = c * vp - sn * vq;
              v[k0 * m + qc] = sn * vp + c * vq;
            }
            if (k1 < m) {
              const double vp = v[k1 * m + pc], vq = v[k1 * m + qc];
              v[k1 * m + pc] = c * vp - sn * vq;
              v[k1 * m + qc] = sn * vp + c * vq;
            }
          }
          if (kindR > 0) {
            const double c = rc[R], sn = rs[R];
            const double x = c * pp - sn * qp, y = sn * pp + c * qp;
            pp = x;
            qp = y;
            const double z = c * pq - sn * qq, u = sn * pq + c * qq;
            pq = z;
            qq = u;
          }
          if (R == C) pq = qp = 0.0;
          a[p * m + pc] = pp;
          if (hasQc) a[p * m + qc] = pq;
          if (hasQ) a[q * m + pc] = qp;
          if (hasQ && hasQc) a[q * m + qc] = qq;
        }
      }
      __syncthreads();
    }
  }
  // stable order by eigenvalue: by rank, or (NaNs have none) by insertion
  if (__syncthreads_or(tid < m && isnan(a[tid * m + tid]))) {
    if (tid == 0) {
      for (int i = 0; i < m; i++) order[i] = i;
      for (int i = 1; i < m; i++) {
        const int o = order[i];
        int j = i;
        while (j > 0 && a[order[j - 1] * m + order[j - 1]] > a[o * m + o]) {
          order[j] = order[j - 1];
          j--;
        }
        order[j] = o;
      }
    }
  } else if (tid < m) {
    const double d = a[tid * m + tid];
    int rank = 0;
    for (int j = 0; j < m; j++) {
      const double e = a[j * m + j];
      rank += e < d || (e == d && j < tid);
    }
    order[rank] = tid;
  }
  __syncthreads();
  if (tid < m) w[tid] = a[order[tid] * m + order[tid]];
  for (int q = tid; q < m * m; q += kBlock) {
    const int k = q / m, j = q % m;
    V[k * m + j] = v[k * m + order[j]];
  }
}

}  // namespace

// ===========================================================================
// launchers

#define DISPATCH_W(W_, ...)                  \
  do {                                       \
    if ((W_) == 1) {                         \
      constexpr int WW = 1;                  \
      __VA_ARGS__;                           \
    } else if ((W_) == 2) {                  \
      constexpr int WW = 2;                  \
      __VA_ARGS__;                           \
    } else {                                 \
      throw HipError("unsupported det width"); \
    }                                        \
  } while (0)

void launchEnergy(const DevSystem& S, const uint64_t* dets, int64_t n, double* out, hipStream_t s) {
  if (n <= 0) return;
  DISPATCH_W(S.W, kEnergy<WW><<<gridFor(n), kBlock, 0, s>>>(S, dets, n, out));
  HIP_CHECK(hipGetLastError());
}

void launchHijPairs(const DevSystem& S, const uint64_t* bra, const uint64_t* ket, int64_t n, double* out,
                    hipStream_t s) {
  if (n <= 0) return;
  DISPATCH_W(S.W, kHijPairs<WW><<<gridFor(n), kBlock, 0, s>>>(S, bra, ket, n, out));
  HIP_CHECK(hipGetLastError());
}

void hashClear(int32_t* table, uint64_t slots, hipStream_t s) {
  kFillNeg<<<gridFor((int64_t)slots), kBlock, 0, s>>>(table, slots);
  HIP_CHECK(hipGetLastError());
}

void hashInsert(const DevSystem& S, const uint64_t* dets, int64_t begin, int64_t end, int32_t* table,
                uint64_t slots, hipStream_t s) {
  if (end <= begin) return;
  DISPATCH_W(S.W, kHashInsert<WW><<<gridFor(end - begin), kBlock, 0, s>>>(dets, begin, end, table, slots - 1));
  HIP_CHECK(hipGetLastError());
}

void launchCmax(const double* ci, int nroots, int64_t ld, int64_t n, double* cmax, hipStream_t s) {
  if (n <= 0) return;
  kCmax<<<gridFor(n), kBlock, 0, s>>>(ci, nroots, ld, n, cmax);
  HIP_CHECK(hipGetLastError());
}

int pairSlices(int64_t nsrc, int nelec) {
  // 32,768 waves (four times what the chip holds) where the sources are
  // fewer, in parts of at least four pairs of electrons, so that a part's own
  // set-up (the lists of occupied and open orbitals) stays small
  const int64_t most = 1 + std::max(1, nelec * (nelec - 1) / 2 / 4);
  return (int)std::max<int64_t>(1, std::min<int64_t>(most, 32768 / std::max<int64_t>(nsrc, 1)));
}

void launchScreen(const DevSystem& S, const uint64_t* dets, int64_t begin, int64_t end, const double* cmax,
                  double eps1, int ncore, int nact, const int32_t* table, uint64_t slots, uint64_t* out,
                  unsigned long long* counter, int64_t cap, hipStream_t s) {
  if (end <= begin) return;
  const int slices = pairSlices(end - begin, S.nelec);
  unsigned g = gridFor((end - begin) * slices, kWaves, 1 << 16);
  DISPATCH_W(S.W, kScreen<WW, 0><<<g, kBlock, 0, s>>>(S, dets, begin, end, cmax, eps1, ncore, nact, table,
                                                         slots - 1, out, counter, cap, 1.0, nullptr, slices));
  HIP_CHECK(hipGetLastError());
}

void buildDenseHeatBath(const DevSystem& S, DevMem* dense, hipStream_t s) {
  const int64_t npair = (int64_t)S.norb * (S.norb + 1) / 2, m = npair * S.norb * S.norb;
  for (int k = 0; k < 2; k++) {
    dense[k].reserve((size_t)m * 4, s);
    kFillNan<<<gridFor(m), kBlock, 0, s>>>(dense[k].as<float>(), m);
    kDenseHeatBath<<<gridFor(npair, 1), kBlock, 0, s>>>(S.hbVal[k], S.hbPair[k], S.hbStart[k], npair, S.norb,
                                                        dense[k].as<float>());
  }
  HIP_CHECK(hipGetLastError());
}

void launchPtGen(const DevSystem& S, const uint64_t* dets, int64_t n, const double* ci, double eps2,
                 const int32_t* table, uint64_t slots, uint32_t nparts, uint32_t part, int slices, const DevMem* dense,
                 int64_t* counts, const int64_t* fillStart, uint64_t* outD, double* outN, hipStream_t s) {
  if (n <= 0) return;
  if (nparts == 0 || part >= nparts) throw HipError("launchPtGen: bad partition");
  unsigned g = gridFor(n * slices, kWaves, 1 << 16);
  const PtStoch st{nullptr, nullptr, 0.0, 0.0, nullptr, nullptr};
  const float *d0 = dense[0].as<float>(), *d1 = dense[1].as<float>();
  if (fillStart)
    DISPATCH_W(S.W, kPtGen<WW, true, false><<<g, kBlock, 0, s>>>(S, dets, n, ci, eps2, table, slots - 1, nparts, part,
                                                                   counts, fillStart, outD, outN, st, slices, d0, d1));
  else
    DISPATCH_W(S.W,
               kPtGen<WW, false, false><<<g, kBlock, 0, s>>>(S, dets, n, ci, eps2, table, slots - 1, nparts, part,
                                                              counts, nullptr, nullptr, nullptr, st, slices, d0, d1));
  HIP_CHECK(hipGetLastError());
}

void launchPtGenStoch(const DevSystem& S, const uint64_t* dets, const uint32_t* src, const double* w, int64_t nsrc,
                      const double* ci, double eps2, double eps2Large, double nmc, const int32_t* table, uint64_t slots,
                      int slices, const DevMem* dense, int64_t* counts, const int64_t* fillStart, uint64_t* outD,
                      double* outN, double* outN2, uint8_t* outP, hipStream_t s) {
  if (nsrc <= 0) return;
  unsigned g = gridFor(nsrc * slices, kWaves, 1 << 16);
  const PtStoch st{src, w, eps2Large, nmc, outN2, outP};
  const float *d0 = dense[0].as<float>(), *d1 = dense[1].as<float>();
  if (fillStart)
    DISPATCH_W(S.W, kPtGen<WW, true, true><<<g, kBlock, 0, s>>>(S, dets, nsrc, ci, eps2, table, slots - 1, 1u, 0u,
                                                                  counts, fillStart, outD, outN, st, slices, d0, d1));
  else
    DISPATCH_W(S.W,
               kPtGen<WW, false, true><<<g, kBlock, 0, s>>>(S, dets, nsrc, ci, eps2, table, slots - 1, 1u, 0u, counts,
                                                             nullptr, nullptr, nullptr, st, slices, d0, d1));
  HIP_CHECK(hipGetLastError());
}

void launchPtStochReduce(const DevSystem& S, const uint64_t* keys, const uint32_t* idx, const double* num,
                         const double* num2, const uint8_t* pres, int64_t m, double e0, double nmc, DevMem& partial,
                         DevMem& counts, DevMem& starts, Workspace& ws, double* out, hipStream_t s) {
  // over the run starts, compacted in order first, as the deterministic sum
  const int64_t nbS = (m + kStartChunk - 1) / kStartChunk;
  counts.reserve((size_t)(nbS + 1) * 8, s);
  starts.reserve((size_t)m * 4, s);
  int64_t* cnt = counts.as<int64_t>();
  HIP_CHECK(hipMemsetAsync(cnt + nbS, 0, 8, s));
  DISPATCH_W(S.W, kPtCountStarts<WW><<<(unsigned)nbS, kBlock, 0, s>>>(keys, m, cnt));
  exclusiveScanI64(cnt, nbS + 1, ws, s);
  DISPATCH_W(S.W, kPtWriteStarts<WW><<<(unsigned)nbS, kBlock, 0, s>>>(keys, m, cnt, starts.as<uint32_t>()));
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(kPtRedBlocks, (m + kBlock - 1) / kBlock));
  partial.reserve((size_t)nb * 2 * sizeof(double));
  const size_t tb = ptTabBytes(S.norb);
  if (tb <= kPtTabMaxBytes)
    DISPATCH_W(S.W, kPtStochReduce<WW, true><<<nb, kBlock, tb, s>>>(S, keys, idx, num, num2, pres,
                                                                    starts.as<uint32_t>(), cnt + nbS, m, e0, nmc,
                                                                    partial.as<double>()));
  else
    DISPATCH_W(S.W, kPtStochReduce<WW, false><<<nb, kBlock, 0, s>>>(S, keys, idx, num, num2, pres,
                                                                     starts.as<uint32_t>(), cnt + nbS, m, e0, nmc,
                                                                     partial.as<double>()));
  kFinalSum<<<2, kBlock, 0, s>>>(partial.as<double>(), nb, 2, 2, out);
  HIP_CHECK(hipGetLastError());
}

size_t rdmScratchDoubles(int norb, int W) {
  const size_t n = norb, NSO = 64 * W;
  return NSO * NSO + n * n * n * n + 2 * n * n * n;
}

void launchRdm(int norb, int W, const uint64_t* dets, const int64_t* rp, const int32_t* cols, const double* bra,
               const double* ket, int64_t n, double* g1, double* g2, double* s1, double* s2, double* scratch,
               hipStream_t s) {
  if (norb > 32 * W) throw HipError("launchRdm: more orbitals than the determinant words hold");
  const int NSO = 64 * W;
  const int64_t nn = norb, n3 = nn * nn * nn;
  double* M = scratch;
  RdmOut o{g1, g2, s1, s2, M + (int64_t)NSO * NSO, M + (int64_t)NSO * NSO + n3 * nn,
           M + (int64_t)NSO * NSO + n3 * nn + n3, norb, 2 * norb, (int64_t)(2 * norb) * (2 * norb + 1) / 2,
           bra == ket};
  HIP_CHECK(hipMemsetAsync(scratch, 0, rdmScratchDoubles(norb, W) * 8, s));
  if (n > 0) {
    const unsigned go = (unsigned)std::min<int64_t>(std::max<int64_t>(n / 64, 1), 2048);
    DISPATCH_W(W, kRdmOcc<WW><<<go, kBlock, 0, s>>>(dets, bra, ket, n, M));
    const unsigned g = gridFor(n, kWaves, 1 << 16);
    DISPATCH_W(W, kRdm<WW><<<g, kBlock, 0, s>>>(o, dets, rp, cols, bra, ket, n));
  }
  kRdmFinish<<<gridFor(n3 * nn), kBlock, 0, s>>>(o);
  kRdmOccScatter<<<gridFor((int64_t)o.nso * o.nso), kBlock, 0, s>>>(o, M, NSO);
  HIP_CHECK(hipGetLastError());
}

int64_t launchTrevBasis(const uint64_t* dets, int64_t i0, int64_t i1, int W, DevMem& flags, uint64_t* block,
                        int64_t base, int64_t* eIdx, int64_t* partner, double* parity, Workspace& ws, hipStream_t s) {
  const int64_t cnt = i1 - i0;
  if (cnt <= 0) return 0;
  flags.reserve((size_t)(cnt + 1) * 8, s);
  int64_t* f = flags.as<int64_t>();
  HIP_CHECK(hipMemsetAsync(f + cnt, 0, 8, s));
  DISPATCH_W(W, kTrevMark<WW><<<gridFor(cnt), kBlock, 0, s>>>(dets, i0, i1, f));
  exclusiveScanI64(f, cnt + 1, ws, s);
  int64_t nu = 0;
  HIP_CHECK(hipMemcpyAsync(&nu, f + cnt, 8, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  if (block)
    DISPATCH_W(W, kTrevBlock<WW><<<gridFor(cnt), kBlock, 0, s>>>(dets, i0, i1, f, base, block, eIdx, partner, parity));
  HIP_CHECK(hipGetLastError());
  return nu;
}

void launchTrevExpand(const double* x, int64_t n, int k, int64_t ld, const int64_t* eIdx, const int64_t* partner,
                      const double* parity, double* xE, int64_t ldE, hipStream_t s) {
  if (n <= 0) return;
  kTrevExpand<<<gridFor(n * k), kBlock, 0, s>>>(x, n, k, ld, eIdx, partner, parity, xE, ldE);
  HIP_CHECK(hipGetLastError());
}

void launchTrevContract(const double* yE, int64_t ldE, int64_t n, int k, const int64_t* eIdx, const int64_t* partner,
                        const double* parity, double* y, int64_t ld, hipStream_t s) {
  if (n <= 0) return;
  kTrevContract<<<gridFor(n * k), kBlock, 0, s>>>(yE, ldE, n, k, eIdx, partner, parity, y, ld);
  HIP_CHECK(hipGetLastError());
}

void launchTrevUnpack(const double* ci, int64_t n, int nroots, int64_t ld, const int64_t* partner,
                      const double* parity, int trev, double* out, int64_t ldE, hipStream_t s) {
  if (n <= 0) return;
  kTrevUnpack<<<gridFor(n * nroots), kBlock, 0, s>>>(ci, n, nroots, ld, partner, parity, trev, out, ldE);
  HIP_CHECK(hipGetLastError());
}


void launchIota(uint32_t* v, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  kIota<<<gridFor(n, kBlock, 8192), kBlock, 0, s>>>(v, n);
  HIP_CHECK(hipGetLastError());
}

static int computeUnits() {
  static int cus = 0;
  if (cus == 0) {
    int dev = 0;
    HIP_CHECK(hipGetDevice(&dev));
    HIP_CHECK(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    if (cus <= 0) cus = 256;
  }
  return cus;
}

void launchPtReduce(const DevSystem& S, const uint64_t* keys, const uint32_t* idx, const double* num, int64_t m,
                    double e0, DevMem& partial, DevMem& counts, DevMem& starts, Workspace& ws, double* out,
                    hipStream_t s) {
  if (m <= 0) {
    HIP_CHECK(hipMemsetAsync(out, 0, 3 * sizeof(double), s));
    return;
  }
  // run starts, compacted in order
  const int64_t nbS = (m + kStartChunk - 1) / kStartChunk;
  counts.reserve((size_t)(nbS + 1) * 8, s);
  int64_t* cnt = counts.as<int64_t>();
  HIP_CHECK(hipMemsetAsync(cnt + nbS, 0, 8, s));
  DISPATCH_W(S.W, kPtCountStarts<WW><<<(unsigned)nbS, kBlock, 0, s>>>(keys, m, cnt));
  exclusiveScanI64(cnt, nbS + 1, ws, s);
  int64_t nu = 0;
  HIP_CHECK(hipMemcpyAsync(&nu, cnt + nbS, 8, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  starts.reserve((size_t)std::max<int64_t>(nu, 1) * 4, s);
  DISPATCH_W(S.W, kPtWriteStarts<WW><<<(unsigned)nbS, kBlock, 0, s>>>(keys, m, cnt, starts.as<uint32_t>()));
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(kPtRedBlocks, (nu + kBlock - 1) / kBlock));
  partial.reserve((size_t)nb * 3 * sizeof(double));
  const size_t tb = ptTabBytes(S.norb);
  if (tb <= kPtTabMaxBytes)
    DISPATCH_W(S.W, kPtReduceStarts<WW, true><<<nb, kBlock, tb, s>>>(S, keys, idx, num, starts.as<uint32_t>(), nu, m,
                                                                     e0, partial.as<double>()));
  else
    DISPATCH_W(S.W, kPtReduceStarts<WW, false><<<nb, kBlock, 0, s>>>(S, keys, idx, num, starts.as<uint32_t>(), nu,
                                                                      m, e0, partial.as<double>()));
  kFinalSum<<<3, kBlock, 0, s>>>(partial.as<double>(), nb, 3, 3, out);
  HIP_CHECK(hipGetLastError());
}

void launchScreenSingles(const DevSystem& S, const uint64_t* dets, int64_t begin, int64_t end, const double* cmax,
                         double eps1, int ncore, int nact, const int32_t* table, uint64_t slots, uint64_t* out,
                         unsigned long long* counter, int64_t cap, hipStream_t s) {
  if (end <= begin) return;
  unsigned g = gridFor(end - begin, kWaves, 1 << 16);
  DISPATCH_W(S.W, kScreen<WW, 1><<<g, kBlock, 0, s>>>(S, dets, begin, end, cmax, eps1, ncore, nact, table,
                                                         slots - 1, out, counter, cap, 1.0, nullptr, 1));
  HIP_CHECK(hipGetLastError());
}

void launchScreenRecords(const DevSystem& S, const uint64_t* dets, int64_t begin, int64_t end, const double* cmax,
                         double eps1, double loosen, int ncore, int nact, CandRecord* rec,
                         unsigned long long* counter, int64_t cap, hipStream_t s) {
  if (end <= begin) return;
  unsigned g = gridFor(end - begin, kWaves, 1 << 16);
  DISPATCH_W(S.W, kScreen<WW, 2><<<g, kBlock, 0, s>>>(S, dets, begin, end, cmax, eps1, ncore, nact, nullptr, 0,
                                                         nullptr, counter, cap, loosen, rec, 1));
  HIP_CHECK(hipGetLastError());
}

void launchCandFeatures(const DevSystem& S, const CandRecord* rec, int64_t n, const uint64_t* dets,
                        const double* cmax, float* X, int din, hipStream_t s) {
  if (n <= 0) return;
  DISPATCH_W(S.W, kCandFeatures<WW><<<gridFor(n * din), kBlock, 0, s>>>(rec, n, dets, S.nso, cmax, X, din));
  HIP_CHECK(hipGetLastError());
}

void launchCandTargets(const CandRecord* rec, int64_t n, const double* cmax, float* t, hipStream_t s) {
  if (n <= 0) return;
  kCandTargets<<<gridFor(n), kBlock, 0, s>>>(rec, n, cmax, t);
  HIP_CHECK(hipGetLastError());
}

void launchCandExact(const DevSystem& S, const CandRecord* rec, int64_t n, const float* score, float tau,
                     const uint64_t* dets, const double* cmax, double eps1, const int32_t* table, uint64_t slots,
                     uint64_t* out, unsigned long long* counter, int64_t cap, unsigned long long* counts,
                     hipStream_t s) {
  if (n <= 0) return;
  DISPATCH_W(S.W, kCandExact<WW><<<gridFor(n), kBlock, 0, s>>>(rec, n, score, tau, dets, cmax, eps1, table,
                                                                  slots - 1, out, counter, cap, counts));
  HIP_CHECK(hipGetLastError());
}

void launchCandSample(const CandRecord* rec, const float* score, const int64_t* idx, int m, const double* cmax,
                      double eps1, float tau, int* flags, float* vals, hipStream_t s) {
  if (m <= 0) return;
  kCandSample<<<gridFor(m), kBlock, 0, s>>>(rec, score, idx, m, cmax, eps1, tau, flags, vals);
  HIP_CHECK(hipGetLastError());
}

void launchGatherRecords(const CandRecord* rec, const int64_t* idx, int64_t m, CandRecord* out, hipStream_t s) {
  if (m <= 0) return;
  kGatherRecords<<<gridFor(m), kBlock, 0, s>>>(rec, idx, m, out);
  HIP_CHECK(hipGetLastError());
}

void buildStringTables(const DevSystem& S, const uint64_t* dets, int64_t n, StringTables& T, Workspace& ws,
                       hipStream_t s) {
  T.n = n;
  const int norb = S.norb;
  T.alpha.reserve(n * 8);
  T.beta.reserve(n * 8);
  T.aIdx.reserve(n * 4);
  T.bIdx.reserve(n * 4);
  T.sortedA.reserve(n * 8);
  T.sortedB.reserve(n * 8);
  T.key.reserve(n * 8);
  T.val.reserve(n * 4);
  T.aMajorDet.reserve(n * 4);
  T.bMajorDet.reserve(n * 4);
  T.aMajorB.reserve(n * 8);
  T.bMajorA.reserve(n * 8);
  DISPATCH_W(S.W, kExtractStrings<WW><<<gridFor(n), kBlock, 0, s>>>(dets, n, T.alpha.as<uint64_t>(),
                                                                        T.beta.as<uint64_t>()));
  HIP_CHECK(hipMemcpyAsync(T.sortedA.p, T.alpha.p, n * 8, hipMemcpyDeviceToDevice, s));
  HIP_CHECK(hipMemcpyAsync(T.sortedB.p, T.beta.p, n * 8, hipMemcpyDeviceToDevice, s));
  radixSortKeys(T.sortedA.as<uint64_t>(), nullptr, n, 1, norb, false, ws, s);
  T.nA = uniqueKeys(T.sortedA.as<uint64_t>(), n, 1, ws, s);
  radixSortKeys(T.sortedB.as<uint64_t>(), nullptr, n, 1, norb, false, ws, s);
  T.nB = uniqueKeys(T.sortedB.as<uint64_t>(), n, 1, ws, s);
  kIndexOf<<<gridFor(n), kBlock, 0, s>>>(T.alpha.as<uint64_t>(), n, T.sortedA.as<uint64_t>(), T.nA,
                                          T.aIdx.as<uint32_t>());
  kIndexOf<<<gridFor(n), kBlock, 0, s>>>(T.beta.as<uint64_t>(), n, T.sortedB.as<uint64_t>(), T.nB,
                                          T.bIdx.as<uint32_t>());
  auto bitsFor = [](uint64_t v) {
    int b = 0;
    while (b < 64 && (v >> b) != 0) b++;
    return b;
  };
  T.aStart.reserve((T.nA + 1) * 8);
  T.bStart.reserve((T.nB + 1) * 8);
  // alpha-major groups, members in increasing determinant index:
  // key = aIdx * n + det
  kGroupKeys<<<gridFor(n), kBlock, 0, s>>>(T.aIdx.as<uint32_t>(), n, T.key.as<uint64_t>(), T.val.as<uint32_t>());
  radixSortKeys(T.key.as<uint64_t>(), T.val.as<uint32_t>(), n, 1, bitsFor((uint64_t)T.nA * n), false, ws, s);
  HIP_CHECK(hipMemcpyAsync(T.aMajorDet.p, T.val.p, n * 4, hipMemcpyDeviceToDevice, s));
  kGroupStarts<<<gridFor(n + 1), kBlock, 0, s>>>(T.key.as<uint64_t>(), n, (uint64_t)n, T.nA,
                                                  T.aStart.as<int64_t>(), T.val.as<uint32_t>(),
                                                  T.beta.as<uint64_t>(), T.aMajorB.as<uint64_t>());
  // beta-major groups: key = bIdx * n + det
  kGroupKeys<<<gridFor(n), kBlock, 0, s>>>(T.bIdx.as<uint32_t>(), n, T.key.as<uint64_t>(), T.val.as<uint32_t>());
  radixSortKeys(T.key.as<uint64_t>(), T.val.as<uint32_t>(), n, 1, bitsFor((uint64_t)T.nB * n), false, ws, s);
  HIP_CHECK(hipMemcpyAsync(T.bMajorDet.p, T.val.p, n * 4, hipMemcpyDeviceToDevice, s));
  kGroupStarts<<<gridFor(n + 1), kBlock, 0, s>>>(T.key.as<uint64_t>(), n, (uint64_t)n, T.nB,
                                                  T.bStart.as<int64_t>(), T.val.as<uint32_t>(),
                                                  T.alpha.as<uint64_t>(), T.bMajorA.as<uint64_t>());
  // alpha-major groups with members ordered by beta string (for lookups of
  // a row's beta singles in large groups): key = aIdx * nB + bIdx (the
  // group starts it writes equal the ones above)
  T.aSortB.reserve(n * 8);
  T.aSortDet.reserve(n * 4);
  kGroupKeys2<<<gridFor(n), kBlock, 0, s>>>(T.aIdx.as<uint32_t>(), T.bIdx.as<uint32_t>(), n, (uint64_t)T.nB,
                                             T.key.as<uint64_t>(), T.val.as<uint32_t>());
  radixSortKeys(T.key.as<uint64_t>(), T.val.as<uint32_t>(), n, 1, bitsFor((uint64_t)T.nA * T.nB), false, ws, s);
  HIP_CHECK(hipMemcpyAsync(T.aSortDet.p, T.val.p, n * 4, hipMemcpyDeviceToDevice, s));
  kGroupStarts<<<gridFor(n + 1), kBlock, 0, s>>>(T.key.as<uint64_t>(), n, (uint64_t)T.nB, T.nA,
                                                  T.aStart.as<int64_t>(), T.val.as<uint32_t>(),
                                                  T.beta.as<uint64_t>(), T.aSortB.as<uint64_t>());
  // Bitmaps of the groups that hold a 32nd of the beta strings and at least
  // 512 (so at most 8 bytes of them per determinant): a lookup there is one
  // load instead of a binary search of 10 to 16 dependent ones, which took
  // half of the enumeration (7,700 steps a row beside 11,500 scanned members
  // on 400,009 determinants of 24 orbitals).
  {
    const int64_t thr = std::max<int64_t>(512, (T.nB + 31) / 32), words = (T.nB + 63) / 64;
    const size_t bytes = (size_t)(n / thr + 1) * words * 16;
    T.bmWords = words;
    T.bmFlag.reserve((size_t)(T.nA + 1) * 8);
    T.bmSlot.reserve((size_t)std::max<int64_t>(T.nA, 1) * 4);
    T.bm.reserve(bytes);
    HIP_CHECK(hipMemsetAsync(T.bm.p, 0, bytes, s));
    kBitmapFlags<<<gridFor(T.nA + 1), kBlock, 0, s>>>(T.aStart.as<int64_t>(), T.nA, thr, T.bmFlag.as<int64_t>());
    exclusiveScanI64(T.bmFlag.as<int64_t>(), T.nA + 1, ws, s);
    kBitmapSet<<<gridFor(n), kBlock, 0, s>>>(T.aIdx.as<uint32_t>(), T.bIdx.as<uint32_t>(), n, T.bmFlag.as<int64_t>(),
                                             words, T.bm.as<uint4>());
    kBitmapCounts<<<gridFor(T.nA, kWaves, 1 << 14), kBlock, 0, s>>>(T.bmFlag.as<int64_t>(), T.nA, words,
                                                                    T.bmSlot.as<int32_t>(), T.bm.as<uint4>());
    HIP_CHECK(hipGetLastError());
  }
  // beta single-excitation adjacency
  {
    T.bSinglesStart.reserve((T.nB + 1) * 8);
    int64_t* bc = T.bSinglesStart.as<int64_t>();
    HIP_CHECK(hipMemsetAsync(bc + T.nB, 0, 8, s));
    kStringSingles<false><<<gridFor(T.nB), kBlock, 0, s>>>(T.sortedB.as<uint64_t>(), T.nB, norb, nullptr, bc,
                                                            nullptr);
    exclusiveScanI64(bc, T.nB + 1, ws, s);
    int64_t tb = 0;
    HIP_CHECK(hipMemcpyAsync(&tb, bc + T.nB, 8, hipMemcpyDeviceToHost, s));
    HIP_CHECK(hipStreamSynchronize(s));
    T.bSingles.reserve(std::max<int64_t>(tb, 1) * 4);
    kStringSingles<true><<<gridFor(T.nB), kBlock, 0, s>>>(T.sortedB.as<uint64_t>(), T.nB, norb, bc, nullptr,
                                                           T.bSingles.as<uint32_t>());
  }
  // alpha single-excitation adjacency
  T.aSinglesStart.reserve((T.nA + 1) * 8);
  int64_t* cnt = T.aSinglesStart.as<int64_t>();
  HIP_CHECK(hipMemsetAsync(cnt + T.nA, 0, 8, s));
  kStringSingles<false><<<gridFor(T.nA), kBlock, 0, s>>>(T.sortedA.as<uint64_t>(), T.nA, norb, nullptr, cnt,
                                                          nullptr);
  exclusiveScanI64(cnt, T.nA + 1, ws, s);
  int64_t tot = 0;
  HIP_CHECK(hipMemcpyAsync(&tot, cnt + T.nA, 8, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  T.aSingles.reserve(std::max<int64_t>(tot, 1) * 4);
  kStringSingles<true><<<gridFor(T.nA), kBlock, 0, s>>>(T.sortedA.as<uint64_t>(), T.nA, norb, cnt, nullptr,
                                                         T.aSingles.as<uint32_t>());
  HIP_CHECK(hipGetLastError());
}

static RowTables rowTables(const StringTables& T) {
  RowTables r;
  r.alpha = T.alpha.as<uint64_t>();
  r.beta = T.beta.as<uint64_t>();
  r.aIdx = T.aIdx.as<uint32_t>();
  r.bIdx = T.bIdx.as<uint32_t>();
  r.aStart = T.aStart.as<int64_t>();
  r.bStart = T.bStart.as<int64_t>();
  r.aMajorDet = T.aMajorDet.as<uint32_t>();
  r.bMajorDet = T.bMajorDet.as<uint32_t>();
  r.aMajorB = T.aMajorB.as<uint64_t>();
  r.bMajorA = T.bMajorA.as<uint64_t>();
  r.aSinglesStart = T.aSinglesStart.as<int64_t>();
  r.aSingles = T.aSingles.as<uint32_t>();
  r.bSinglesStart = T.bSinglesStart.as<int64_t>();
  r.bSingles = T.bSingles.as<uint32_t>();
  r.sortedB = T.sortedB.as<uint64_t>();
  r.aSortB = T.aSortB.as<uint64_t>();
  r.aSortDet = T.aSortDet.as<uint32_t>();
  r.n = T.n;
  r.bmSlot = T.bmSlot.as<int32_t>();
  r.bm = T.bm.as<uint4>();
  r.bmWords = T.bmWords;
  return r;
}

void launchCsrCount(const DevSystem& S, const uint64_t* dets, const StringTables& T, int64_t nOld, int64_t* rowCount,
                    hipStream_t s, bool lower) {
  if (T.n <= 0) return;
  unsigned g = gridFor(T.n, kWaves, 1 << 16);
  RowTables r = rowTables(T);
  if (lower)
    DISPATCH_W(S.W, kCsrRows<WW, false, false, true><<<g, kBlock, 0, s>>>(S, dets, r, nOld, rowCount, nullptr,
                                                                          nullptr, nullptr, nullptr, nullptr));
  else
    DISPATCH_W(S.W, kCsrRows<WW, false, false, false><<<g, kBlock, 0, s>>>(S, dets, r, nOld, rowCount, nullptr,
                                                                           nullptr, nullptr, nullptr, nullptr));
  HIP_CHECK(hipGetLastError());
}

void launchCsrFill(const DevSystem& S, const uint64_t* dets, const StringTables& T, int64_t nOld,
                   const int64_t* fillStart, int32_t* cols, double* vals, hipStream_t s, bool lower) {
  if (T.n <= 0) return;
  unsigned g = gridFor(T.n, kWaves, 1 << 16);
  RowTables r = rowTables(T);
  if (lower)
    DISPATCH_W(S.W, kCsrRows<WW, true, false, true><<<g, kBlock, 0, s>>>(S, dets, r, nOld, nullptr, fillStart, cols,
                                                                         vals, nullptr, nullptr));
  else
    DISPATCH_W(S.W, kCsrRows<WW, true, false, false><<<g, kBlock, 0, s>>>(S, dets, r, nOld, nullptr, fillStart, cols,
                                                                          vals, nullptr, nullptr));
  HIP_CHECK(hipGetLastError());
}

void launchCsrFillSplit(const DevSystem& S, const uint64_t* dets, const StringTables& T, int64_t nOld,
                        const int64_t* fillStart, int32_t* cols, float* hi, float* lo, hipStream_t s, bool lower) {
  if (T.n <= 0) return;
  unsigned g = gridFor(T.n, kWaves, 1 << 16);
  RowTables r = rowTables(T);
  if (lower)
    DISPATCH_W(S.W, kCsrRows<WW, true, true, true><<<g, kBlock, 0, s>>>(S, dets, r, nOld, nullptr, fillStart, cols,
                                                                        nullptr, hi, lo));
  else
    DISPATCH_W(S.W, kCsrRows<WW, true, true, false><<<g, kBlock, 0, s>>>(S, dets, r, nOld, nullptr, fillStart, cols,
                                                                         nullptr, hi, lo));
  HIP_CHECK(hipGetLastError());
}

void launchLowerRowPtr(const int64_t* cnt, int64_t nOld, int64_t n, int64_t* rowPtr, hipStream_t s) {
  if (n + 1 - nOld <= 0) return;
  kLowerRowPtr<<<gridFor(n + 1 - nOld), kBlock, 0, s>>>(cnt, nOld, n, rowPtr);
  HIP_CHECK(hipGetLastError());
}

void launchSigmaLowerF64(const int64_t* rowPtr, const int32_t* cols, const double* vals, const double* diag, int64_t n,
                         const double* x, double* y, int k, int64_t ld, hipStream_t s) {
  if (n <= 0 || k <= 0) return;
  kZeroVectors<<<gridFor(n * k), kBlock, 0, s>>>(y, k, ld, n);
  kSigmaLower<double, false><<<gridFor(n, kWaves), kBlock, 0, s>>>(rowPtr, cols, vals, nullptr, diag, n, x, y, k, ld);
  HIP_CHECK(hipGetLastError());
}

void launchSigmaLowerF32(const int64_t* rowPtr, const int32_t* cols, const float* vals, const float* lo,
                         const double* diag, int64_t n, const double* x, double* y, int k, int64_t ld, hipStream_t s) {
  if (n <= 0 || k <= 0) return;
  kZeroVectors<<<gridFor(n * k), kBlock, 0, s>>>(y, k, ld, n);
  if (lo)
    kSigmaLower<float, true><<<gridFor(n, kWaves), kBlock, 0, s>>>(rowPtr, cols, vals, lo, diag, n, x, y, k, ld);
  else
    kSigmaLower<float, false><<<gridFor(n, kWaves), kBlock, 0, s>>>(rowPtr, cols, vals, nullptr, diag, n, x, y, k,
                                                                    ld);
  HIP_CHECK(hipGetLastError());
}

void launchSigmaDirect(const DevSystem& S, const uint64_t* dets, const StringTables& T, const double* diag,
                       const double* x, double* y, int k, int64_t ld, hipStream_t s) {
  if (T.n <= 0 || k <= 0) return;
  unsigned g = gridFor(T.n, kWaves, 1 << 16);
  RowTables r = rowTables(T);
  for (int c0 = 0; c0 < k; c0 += 8) {
    const int kk = std::min(8, k - c0);
    DISPATCH_W(S.W, kSigmaDirect<WW><<<g, kBlock, 0, s>>>(S, dets, r, diag, x + (int64_t)c0 * ld,
                                                             y + (int64_t)c0 * ld, kk, ld));
  }
  HIP_CHECK(hipGetLastError());
}

void launchNewRowLengths(const int64_t* oldRowPtr, int64_t nOld, int64_t n, int64_t* cnt, hipStream_t s) {
  if (nOld <= 0) return;
  kNewRowLengths<<<gridFor(n), kBlock, 0, s>>>(oldRowPtr, nOld, n, cnt);
  HIP_CHECK(hipGetLastError());
}

void launchFillStart(const int64_t* oldRowPtr, int64_t nOld, int64_t n, const int64_t* rowPtr, int64_t* fs,
                     hipStream_t s) {
  kFillStart<<<gridFor(n), kBlock, 0, s>>>(oldRowPtr, nOld, n, rowPtr, fs);
  HIP_CHECK(hipGetLastError());
}

void launchCopyOldRowsF64(const int64_t* oldRowPtr, const int32_t* oldCols, const double* oldVals, int64_t nOld,
                          const int64_t* rowPtr, int32_t* cols, double* vals, hipStream_t s) {
  if (nOld <= 0) return;
  kCopyOldRows<double><<<gridFor(nOld, kWaves, 1 << 16), kBlock, 0, s>>>(oldRowPtr, oldCols, oldVals, nullptr, nOld,
                                                                          rowPtr, cols, vals, nullptr);
  HIP_CHECK(hipGetLastError());
}

void launchCopyOldRowsF32(const int64_t* oldRowPtr, const int32_t* oldCols, const float* oldHi, const float* oldLo,
                          int64_t nOld, const int64_t* rowPtr, int32_t* cols, float* hi, float* lo, hipStream_t s) {
  if (nOld <= 0) return;
  kCopyOldRows<float><<<gridFor(nOld, kWaves, 1 << 16), kBlock, 0, s>>>(oldRowPtr, oldCols, oldHi, oldLo, nOld, rowPtr,
                                                                         cols, hi, lo);
  HIP_CHECK(hipGetLastError());
}

void launchCastValues(const double* v, float* out, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  kCast<<<gridFor(n), kBlock, 0, s>>>(v, out, n);
  HIP_CHECK(hipGetLastError());
}

void launchSortRows(const int64_t* rowPtr, int64_t n, int32_t* cols, double* vals, hipStream_t s) {
  if (n <= 0) return;
  kSortRows<<<gridFor(n, 64), 64, 0, s>>>(rowPtr, n, cols, vals);
  HIP_CHECK(hipGetLastError());
}

template <typename VT, bool LO>
static void launchSigmaT(const int64_t* rowPtr, const int32_t* cols, const VT* vals, const float* lo,
                         const double* diag, int64_t n, const double* x, double* y, int k, int64_t ld, hipStream_t s) {
  if (n <= 0) return;
  const int64_t blocks = std::min<int64_t>((n + kWaves - 1) / kWaves, 1 << 15);
  kSigma<VT, LO><<<(unsigned)blocks, kBlock, 0, s>>>(rowPtr, cols, vals, lo, diag, n, x, y, k, ld);
  HIP_CHECK(hipGetLastError());
}

void launchSigmaF64(const int64_t* rowPtr, const int32_t* cols, const double* vals, const double* diag, int64_t n,
                    const double* x, double* y, int k, int64_t ld, hipStream_t s) {
  launchSigmaT<double, false>(rowPtr, cols, vals, nullptr, diag, n, x, y, k, ld, s);
}

void launchSigmaF32(const int64_t* rowPtr, const int32_t* cols, const float* vals, const float* lo,
                    const double* diag, int64_t n, const double* x, double* y, int k, int64_t ld, hipStream_t s) {
  if (lo)
    launchSigmaT<float, true>(rowPtr, cols, vals, lo, diag, n, x, y, k, ld, s);
  else
    launchSigmaT<float, false>(rowPtr, cols, vals, nullptr, diag, n, x, y, k, ld, s);
}

__global__ void kSplitHiLo(const double* v, float* hi, float* lo, int64_t n) {
  for (int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (int64_t)gridDim.x * blockDim.x) {
    const double d = v[i];
    const float h = (float)d;
    hi[i] = h;
    lo[i] = (float)(d - (double)h);
  }
}

void launchSplitHiLo(const double* v, float* hi, float* lo, int64_t n, hipStream_t s) {
  if (n <= 0) return;
  kSplitHiLo<<<gridFor(n), kBlock, 0, s>>>(v, hi, lo, n);
  HIP_CHECK(hipGetLastError());
}

void launchInversePerm(const uint32_t* perm, int64_t n, uint32_t* pos, hipStream_t s) {
  if (n <= 0) return;
  kInversePerm<<<gridFor(n), kBlock, 0, s>>>(perm, n, pos);
  HIP_CHECK(hipGetLastError());
}

void launchPermRowLengths(const int64_t* rowPtr, const uint32_t* perm, int64_t n, int64_t* len, hipStream_t s) {
  if (n <= 0) return;
  kPermRowLengths<<<gridFor(n), kBlock, 0, s>>>(rowPtr, perm, n, len);
  HIP_CHECK(hipGetLastError());
}

void launchPermRowsF64(const int64_t* rowPtr, const int32_t* cols, const double* vals, const uint32_t* perm,
                       const uint32_t* pos, const uint32_t* bIdx, const uint32_t* bPos, int64_t n,
                       const int64_t* rpP, int32_t* colsP, double* valsP, hipStream_t s) {
  if (n <= 0) return;
  if (bIdx && 2 * n > 0x7fffffffLL) throw HipError("too many rows for the split relabelled columns");
  kPermRows<double><<<gridFor(n, kWaves, 1 << 16), kBlock, 0, s>>>(rowPtr, cols, vals, perm, pos, bIdx, bPos, n, rpP,
                                                                     colsP, valsP);
  HIP_CHECK(hipGetLastError());
}

void launchPermRowsF32(const int64_t* rowPtr, const int32_t* cols, const float* vals, const uint32_t* perm,
                       const uint32_t* pos, const uint32_t* bIdx, const uint32_t* bPos, int64_t n,
                       const int64_t* rpP, int32_t* colsP, float* valsP, hipStream_t s) {
  if (n <= 0) return;
  if (bIdx && 2 * n > 0x7fffffffLL) throw HipError("too many rows for the split relabelled columns");
  kPermRows<float><<<gridFor(n, kWaves, 1 << 16), kBlock, 0, s>>>(rowPtr, cols, vals, perm, pos, bIdx, bPos, n, rpP,
                                                                    colsP, valsP);
  HIP_CHECK(hipGetLastError());
}

void* XScratch::get(size_t bytes) const {
  if (mem) {
    mem->reserve(bytes);
    return mem->p;
  }
  if (bytes > fixedBytes)
    throw HipError("sigma needs " + std::to_string(bytes) + " bytes of x scratch, more than the fixed " +
                   std::to_string(fixedBytes));
  return fixed;
}

size_t sigmaPermScratchBytes(int64_t n, bool split, int k, size_t xBytes) {
  const int K = k <= 1 ? 1 : k == 2 ? 2 : k <= 4 ? 4 : 8;
  return (size_t)(split ? 2 * n : n) * K * xBytes;
}

// Fixed scratch of the allocation-free sigma: 256 bytes of work counters,
// then up to 64 MiB of permuted x (one FP64 vector of up to 4,194,304
// determinants with split columns, or n * vectors per pass up to that).
// Each GPU holds its own copy for the life of the process.
constexpr size_t kFixedScratchBytes = ((size_t)64 << 20) + 256;
static __device__ __align__(256) unsigned char scratch[kFixedScratchBytes];

void* fixedSigmaScratch(size_t* bytes) {
  static std::mutex mu;
  static void* addr[64] = {};
  int dev = 0;
  HIP_CHECK(hipGetDevice(&dev));
  if (dev < 0 || dev >= 64) throw HipError("device index out of range for the fixed sigma scratch");
  std::lock_guard<std::mutex> lock(mu);
  if (!addr[dev]) {
    void* p = nullptr;
    HIP_CHECK(hipGetSymbolAddress(&p, HIP_SYMBOL(scratch)));
    if (!p) throw HipError("hipGetSymbolAddress returned no address for the fixed sigma scratch");
    addr[dev] = p;
  }
  if (bytes) *bytes = kFixedScratchBytes;
  return addr[dev];
}

template <typename VT, typename XT, int CHUNK, bool PERSIST>
static void sigmaPermChunk(const int64_t* rp, const int32_t* cols, const VT* vals, const double* diag,
                           const uint32_t* perm, const uint32_t* bPerm, int64_t n, const double* x, double* y, int k,
                           int64_t ld, const XScratch& xP, unsigned* counter, hipStream_t s) {
  const int64_t nx = bPerm ? 2 * n : n;
  const int64_t chunks = (n + CHUNK - 1) / CHUNK;
  if (chunks > 0x7fffffffLL) throw HipError("too many rows for the relabelled sigma");
  unsigned grid = (unsigned)chunks;
  if (PERSIST) grid = (unsigned)std::min<int64_t>(chunks, (int64_t)computeUnits() * 8);
  for (int c0 = 0; c0 < k;) {
    const int kk = k - c0;
    const double* xc = x + (int64_t)c0 * ld;
    double* yc = y + (int64_t)c0 * ld;
    auto spmm = [&](auto KT) {
      constexpr int K = decltype(KT)::value;
      const int take = kk < K ? kk : K;
      XT* xs = (XT*)xP.get((size_t)nx * K * sizeof(XT));
      kGatherPerm<XT, K><<<gridFor(nx), kBlock, 0, s>>>(xc, take, ld, perm, bPerm, n, xs, counter);
      kSpmmPerm<VT, XT, K, CHUNK, PERSIST><<<grid, kBlock, 0, s>>>(rp, cols, vals, diag, perm, n, xs, xc, yc, take,
                                                                     ld, counter);
      return take;
    };
    if (kk == 1) {
      XT* xs = (XT*)xP.get((size_t)nx * sizeof(XT));
      kGatherPerm<XT, 1><<<gridFor(nx), kBlock, 0, s>>>(xc, 1, ld, perm, bPerm, n, xs, counter);
      kSigmaPerm<VT, XT, CHUNK, PERSIST><<<grid, kBlock, 0, s>>>(rp, cols, vals, diag, perm, n, xs, nx, xc, yc, 1,
                                                                   ld, counter);
      c0 += 1;
    } else if (kk == 2) {
      c0 += spmm(std::integral_constant<int, 2>());
    } else if (kk <= 4) {
      c0 += spmm(std::integral_constant<int, 4>());
    } else {
      c0 += spmm(std::integral_constant<int, 8>());
    }
    HIP_CHECK(hipGetLastError());
  }
}

template <typename VT, typename XT>
static void launchSigmaPermT(const int64_t* rp, const int32_t* cols, const VT* vals, const double* diag,
                             const uint32_t* perm, const uint32_t* bPerm, int64_t n, const double* x, double* y, int k, int64_t ld,
                             const XScratch& xP, const SigmaConfig& cfg, unsigned* counter, hipStream_t s) {
  if (n <= 0 || k <= 0) return;
  if (cfg.persistent && !counter) throw HipError("persistent sigma needs a work counter");
  switch (cfg.chunk * 2 + (cfg.persistent ? 1 : 0)) {
    case 8: sigmaPermChunk<VT, XT, 4, false>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, counter, s); break;
    case 9: sigmaPermChunk<VT, XT, 4, true>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, counter, s); break;
    case 16: sigmaPermChunk<VT, XT, 8, false>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, counter, s); break;
    case 17: sigmaPermChunk<VT, XT, 8, true>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, counter, s); break;
    case 32: sigmaPermChunk<VT, XT, 16, false>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, counter, s); break;
    case 33: sigmaPermChunk<VT, XT, 16, true>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, counter, s); break;
    case 64: sigmaPermChunk<VT, XT, 32, false>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, counter, s); break;
    case 65: sigmaPermChunk<VT, XT, 32, true>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, counter, s); break;
    default: throw HipError("unsupported sigma configuration");
  }
}

void launchSigmaPermF64(const int64_t* rp, const int32_t* cols, const double* vals, const double* diag,
                        const uint32_t* perm, const uint32_t* bPerm, int64_t n, const double* x, double* y, int k,
                        int64_t ld, const XScratch& xP, const SigmaConfig& cfg, unsigned* counter, hipStream_t s) {
  launchSigmaPermT<double, double>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, cfg, counter, s);
}

void launchSigmaPermF32(const int64_t* rp, const int32_t* cols, const float* vals, const double* diag,
                        const uint32_t* perm, const uint32_t* bPerm, int64_t n, const double* x, double* y, int k,
                        int64_t ld, const XScratch& xP, const SigmaConfig& cfg, unsigned* counter, hipStream_t s) {
  launchSigmaPermT<float, float>(rp, cols, vals, diag, perm, bPerm, n, x, y, k, ld, xP, cfg, counter, s);
}

void TiledHam::release() {
  for (DevMem* m : tables()) m->release();
  n = -1;
  hasLo = false;
}

// With half storage only the next build would want them, and it begins by
// releasing the copy; with full storage it fills the segment tables again, so
// they stay, but not the bitmaps, whose size is quadratic in n.
void TiledHam::releaseBuildTables(bool sym) {
  tileBits.release();
  if (!sym) return;
  for (DevMem* m : {&segBase, &segTile, &segCnt, &segStart, &segInst, &segTotal, &fill, &blockI, &inst, &order, &blockOf,
                    &bigI, &smallI, &lead, &unitStart})
    m->release();
}

size_t TiledHam::heldBytes() {
  size_t b = 0;
  for (DevMem* m : tables()) b += m->bytes;
  return b;
}

// the half-storage sigma's order of a tiled copy and its work units
static void buildSymOrder(TiledHam& T, int bigMin, Workspace& ws, hipStream_t s);

size_t tiledHamBytes(int64_t n, int64_t nnz, bool f32, bool sym) {
  const int64_t blocks = (n + kTileRows - 1) / kTileRows;
  // entries, one instruction per 32 entries at most on average plus one per
  // segment, segment tables (48 bytes) with at most one segment per 64
  // entries or per block, and the bitmaps of the blocks' tiles; sym: the
  // instructions once more and 40 bytes per segment, in its own order
  const int64_t segs = nnz / 64 + blocks;
  const size_t bitmap = (size_t)((2 * n + kTileCols - 1) / kTileCols + 31) / 32 * 4;
  return (size_t)nnz * (4 + (f32 ? 4 : 8)) + (size_t)(nnz / 32 + segs) * (sym ? 16 : 8) +
         (size_t)segs * (sym ? 88 : 48) + (size_t)(blocks + 1) * ((sym ? 40 : 24) + bitmap);
}

bool buildTiledHam(TiledHam& T, const int64_t* rowPtr, const int32_t* cols, const double* vals64,
                   const float* vals32, const uint32_t* perm, const uint32_t* pos, const uint32_t* bIdx,
                   const uint32_t* bPos, int64_t n, int64_t nnz, Workspace& ws, hipStream_t s, bool splitCols,
                   int stageMin, const float* valsLo, bool sym) {
  T.n = -1;
  T.hasLo = false;
  if (n <= 0) return false;
  const bool split = pos ? bIdx != nullptr : splitCols;
  const int64_t nx = split ? 2 * n : n;
  const int64_t tiles = (nx + kTileCols - 1) / kTileCols;
  const int nwords = (int)((tiles + 31) / 32);
  if (nwords > kTileMaxWords) return false;
  const int64_t blocks = (n + kTileRows - 1) / kTileRows;
  if (blocks > 0x7fffffffLL) return false;
  const unsigned grid = (unsigned)blocks;
  T.segBase.reserve((size_t)(blocks + 1) * 8);
  int64_t* segBase = T.segBase.as<int64_t>();
  HIP_CHECK(hipMemsetAsync(segBase + blocks, 0, 8, s));
  T.tileBits.reserve((size_t)blocks * nwords * 4);
  uint32_t* tileBits = T.tileBits.as<uint32_t>();
  const size_t ldsBits = (size_t)nwords * 4;
  kTileMark<<<grid, kBlock, ldsBits, s>>>(rowPtr, cols, perm, pos, bIdx, bPos, n, nwords, segBase, tileBits);
  HIP_CHECK(hipGetLastError());
  exclusiveScanI64(segBase, blocks + 1, ws, s);
  int64_t S = 0;
  HIP_CHECK(hipMemcpyAsync(&S, segBase + blocks, 8, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  const size_t sb = (size_t)std::max<int64_t>(S, 1);
  T.segTile.reserve(sb * 4);
  T.segCnt.reserve(sb * 16);
  T.segStart.reserve(sb * 4);
  T.segInst.reserve(sb * 4);
  T.segTotal.reserve(sb * 4);
  T.fill.reserve(sb * 16);
  T.blockE.reserve((size_t)(blocks + 1) * 8);
  T.blockI.reserve((size_t)(blocks + 1) * 8);
  HIP_CHECK(hipMemsetAsync(T.segCnt.p, 0, sb * 16, s));
  int64_t* blockE = T.blockE.as<int64_t>();
  int64_t* blockI = T.blockI.as<int64_t>();
  HIP_CHECK(hipMemsetAsync(blockE + blocks, 0, 8, s));
  HIP_CHECK(hipMemsetAsync(blockI + blocks, 0, 8, s));
  kTileCount<<<grid, kBlock, 2 * ldsBits, s>>>(
      rowPtr, cols, perm, pos, bIdx, bPos, n, nwords, tileBits, segBase, T.segTile.as<uint32_t>(),
      T.segCnt.as<uint32_t>(), T.segStart.as<uint32_t>(), T.segInst.as<uint32_t>(), T.segTotal.as<uint32_t>(),
      T.fill.as<uint32_t>(), blockE, blockI);
  HIP_CHECK(hipGetLastError());
  exclusiveScanI64(blockE, blocks + 1, ws, s);
  exclusiveScanI64(blockI, blocks + 1, ws, s);
  int64_t E = 0, I = 0;
  HIP_CHECK(hipMemcpyAsync(&E, blockE + blocks, 8, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipMemcpyAsync(&I, blockI + blocks, 8, hipMemcpyDeviceToHost, s));
  HIP_CHECK(hipStreamSynchronize(s));
  if (E != nnz) throw HipError("tiled Hamiltonian: entry count " + std::to_string(E) + " != " + std::to_string(nnz));
  const bool f32 = vals64 == nullptr;
  T.idx.reserve((size_t)std::max<int64_t>(E, 1) * 4);
  T.vals.reserve((size_t)std::max<int64_t>(E, 1) * (f32 ? 4 : 8));
  const bool withLo = f32 && valsLo;
  if (withLo) T.lo.reserve((size_t)std::max<int64_t>(E, 1) * 4);
  // kSigmaTiled reads up to kTileInstPad descriptors past a block's last
  // one: zero padding after the last block (count 0, tile 0)
  T.inst.reserve((size_t)(I + kTileInstPad) * 8);
  HIP_CHECK(hipMemsetAsync(T.inst.as<uint2>() + I, 0, (size_t)kTileInstPad * 8, s));
  if (f32)
    kTileFill<float><<<grid, kBlock, 2 * ldsBits, s>>>(
        rowPtr, cols, vals32, perm, pos, bIdx, bPos, n, nwords, tileBits, segBase, T.segTile.as<uint32_t>(),
        T.segStart.as<uint32_t>(), T.segInst.as<uint32_t>(), T.segTotal.as<uint32_t>(), T.fill.as<uint32_t>(), blockE,
        blockI, T.idx.as<uint32_t>(), T.vals.as<float>(), T.inst.as<uint2>(), stageMin, withLo ? valsLo : nullptr,
        withLo ? T.lo.as<float>() : nullptr);
  else
    kTileFill<double><<<grid, kBlock, 2 * ldsBits, s>>>(
        rowPtr, cols, vals64, perm, pos, bIdx, bPos, n, nwords, tileBits, segBase, T.segTile.as<uint32_t>(),
        T.segStart.as<uint32_t>(), T.segInst.as<uint32_t>(), T.segTotal.as<uint32_t>(), T.fill.as<uint32_t>(), blockE,
        blockI, T.idx.as<uint32_t>(), T.vals.as<double>(), T.inst.as<uint2>(), stageMin, nullptr, nullptr);
  HIP_CHECK(hipGetLastError());
  kTileRunBits<<<grid, kBlock, 0, s>>>(T.inst.as<uint2>(), blockI, blockE, T.idx.as<uint32_t>());
  HIP_CHECK(hipGetLastError());
  T.n = n;
  T.blocks = blocks;
  T.segments = S;
  T.nnz = E;
  T.instructions = I;
  T.f32 = f32;
  T.split = split;
  T.hasLo = withLo;
  if (sym) buildSymOrder(T, stageMin, ws, s);
  return true;
}

template <typename VT, typename XT, bool PERSIST, bool STAGE>
static void sigmaTiledS(int step, unsigned grid, const TiledHam& T, const double* diag, const uint32_t* perm,
                        int64_t n, const XT* xs, int64_t nx, const double* x, double* y, unsigned* counter,
                        hipStream_t s) {
  if (step >= 16)
    kSigmaTiled<VT, XT, PERSIST, 16, STAGE><<<grid, kBlock, 0, s>>>(
        T.inst.as<uint2>(), T.blockI.as<int64_t>(), T.blockE.as<int64_t>(), T.idx.as<uint32_t>(), T.vals.as<VT>(),
        diag, perm, n, T.blocks, xs, nx, x, y, counter);
  else
    kSigmaTiled<VT, XT, PERSIST, 8, STAGE><<<grid, kBlock, 0, s>>>(
        T.inst.as<uint2>(), T.blockI.as<int64_t>(), T.blockE.as<int64_t>(), T.idx.as<uint32_t>(), T.vals.as<VT>(),
        diag, perm, n, T.blocks, xs, nx, x, y, counter);
}

template <typename VT, typename XT, bool PERSIST>
static void sigmaTiledU(int step, bool stage, unsigned grid, const TiledHam& T, const double* diag,
                        const uint32_t* perm, int64_t n, const XT* xs, int64_t nx, const double* x, double* y,
                        unsigned* counter, hipStream_t s) {
  if (stage)
    sigmaTiledS<VT, XT, PERSIST, true>(step, grid, T, diag, perm, n, xs, nx, x, y, counter, s);
  else
    sigmaTiledS<VT, XT, PERSIST, false>(step, grid, T, diag, perm, n, xs, nx, x, y, counter, s);
}

void launchSigmaTiled(const TiledHam& T, const double* diag, const uint32_t* perm, const uint32_t* bPerm,
                      const double* x, double* y, const XScratch& xP, bool persistent, unsigned* counter,
                      hipStream_t s, int step, bool stage) {
  const int64_t n = T.n;
  if (n <= 0) return;
  if (T.split != (bPerm != nullptr)) throw HipError("tiled sigma: split columns need the beta-major order");
  const int64_t nx = bPerm ? 2 * n : n;
  const unsigned grid =
      (unsigned)(persistent ? std::min<int64_t>(T.blocks, (int64_t)computeUnits() * 8) : T.blocks);
  if (persistent && !counter) throw HipError("persistent sigma needs a work counter");
  if (T.f32) {
    float* xs = (float*)xP.get((size_t)nx * 4);
    kGatherPerm<float, 1><<<gridFor(nx), kBlock, 0, s>>>(x, 1, n, perm, bPerm, n, xs, counter);
    if (persistent)
      sigmaTiledU<float, float, true>(step, stage, grid, T, diag, perm, n, xs, nx, x, y, counter, s);
    else
      sigmaTiledU<float, float, false>(step, stage, grid, T, diag, perm, n, xs, nx, x, y, counter, s);
  } else {
    double* xs = (double*)xP.get((size_t)nx * 8);
    kGatherPerm<double, 1><<<gridFor(nx), kBlock, 0, s>>>(x, 1, n, perm, bPerm, n, xs, counter);
    if (persistent)
      sigmaTiledU<double, double, true>(step, stage, grid, T, diag, perm, n, xs, nx, x, y, counter, s);
    else
      sigmaTiledU<double, double, false>(step, stage, grid, T, diag, perm, n, xs, nx, x, y, counter, s);
  }
  HIP_CHECK(hipGetLastError());
}

// the half-storage sigma's order of a tiled copy and its work units
static void buildSymOrder(TiledHam& T, int bigMin, Workspace& ws, hipStream_t s) {
  const int64_t S = T.segments, supers = (T.blocks + kSymBlocks - 1) / kSymBlocks;
  if (T.instructions >= 0xffffffffLL) throw HipError("tiled Hamiltonian: too many instructions");
  T.order.reserve((size_t)std::max<int64_t>(S, 1) * 4);
  T.blockOf.reserve((size_t)std::max<int64_t>(S, 1) * 4);
  for (DevMem* m : {&T.bigI, &T.smallI, &T.lead}) {
    m->reserve((size_t)(S + 1) * 8);
    HIP_CHECK(hipMemsetAsync(m->as<int64_t>() + S, 0, 8, s));
  }
  T.groups.reserve((size_t)(S + 1) * 8);
  T.symInst.reserve((size_t)std::max<int64_t>(T.instructions, 1) * 8);
  T.unitStart.reserve((size_t)(supers + 1) * 8);
  const int64_t* segBase = T.segBase.as<int64_t>();
  kSymRank<<<gridFor(S), kBlock, 0, s>>>(segBase, T.blocks, S, T.segTile.as<uint32_t>(), T.segTotal.as<uint32_t>(),
                                         (uint32_t)bigMin, T.order.as<uint32_t>(), T.blockOf.as<uint32_t>(),
                                         T.bigI.as<int64_t>(), T.smallI.as<int64_t>(), T.lead.as<int64_t>());
  HIP_CHECK(hipGetLastError());
  for (DevMem* m : {&T.bigI, &T.smallI, &T.lead}) exclusiveScanI64(m->as<int64_t>(), S + 1, ws, s);
  kSymEmit<<<gridFor(S), kBlock, 0, s>>>(S, T.order.as<uint32_t>(), T.blockOf.as<uint32_t>(), T.blockE.as<int64_t>(),
                                         T.segTile.as<uint32_t>(), T.segTotal.as<uint32_t>(),
                                         T.segStart.as<uint32_t>(), T.bigI.as<int64_t>(), T.smallI.as<int64_t>(),
                                         T.lead.as<int64_t>(), T.symInst.as<uint2>(), T.groups.as<uint2>());
  HIP_CHECK(hipGetLastError());
  // Units of I / (8 CUs) instructions: two workgroups for each of the four
  // that a CU holds, between 64 (two steps for each wave) and 1,024; 57,963
  // determinants of 40 orbitals: 89 us in the 190 this gives, 95 in units of
  // 512, 128 of 1,024; 1,000,003 of 24 orbitals: 1,790 us in units of 256,
  // 1,711 of 512, 1,713 of 1,024, 1,701 of 2,048.
  const int64_t per = std::min<int64_t>(1024, std::max<int64_t>(64, T.instructions / ((int64_t)computeUnits() * 8)));
  T.unitCap = 2 * supers + T.instructions / per;
  T.units.reserve((size_t)T.unitCap * sizeof(SymUnit));
  kSymUnits<<<gridFor(supers), kBlock, 0, s>>>(segBase, T.blocks, supers, S, T.bigI.as<int64_t>(),
                                               T.smallI.as<int64_t>(), T.lead.as<int64_t>(), T.groups.as<uint2>(),
                                               per, T.unitStart.as<int64_t>(), nullptr, 0);
  exclusiveScanI64(T.unitStart.as<int64_t>(), supers + 1, ws, s);
  kSymUnits<<<gridFor(supers), kBlock, 0, s>>>(segBase, T.blocks, supers, S, T.bigI.as<int64_t>(),
                                               T.smallI.as<int64_t>(), T.lead.as<int64_t>(), T.groups.as<uint2>(),
                                               per, T.unitStart.as<int64_t>(), T.units.as<SymUnit>(), T.unitCap);
  HIP_CHECK(hipGetLastError());
}

template <typename VT, typename XT, bool LO, bool ABS>
static void runSymTiles(const TiledHam& T, int64_t nx, const XT* xs, unsigned long long* yT,
                        const unsigned long long* bound, hipStream_t s) {
  kSigmaTiledSym<VT, XT, LO, ABS><<<(unsigned)T.unitCap, kSymThreads, 0, s>>>(
      T.units.as<SymUnit>(), T.symInst.as<uint2>(), T.groups.as<uint2>(), T.blockE.as<int64_t>(),
      T.idx.as<uint32_t>(), T.vals.as<VT>(), LO ? T.lo.as<float>() : nullptr, T.n, nx, xs, yT, bound);
}

void launchSigmaTiledSym(const TiledHam& T, const double* diag, const uint32_t* perm, const uint32_t* bPerm,
                         const uint32_t* pos, const uint32_t* bPos, const double* x, double* y, const XScratch& xP,
                         unsigned long long* yT, const unsigned long long* bound, hipStream_t s, bool exact) {
  const int64_t n = T.n;
  if (n <= 0) return;
  if (T.split != (bPerm != nullptr) || T.split != (bPos != nullptr))
    throw HipError("tiled sigma: split columns need the beta-major order");
  if (exact && T.f32 && !T.hasLo) throw HipError("tiled sigma: the exact FP32 form needs the lo values");
  const int64_t nx = bPerm ? 2 * n : n;
  kFillZeroU64<<<gridFor(nx + 1), kBlock, 0, s>>>(yT, nx + 1);
  if (T.f32 && !exact) {
    float* xs = (float*)xP.get((size_t)nx * 4);
    kGatherPermMax<float><<<gridFor(nx, kBlock, 1024), kBlock, 0, s>>>(x, perm, bPerm, n, xs, yT + nx);
    runSymTiles<float, float, false, false>(T, nx, xs, yT, bound, s);
  } else {
    double* xs = (double*)xP.get((size_t)nx * 8);
    kGatherPermMax<double><<<gridFor(nx, kBlock, 1024), kBlock, 0, s>>>(x, perm, bPerm, n, xs, yT + nx);
    if (T.f32)  // the exact FP32 form: hi + lo values, x in FP64
      runSymTiles<float, double, true, false>(T, nx, xs, yT, bound, s);
    else
      runSymTiles<double, double, false, false>(T, nx, xs, yT, bound, s);
  }
  kSymFinish<<<gridFor(n), kBlock, 0, s>>>(diag, x, y, yT, bound, pos, bPos, n, nx);
  HIP_CHECK(hipGetLastError());
}

void launchSymRowBound(const TiledHam& T, const uint32_t* pos, const uint32_t* bPos, unsigned long long* yT,
                       unsigned long long* bound, hipStream_t s) {
  const int64_t n = T.n, nx = bPos ? 2 * n : n;
  if (n <= 0) return;
  kFillZeroU64<<<gridFor(nx), kBlock, 0, s>>>(yT, nx);
  kFillZeroU64<<<1, 64, 0, s>>>(bound, 1);
  if (T.f32)
    runSymTiles<float, float, false, true>(T, nx, nullptr, yT, nullptr, s);
  else
    runSymTiles<double, double, false, true>(T, nx, nullptr, yT, nullptr, s);
  kMaxU64<<<gridFor(n, kBlock, 1024), kBlock, 0, s>>>(yT, pos, bPos, n, bound);
  kU64ScaledToDouble<<<1, 64, 0, s>>>(bound);
  HIP_CHECK(hipGetLastError());
}

void launchDot(const double* a, const double* b, int64_t n, double* out, DevMem& partial, hipStream_t s) {
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(kRedBlocks, (n + kBlock - 1) / kBlock));
  partial.reserve((size_t)nb * sizeof(double));
  kDot<<<nb, kBlock, 0, s>>>(a, b, n, partial.as<double>());
  kFinalSum<<<1, kBlock, 0, s>>>(partial.as<double>(), nb, 1, 1, out);
  HIP_CHECK(hipGetLastError());
}

void launchGramTiled(const double* A, int ma, const double* B, int mb, int64_t n, int64_t ld, bool upper,
                     double* G, DevMem& partial, hipStream_t s) {
  if (ma > 64 || mb > 64 || (upper && ma != mb)) throw HipError("launchGramTiled: bad block");
  if (ma <= 0 || mb <= 0) return;
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(kRedBlocks / 2, (n + kBlock - 1) / kBlock));
  const int tiles = ((ma + 7) / 8) * ((mb + 7) / 8);
  partial.reserve((size_t)tiles * nb * 64 * sizeof(double));
  kGramTile<<<dim3(nb, tiles), kBlock, 0, s>>>(A, ma, B, mb, n, ld, upper, partial.as<double>());
  kGramTileFinal<<<ma * mb, kBlock, 0, s>>>(partial.as<double>(), nb, ma, mb, upper, G);
  HIP_CHECK(hipGetLastError());
}

void launchGemmTS(const double* A, int ma, const double* W, int mb, int64_t n, int64_t lda, double* out,
                  int64_t ldo, double alpha, double beta, hipStream_t s) {
  if (ma > 64 || mb > 64) throw HipError("launchGemmTS: block too large");
  if (n <= 0 || mb <= 0) return;
  kGemmTS<<<dim3(gridFor(n, kBlock, 4096), (mb + 7) / 8), kBlock, 0, s>>>(A, ma, W, mb, n, lda, out, ldo, alpha, beta);
  HIP_CHECK(hipGetLastError());
}

__global__ void kSubMatrix(const double* C, int ldc, int rows, int cols, double* out) {
  for (int q = threadIdx.x; q < rows * cols; q += blockDim.x) out[q] = C[(q / cols) * ldc + q % cols];
}

void launchSubMatrix(const double* C, int ldc, int rows, int cols, double* out, hipStream_t s) {
  if (rows <= 0 || cols <= 0) return;
  kSubMatrix<<<1, kBlock, 0, s>>>(C, ldc, rows, cols, out);
  HIP_CHECK(hipGetLastError());
}

void launchResidual(const double* sig, const double* b, const double* e, int64_t n, double* r, double* out,
                    DevMem& partial, hipStream_t s) {
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(kRedBlocks, (n + kBlock - 1) / kBlock));
  partial.reserve((size_t)nb * sizeof(double));
  kResidual<<<nb, kBlock, 0, s>>>(sig, b, e, n, r, partial.as<double>());
  kFinalSum<<<1, kBlock, 0, s>>>(partial.as<double>(), nb, 1, 1, out);
  HIP_CHECK(hipGetLastError());
}

void launchPrecondition(double* r, const double* diag, const double* e, int64_t n, hipStream_t s) {
  kPrecondition<<<gridFor(n, kBlock, 8192), kBlock, 0, s>>>(r, diag, e, n);
  HIP_CHECK(hipGetLastError());
}

void launchDot2(const double* b, const double* r, int64_t n, double* out, DevMem& partial, hipStream_t s) {
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(kRedBlocks, (n + kBlock - 1) / kBlock));
  partial.reserve((size_t)nb * 2 * sizeof(double));
  kDot2<<<nb, kBlock, 0, s>>>(b, r, n, partial.as<double>());
  kFinalSum<<<2, kBlock, 0, s>>>(partial.as<double>(), nb, 2, 2, out);
  HIP_CHECK(hipGetLastError());
}

void launchOrthoStep(double* r, const double* b, const double* d, int64_t n, hipStream_t s) {
  kOrthoStep<<<gridFor(n, kBlock, 8192), kBlock, 0, s>>>(r, b, d, n);
  HIP_CHECK(hipGetLastError());
}

void launchNorm2(const double* x, int64_t n, double* out, DevMem& partial, hipStream_t s) {
  const int nb = (int)std::max<int64_t>(1, std::min<int64_t>(kRedBlocks, (n + kBlock - 1) / kBlock));
  partial.reserve((size_t)nb * sizeof(double));
  kNorm2<<<nb, kBlock, 0, s>>>(x, n, partial.as<double>());
  kFinalSum<<<1, kBlock, 0, s>>>(partial.as<double>(), nb, 1, 1, out);
  HIP_CHECK(hipGetLastError());
}

void launchScaleInto(double* dst, const double* src, const double* nrm2, int64_t n, hipStream_t s) {
  kScaleInto<<<gridFor(n, kBlock, 8192), kBlock, 0, s>>>(dst, src, nrm2, n);
  HIP_CHECK(hipGetLastError());
}

void launchAxpy(double* x, const double* y, double alpha, int64_t n, hipStream_t s) {
  kAxpy<<<gridFor(n, kBlock, 8192), kBlock, 0, s>>>(x, y, alpha, n);
  HIP_CHECK(hipGetLastError());
}

void launchJacobiRR(const double* A, int m, double* w, double* V, hipStream_t s) {
  if (m > kJacobiMax) throw HipError("launchJacobiRR: subspace too large");
  kJacobiRR<<<1, kBlock, 0, s>>>(A, m, w, V);
  HIP_CHECK(hipGetLastError());
}

static int redGrid(int64_t n) {
  return (int)std::max<int64_t>(1, std::min<int64_t>(kRedBlocks, (n + kBlock - 1) / kBlock));
}

void launchRayleighRitz(double* B, double* S, int m, int64_t n, double* w, double* V, int last, double* r,
                        DevMem& partial, double* host, hipStream_t s) {
  if (m < 1 || m > 12 || last < 0 || last >= m || last >= kResMax) throw HipError("launchRayleighRitz: bad subspace");
  const int nb = redGrid(n);
  partial.reserve((size_t)nb * 78 * sizeof(double));
  double* p = partial.as<double>();
#define GRAM_CASE(M) \
  case M: kGramUpper<M><<<nb, kBlock, 0, s>>>(B, S, n, n, p); break
  switch (m) {
    GRAM_CASE(1);
    GRAM_CASE(2);
    GRAM_CASE(3);
    GRAM_CASE(4);
    GRAM_CASE(5);
    GRAM_CASE(6);
    GRAM_CASE(7);
    GRAM_CASE(8);
    GRAM_CASE(9);
    GRAM_CASE(10);
    GRAM_CASE(11);
    GRAM_CASE(12);
  }
#undef GRAM_CASE
  kGramJacobi<<<1, kGramThreads, 0, s>>>(p, nb, m, w, V);
  kRotateResidual<<<nb, kBlock, 0, s>>>(B, S, m, n, n, V, w, last, r, p);
  kResidualSums<<<1, kBlock, 0, s>>>(p, nb, last + 1, w, m, host);
  HIP_CHECK(hipGetLastError());
}

void launchCorrection(double* r, const double* diag, const double* e, const double* B, int m, int64_t n, double* dst,
                      DevMem& partial, hipStream_t s) {
  const int nb = redGrid(n);
  partial.reserve((size_t)nb * 4 * sizeof(double));
  double* p[2] = {partial.as<double>(), partial.as<double>() + 2 * nb};
  kPreconditionDot<<<nb, kBlock, 0, s>>>(r, diag, e, B, n, p[0]);
  for (int i = 0; i < m; i++)
    kOrthoDot<<<nb, kBlock, 0, s>>>(r, B + (int64_t)i * n, i + 1 < m ? B + (int64_t)(i + 1) * n : nullptr, n, p[i & 1],
                                    p[(i + 1) & 1]);
  kScaleSum<<<nb, kBlock, 0, s>>>(dst, r, n, p[m & 1]);
  HIP_CHECK(hipGetLastError());
}

}  // namespace shci
