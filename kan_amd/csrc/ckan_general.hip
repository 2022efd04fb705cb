// The ChebyKAN layer for any degree, in fp32 or fp64, on the fp32 / fp64
// matrix instructions (v_mfma_f32_16x16x4_f32, v_mfma_f64_16x16x4_f64):
//   forward  y[b, o]     = sum_{i, d} P_d(t[b, i]) C[i, o, d],  t = tanh(x)
//   dx       dx[b, i]    = t'(x) sum_d G[b, i, d] P_d'(t),
//                          G[b, i, d] = sum_o dy[b, o] C[i, o, d]
//   dC       dC[i, o, d] = sum_b P_d(t[b, i]) dy[b, o]
// with P_d = T_d (the Chebyshev layers) or any basis of a three-term
// recurrence P_d = (a_d u + b_d) P_{d-1} - c_d P_{d-2} at u = s t (the Jacobi
// and Hermite layers, kan/basis/jacobi.py:131-188,
// kan/basis/hermite.py:158-233), whose coefficients come from a recurrence
// block (in fp32, the packed buffer's).  t = tanh(x), or the affine map a x + b
// of a finite-domain Hermite layer (kan/basis/hermite.py:102-112).
// It serves the fp64 layer (the reference computes in fp64 when its
// parameter is fp64: kan/layers/chebykan.py:48-51 after .double()) and fp32
// layers above the packed kernels' degree 16 (the reference layers take any
// degree, kan/layers/chebykan.py:21-51).  C is read in its own [I, O, D]
// layout; t is [B, I].
//
// How the contractions meet the 16x16x4 instruction.  Lane l holds row (or
// column) l % 16 of an operand at reduction slot g = l / 16.  Which reduction
// index a slot carries is free, so every basis value is made in the register
// of the lane that feeds it, by that lane's own recurrence, one step per
// matrix instruction:
//   forward: slot g of one instruction is input i0 + g at one degree, so lane
//     (row, g) walks the degrees of its (row, input) pair;
//   dC: the operand rows are 16 inputs and slot g is batch row b0 + g, so lane
//     (input, g) walks the degrees of its (input, row) pair, one accumulator
//     per degree;
//   dx: the result columns are 16 inputs with one accumulator per degree, so
//     each lane holds every G[b, i, d] of its own (b, i) pairs and the degree
//     sum needs no exchange.
// The basis never passes through LDS or memory, and one or two recurrence
// FMAs ride beside up to eight matrix instructions; what bounds the kernels is
// the matrix pipe (64 clk per fp64 instruction, 32 per fp32) and, at small
// sizes, how far the reduction can be split to fill it.  Against the
// vector-ALU register tiles that these kernels replaced (which put 64-128
// blocks on the chip at these sizes), forward / dx / dC:
//   2048 x 256 -> 256, degree 8, fp64:  483 / 112 / 532 -> 67 / 51 / 51 us
//   4096 x 256 -> 128, degree 24, fp32: 1013 / 191 / 1534 -> 90 / 75 / 86 us
// (36-47 TFLOP/s of products in fp64; 74-87 in fp32).
#include "ckan_kernels.hpp"

#include <math.h>

#include <atomic>
#include <type_traits>

namespace ckan {

typedef __attribute__((ext_vector_type(4))) double f64x4_t;

template <typename T> __device__ __forceinline__ T vtanh(T x);
template <> __device__ __forceinline__ float vtanh<float>(float x) { return tanhf(x); }
template <> __device__ __forceinline__ double vtanh<double>(double x) { return tanh(x); }

// t = tanh(x), or ima x + imb with the affine map.
template <typename T>
__global__ void __launch_bounds__(256)
k_tanh_v(const T* __restrict__ x, T* __restrict__ t, int64_t n, int imap, float ima, float imb) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x)
    t[q] = imap ? fma((T)ima, x[q], (T)imb) : vtanh<T>(x[q]);
}

template <typename T>
__device__ __forceinline__ T buffer_load(__amdgpu_buffer_rsrc_t rs, int voff, int soff) {
  if constexpr (sizeof(T) == 8)
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b64(rs, voff, soff, 0));
  else
    return __builtin_bit_cast(T, __builtin_amdgcn_raw_buffer_load_b32(rs, voff, soff, 0));
}

// The 16x16x4 matrix instruction of each type, and the result row of
// accumulator value v in lane group g (the column is lane % 16).
template <typename T> struct Mx;
template <> struct Mx<float> {
  typedef f32x4_t acc_t;
  static __device__ __forceinline__ acc_t mma(float a, float b, acc_t c) {
    return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int v, int g) { return 4 * g + v; }
};
template <> struct Mx<double> {
  typedef f64x4_t acc_t;
  static __device__ __forceinline__ acc_t mma(double a, double b, acc_t c) {
    return __builtin_amdgcn_mfma_f64_16x16x4f64(a, b, c, 0, 0, 0);
  }
  static __device__ __forceinline__ int row(int v, int g) { return 4 * v + g; }
};

// One basis recurrence.  Chebyshev (GEN = false): T_{d+1} = 2t T_d - T_{d-1},
// w = 2t, started from T_{-1} = t so that the first step gives 2t - t = t =
// T_1 exactly and every step is the same FMA.  GEN: P_{d+1} = (a_{d+1} w +
// b_{d+1}) P_d - c_{d+1} P_{d-1}, w = u = s t, started from P_{-1} = 0 (c_1 =
// 0); rs holds a[D], b[D], c[D], s.  A cleared recurrence stays zero.
template <typename T, bool GEN> struct Rec {
  T w, pm, pc;
  __device__ __forceinline__ void init(T t, const T* rs, int D) {
    if constexpr (GEN) {
      w = rs[3 * D] * t;
      pm = T(0);
    } else {
      w = t + t;
      pm = t;
    }
    pc = T(1);
  }
  __device__ __forceinline__ void clear() { w = pm = pc = T(0); }
  // To degree n (n past the layer's last degree reads in-range coefficients
  // whose result no caller uses).
  __device__ __forceinline__ void step(const T* rs, int D, int n) {
    T nx;
    if constexpr (GEN) {
      const int k = n < D ? n : D - 1;
      nx = fma(fma(rs[k], w, rs[D + k]), pc, -rs[2 * D + k] * pm);
    } else {
      nx = fma(w, pc, -pm);
    }
    pm = pc;
    pc = nx;
  }
  // To degree n + 1 from n - 1, in place (a rolled loop of single steps would
  // move registers as often as it computes).
  __device__ __forceinline__ void step2(const T* rs, int D, int n) {
    if constexpr (GEN) {
      pm = fma(fma(rs[n], w, rs[D + n]), pc, -rs[2 * D + n] * pm);
      pc = fma(fma(rs[n + 1], w, rs[D + n + 1]), pm, -rs[2 * D + n + 1] * pc);
    } else {
      pm = fma(w, pc, -pm);
      pc = fma(w, pm, -pc);
    }
  }
};

// The recurrence block in LDS (families only); the kind flag (0: Chebyshev)
// is uniform over a launch and selects the kernel body.
template <typename T>
__device__ __forceinline__ bool stage_rec(T* rs, const T* __restrict__ rec, int D) {
  if (rec == nullptr || rec[3 * D + 1] == T(0)) return false;
  for (int k = threadIdx.x; k < 3 * D + 2; k += blockDim.x) rs[k] = rec[k];
  return true;
}
// LDS elements reserved for it (16-byte multiple).
static int rec_lds_elems(bool has_rec, int D) { return has_rec ? (3 * D + 2 + 3) / 4 * 4 : 0; }

// Blocks are 8 waves.  kWaves = WM * WK: WM waves share a C tile along the
// rows, WK groups split the reduction and are summed in a fixed order.
constexpr int kWaves = 8;

// Block -> tile with consecutive tiles on one XCD (workgroups go round-robin
// over the 8 XCDs), so that tiles sharing operands meet in one L2.
__device__ __forceinline__ unsigned xcd_tile(unsigned id, unsigned n) {
  const unsigned per = n / 8, rem = n % 8, x = id % 8, k = id / 8;
  return x * per + (x < rem ? x : rem) + k;
}

// 16 bytes of consecutive elements at the elements' own alignment (C's runs
// start anywhere; the memory system takes unaligned 16-byte loads).
template <typename T> struct Run {
  static constexpr int V = 16 / (int)sizeof(T);
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T)), aligned(sizeof(T))));
};
// n (uniform, at most MAX) consecutive elements of C from src into dst, 16
// bytes at a time where that stays inside C (it ends at cend), else one by
// one.  Whole vectors: elements past n hold what follows in C.  !ok: zeros.
template <typename T, int MAX>
__device__ __forceinline__ void load_run(const T* src, const T* cend, int n, bool ok, T* dst) {
  constexpr int V = Run<T>::V, NV = (MAX + V - 1) / V;
  if (src + (n + V - 1) / V * V <= cend) {
#pragma unroll
    for (int v = 0; v < NV; ++v) {
      if (v * V < n) {
        const typename Run<T>::vec x = *reinterpret_cast<const typename Run<T>::vec*>(src + v * V);
#pragma unroll
        for (int e = 0; e < V; ++e)
          if (v * V + e < MAX) dst[v * V + e] = x[e];
      }
    }
  } else {
#pragma unroll
    for (int d = 0; d < MAX; ++d) dst[d] = src[d < n ? d : n - 1];
  }
  if (!ok) {
#pragma unroll
    for (int d = 0; d < MAX; ++d) dst[d] = T(0);
  }
}

// ---- forward ------------------------------------------------------------------
// Wave tile 16 NM rows x 16 NN outputs.  A step is 4 inputs x every degree
// (WHOLE), or one chunk of at most kFwdDC degrees where LDS or registers do not
// hold them: its C tile goes through registers into one of two LDS buffers
// while the other one's step runs.  A WHOLE tile is 4 contiguous pieces of C,
// read 16 bytes a lane in order; runs of a chunk are read by one thread each,
// whose strided loads touch every line of the tile once per 16 bytes of run
// and lose the L1 to each other (4096 x 256 -> 128, degree 24, fp32: 106 -> 90 us;
// 2048 x 256 -> 256, degree 8, fp64: 70 -> 67).  LDS image: element (ii, o, d) at
// ii * S + o * DP + d with DP odd and S = 16 DP (mod 64), so that the 64 lanes
// of a read (16 outputs x 4 inputs at one degree) take distinct banks.
template <typename T> constexpr int kFwdDC = sizeof(T) == 8 ? 9 : 17;
struct GenFwd {
  int wk;              // reduction groups
  int dc, nch;         // degrees per chunk, chunks
  int dp, s;           // LDS strides (elements)
  int rec_elems;
  int mblocks;
};
constexpr int kFwdVecs = 9;  // 16-byte pieces of a WHOLE tile that a thread stages
template <int NN> __host__ __device__ constexpr int fwd_stride(int dp) {
  return 16 * NN * dp + (16 * dp * (NN == 4 ? 1 : NN == 2 ? 3 : 0)) % 64;
}

template <typename T, int NM, int NN, bool WHOLE, bool GEN>
__device__ __forceinline__ void gen_fwd_body(const T* __restrict__ t, const T* __restrict__ C,
                                             T* __restrict__ y, int64_t B, int I, int O, int D,
                                             const GenFwd f, T* lds, const T* rs) {
  typedef typename Mx<T>::acc_t acc_t;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, l15 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int WM = kWaves / f.wk, wm = wave % WM, wk = wave / WM;
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
  const int64_t b0 = ((int64_t)(tile % f.mblocks) * WM + wm) * (16 * NM);
  const int o0 = (int)(tile / f.mblocks) * (16 * NN);
  const int stage = 4 * f.s;
  T* buf = lds + f.rec_elems + wk * stage;
  const int half = f.wk * stage;  // elements from buffer 0 to buffer 1

  acc_t acc[NM][NN];
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int n = 0; n < NN; ++n) acc[m][n] = acc_t{0, 0, 0, 0};

  // this lane's rows, clamped (results of rows past B are not stored)
  const T* trow[NM];
#pragma unroll
  for (int m = 0; m < NM; ++m) {
    const int64_t b = b0 + 16 * m + l15;
    trow[m] = t + (b < B ? b : 0) * I;
  }

  const T* cend = C + (size_t)I * O * D;
  constexpr int V = Run<T>::V;
  typedef typename Run<T>::vec vec;
  // WHOLE: thread q stages pieces q, q + nth, ...: piece -> (input ii, element e
  // of its 16 NN D); an even D leaves one element of LDS after each output
  const int per_in = 16 * NN * D / V, nth = 64 * WM, total = 4 * per_in;
  int goff[WHOLE ? kFwdVecs : 1], loff[WHOLE ? kFwdVecs : 1], dv[WHOLE ? kFwdVecs : 1];
  vec pv[WHOLE ? kFwdVecs : 1];
  if constexpr (WHOLE) {
#pragma unroll
    for (int k = 0; k < kFwdVecs; ++k) {
      const int q = k * nth + wm * 64 + lane, qc = q < total ? q : 0;
      const int ii = qc / per_in, e = (qc - ii * per_in) * V, od = e / D;
      goff[k] = ii * O * D + e;
      loff[k] = ii * f.s + e + (D & 1 ? 0 : od);
      dv[k] = e - od * D;
    }
  }
  // chunked: C's tile is 64 NN runs of dn degrees, (input q / 16 NN, output
  // q % 16 NN); thread q of the group's first NN waves stages run q (two runs
  // where a group has NN / 2 waves)
  constexpr int kRuns = NN > 1 ? 2 : 1;
  T pre[WHOLE ? 1 : kRuns][WHOLE ? 1 : kFwdDC<T>], tn[NM];
  auto load_tile = [&](int i0, int d0, int dn) {
    if constexpr (WHOLE) {
      const T* base = C + ((size_t)i0 * O + o0) * D;
      if (i0 + 4 <= I && base + 3 * (size_t)O * D + 16 * NN * D <= cend) {
#pragma unroll
        for (int k = 0; k < kFwdVecs; ++k)
          if (k * nth < total) pv[k] = *reinterpret_cast<const vec*>(base + goff[k]);
      } else {
        // the layer's last inputs or outputs, element by element: zeros past the
        // inputs; past the outputs, whatever C holds there (results not stored)
        const int64_t left = cend - base;
        const int last = (int)(left > (1 << 30) ? (1 << 30) : left) - 1, ni = I - i0;
#pragma unroll
        for (int k = 0; k < kFwdVecs; ++k) {
          if (k * nth < total) {
            int e0 = goff[k];
            asm volatile("" : "+v"(e0));  // addresses formed here, not kept across the loop
            const bool ok = ni > 0 && (k * nth + wm * 64 + lane) < ni * per_in;
#pragma unroll
            for (int v = 0; v < V; ++v) {
              const T x = ok ? base[e0 + v < last ? e0 + v : last] : T(0);
              pv[k][v] = x;
            }
          }
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < kRuns; ++r) {
        if (r * WM + wm < NN) {
          const int q = (r * WM + wm) * 64 + lane, i = i0 + q / (16 * NN), o = o0 + q % (16 * NN);
          const bool ok = i < I && o < O;
          load_run<T, kFwdDC<T>>(ok ? C + ((size_t)i * O + o) * D + d0 : C, cend, dn, ok, pre[r]);
        }
      }
    }
  };
  auto store_tile = [&](T* dst, int dn) {
    if constexpr (WHOLE) {
#pragma unroll
      for (int k = 0; k < kFwdVecs; ++k) {
        if (k * nth < total && k * nth + wm * 64 + lane < total) {
          if (D & 1) {
            *reinterpret_cast<vec*>(dst + loff[k]) = pv[k];
          } else {
#pragma unroll
            for (int v = 0; v < V; ++v) dst[loff[k] + v + (dv[k] + v >= D)] = pv[k][v];
          }
        }
      }
    } else {
#pragma unroll
      for (int r = 0; r < kRuns; ++r) {
        if (r * WM + wm < NN) {
          const int q = (r * WM + wm) * 64 + lane;
          T* run = dst + (q / (16 * NN)) * f.s + (q % (16 * NN)) * f.dp;
#pragma unroll
          for (int d = 0; d < kFwdDC<T>; ++d)
            if (d < dn) run[d] = pre[r][d];
        }
      }
    }
  };
  auto load_t = [&](int i0) {
    const int i = i0 + g < I ? i0 + g : 0;
#pragma unroll
    for (int m = 0; m < NM; ++m) tn[m] = trow[m][i];
  };

  const int groups = (I + 3) / 4, iters = (groups + f.wk - 1) / f.wk;
  Rec<T, GEN> r[NM];
  load_tile(4 * wk, 0, min(f.dc, D));
  load_t(4 * wk);
  store_tile(buf, min(f.dc, D));
  __syncthreads();
  int cur = 0;
  for (int it = 0; it < iters; ++it) {
    const int i0 = 4 * (it * f.wk + wk);
#pragma unroll
    for (int m = 0; m < NM; ++m) r[m].init(tn[m], rs, D);
    if (i0 + 4 > I) {  // inputs past I meet zero coefficients: keep their basis finite
#pragma unroll
      for (int m = 0; m < NM; ++m)
        if (i0 + g >= I) r[m].clear();
    }
    for (int c = 0; c < f.nch; ++c) {
      const int d0 = c * f.dc, dn = min(f.dc, D - d0);
      const bool last_c = c + 1 == f.nch, more = !(last_c && it + 1 == iters);
      const int nd0 = last_c ? 0 : d0 + f.dc, ndn = min(f.dc, D - nd0);
      const int ni0 = last_c ? i0 + 4 * f.wk : i0;
      if (more) {
        load_tile(ni0, nd0, ndn);
        if (last_c) load_t(ni0);
      }
      const T* bp = buf + cur * half + g * f.s + l15 * f.dp;
      T bv[NN];
#pragma unroll
      for (int n = 0; n < NN; ++n) bv[n] = bp[n * 16 * f.dp];
#pragma unroll 2
      for (int d = 0; d < dn; ++d) {
        T bn[NN];  // the next degree's (the last one's read stays inside the LDS tile and is dropped)
#pragma unroll
        for (int n = 0; n < NN; ++n) bn[n] = bp[n * 16 * f.dp + (d + 1 < dn ? d + 1 : d)];
#pragma unroll
        for (int m = 0; m < NM; ++m)
#pragma unroll
          for (int n = 0; n < NN; ++n) acc[m][n] = Mx<T>::mma(r[m].pc, bv[n], acc[m][n]);
#pragma unroll
        for (int m = 0; m < NM; ++m) r[m].step(rs, D, d0 + d + 1);
#pragma unroll
        for (int n = 0; n < NN; ++n) bv[n] = bn[n];
      }
      if (more) store_tile(buf + (cur ^ 1) * half, ndn);
      cur ^= 1;
      __syncthreads();
    }
  }
  // sum the reduction groups in order through LDS (the tile buffers are done)
  T* red = lds + f.rec_elems + (size_t)wm * (64 * NM * NN * 4) + lane;
  for (int k = 1; k < f.wk; ++k) {
    if (wk == k) {
#pragma unroll
      for (int q = 0; q < NM * NN * 4; ++q) red[q * 64] = acc[q / 4 / NN][q / 4 % NN][q % 4];
    }
    __syncthreads();
    if (wk == 0) {
#pragma unroll
      for (int q = 0; q < NM * NN * 4; ++q) acc[q / 4 / NN][q / 4 % NN][q % 4] += red[q * 64];
    }
    __syncthreads();
  }
  if (wk != 0) return;
#pragma unroll
  for (int m = 0; m < NM; ++m)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int64_t b = b0 + 16 * m + Mx<T>::row(v, g);
      if (b >= B) continue;
#pragma unroll
      for (int n = 0; n < NN; ++n) {
        const int o = o0 + 16 * n + l15;
        if (o < O) y[b * O + o] = acc[m][n][v];
      }
    }
}

template <typename T> __device__ __forceinline__ T* dyn_lds() {
  extern __shared__ __align__(16) char gen_lds[];
  return reinterpret_cast<T*>(gen_lds);
}

template <typename T, int NM, int NN, bool WHOLE>
__global__ void __launch_bounds__(512)
k_gen_fwd(const T* __restrict__ t, const T* __restrict__ C, T* __restrict__ y, int64_t B, int I,
          int O, int D, GenFwd f, const T* __restrict__ rec) {
  T* lds = dyn_lds<T>();
  const bool gen = stage_rec<T>(lds, rec, D);
  __syncthreads();
  if (gen) gen_fwd_body<T, NM, NN, WHOLE, true>(t, C, y, B, I, O, D, f, lds, lds);
  else gen_fwd_body<T, NM, NN, WHOLE, false>(t, C, y, B, I, O, D, f, lds, lds);
}

// ---- dx -------------------------------------------------------------------------
// Wave tile 16 rows x 16 inputs, DM degrees at a time with one accumulator per
// degree; a chunk's G is folded into dx by the lane that holds it before the
// next chunk starts.  A step is 16 outputs: lane group g takes outputs 4 g ..
// 4 g + 3 of it, so a lane reads 4 consecutive dy values.  C's tile [16
// inputs][16 outputs][degrees] goes through registers into one of two LDS
// buffers; element (i, o = 4 g + s, d) at i * S + g * Q + s * ds + d with S odd
// and Q = 16 S (mod 64): the 64 lanes of a read take distinct banks.  WHOLE
// (every degree in one chunk, ds = D <= DM): 16 contiguous pieces of C, read 16
// bytes a lane in order; else one (input, output) run of degrees per thread,
// ds = DM.  A second row fragment per wave would halve
// the LDS reads, which are far from the bound (4 per SIMD round of one matrix
// instruction each), and spills.  With few outputs or many chunks a wave is bound
// by its own chain of loads and recurrence steps: t is read ahead of the
// products, and the recurrences go on from chunk to chunk.  dx alone, us, vector-ALU
// tiles / t and the recurrences from degree 0 after each chunk / now:
//   100000 x 64 -> 1, degree 4, fp64:  58 / 75 / 60
//   16 x 64 -> 64, degree 500, fp64:   1292 / 1518 / 484
//   16 x 64 -> 64, degree 1024, fp32:  2967 / 1913 / 469
// Still behind the vector-ALU tiles where most of the 16 input columns are
// padding: 100000 x 4 -> 4, degree 5, fp64, 19 / 23 / 21 (its dC 32349 -> 1364),
// 100000 x 1 -> 16, degree 8, 14 / 29 / 27.
template <int DM> struct GenDxLds {
  static constexpr int Q = (4 * DM + 15) / 32 * 32 + 16;      // 16 (mod 32), >= 4 DM
  static constexpr int S = 4 * Q + (Q % 64 == 16 ? 1 : 3);    // odd, 16 S = Q (mod 64)
  static_assert(Q >= 4 * DM && Q % 32 == 16 && (16 * S - Q) % 64 == 0, "LDS strides");
  static constexpr int kStage = 16 * S;
};
struct GenDx {
  int wk, nch, rec_elems, mblocks;
  int imap;
  float ima;
};

template <typename T, int DM, bool WHOLE, bool GEN>
__device__ __forceinline__ void gen_dx_body(const T* __restrict__ t, const T* __restrict__ C,
                                            const T* __restrict__ dy, T* __restrict__ dx, int64_t B,
                                            int I, int O, int D, const GenDx f, T* lds,
                                            const T* rs) {
  typedef typename Mx<T>::acc_t acc_t;
  typedef GenDxLds<DM> L;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, l15 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int WM = kWaves / f.wk, wm = wave % WM, wk = wave / WM;
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x);
  const int64_t b0 = ((int64_t)(tile % f.mblocks) * WM + wm) * 16;
  const int i0 = (int)(tile / f.mblocks) * 16;
  T* buf = lds + f.rec_elems + wk * L::kStage;
  const int half = f.wk * L::kStage;

  const T* yrow = dy + (b0 + l15 < B ? b0 + l15 : 0) * O + 4 * g;  // rows past B are not stored
  // waves 0-3 of a group stage its C tile: pieces q, q + 256, ... (WHOLE), or
  // thread q the run of degrees of (input q / 16, output q % 16)
  const bool stager = wm < 4;
  const int q = (wm & 3) * 64 + lane;
  const T* cend = C + (size_t)I * O * D;
  constexpr int V = Run<T>::V, NV = (DM + V - 1) / V;
  typedef typename Run<T>::vec vec;
  const int per_in = 16 * D / V, total = 16 * per_in;  // D / V pieces a thread
  int goff[WHOLE ? NV : 1], loff[WHOLE ? NV : 1];
  vec pv[WHOLE ? NV : 1];
  if constexpr (WHOLE) {
#pragma unroll
    for (int k = 0; k < NV; ++k) {
      const int qc = k * 256 + q < total ? k * 256 + q : 0;
      const int ii = qc / per_in, e = (qc - ii * per_in) * V, gg = e / (4 * D);
      goff[k] = ii * O * D + e;
      loff[k] = ii * L::S + gg * L::Q + (e - gg * 4 * D);
    }
  }
  const bool iok = i0 + (q >> 4) < I;
  const T* crun = C + (size_t)(iok ? i0 + (q >> 4) : 0) * O * D;
  T* cdst = buf + (q >> 4) * L::S + ((q >> 2) & 3) * L::Q + (q & 3) * DM;

  // this lane's (b, i) pairs: rows b0 + row(v, g), input i0 + l15; their t is
  // read up front, ahead of its use after the products
  T s[4], tv[4];
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int64_t b = b0 + Mx<T>::row(v, g);
    tv[v] = b < B && i0 + l15 < I ? t[b * I + i0 + l15] : T(0);
    s[v] = T(0);
  }
  // their recurrences at the chunk's first degree, kept from chunk to chunk
  // (one chunk: made in place): (up, u) = (U_{n-2}, U_{n-1}) at degree n, from
  // n = 1; GEN: (pm, pc) = (P_{n-1}, P_n) and their derivatives (qm, qc) in u,
  // from n = 0
  constexpr int NR = WHOLE ? 1 : 4;
  T rp[NR][2], rq[GEN ? NR : 1][2];
  auto rec0 = [&](int r) __attribute__((always_inline)) {
    rp[r][0] = T(0);
    rp[r][1] = T(1);
    if constexpr (GEN) rq[r][0] = rq[r][1] = T(0);
  };
#pragma unroll
  for (int r = 0; r < NR; ++r) rec0(r);

  T pre[WHOLE ? 1 : DM], an[4];
  auto load_step = [&](int ob, int d0, int dn) {
    if (stager && WHOLE) {
      const T* base = C + ((size_t)i0 * O + ob) * D;
      if (i0 + 16 <= I && ob + 16 <= O) {
#pragma unroll
        for (int k = 0; k < NV; ++k)
          if (k * 256 < total) pv[k] = *reinterpret_cast<const vec*>(base + goff[k]);
      } else {  // zeros past the layer's inputs and outputs
        const int lim = (O - ob) * D, ni = I - i0;
#pragma unroll
        for (int k = 0; k < NV; ++k) {
          if (k * 256 < total) {
            int e0 = goff[k], qk = k * 256 + q;
            asm volatile("" : "+v"(e0), "+v"(qk));  // addresses formed here, not kept across the loop
            const int e = (qk % per_in) * V;
            const bool ok = qk < total && qk < ni * per_in;
#pragma unroll
            for (int v = 0; v < V; ++v) pv[k][v] = ok && e + v < lim ? base[e0 + v] : T(0);
          }
        }
      }
    } else if (stager) {
      const int o = ob + (q & 15);
      const bool ok = iok && o < O;
      if constexpr (!WHOLE) load_run<T, DM>(ok ? crun + (size_t)o * D + d0 : C, cend, dn, ok, pre);
    }
    if (ob + 16 <= O) {
      constexpr int V = Run<T>::V;
#pragma unroll
      for (int v = 0; v < 4 / V; ++v) {
        const typename Run<T>::vec x = *reinterpret_cast<const typename Run<T>::vec*>(yrow + ob + v * V);
#pragma unroll
        for (int e = 0; e < V; ++e) an[v * V + e] = x[e];
      }
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) an[k] = ob + 4 * g + k < O ? yrow[ob + k] : T(0);
    }
  };
  auto store_step = [&](int b) {
    if (stager && WHOLE) {
#pragma unroll
      for (int k = 0; k < NV; ++k) {
        if (k * 256 < total && k * 256 + q < total) {
#pragma unroll
          for (int v = 0; v < V; ++v) buf[b * half + loff[k] + v] = pv[k][v];
        }
      }
    } else if (stager) {
#pragma unroll
      for (int k = 0; k < DM; ++k) cdst[b * half + k] = pre[WHOLE ? 0 : k];
    }
  };

  const int osteps = (O + 15) / 16, iters = (osteps + f.wk - 1) / f.wk;
  load_step(16 * wk, 0, min(DM, D));
  store_step(0);
  __syncthreads();
  int cur = 0;
  for (int c = 0; c < f.nch; ++c) {
    const int d0 = c * DM, dn = min(DM, D - d0);
    acc_t acc[DM];
#pragma unroll
    for (int d = 0; d < DM; ++d) acc[d] = acc_t{0, 0, 0, 0};
    for (int it = 0; it < iters; ++it) {
      T a[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) a[k] = an[k];
      const bool last = it + 1 == iters, more = !(last && c + 1 == f.nch);
      if (more) {
        const int nd0 = last ? d0 + DM : d0;
        load_step(16 * (last ? wk : (it + 1) * f.wk + wk), nd0, min(DM, D - nd0));
      }
      const T* bp = buf + cur * half + l15 * L::S + g * L::Q;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const T* bk = bp + k * (WHOLE ? D : DM);  // (degrees past D: values no one uses)
#pragma unroll
        for (int d = 0; d < DM; ++d) acc[d] = Mx<T>::mma(a[k], bk[d], acc[d]);
      }
      if (more) store_step(cur ^ 1);
      cur ^= 1;
      __syncthreads();
    }
    // s += sum_d G_d P_d'(t) over the chunk (this reduction group's share of G);
    // a WHOLE chunk in two sums, as two chunks would be
    const int dh = WHOLE && sizeof(T) == 4 ? (D + 1) / 2 : 0;
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int r = WHOLE ? 0 : v;
      if (WHOLE) rec0(r);
      T sum = T(0);
      if constexpr (GEN) {
        // P_n' = a_n P_{n-1} + (a_n u + b_n) P_{n-1}' - c_n P_{n-2}'
        const T u = rs[3 * D] * tv[v];
#pragma unroll
        for (int d = 0; d < DM; ++d) {
          if (d > 0 && d == dh) {
            s[v] += sum;  // du/dt once, at the store
            sum = T(0);
          }
          if (d < dn) {
            sum = fma(acc[d][v], rq[r][1], sum);
            asm volatile("" ::: "memory");  // coefficients read per step, not hoisted
            const int n = d0 + d + 1, k = n < D ? n : D - 1;
            const T a_n = rs[k], fn = fma(a_n, u, rs[D + k]), cn = rs[2 * D + k];
            const T pn = fma(fn, rp[r][1], -cn * rp[r][0]);
            const T qn = fma(a_n, rp[r][1], fma(fn, rq[r][1], -cn * rq[r][0]));
            rp[r][0] = rp[r][1];
            rp[r][1] = pn;
            rq[r][0] = rq[r][1];
            rq[r][1] = qn;
          }
        }
      } else {
        // dT_n/dt = n U_{n-1}; degree 0 has no derivative
        const T t2 = tv[v] + tv[v];
        T deg = (T)d0;  // counted in T (exact)
#pragma unroll
        for (int d = 0; d < DM; ++d) {
          if (d > 0 && d == dh) {
            s[v] += sum;
            sum = T(0);
          }
          if (d < dn && (d > 0 || d0 > 0)) {
            sum = fma(acc[d][v] * deg, rp[r][1], sum);
            const T un = fma(t2, rp[r][1], -rp[r][0]);
            rp[r][0] = rp[r][1];
            rp[r][1] = un;
          }
          deg += T(1);
        }
      }
      s[v] += sum;
    }
  }
  // sum the reduction groups in order, apply t'(x), store
  T* red = lds + f.rec_elems + wm * 256 + lane;
  for (int k = 1; k < f.wk; ++k) {
    if (wk == k) {
#pragma unroll
      for (int v = 0; v < 4; ++v) red[v * 64] = s[v];
    }
    __syncthreads();
    if (wk == 0) {
#pragma unroll
      for (int v = 0; v < 4; ++v) s[v] += red[v * 64];
    }
    __syncthreads();
  }
  if (wk != 0 || i0 + l15 >= I) return;
#pragma unroll
  for (int v = 0; v < 4; ++v) {
    const int64_t b = b0 + Mx<T>::row(v, g);
    if (b >= B) continue;
    const T slope = f.imap ? (T)f.ima : T(1) - tv[v] * tv[v];
    dx[b * I + i0 + l15] = (GEN ? s[v] * rs[3 * D] : s[v]) * slope;  // du/dt = rs[3 D] for a family
  }
}

template <typename T, int DM, bool WHOLE>
__global__ void __launch_bounds__(512)
k_gen_dx(const T* __restrict__ t, const T* __restrict__ C, const T* __restrict__ dy,
         T* __restrict__ dx, int64_t B, int I, int O, int D, GenDx f, const T* __restrict__ rec) {
  T* lds = dyn_lds<T>();
  const bool gen = stage_rec<T>(lds, rec, D);
  __syncthreads();
  if (gen) gen_dx_body<T, DM, WHOLE, true>(t, C, dy, dx, B, I, O, D, f, lds, lds);
  else gen_dx_body<T, DM, WHOLE, false>(t, C, dy, dx, B, I, O, D, f, lds, lds);
}

// ---- dC ---------------------------------------------------------------------------
template <typename T> struct DcWrite;
template <> struct DcWrite<float> {  // the dC write modes of the MFMA kernels
  static __device__ __forceinline__ void put(float* d, float v, const DcOut& om) { dc_write(d, v, om); }
};
template <> struct DcWrite<double> {  // store or accumulate
  static __device__ __forceinline__ void put(double* d, double v, const DcOut& om) {
    *d = om.mode == kDcAccumulate ? *d + v : v;
  }
};

// Wave tile 16 inputs x 16 NN outputs x DM degrees (one chunk of the degree
// axis), the reduction over the batch rows split between the WK waves of a
// block that share the tile.  Both operands come straight from memory: 16
// lanes read 16 consecutive t (or dy) values of a row, and the waves of a
// block reuse each other's lines in L1.  The next unit of rows is loaded while
// one is used.  The WK partial sums meet in LDS by halves (a fixed order).
struct GenDc {
  int wk, nch, rec_elems;
  int iblocks, otiles;   // 16-input blocks, output tiles of 16 NN
  int64_t units;         // row units per reduction group
};
// Rows a wave loads ahead, 4 per matrix instruction: as many as the registers
// beside the accumulators hold (twice as many on the narrow tiles measured
// the same).
template <typename T> constexpr int kDcUnit = sizeof(T) == 8 ? 8 : 16;

template <typename T, int DM, int NN, bool GEN>
__device__ __forceinline__ void gen_dc_body(const T* __restrict__ t, const T* __restrict__ dy,
                                            T* __restrict__ dC, int64_t B, int I, int O, int D,
                                            const GenDc f, const DcOut& om, T* lds, const T* rs) {
  typedef typename Mx<T>::acc_t acc_t;
  constexpr int kU = kDcUnit<T>, KU = kU / 4;
  const int tid = threadIdx.x, lane = tid & 63, g = lane >> 4, l15 = lane & 15;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int WT = kWaves / f.wk, wt = wave % WT, wk = wave / WT;
  // tiles: output tile fastest, then input block, then chunk
  const unsigned ntiles = (unsigned)f.otiles * f.iblocks * f.nch;
  const unsigned tile = xcd_tile(blockIdx.x, gridDim.x) * WT + wt;
  const bool live = tile < ntiles;  // a block's last waves may have no tile
  const unsigned tl = live ? tile : 0;
  const int o0 = (int)(tl % f.otiles) * (16 * NN);
  const int i0 = (int)(tl / f.otiles % f.iblocks) * 16;
  const int d0 = (int)(tl / f.otiles / f.iblocks) * DM;
  const int i = i0 + l15;
  const bool iok = i < I;

  acc_t acc[DM][NN];
#pragma unroll
  for (int d = 0; d < DM; ++d)
#pragma unroll
    for (int n = 0; n < NN; ++n) acc[d][n] = acc_t{0, 0, 0, 0};

  const int64_t ub = (int64_t)wk * f.units, ue0 = ub + f.units, nu = (B + kU - 1) / kU;
  const int64_t ue = live ? (ue0 < nu ? ue0 : nu) : 0;
  // Loads go through a buffer descriptor of the unit's rows, rebuilt in
  // scalar registers each unit: a lane's byte offset is fixed for the kernel,
  // the row offset is scalar, and rows past B read as zeros (dy = 0 drops
  // them).  Inputs and outputs past the layer's read column 0; their results
  // are not stored.
  const int esz = (int)sizeof(T);
  const int toff = (g * I + (iok ? i : 0)) * esz;
  int yoff[NN];
#pragma unroll
  for (int n = 0; n < NN; ++n) yoff[n] = (g * O + (o0 + 16 * n + l15 < O ? o0 + 16 * n + l15 : 0)) * esz;
  T tn[KU], yn[KU][NN];
  auto load = [&](int64_t u) {
    const int64_t left = B - u * kU;
    const int rows = (int)(left < kU ? left : kU);
    const __amdgpu_buffer_rsrc_t rt = buffer_rsrc(t + u * kU * I, rows * I * esz);
    const __amdgpu_buffer_rsrc_t ry = buffer_rsrc(dy + u * kU * O, rows * O * esz);
#pragma unroll
    for (int k = 0; k < KU; ++k) {
      tn[k] = buffer_load<T>(rt, toff, 4 * k * I * esz);
#pragma unroll
      for (int n = 0; n < NN; ++n) yn[k][n] = buffer_load<T>(ry, yoff[n], 4 * k * O * esz);
    }
  };
  if (ub < ue) load(ub);
  for (int64_t u = ub; u < ue; ++u) {
    Rec<T, GEN> r[KU];
    T yc[KU][NN];
#pragma unroll
    for (int k = 0; k < KU; ++k) {
      r[k].init(tn[k], rs, D);
#pragma unroll
      for (int n = 0; n < NN; ++n) yc[k][n] = yn[k][n];
    }
    if ((u + 1) * kU > B) {  // a basis value of a row past B may not be finite
#pragma unroll
      for (int k = 0; k < KU; ++k)
        if (u * kU + 4 * k + g >= B) r[k].clear();
    }
    load(u + 1 < ue ? u + 1 : u);
    // to the chunk's first degree, the rows side by side
    if (d0 & 1) {
#pragma unroll
      for (int k = 0; k < KU; ++k) r[k].step(rs, D, 1);
    }
    for (int n = 1 + (d0 & 1); n <= d0; n += 2) {
#pragma unroll
      for (int k = 0; k < KU; ++k) r[k].step2(rs, D, n);
    }
#pragma unroll
    for (int k = 0; k < KU; ++k) {
#pragma unroll
      for (int d = 0; d < DM; ++d) {
#pragma unroll
        for (int n = 0; n < NN; ++n) acc[d][n] = Mx<T>::mma(r[k].pc, yc[k][n], acc[d][n]);
        if (d + 1 < DM) r[k].step(rs, D, d0 + d + 1);
      }
    }
  }
  constexpr int kAcc = DM * NN * 4;
  for (int h = f.wk / 2; h >= 1; h /= 2) {
    T* red = lds + f.rec_elems + (size_t)((wk % h) * WT + wt) * (64 * kAcc) + lane;
    if (wk >= h && wk < 2 * h) {
#pragma unroll
      for (int q = 0; q < kAcc; ++q) red[q * 64] = acc[q / 4 / NN][q / 4 % NN][q % 4];
    }
    __syncthreads();
    if (wk < h) {
#pragma unroll
      for (int q = 0; q < kAcc; ++q) acc[q / 4 / NN][q / 4 % NN][q % 4] += red[q * 64];
    }
    __syncthreads();
  }
  if (wk != 0 || !live) return;
#pragma unroll
  for (int n = 0; n < NN; ++n)
#pragma unroll
    for (int v = 0; v < 4; ++v) {
      const int io = i0 + Mx<T>::row(v, g), o = o0 + 16 * n + l15;
      if (io >= I || o >= O) continue;
      T* dst = dC + ((size_t)io * O + o) * D + d0;
#pragma unroll
      for (int d = 0; d < DM; ++d)
        if (d0 + d < D) DcWrite<T>::put(dst + d, acc[d][n][v], om);
    }
}

template <typename T, int DM, int NN>
__global__ void __launch_bounds__(512)
k_gen_dc(const T* __restrict__ t, const T* __restrict__ dy, T* __restrict__ dC, int64_t B, int I,
         int O, int D, GenDc f, DcOut om, const T* __restrict__ rec) {
  T* lds = dyn_lds<T>();
  const bool gen = stage_rec<T>(lds, rec, D);
  __syncthreads();
  if (gen) gen_dc_body<T, DM, NN, true>(t, dy, dC, B, I, O, D, f, om, lds, lds);
  else gen_dc_body<T, DM, NN, false>(t, dy, dC, B, I, O, D, f, om, lds, lds);
}

// dst = float(src) (or dst += float(src)), src fp32 or bf16: the coefficient
// copy of this path.
__global__ void __launch_bounds__(256)
k_to_f32(const void* __restrict__ src, int src_bf16, float* __restrict__ dst, int64_t n,
         int accumulate) {
  for (int64_t q = blockIdx.x * (int64_t)blockDim.x + threadIdx.x; q < n;
       q += (int64_t)gridDim.x * blockDim.x) {
    const float v = src_bf16 ? __uint_as_float((uint32_t)static_cast<const uint16_t*>(src)[q] << 16)
                             : static_cast<const float*>(src)[q];
    dst[q] = accumulate ? dst[q] + v : v;
  }
}

static unsigned vgrid(int64_t n) {
  int64_t g = (n + 255) / 256;
  if (g > 65536) g = 65536;
  return (unsigned)(g < 1 ? 1 : g);
}

void launch_to_f32(const void* src, bool src_bf16, float* dst, int64_t n, hipStream_t s,
                   bool accumulate) {
  if (n > 0)
    hipLaunchKernelGGL(k_to_f32, dim3(vgrid(n)), dim3(256), 0, s, src, src_bf16 ? 1 : 0, dst, n,
                       accumulate ? 1 : 0);
}

// ---- launch shapes ----------------------------------------------------------------
// Waves that give every SIMD two: below it, tiles shrink and the reduction is
// split until the launch has as many (or nothing is left to split).  Four per
// SIMD measured slower: the smaller tiles stage more of C for each product
// (2048 x 256 -> 256 in fp64: forward 73 -> 84 us, backward 103 -> 117; 4096 x
// 256 -> 128, degree 24: forward 108 -> 134).
constexpr int64_t kWantWaves = 2 * 4 * kNumCUs;
constexpr int kMaxLds = 160 * 1024;

// Degrees per chunk: the fewest chunks of at most `cap` degrees, evenly sized.
static int even_chunk(int D, int cap) {
  const int n = (D + cap - 1) / cap;
  return (D + n - 1) / n;
}

template <typename T, int NM, int NN, bool WHOLE>
static bool gen_fwd_launch(const T* t, const T* C, T* y, int64_t B, int I, int O, int D,
                           const T* rec, hipStream_t s, bool must) {
  static std::atomic<uint32_t> lds_done{0};
  GenFwd f;
  f.dc = WHOLE ? D : even_chunk(D, kFwdDC<T>);
  f.nch = (D + f.dc - 1) / f.dc;
  f.dp = f.dc | 1;
  f.s = fwd_stride<NN>(f.dp);
  f.rec_elems = rec_lds_elems(rec != nullptr, D);
  const int64_t mt = (B + 16 * NM - 1) / (16 * NM), nt = (O + 16 * NN - 1) / (16 * NN);
  auto bytes = [&](int wk) {
    const int64_t st = 2LL * wk * 4 * f.s, red = wk > 1 ? (int64_t)(kWaves / wk) * 64 * NM * NN * 4 : 0;
    return (f.rec_elems + (st > red ? st : red)) * (int64_t)sizeof(T);
  };
  // what a thread stages, and the 32-bit offsets of a WHOLE tile
  auto fits = [&](int wk) {
    const int WM = kWaves / wk;
    return bytes(wk) <= kMaxLds &&
           (WHOLE ? NN * D <= kFwdVecs * Run<T>::V * WM && (int64_t)O * D < (1 << 28) : WM >= NN / 2);
  };
  int wk = 1;
  while (wk < 8 && mt * nt * wk < kWantWaves && 2 * wk <= (I + 3) / 4 && fits(2 * wk)) wk *= 2;
  if (!fits(wk) || (!must && mt * nt * wk < kWantWaves)) return false;
  f.wk = wk;
  const int WM = kWaves / wk;
  f.mblocks = (int)((mt + WM - 1) / WM);
  ensure_lds_limit(reinterpret_cast<const void*>(&k_gen_fwd<T, NM, NN, WHOLE>), kMaxLds, lds_done);
  hipLaunchKernelGGL((k_gen_fwd<T, NM, NN, WHOLE>), dim3((unsigned)f.mblocks * (unsigned)nt), dim3(512),
                     (size_t)bytes(wk), s, t, C, y, B, I, O, D, f, rec);
  return true;
}

template <typename T>
void launch_forward_general(const T* x, const T* C, T* y, T* t, int64_t B, int I, int O, int deg,
                            hipStream_t s, const T* rec, int imap, float ima, float imb) {
  if (B == 0) return;
  hipLaunchKernelGGL(k_tanh_v<T>, dim3(vgrid(B * I)), dim3(256), 0, s, x, t, B * I, imap, ima, imb);
  const int D = deg + 1;
  // the largest wave tile whose launch still fills the chip, WHOLE where it fits
  if (gen_fwd_launch<T, 2, 4, true>(t, C, y, B, I, O, D, rec, s, false)) return;
  if (gen_fwd_launch<T, 2, 2, true>(t, C, y, B, I, O, D, rec, s, false)) return;
  if (gen_fwd_launch<T, 2, 4, false>(t, C, y, B, I, O, D, rec, s, false)) return;
  if (gen_fwd_launch<T, 2, 2, false>(t, C, y, B, I, O, D, rec, s, false)) return;
  if (gen_fwd_launch<T, 1, 1, true>(t, C, y, B, I, O, D, rec, s, true)) return;
  gen_fwd_launch<T, 1, 1, false>(t, C, y, B, I, O, D, rec, s, true);
}

template <typename T, int DM, bool WHOLE>
static void gen_dx(const T* t, const T* C, const T* dy, T* dx, int64_t B, int I, int O, int D,
                   const T* rec, int imap, float ima, hipStream_t s) {
  static std::atomic<uint32_t> lds_done{0};
  GenDx f;
  f.nch = (D + DM - 1) / DM;
  f.rec_elems = rec_lds_elems(rec != nullptr, D);
  f.imap = imap;
  f.ima = ima;
  const int64_t mt = (B + 15) / 16, it = (I + 15) / 16;
  // two reduction groups at most: a group's 4 waves stage one run per thread
  f.wk = mt * it < kWantWaves && O > 16 ? 2 : 1;
  const int WM = kWaves / f.wk;
  f.mblocks = (int)((mt + WM - 1) / WM);
  const size_t bytes = (f.rec_elems + 2 * (size_t)f.wk * GenDxLds<DM>::kStage) * sizeof(T);
  ensure_lds_limit(reinterpret_cast<const void*>(&k_gen_dx<T, DM, WHOLE>), kMaxLds, lds_done);
  hipLaunchKernelGGL((k_gen_dx<T, DM, WHOLE>), dim3((unsigned)(f.mblocks * it)), dim3(512), bytes, s, t, C,
                     dy, dx, B, I, O, D, f, rec);
}

template <typename T, int DM, int NN>
static bool gen_dc_launch(const T* t, const T* dy, T* dC, DcOut om, int64_t B, int I, int O, int D,
                          const T* rec, hipStream_t s, bool must) {
  static std::atomic<uint32_t> lds_done{0};
  GenDc f;
  f.nch = (D + DM - 1) / DM;
  f.rec_elems = rec_lds_elems(rec != nullptr, D);
  f.iblocks = (I + 15) / 16;
  f.otiles = (O + 16 * NN - 1) / (16 * NN);
  const int64_t tiles = (int64_t)f.iblocks * f.otiles * f.nch;
  const int64_t nu = (B + kDcUnit<T> - 1) / kDcUnit<T>;
  auto bytes = [&](int wk) {
    const int64_t red = wk > 1 ? 4LL * 64 * DM * NN * 4 : 0;
    return (f.rec_elems + red) * (int64_t)sizeof(T);
  };
  int wk = 1;
  while (wk < kWaves && tiles * wk < kWantWaves && 2 * wk <= nu && bytes(2 * wk) <= kMaxLds) wk *= 2;
  if (!must && tiles * wk < kWantWaves) return false;
  f.wk = wk;
  f.units = (nu + wk - 1) / wk;
  const int WT = kWaves / wk;
  ensure_lds_limit(reinterpret_cast<const void*>(&k_gen_dc<T, DM, NN>), kMaxLds, lds_done);
  hipLaunchKernelGGL((k_gen_dc<T, DM, NN>), dim3((unsigned)((tiles + WT - 1) / WT)), dim3(512),
                     (size_t)bytes(wk), s, t, dy, dC, B, I, O, D, f, om, rec);
  return true;
}
template <typename T, int DM>
static void gen_dc(const T* t, const T* dy, T* dC, DcOut om, int64_t B, int I, int O, int D,
                   const T* rec, hipStream_t s) {
  // accumulators: DM x NN x 4 values a lane, at most 144 registers
  constexpr int kBig = DM * 4 * 4 * (int)sizeof(T) / 4 <= 150 ? 4 : 2;
  if (gen_dc_launch<T, DM, kBig>(t, dy, dC, om, B, I, O, D, rec, s, false)) return;
  gen_dc_launch<T, DM, 1>(t, dy, dC, om, B, I, O, D, rec, s, true);
}

// Calls f with the accumulators' degree capacity as a constant: the first of
// the list that holds n (its last one does).
template <int A, int... R, typename F> static void with_degrees(int n, F f) {
  if constexpr (sizeof...(R) > 0) {
    if (n > A) return with_degrees<R...>(n, f);
  }
  f(std::integral_constant<int, A>());
}

// Degrees of dx in one chunk: what fits the registers beside the staging.
template <typename T> constexpr int kDxDegrees = sizeof(T) == 8 ? 9 : 27;

template <typename T>
void launch_backward_general(const T* t, const T* C, const T* dy, T* dx, T* dC, DcOut om, int64_t B,
                             int I, int O, int deg, hipStream_t s, const T* rec, int imap,
                             float ima) {
  const int D = deg + 1;
  constexpr bool F64 = sizeof(T) == 8;
  if (dx && B > 0) {
    // one chunk, staged whole (32-bit offsets), or the fewest chunks of equal size
    const bool whole = D <= kDxDegrees<T> && (int64_t)O * D < (1 << 26);
    auto go = [&](auto dm) { gen_dx<T, decltype(dm)::value, true>(t, C, dy, dx, B, I, O, D, rec, imap, ima, s); };
    auto chunks = [&](auto dm) { gen_dx<T, decltype(dm)::value, false>(t, C, dy, dx, B, I, O, D, rec, imap, ima, s); };
    const int c = even_chunk(D, kDxDegrees<T>);
    if constexpr (F64) {
      if (whole) with_degrees<2, 3, 4, 5, 6, 7, 8, 9>(D, go);
      else with_degrees<3, 5, 6, 7, 8, 9>(c, chunks);
    } else {  // D >= 18
      if (whole) with_degrees<19, 21, 23, 25, 27>(D, go);
      else with_degrees<15, 17, 21, 25, 27>(c, chunks);
    }
  }
  if (dC) {
    auto go = [&](auto dm) { gen_dc<T, decltype(dm)::value>(t, dy, dC, om, B, I, O, D, rec, s); };
    if constexpr (F64) with_degrees<3, 5, 6, 7, 8, 9>(even_chunk(D, 9), go);
    else with_degrees<9, 11, 13, 15, 17>(even_chunk(D, 17), go);
  }
}

template void launch_forward_general<float>(const float*, const float*, float*, float*, int64_t, int,
                                         int, int, hipStream_t, const float*, int, float, float);
template void launch_forward_general<double>(const double*, const double*, double*, double*, int64_t,
                                          int, int, int, hipStream_t, const double*, int, float,
                                          float);
template void launch_backward_general<float>(const float*, const float*, const float*, float*, float*,
                                          DcOut, int64_t, int, int, int, hipStream_t, const float*,
                                          int, float);
template void launch_backward_general<double>(const double*, const double*, const double*, double*,
                                           double*, DcOut, int64_t, int, int, int, hipStream_t,
                                           const double*, int, float);

}  // namespace ckan

