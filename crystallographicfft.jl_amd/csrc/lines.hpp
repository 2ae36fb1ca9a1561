// Line-matrix chain of path QS (gfx950): the diffusion operator of a
// separable plan as one real H x H matrix per channel and axis, applied with
// the FP64 matrix instructions.
//
// The fold splits a subgrid field into real channels
//   g_o(x) = sum_e (-1)^(o.e) f(x + H e),  x < H,  o the channel's parity
// (no twiddle: the phase exp(-2 pi i o x / M) that makes a channel's FFT the
// M-grid spectrum at q = 2k + o goes into the matrices).  With an orthogonal
// cell and diagonal representative ops the Q-fused multiply
// (src/q_fused_krfft.jl:518-667) acts on channel c as
//   G'(q) = prod_d (F_d[0][q_d] + chi_{c,d} F_d[1][q_d] flip_d) G(q),
// chi = -1 where the ops' half-cell glides change sign on the channel, so in
// real space it is A_x A_y A_z, one real matrix per axis:
//   A[x'][x] = (1/H) sum_{q = o mod 2} Re(F_0(q) e^{2 pi i q (x' - x)/M}
//                                       + chi F_1(q) e^{2 pi i q (x' + x)/M}).
// The A_d of different axes commute, so the contour chain
//   ... E U (A_x A_y A_z) F E  E U (A_x A_y A_z) F E ...   (F fold, U unfold)
// runs as ONE kernel per step: the kernels alternate between y-lines
// (planes of fixed z) and z-lines (planes of fixed y); each applies A_x and
// its line matrix to its input, then unfold, E, fold at its points, then its
// line matrix again, which leaves A_x and the other line matrix to the next
// kernel.  A workgroup takes the line axis in full and kCW x-values of one
// plane; A_x reads the plane's other x-values too.  Source and destination channels alternate
// between the two halves of the plan's channel buffer.
#pragma once

#include <hip/hip_runtime.h>

#include "pipeline.hpp"
#include "plan.hpp"

namespace cfft {

typedef double mfma_d4 __attribute__((ext_vector_type(4)));

// Channel lengths of the chain: at every one it beats the plane-pair chain, in
// each centring, precision and batch.  Steps of one field, FP64, plane pairs ->
// line matrices: Pmmm H = 8 10.0 -> 3.6 us, 16 11.4 -> 4.3, 32 18.2 -> 8.0, 48
// 41.2 -> 15.7; Pm-3m H = 64 71.1 -> 24.3; Im-3m H = 48 31.6 -> 10.1, 64 52.0 ->
// 14.7; Fm-3m H = 48 27.0 -> 8.5, 64 49.0 -> 13.0; eight fields of Pmmm, H = 32
// 45.3 -> 15.3; two of Im-3m, H = 64 89.0 -> 26.5 (mixed 63.4 -> 23.6).
constexpr int kLineLens[] = {8, 12, 16, 24, 32, 48, 64};
inline bool line_len_ok(int H) {
  for (int v : kLineLens)
    if (v == H) return true;
  return false;
}

// Interaction factors of batch entry b: e1 for steps < sw, then e2.
struct LineEnt {
  struct Entry {
    const double *e1, *e2;
    long sw;
  } ent[kMaxEPtr];
};

// Arguments of the chain's kernels besides LineEnt, in the order the kernels
// take them: the first 14 dwords reach a wave in scalar registers, so its
// first loads wait for no argument fetch.
struct LineP {
  void* ch;                // channels: two halves of batch x n_ch x H^3 reals
  const double* mats;      // matrix table
  unsigned long long axv;  // matrix variant of channel c on axis d: bits 6 c + 2 d
  int batch, step;
  int flags;               // kLineFlip, kLineContig, kLineZ
  const double* E;         // kLineContig: one array of batch x M^3 factors (nullptr: none)
  const void* f0_in;
  void* f0_out;
};
enum { kLineFlip = 1, kLineContig = 2, kLineZ = 4 };  // half of ch read; factors in E, not LineEnt; z-lines

// Matrix table: entry [axis][variant][tile t][k-step i][lane] with variant =
// o | (chi < 0) << 1, tiles of 16 matrix rows, H/4 k-steps; lane l holds
// A[16 t + l % 16][4 i + l / 16], the order in which the matrix instruction
// takes its operands and leaves its result.  Rows past H are 0.  An even
// number of k-steps is stored in pairs, one 16-byte load each.
constexpr int line_tiles(int H) { return (H + 15) / 16; }
constexpr int line_variant_len(int H) { return line_tiles(H) * (H / 4) * 64; }
constexpr int line_entry(int H, int t, int i, int lane) {
  const int KS = H / 4;
  return KS % 2 == 0 ? (t * KS + (i & ~1)) * 64 + 2 * lane + (i & 1) : (t * KS + i) * 64 + lane;
}
// The k-steps of one matrix tile for this lane.
template <int KS>
__device__ __forceinline__ void load_matrix(const double* __restrict__ m, int lane, double (&v)[KS]) {
  if constexpr (KS % 2 == 0) {
    const double2* q = reinterpret_cast<const double2*>(m) + lane;
#pragma unroll
    for (int i = 0; i < KS / 2; ++i) {
      const double2 w = q[64 * i];
      v[2 * i] = w.x;
      v[2 * i + 1] = w.y;
    }
  } else {
#pragma unroll
    for (int i = 0; i < KS; ++i) v[i] = m[64 * i + lane];
  }
}

// One channel of a plane, H rows of W values (all H, or half of them in each of
// two rounds where H > 32), staged in LDS by its wave: rows are read in 16-byte
// chunks, whole rows by neighbouring lanes (measured 63 bytes per cycle and
// CU; the matrix operand's own pattern, 16 rows of 64 bytes per load, takes
// 17, and loads straight into LDS issue at one per 120 cycles), and written
// with chunk c of row r at chunk (c + s(r)) mod the row's chunks, s(r) chosen
// so that the 16 rows an operand read touches lie on different banks.  The
// chunks pass between the lanes of one wave: no workgroup barrier, but a
// wave_sync() between the writes and the reads, and before the second round's
// writes over rows that other lanes have read.
template <typename T, int H>
struct LineStage {
  static constexpr int E = 16 / (int)sizeof(T);        // values per chunk
  static constexpr int W = H <= 32 ? H : H / 2, ROUNDS = H / W;
  static constexpr int C = W / E;                      // chunks per row
  static constexpr int N = H * C, NI = (N + 63) / 64;  // chunks, loads of 64 lanes
  static constexpr int G = C % 16 == 0 ? 16 : (C % 8 == 0 ? 8 : (C % 4 == 0 ? 4 : (C % 2 == 0 ? 2 : 1)));
  static constexpr int BYTES = 16 * N;
  static_assert(W % E == 0 && W % 4 == 0, "rows of whole chunks and k-steps");
  __device__ static __forceinline__ int shift(int row) { return row * G / 16; }
};

template <typename T, int H>
struct LineRows {  // a round's chunks on their way to LDS
  typedef T vec __attribute__((ext_vector_type(16 / sizeof(T))));
  vec v[LineStage<T, H>::NI];
};
template <typename T, int H>
__device__ __forceinline__ void load_rows(const T* __restrict__ src, unsigned rs, int lane, LineRows<T, H>& q) {
  typedef LineStage<T, H> S;
#pragma unroll
  for (int j = 0; j < S::NI; ++j) {
    const int k0 = 64 * j + lane, k = S::N % 64 == 0 || k0 < S::N ? k0 : S::N - 1;
    q.v[j] = *reinterpret_cast<const typename LineRows<T, H>::vec*>(
        src + ((unsigned)(k / S::C) * rs + (unsigned)(k % S::C * S::E)));
  }
}
template <typename T, int H>
__device__ __forceinline__ void stage_rows(const LineRows<T, H>& q, int lane, unsigned char* lds) {
  typedef LineStage<T, H> S;
#pragma unroll
  for (int j = 0; j < S::NI; ++j) {
    const int k = 64 * j + lane, row = k / S::C, c = (k % S::C + S::shift(row)) % S::C;
    if (S::N % 64 == 0 || k < S::N) reinterpret_cast<typename LineRows<T, H>::vec*>(lds)[row * S::C + c] = q.v[j];
  }
}

// Value x < W of row `row`.
template <typename T, int H>
__device__ __forceinline__ double staged(const unsigned char* lds, int row, int x) {
  typedef LineStage<T, H> S;
  const int c = (x / S::E + S::shift(row)) % S::C;
  return (double)reinterpret_cast<const T*>(lds)[(row * S::C + c) * S::E + x % S::E];
}

// Channels of a lattice centring (plan.hpp's Centering) as a group of
// parities: channel c = sum of the generators gen(k) of its bits.  A corner e
// of the fold only enters as its class, bit k = parity of gen(k) & e: a field
// with the centring takes one value per class, and fold and unfold are
// Walsh-Hadamard transforms of length n_ch between channels and classes.
template <int CENT>
struct LineCent;
template <>
struct LineCent<CENT_P> {
  static constexpr int NCH = 8, gen[3] = {1, 2, 4};
};
template <>
struct LineCent<CENT_I> {
  static constexpr int NCH = 4, gen[3] = {3, 5, 0};
};
template <>
struct LineCent<CENT_C> {
  static constexpr int NCH = 4, gen[3] = {3, 4, 0};
};
template <>
struct LineCent<CENT_A> {
  static constexpr int NCH = 4, gen[3] = {6, 1, 0};
};
template <>
struct LineCent<CENT_F> {
  static constexpr int NCH = 2, gen[3] = {7, 0, 0};
};
template <int CENT>
constexpr int line_parity(int c) {  // parity offset of channel c
  int o = 0;
  for (int k = 0; k < 3; ++k)
    if ((c >> k) & 1) o ^= LineCent<CENT>::gen[k];
  return o;
}
template <int CENT>
__host__ __device__ constexpr int line_class(int e) {
  int v = 0;
  for (int k = 0; k < 3; ++k) {
    const int m = LineCent<CENT>::gen[k] & e;
    v |= ((m ^ (m >> 1) ^ (m >> 2)) & 1) << k;
  }
  return v;
}

enum { kLinesIn = 1, kLinesOut = 2, kLinesStore = 4 };

// x-values per workgroup: the matrix instructions' tile.  Measured against 8
// (every CU at work from half the fields, half of each tile wasted) and 32
// (a plane's rows read once): Im-3m 128^3 FP64 at 1, 2 and 8 fields 5.58, 6.01,
// 12.1 us (8), 5.75, 6.11, 8.9 us (16), 7.7, 8.1, 9.6 us (32); at 16 fields
// 15.7 us (16), 14.8 us (32).
constexpr int kCW = 16;
constexpr int line_parts(int H) { return (H + kCW - 1) / kCW; }

// LDS of a workgroup: per channel its staged plane, then its H x kCW points.
template <typename T, int H, int CENT, int MODE>
struct LineLds {
  static constexpr int PTS = 8 * H * kCW, ST = (MODE & kLinesIn) ? LineStage<T, H>::BYTES : 0;
  static constexpr int CH = PTS > ST ? PTS : ST, BYTES = LineCent<CENT>::NCH * CH;
};

// VX neighbouring values of a caller's array, which is aligned to its element
// only (the plan's own channels are aligned to whole vectors).
template <typename T, int VX>
struct CallerVec {
  typedef T type __attribute__((ext_vector_type(VX), aligned(sizeof(T))));
};

template <int N>
__device__ __forceinline__ void wht(double (&v)[N]) {
#pragma unroll
  for (int bit = 1; bit < N; bit <<= 1)
#pragma unroll
    for (int e = 0; e < N; ++e)
      if (!(e & bit)) {
        const double a = v[e], c = v[e | bit];
        v[e] = a + c;
        v[e | bit] = a - c;
      }
}

// VX neighbouring points (x, x + 1) between two steps: channel values g ->
// corner values (unfold, factor eo), to f at the points' offset `at` when ST,
// times en, folded back into g.  Without IN the corner values are f_in;
// without OUT g is left alone.  No contraction: every kernel that inlines
// this rounds alike.
template <typename T, int H, int CENT, int VX, bool IN, bool OUT, bool ST>
__device__ __forceinline__ void line_point(double (&g)[LineCent<CENT>::NCH][VX], const double (&f_in)[8][VX],
                                           const double (&eo)[8][VX], const double (&en)[8][VX], T* __restrict__ f,
                                           unsigned at) {
#pragma clang fp contract(off)
  constexpr int NCH = LineCent<CENT>::NCH;
  constexpr unsigned M = 2 * H;
  typedef typename CallerVec<T, VX>::type vec;
  double u[VX][NCH], h[VX][NCH];
  bool seen[NCH] = {};
#pragma unroll
  for (int v = 0; v < VX; ++v) {
#pragma unroll
    for (int c = 0; c < NCH; ++c) {
      u[v][c] = IN ? g[c][v] : 0.0;
      h[v][c] = 0.0;
    }
    if constexpr (IN) {
      wht<NCH>(u[v]);
#pragma unroll
      for (int c = 0; c < NCH; ++c) u[v][c] = 0.125 * u[v][c];
    }
  }
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = line_class<CENT>(e);
    vec out;
#pragma unroll
    for (int v = 0; v < VX; ++v) {
      const double q = IN ? u[v][k] * eo[e][v] : f_in[e][v];
      out[v] = (T)q;
      if constexpr (OUT) {
        const double w = q * en[e][v];
        h[v][k] = seen[k] ? h[v][k] + w : w;
      }
    }
    seen[k] = true;
    if constexpr (ST) {
      vec* q = reinterpret_cast<vec*>(f + at + (unsigned)(((e & 1) + ((e >> 1) & 1) * M + (e >> 2) * M * M) * H));
      if constexpr (OUT) __builtin_nontemporal_store(out, q);  // a stored sweep's slice: read after the sweep only
      else *q = out;
    }
  }
  if constexpr (OUT) {
#pragma unroll
    for (int v = 0; v < VX; ++v) {
      wht<NCH>(h[v]);
#pragma unroll
      for (int c = 0; c < NCH; ++c) g[c][v] = h[v][c];
    }
  }
}

// Corner e of the VX points at offset `at` of one M^3 array.
template <typename T, int H, int VX>
__device__ __forceinline__ void load_corner(const T* __restrict__ f, unsigned at, int e, double (&v)[VX]) {
  constexpr unsigned M = 2 * H;
  typedef typename CallerVec<T, VX>::type vec;
  const unsigned corner = (unsigned)(((e & 1) + ((e >> 1) & 1) * M + (e >> 2) * M * M) * H);
  const vec t = *reinterpret_cast<const vec*>(f + at + corner);
#pragma unroll
  for (int i = 0; i < VX; ++i) v[i] = (double)t[i];
}

template <int VX>
__device__ __forceinline__ void ones(double (&v)[8][VX]) {
#pragma unroll
  for (int e = 0; e < 8; ++e)
#pragma unroll
    for (int i = 0; i < VX; ++i) v[e][i] = 1.0;
}

// One workgroup of n_ch waves (wave c: channel c): the points (line position
// a < H, x = kCW part + 0 .. kCW - 1) of plane `plane` of batch entry b, with
// the entry's factors at E of `step` (Eo) and of step + 1 (En).  y-lines of
// the plane z = plane, or (kLineZ) z-lines of the plane y = plane.  MODE:
// kLinesIn: the input is the channels, A_x and the line matrix applied (else
// the field f0_in); kLinesOut: folded, the line matrix applied, stored to the
// other half; kLinesStore (and always without kLinesOut): the field after Eo
// goes to f0_out.
//
// A workgroup's time is a memory latency and three passes of H/16 * H/4
// matrix instructions of 64 cycles, so the loads are ordered by use: rows,
// A_x, the line matrix, and the factors between the matrix instructions of
// the second pass.  No value test guards a load (the factor pointers are
// tested once per array): loads behind per-value tests cost 9300 of 17000
// cycles at H = 32.
template <typename T, int H, int CENT, int MODE>
__device__ __forceinline__ void ph_lines(const LineP& p, const double* Eo, const double* En, int b, int plane,
                                         int part, unsigned char* lds_raw) {
  constexpr int NCH = LineCent<CENT>::NCH;
  constexpr bool IN = (MODE & kLinesIn) != 0, OUT = (MODE & kLinesOut) != 0, ST = (MODE & kLinesStore) != 0 || !OUT;
  constexpr int NT = line_tiles(H), KS = H / 4, VAR = line_variant_len(H);
  constexpr int NTH = 64 * NCH, VX = kCW * H > NTH ? 2 : 1, XV = kCW / VX;  // VX neighbouring points per thread
  constexpr int NP = kCW * H / VX, NPT = (NP + NTH - 1) / NTH;
  constexpr bool FULL = H % kCW == 0;  // no columns past H
  constexpr unsigned M = 2 * H, H2 = (unsigned)H * H, H3 = H2 * H;
  constexpr long M3 = 8L * H3;
  typedef double vecd __attribute__((ext_vector_type(VX)));
  typedef LineStage<T, H> S;
  const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int c = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int x0 = kCW * part, line = (p.flags & kLineZ) ? 2 : 1, flip = p.flags & kLineFlip;
  const long half = (long)p.batch * NCH * H3;
  const long cb = ((long)b * NCH + c) * H3 + (line == 1 ? (unsigned)plane * H2 : (unsigned)plane * H);
  const unsigned rs = line == 1 ? (unsigned)H : H2;
  const unsigned sy = line == 1 ? M : M * M, sp = line == 1 ? M * M : M;  // strides of line position and plane
  const int av = (int)(p.axv >> (6 * c));

  // a wave's rows are staged in the bytes that then hold its channel's points
  unsigned char* own = lds_raw + c * LineLds<T, H, CENT, MODE>::CH;
  double* lds = reinterpret_cast<double*>(lds_raw);
  constexpr int LC = LineLds<T, H, CENT, MODE>::CH / 8;  // doubles per channel
  double mx[KS], ml[NT][KS];
  const T* src = static_cast<const T*>(p.ch) + flip * half + cb;
  LineRows<T, H> rows;
  if constexpr (IN) {
    load_rows<T, H>(src, rs, lane, rows);
    load_matrix<KS>(p.mats + (av & 3) * VAR + part * (KS * 64), lane, mx);
  }
  const bool other_E = IN && OUT && En != Eo;
  const double* tl = p.mats + (line * 4 + ((av >> (2 * line)) & 3)) * VAR;
  // eight waves of a workgroup leave 256 registers each, and 128 of line matrix
  // beside the staged FP64 rows spilled up to 37: read where a pass takes it, not
  // held across the others (Pm-3m 256^3, 1 and 2 fields 29.3, 54.8 -> 24.3, 44.2 us)
  constexpr bool LATE = NT * KS >= 64 && NCH == 8 && sizeof(T) == 8;
  if constexpr (!LATE) {
#pragma unroll
    for (int t = 0; t < NT; ++t) load_matrix<KS>(tl + t * (KS * 64), lane, ml[t]);
  }
  // en: the factor of the fold when it is another array (or the field, without IN)
  double eo[NPT][8][VX], en[NPT][8][VX];
  unsigned at[NPT];
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    const int pt0 = (int)threadIdx.x + k * NTH, pt = NP % NTH == 0 || pt0 < NP ? pt0 : NP - 1;
    const int xx = x0 + VX * (pt % XV);
    at[k] = (unsigned)(FULL || xx < H ? xx : H - VX) + (unsigned)(pt / XV) * sy + (unsigned)plane * sp;
    ones<VX>(eo[k]);
  }
  if constexpr (!IN) {
    if (Eo) {
#pragma unroll
      for (int k = 0; k < NPT; ++k)
#pragma unroll
        for (int e = 0; e < 8; ++e) load_corner<double, H, VX>(Eo, at[k], e, eo[k][e]);
    }
#pragma unroll
    for (int k = 0; k < NPT; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e)
        load_corner<T, H, VX>(static_cast<const T*>(p.f0_in) + b * M3, at[k], e, en[k][e]);
  }

  if constexpr (IN) {
    stage_rows<T, H>(rows, lane, own);
    wave_sync();
    mfma_d4 a1[NT], a2[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      a1[t] = mfma_d4{0.0, 0.0, 0.0, 0.0};
      a2[t] = mfma_d4{0.0, 0.0, 0.0, 0.0};
    }
    // A_x: rows of the plane (line positions) times 16 columns of A_x^T
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      if (i > 0 && 4 * i % S::W == 0) {  // the next round's columns, over the ones just read
        load_rows<T, H>(src + 4 * i, rs, lane, rows);
        wave_sync();
        stage_rows<T, H>(rows, lane, own);
        wave_sync();
      }
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int row = 16 * t + r;
        const double gv = staged<T, H>(own, H % 16 == 0 || row < H ? row : H - 1, 4 * i % S::W + g);
        a1[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(gv, mx[i], a1[t], 0, 0, 0);
      }
    }
    if constexpr (LATE) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < NT; ++t) load_matrix<KS>(tl + t * (KS * 64), lane, ml[t]);
    }
    // the line matrix: result register j of tile t is line position
    // 16 t + 4 j + l / 16, the B operand of k-step 4 t + j
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      // the factors' loads between the matrix instructions: a wave that issues
      // them ahead of phase 1 stands still until the CU has taken them
      __builtin_amdgcn_sched_barrier(0);
      if (Eo) {
#pragma unroll
        for (int j = i * NPT * 8 / KS; j < (i + 1) * NPT * 8 / KS; ++j)
          load_corner<double, H, VX>(Eo, at[j / 8], j % 8, eo[j / 8][j % 8]);
      }
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < NT; ++t)
        a2[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ml[t][i], a1[i / 4][i % 4], a2[t], 0, 0, 0);
    }
    if (other_E) {
#pragma unroll
      for (int k = 0; k < NPT; ++k) ones<VX>(en[k]);
      if (En) {
#pragma unroll
        for (int k = 0; k < NPT; ++k)
#pragma unroll
          for (int e = 0; e < 8; ++e) load_corner<double, H, VX>(En, at[k], e, en[k][e]);
      }
    }
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (16 * t + 4 * j < H) lds[c * LC + (16 * t + 4 * j + g) * kCW + r] = a2[t][j];
    __syncthreads();
  }
  T* f_out = static_cast<T*>(p.f0_out) + b * M3;
  vecd* ldv = reinterpret_cast<vecd*>(lds);
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    const int pt = (int)threadIdx.x + k * NTH;
    if (NP % NTH != 0 && pt >= NP) continue;
    double v[NCH][VX];
    if constexpr (IN) {
#pragma unroll
      for (int cc = 0; cc < NCH; ++cc) {
        const vecd w = ldv[cc * (LC / VX) + pt];
#pragma unroll
        for (int i = 0; i < VX; ++i) v[cc][i] = w[i];
      }
    }
    // columns past H (part-filled tiles) hold no field point
    const bool out = ST && (FULL || x0 + VX * (pt % XV) < H);
    auto point = [&](const double(&a)[8][VX], const double(&w)[8][VX]) {
      if (out) line_point<T, H, CENT, VX, IN, OUT, ST>(v, en[k], a, w, f_out, at[k]);
      else line_point<T, H, CENT, VX, IN, OUT, false>(v, en[k], a, w, f_out, at[k]);
    };
    if (other_E) {
      point(eo[k], en[k]);
    } else {
      // taken here, not where the loads are issued: a copy of eo into en's
      // registers up there would wait for it
      double w[8][VX];
#pragma unroll
      for (int e = 0; e < 8; ++e)
#pragma unroll
        for (int i = 0; i < VX; ++i) {
          w[e][i] = eo[k][e][i];
          asm volatile("" : "+v"(w[e][i]));
        }
      point(eo[k], w);
    }
    if constexpr (OUT) {
#pragma unroll
      for (int cc = 0; cc < NCH; ++cc) {
        vecd w;
#pragma unroll
        for (int i = 0; i < VX; ++i) w[i] = v[cc][i];
        ldv[cc * (LC / VX) + pt] = w;
      }
    }
  }
  if constexpr (OUT) {
    if constexpr (LATE) {
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int t = 0; t < NT; ++t) load_matrix<KS>(tl + t * (KS * 64), lane, ml[t]);
    }
    __syncthreads();
    mfma_d4 a3[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) a3[t] = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const double w = lds[c * LC + (4 * i + g) * kCW + r];
#pragma unroll
      for (int t = 0; t < NT; ++t) a3[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ml[t][i], w, a3[t], 0, 0, 0);
    }
    T* dst = static_cast<T*>(p.ch) + (1 - flip) * half + cb;
    const int x = x0 + r;
    if (FULL || x < H) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (16 * t + 4 * j < H) dst[(unsigned)(16 * t + 4 * j + g) * rs + (unsigned)x] = (T)a3[t][j];
    }
  }
}

// Workgroup -> (plane of all batch entries, x part).  The parts of a plane
// read the whole plane: blocks go to the 8 XCDs round robin, so the parts of
// plane 8 j + i are the blocks of that i in group j and share an L2.
__host__ __device__ __forceinline__ void lines_item(unsigned parts, unsigned blk, unsigned n_planes, unsigned& pl,
                                                    unsigned& part) {
  if (parts > 1 && n_planes % 8 == 0) {
    const unsigned j = blk >> 3;
    part = j % parts;
    pl = (j / parts) * 8 + (blk & 7);
  } else {
    part = blk % parts;
    pl = blk / parts;
  }
}

// Factors of batch entry b at `step`.
__device__ __forceinline__ const double* line_E(const LineEnt::Entry& e, int step) { return step < e.sw ? e.e1 : e.e2; }

// Three waves per SIMD for H <= 32: below that the compiler moves the
// accumulators through the second register file (Im-3m 128^3, 2 fields FP64
// 6.1 -> 5.8 us, 16 fields mixed 13.6 -> 11.9).  Two with two channels, whose
// threads hold two pairs of points at H = 24 and 32: three spilled 4 to 124
// registers (Fm-3m 128^3, 1, 2, 8 fields FP64 6.5, 6.8, 11.5 -> 5.4, 5.6, 8.6 us,
// mixed 5.4, 5.6, 8.8 -> 5.1, 5.2, 7.8; 96^3 5.28, 5.34, 7.4 -> 5.12, 5.19, 7.2).
// No instance has scratch memory.
constexpr int line_waves(int H, int nch) { return H <= 32 ? (H > 16 && nch == 2 ? 2 : 3) : 1; }

template <typename T, int H, int CENT, int MODE>
__global__ void __launch_bounds__(64 * LineCent<CENT>::NCH, line_waves(H, LineCent<CENT>::NCH))
    k_lines(void* ch, const double* mats, unsigned long long axv, int batch, int step, int flags, const double* E,
            const void* f0_in, void* f0_out, LineEnt ents) {
  __shared__ __align__(16) unsigned char lds[LineLds<T, H, CENT, MODE>::BYTES];
  constexpr long M3 = 8L * H * H * H;
  unsigned pl, part;
  lines_item(line_parts(H), blockIdx.x, (unsigned)(batch * H), pl, part);
  const int b = (int)(pl / H);
  const LineEnt::Entry ent = ents.ent[(flags & kLineContig) ? 0 : b];
  const double* all = E ? E + b * M3 : nullptr;
  const double* Eo = (flags & kLineContig) ? all : line_E(ent, step);
  const double* En = (flags & kLineContig) ? all : line_E(ent, step + 1);
  ph_lines<T, H, CENT, MODE>(LineP{ch, mats, axv, batch, step, flags, E, f0_in, f0_out}, Eo, En, b, (int)(pl % H),
                                 (int)part, lds);
}

// Launches k_lines over every plane of the plan (lines.hip).
template <typename T>
void launch_lines_prec(int H, int cent, int mode, const LineP& p, const LineEnt& e, hipStream_t s);
extern template void launch_lines_prec<double>(int, int, int, const LineP&, const LineEnt&, hipStream_t);
extern template void launch_lines_prec<float>(int, int, int, const LineP&, const LineEnt&, hipStream_t);
void launch_lines(int prec, int H, int cent, int mode, const LineP& p, const LineEnt& e, hipStream_t s);

}  // namespace cfft
