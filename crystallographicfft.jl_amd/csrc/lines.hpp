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
// kernel.  A workgroup takes the line axis in full and 16 x-values of one
// plane; A_x reads the plane's other x-values (shared by the plane's
// workgroups through the L2).  Source and destination channels alternate
// between the two halves of the plan's channel buffer.
#pragma once

#include <hip/hip_runtime.h>

#include "pipeline.hpp"
#include "plan.hpp"

namespace cfft {

typedef double mfma_d4 __attribute__((ext_vector_type(4)));

constexpr int kLineLens[] = {8, 12, 16, 24, 32, 48, 64};
inline bool line_len_ok(int H) {
  for (int v : kLineLens)
    if (v == H) return true;
  return false;
}

// Matrix table (B.lines): entry [axis][variant][tile t][k-step i][lane] with
// variant = o | (chi < 0) << 1, tiles of 16 matrix rows, H/4 k-steps.  Lane l
// of axis 0 holds A[16 t + l % 16][(H/4) (l / 16) + i] (the contraction order
// of rows read from memory, (H/4) consecutive values per lane), lane l of
// axes 1, 2 holds A[16 t + l % 16][4 i + l / 16] (the order in which the
// matrix instruction leaves its result); rows past H are 0.  An even number
// of k-steps is stored in pairs, one 16-byte load each.
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

// KS consecutive values at p (aligned to their power-of-two part) as doubles.
template <typename T, int KS>
__device__ __forceinline__ void load_run(const T* __restrict__ p, double (&v)[KS]) {
  constexpr int BYTES = KS * (int)sizeof(T);
  constexpr int VB = BYTES % 16 == 0 ? 16 : (BYTES % 8 == 0 ? 8 : 4);
  constexpr int VE = VB / (int)sizeof(T);
  typedef T vec __attribute__((ext_vector_type(VE)));
  if constexpr (VE == 1) {
#pragma unroll
    for (int i = 0; i < KS; ++i) v[i] = (double)p[i];
  } else {
    vec t[KS / VE];
#pragma unroll
    for (int i = 0; i < KS / VE; ++i) t[i] = reinterpret_cast<const vec*>(p)[i];
#pragma unroll
    for (int i = 0; i < KS / VE; ++i)
#pragma unroll
      for (int j = 0; j < VE; ++j) v[i * VE + j] = (double)t[i][j];
  }
}

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

// One point between two steps: channel values g -> corner values (unfold,
// factor eo), to f[off of the corner] when ST, times en, folded back into g.
// Without IN the corner values are f_in; without OUT g is left alone.  No
// contraction: every kernel that inlines this rounds alike.
template <typename T, int H, int CENT, bool IN, bool OUT, bool ST>
__device__ __forceinline__ void line_point(double (&g)[LineCent<CENT>::NCH], const double (&f_in)[8],
                                           const double (&eo)[8], const double (&en)[8], T* __restrict__ f,
                                           unsigned at) {
#pragma clang fp contract(off)
  constexpr int NCH = LineCent<CENT>::NCH;
  constexpr unsigned M = 2 * H;
  if constexpr (IN) {
    wht<NCH>(g);
#pragma unroll
    for (int c = 0; c < NCH; ++c) g[c] = 0.125 * g[c];
  }
  double h[NCH];
#pragma unroll
  for (int c = 0; c < NCH; ++c) h[c] = 0.0;
  bool seen[NCH] = {};
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const int k = line_class<CENT>(e);
    const double u = IN ? g[k] * eo[e] : f_in[e];
    if constexpr (ST) {
      T* q = f + at + (unsigned)(((e & 1) + ((e >> 1) & 1) * M + (e >> 2) * M * M) * H);
      if constexpr (OUT) __builtin_nontemporal_store((T)u, q);  // a stored sweep's slice: read after the sweep only
      else *q = (T)u;
    }
    if constexpr (OUT) {
      const double w = u * en[e];
      h[k] = seen[k] ? h[k] + w : w;
      seen[k] = true;
    }
  }
  if constexpr (OUT) {
    wht<NCH>(h);
#pragma unroll
    for (int c = 0; c < NCH; ++c) g[c] = h[c];
  }
}

// The 8 corner values of the point at offset `at` of one M^3 array.
template <typename T, int H>
__device__ __forceinline__ void load_corners(const T* __restrict__ f, unsigned at, double (&v)[8]) {
  constexpr unsigned M = 2 * H;
#pragma unroll
  for (int e = 0; e < 8; ++e) v[e] = (double)f[at + (unsigned)(((e & 1) + ((e >> 1) & 1) * M + (e >> 2) * M * M) * H)];
}

enum { kLinesIn = 1, kLinesOut = 2, kLinesStore = 4 };

// One workgroup of n_ch waves (wave c: channel c): the points (line position
// a < H, x = 16 part + 0..15) of plane `plane` of batch entry b.  line = 1:
// y-lines of the plane z = plane; line = 2: z-lines of the plane y = plane.
// MODE: kLinesIn: the input is the channels at half `flip` of B.ch, A_x and
// the line matrix applied (else the field B.f0_in); kLinesOut: folded, the
// line matrix applied, stored to the other half; kLinesStore (and always
// without kLinesOut): the field after E of `step` goes to B.f0_out.
//
// Every load is issued before the first use: per plane and step the
// dependent chain is one memory latency, three passes of H/16 * H/4 matrix
// instructions (64 cycles each) and two LDS exchanges.  Loads behind
// per-value tests of the factor pointers cost 9300 of the kernel's 17000
// cycles at H = 32; tested once per array they overlap.
template <typename T, int H, int CENT, int MODE>
__device__ __forceinline__ void ph_lines(const PipeP& p, const PipeBufs& B, int b, int plane, int part, int step,
                                         int line, int flip, double* lds) {
  constexpr int NCH = LineCent<CENT>::NCH;
  constexpr bool IN = (MODE & kLinesIn) != 0, OUT = (MODE & kLinesOut) != 0, ST = (MODE & kLinesStore) != 0 || !OUT;
  constexpr int NT = line_tiles(H), KS = H / 4, VAR = line_variant_len(H);
  constexpr int NTH = 64 * NCH, NP = 16 * H, NPT = (NP + NTH - 1) / NTH;
  constexpr unsigned M = 2 * H, H2 = (unsigned)H * H, H3 = H2 * H;
  constexpr long M3 = 8L * H3;
  const int lane = threadIdx.x & 63, g = lane >> 4, r = lane & 15;
  const int c = __builtin_amdgcn_readfirstlane((int)threadIdx.x >> 6);
  const int x0 = 16 * part;
  const long half = (long)p.batch * NCH * H3;
  const long cb = ((long)b * NCH + c) * H3 + (line == 1 ? (unsigned)plane * H2 : (unsigned)plane * H);
  const unsigned rs = line == 1 ? (unsigned)H : H2;
  const unsigned sy = line == 1 ? M : M * M, sp = line == 1 ? M * M : M;  // strides of line position and plane
  const int av = p.axv[c];

  double gv[NT][KS], mx[KS], ml[NT][KS];
  if constexpr (IN) {
    const T* src = static_cast<const T*>(B.ch) + flip * half + cb;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int row = 16 * t + r;
      load_run<T, KS>(src + ((unsigned)(H % 16 == 0 || row < H ? row : H - 1) * rs + (unsigned)(KS * g)), gv[t]);
    }
  }
  const double* Eo = pipe_E(p, b, step, M3);
  const double* En = IN ? pipe_E(p, b, step + 1, M3) : Eo;
  const bool other_E = IN && OUT && En != Eo;
  double eo[NPT][8], en[NPT][8];  // en: the factor of the fold when it is another array (or the field, without IN)
  unsigned at[NPT];
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    const int pt0 = (int)threadIdx.x + k * NTH, pt = NP % NTH == 0 || pt0 < NP ? pt0 : NP - 1;
    const int xx = x0 + (pt & 15);
    at[k] = (unsigned)(H % 16 == 0 || xx < H ? xx : H - 1) + (unsigned)(pt >> 4) * sy + (unsigned)plane * sp;
  }
  if (Eo) {
#pragma unroll
    for (int k = 0; k < NPT; ++k) load_corners<double, H>(Eo, at[k], eo[k]);
  } else {
#pragma unroll
    for (int k = 0; k < NPT; ++k)
#pragma unroll
      for (int e = 0; e < 8; ++e) eo[k][e] = 1.0;
  }
  if constexpr (IN) {
    load_matrix<KS>(B.lines + (long)(av & 3) * VAR + part * (KS * 64), lane, mx);
    if (other_E) {
      if (En) {
#pragma unroll
        for (int k = 0; k < NPT; ++k) load_corners<double, H>(En, at[k], en[k]);
      } else {
#pragma unroll
        for (int k = 0; k < NPT; ++k)
#pragma unroll
          for (int e = 0; e < 8; ++e) en[k][e] = 1.0;
      }
    }
  } else {
#pragma unroll
    for (int k = 0; k < NPT; ++k) load_corners<T, H>(static_cast<const T*>(B.f0_in) + b * M3, at[k], en[k]);
  }
  const double* tl = B.lines + ((long)line * 4 + ((av >> (2 * line)) & 3)) * VAR;
#pragma unroll
  for (int t = 0; t < NT; ++t) load_matrix<KS>(tl + t * (KS * 64), lane, ml[t]);

  if constexpr (IN) {
    mfma_d4 a1[NT], a2[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      a1[t] = mfma_d4{0.0, 0.0, 0.0, 0.0};
      a2[t] = mfma_d4{0.0, 0.0, 0.0, 0.0};
    }
    // A_x: rows of the plane (line positions) times the part's 16 columns of A_x^T
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t) a1[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(gv[t][i], mx[i], a1[t], 0, 0, 0);
    // the line matrix: result register j of tile t is line position
    // 16 t + 4 j + l / 16, the B operand of k-step 4 t + j
#pragma unroll
    for (int i = 0; i < KS; ++i)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        a2[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ml[t][i], a1[i / 4][i % 4], a2[t], 0, 0, 0);
#pragma unroll
    for (int t = 0; t < NT; ++t)
#pragma unroll
      for (int j = 0; j < 4; ++j)
        if (16 * t + 4 * j < H) lds[(c * H + 16 * t + 4 * j + g) * 16 + r] = a2[t][j];
    __syncthreads();
  }
  T* f_out = static_cast<T*>(B.f0_out) + b * M3;
#pragma unroll
  for (int k = 0; k < NPT; ++k) {
    const int pt = (int)threadIdx.x + k * NTH;
    if (NP % NTH != 0 && pt >= NP) continue;
    double v[NCH];
    if constexpr (IN) {
#pragma unroll
      for (int cc = 0; cc < NCH; ++cc) v[cc] = lds[cc * NP + pt];
    }
    // columns past H (part-filled tiles) hold no field point
    const bool out = ST && (H % 16 == 0 || x0 + (pt & 15) < H);
    auto point = [&](const double(&a)[8], const double(&w)[8]) {
      if (out) line_point<T, H, CENT, IN, OUT, ST>(v, en[k], a, w, f_out, at[k]);
      else line_point<T, H, CENT, IN, OUT, false>(v, en[k], a, w, f_out, at[k]);
    };
    if (other_E) {
      point(eo[k], en[k]);
    } else {
      // taken here, not where the loads are issued: a copy of eo into en's
      // registers up there would wait for it
      double w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) {
        w[e] = eo[k][e];
        asm volatile("" : "+v"(w[e]));
      }
      point(eo[k], w);
    }
    if constexpr (OUT) {
#pragma unroll
      for (int cc = 0; cc < NCH; ++cc) lds[cc * NP + pt] = v[cc];
    }
  }
  if constexpr (OUT) {
    __syncthreads();
    mfma_d4 a3[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) a3[t] = mfma_d4{0.0, 0.0, 0.0, 0.0};
#pragma unroll
    for (int i = 0; i < KS; ++i) {
      const double w = lds[(c * H + 4 * i + g) * 16 + r];
#pragma unroll
      for (int t = 0; t < NT; ++t) a3[t] = __builtin_amdgcn_mfma_f64_16x16x4f64(ml[t][i], w, a3[t], 0, 0, 0);
    }
    T* dst = static_cast<T*>(B.ch) + (1 - flip) * half + cb;
    if (H % 16 == 0 || x0 + r < H) {
#pragma unroll
      for (int t = 0; t < NT; ++t)
#pragma unroll
        for (int j = 0; j < 4; ++j)
          if (16 * t + 4 * j < H) dst[(unsigned)(16 * t + 4 * j + g) * rs + (unsigned)(x0 + r)] = (T)a3[t][j];
    }
  }
}

// Workgroup -> (plane of all batch entries, x part).  The parts of a plane
// read the whole plane: blocks go to the 8 XCDs round robin, so the parts of
// plane 8 j + i are the blocks of that i in group j and share an L2.
template <int NT>
__host__ __device__ __forceinline__ void lines_item(unsigned blk, unsigned n_planes, unsigned& pl, unsigned& part) {
  if (NT > 1 && n_planes % 8 == 0) {
    const unsigned j = blk >> 3;
    part = j % NT;
    pl = (j / NT) * 8 + (blk & 7);
  } else {
    part = blk % NT;
    pl = blk / NT;
  }
}

template <typename T, int H, int CENT, int MODE>
__global__ void __launch_bounds__(64 * LineCent<CENT>::NCH) k_lines(PipeP p, PipeBufs B, int step, int line, int flip) {
  __shared__ double lds[LineCent<CENT>::NCH * H * 16];
  unsigned pl, part;
  lines_item<line_tiles(H)>(blockIdx.x, (unsigned)(p.batch * H), pl, part);
  ph_lines<T, H, CENT, MODE>(p, B, (int)(pl / H), (int)(pl % H), (int)part, step, line, flip, lds);
}

// Launches k_lines over every plane of the plan (lines.hip).
void launch_lines(int prec, int H, int cent, int mode, const PipeP& p, const PipeBufs& B, int step, int line,
                  int flip, hipStream_t s);

}  // namespace cfft
