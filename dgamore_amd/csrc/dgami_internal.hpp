// Shared device/host helpers for libdgami (gfx950, CDNA4).
//
// Complex numbers are interleaved (re, im) doubles, i.e. the memory layout of
// numpy.complex128; on the device they are handled as HIP's double2.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>
#include <cstdio>
#include <string>

namespace dgami {

// ----------------------------------------------------------------------------
// complex double helpers
// ----------------------------------------------------------------------------
__host__ __device__ __forceinline__ double2 cmk(double r, double i) { return make_double2(r, i); }
__host__ __device__ __forceinline__ double2 cadd(double2 a, double2 b) { return make_double2(a.x + b.x, a.y + b.y); }
__host__ __device__ __forceinline__ double2 csub(double2 a, double2 b) { return make_double2(a.x - b.x, a.y - b.y); }
__host__ __device__ __forceinline__ double2 cmul(double2 a, double2 b) {
  return make_double2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__host__ __device__ __forceinline__ double2 cscale(double2 a, double s) { return make_double2(a.x * s, a.y * s); }
__host__ __device__ __forceinline__ double2 cconj(double2 a) { return make_double2(a.x, -a.y); }
// a - b*c
__host__ __device__ __forceinline__ double2 cfms(double2 a, double2 b, double2 c) {
  double re = fma(-b.x, c.x, a.x);
  re = fma(b.y, c.y, re);
  double im = fma(-b.x, c.y, a.y);
  im = fma(-b.y, c.x, im);
  return make_double2(re, im);
}
// a + b*c
__host__ __device__ __forceinline__ double2 cfma(double2 a, double2 b, double2 c) {
  double re = fma(b.x, c.x, a.x);
  re = fma(-b.y, c.y, re);
  double im = fma(b.x, c.y, a.y);
  im = fma(b.y, c.x, im);
  return make_double2(re, im);
}
// 1/b with Smith's scaling (robust against over/underflow of |b|^2)
__host__ __device__ __forceinline__ double2 cinv(double2 b) {
  if (fabs(b.x) >= fabs(b.y)) {
    double r = b.y / b.x;
    double d = b.x + b.y * r;
    return make_double2(1.0 / d, -r / d);
  }
  double r = b.x / b.y;
  double d = b.x * r + b.y;
  return make_double2(r / d, -1.0 / d);
}
__host__ __device__ __forceinline__ double cabs1(double2 a) { return fabs(a.x) + fabs(a.y); }

// complex float (interleaved, numpy.complex64 layout)
__host__ __device__ __forceinline__ float2 cadd(float2 a, float2 b) { return make_float2(a.x + b.x, a.y + b.y); }
__host__ __device__ __forceinline__ float2 csub(float2 a, float2 b) { return make_float2(a.x - b.x, a.y - b.y); }
__host__ __device__ __forceinline__ float2 cmul(float2 a, float2 b) {
  return make_float2(a.x * b.x - a.y * b.y, a.x * b.y + a.y * b.x);
}
__host__ __device__ __forceinline__ float2 cfms(float2 a, float2 b, float2 c) {
  float re = fmaf(-b.x, c.x, a.x);
  re = fmaf(b.y, c.y, re);
  float im = fmaf(-b.x, c.y, a.y);
  im = fmaf(-b.y, c.x, im);
  return make_float2(re, im);
}
__host__ __device__ __forceinline__ float2 cfma(float2 a, float2 b, float2 c) {
  float re = fmaf(b.x, c.x, a.x);
  re = fmaf(-b.y, c.y, re);
  float im = fmaf(b.x, c.y, a.y);
  im = fmaf(b.y, c.x, im);
  return make_float2(re, im);
}
__host__ __device__ __forceinline__ float2 cinv(float2 b) {
  if (fabsf(b.x) >= fabsf(b.y)) {
    float r = b.y / b.x;
    float d = b.x + b.y * r;
    return make_float2(1.0f / d, -r / d);
  }
  float r = b.x / b.y;
  float d = b.x * r + b.y;
  return make_float2(r / d, -1.0f / d);
}
__host__ __device__ __forceinline__ float cabs1(float2 a) { return fabsf(a.x) + fabsf(a.y); }

// conversions and zero of the two storage types
template <typename S>
__host__ __device__ __forceinline__ S czero();
template <>
__host__ __device__ __forceinline__ double2 czero<double2>() { return make_double2(0.0, 0.0); }
template <>
__host__ __device__ __forceinline__ float2 czero<float2>() { return make_float2(0.0f, 0.0f); }
template <typename S>
__host__ __device__ __forceinline__ S from_c128(double2 v);
template <>
__host__ __device__ __forceinline__ double2 from_c128<double2>(double2 v) { return v; }
template <>
__host__ __device__ __forceinline__ float2 from_c128<float2>(double2 v) {
  return make_float2(static_cast<float>(v.x), static_cast<float>(v.y));
}
__host__ __device__ __forceinline__ double2 to_c128(double2 v) { return v; }
__host__ __device__ __forceinline__ double2 to_c128(float2 v) {
  return make_double2(static_cast<double>(v.x), static_cast<double>(v.y));
}

// ----------------------------------------------------------------------------
// XCD-aware tile order. Workgroups are dispatched round-robin over MI355X's 8 XCDs, each
// with its own L2. With a grid of xcd_grid(nprob, per) workgroups, xcd_tile maps the
// linear id so that all `per` tiles of one problem run on the same XCD and share its L2
// copy of the problem's operand panels. Returns false for the padding ids.
// ----------------------------------------------------------------------------
constexpr int NUM_XCD = 8;

inline size_t xcd_grid(size_t nprob, size_t per) { return (nprob + NUM_XCD - 1) / NUM_XCD * NUM_XCD * per; }

__device__ __forceinline__ bool xcd_tile(unsigned id, int nprob, int per, int& prob, int& tile) {
  const unsigned x = id % NUM_XCD, slot = id / NUM_XCD;
  const unsigned j = slot / per;
  tile = static_cast<int>(slot - j * per);
  prob = static_cast<int>(j * NUM_XCD + x);
  return prob < nprob;
}

// ----------------------------------------------------------------------------
// Wavefront maximum of a 32-bit key with DPP row shifts and row broadcasts (the result
// collects in lane 63 and is returned uniform). Pivot searches reduce the key
// (upper word of the FP64 magnitude) + 1, then pick the lowest lane holding the maximum.
// ----------------------------------------------------------------------------
__device__ __forceinline__ unsigned wave_max_u32(unsigned v) {
  v = max(v, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x111, 0xf, 0xf, false)));
  v = max(v, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x112, 0xf, 0xf, false)));
  v = max(v, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x114, 0xf, 0xf, false)));
  v = max(v, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x118, 0xf, 0xf, false)));
  v = max(v, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x142, 0xa, 0xf, false)));
  v = max(v, static_cast<unsigned>(__builtin_amdgcn_update_dpp(0, static_cast<int>(v), 0x143, 0xc, 0xf, false)));
  return static_cast<unsigned>(__builtin_amdgcn_readlane(static_cast<int>(v), 63));
}

__device__ __forceinline__ unsigned pivot_key(double mag, bool valid) {
  return valid ? static_cast<unsigned>(__double_as_longlong(mag) >> 32) + 1u : 0u;
}

// ----------------------------------------------------------------------------
// error reporting (thread-local last error; host side)
// ----------------------------------------------------------------------------
void set_error(const std::string& msg);
const char* last_error();

#define DGAMI_ARG_CHECK(cond, msg)      \
  do {                                  \
    if (!(cond)) {                      \
      ::dgami::set_error(msg);          \
      return -1;                        \
    }                                   \
  } while (0)

#define DGAMI_HIP_CHECK(expr)                                                              \
  do {                                                                                     \
    hipError_t _e = (expr);                                                                \
    if (_e != hipSuccess) {                                                                \
      ::dgami::set_error(std::string("HIP error in " #expr ": ") + hipGetErrorString(_e)); \
      return -2;                                                                           \
    }                                                                                      \
  } while (0)

// Kernel timing (dgami_profile_enable): profile_begin records a start event on the stream,
// profile_end the stop event together with the launch's algorithmic bytes and flops.
bool profile_on();
int profile_begin(hipStream_t stream, hipEvent_t* start);
int profile_end(hipStream_t stream, hipEvent_t start, double bytes, double flops);

// Grow-only device scratch owned by the library, one slot per purpose id.
// Returns nullptr (and sets the error) when the allocation fails.
void* workspace(int slot, size_t bytes);
// Bytes the slot holds on the current device now.
size_t workspace_bytes(int slot);

inline unsigned ceil_div(size_t a, size_t b) { return static_cast<unsigned>((a + b - 1) / b); }

// A grid of `blocks` workgroups in two dimensions (a launch holds fewer than 2^32 work-items in one):
// workgroup flat_block() of it, those from `blocks` on are padding.
inline dim3 flat_grid(size_t blocks) {
  const size_t x = blocks < (size_t(1) << 20) ? blocks : size_t(1) << 20;
  return dim3(static_cast<unsigned>(x), static_cast<unsigned>((blocks + x - 1) / x));
}
__device__ __forceinline__ unsigned flat_block() { return blockIdx.y * gridDim.x + blockIdx.x; }

// Allow a kernel to use more than the default 64 KiB of dynamic LDS (gfx950 has 160 KiB per CU).
template <typename K>
inline void allow_lds(K kernel, size_t bytes) {
  if (bytes > 48 * 1024)
    (void)hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize,
                              static_cast<int>(bytes));
}

// ----------------------------------------------------------------------------
// in-LDS mixed-radix momentum FFT (radices 2, 3, 4, 5, 6, 8), Stockham autosort
// ----------------------------------------------------------------------------
// One block holds one [nx][ny][nz] slab. What bounds it is LDS traffic and, before that, index
// arithmetic: with the stage shapes known only at run time, dividing every butterfly number by
// them cost more than the transform. The plan therefore carries the reciprocals (fft_div), few
// stages with large radices (24 = 6 4, 64 = 8 8: two passes over the slab per axis), and an LDS
// row length made odd, so that 16 lanes on 16 rows touch 16 different bank groups. The first axis
// is the slowest one, whose lanes run along the contiguous index: a caller's load function reads
// global memory in order and the slab's first pass over LDS is a write.
constexpr int FFT_MAX_STAGES = 12;  // a grid of at most 4096 points, each stage at least radix 2
constexpr int FFT_MAX_POINTS = 4096;
constexpr int FFT_MAX_THREADS = 512;
constexpr int FFT_MAX_ELEMS = 9;  // slab elements per thread at the planned block size

// Butterflies per thread of one stage at the planned block size (fft_block_threads): N / R
// butterflies over at least N / 9 threads, N / 8 where a radix-8 stage occurs.
__host__ __device__ constexpr int fft_max_bfly(int R) { return R == 8 ? 1 : R >= 5 ? 2 : R >= 3 ? 3 : 5; }

struct FftStage {
  int radix, len, ns;  // radix, axis length, product of the axis' earlier radices
  int nfft, nf2;       // transforms in the slab; transform f starts at (f / nf2) s1 + f % nf2 (row
  int s1, xs;          // stage: f s1), its elements are xs apart in LDS
  int tw;              // offset of the axis' twiddles
  float r_nfft, r_ns, r_nf2;
};

// Momentum-grid FFT plan: LDS layout and the stages of all axes in order.
struct FftPlan3D {
  int n[3];
  int ntot;
  int nrow;    // length of the contiguous axis
  int rowlen;  // its padded LDS length (odd)
  int nlds;    // complex elements of the LDS slab
  int ntw;     // complex elements of the twiddle tables
  int axis[3], axis_tw[3];  // lengths of the axes longer than 1, slowest first, and their tables
  int naxis;
  int nstage;
  int threads;  // block size the butterfly budget holds for
  float r_nrow;
  FftStage st[FFT_MAX_STAGES];
};

// b / d with the stored reciprocal 1.0f / d: (b + 1/2) / d stays 1/(2 d) away from the next
// integer, more than the rounding of a product below 2^12, so the quotient is exact for
// b <= 4096.
__device__ __forceinline__ int fft_div(int b, float rd) { return static_cast<int>((b + 0.5f) * rd); }

// Radices of one axis: the fewest stages, then the smallest largest radix; largest first, so that
// the stages with twiddles are the cheap ones. Returns the number of stages, 0 if len does not
// factor into 2, 3 and 5.
inline int fft_radices(int len, int* radix) {
  static const int all[6] = {8, 6, 5, 4, 3, 2};
  int best = 0, best_max = 0;
  int cur[FFT_MAX_STAGES + 1];
  struct Search {
    int* cur;
    int* radix;
    int* best;
    int* best_max;
    void run(int m, int depth, int from) {
      if (m == 1) {
        if (*best == 0 || depth < *best || (depth == *best && cur[0] < *best_max)) {
          *best = depth;
          *best_max = cur[0];
          for (int i = 0; i < depth; ++i) radix[i] = cur[i];
        }
        return;
      }
      if (depth == FFT_MAX_STAGES || (*best && depth + 1 > *best)) return;
      for (int i = from; i < 6; ++i)
        if (m % all[i] == 0) {
          cur[depth] = all[i];
          run(m / all[i], depth + 1, i);
        }
    }
  } search{cur, radix, &best, &best_max};
  search.run(len, 0, 0);
  return best;
}

// False if a length does not factor into 2, 3 and 5. A grid above FFT_MAX_POINTS gets no stages
// (fft_grid_fits is false for it).
inline bool fft_plan_3d(int nx, int ny, int nz, FftPlan3D* p) {
  *p = FftPlan3D{};
  const int n[3] = {nx, ny, nz};
  int64_t total = 1;
  for (int d = 0; d < 3; ++d) {
    p->n[d] = n[d];
    total *= n[d];
    int m = n[d];
    while (m % 2 == 0) m /= 2;
    while (m % 3 == 0) m /= 3;
    while (m % 5 == 0) m /= 5;
    if (m != 1 || total >= (int64_t(1) << 31)) return false;
  }
  p->ntot = static_cast<int>(total);
  for (int d = 0; d < 3; ++d)
    if (n[d] > 1) p->axis[p->naxis++] = n[d];
  p->nrow = p->naxis ? p->axis[p->naxis - 1] : 1;
  p->r_nrow = 1.0f / p->nrow;
  p->rowlen = p->nrow | 1;
  if (total > FFT_MAX_POINTS) return true;
  p->nlds = p->ntot / p->nrow * p->rowlen;
  int elems = FFT_MAX_ELEMS;
  int inner = p->ntot;  // points of the axes after this one
  for (int d = 0; d < p->naxis; ++d) {
    const int len = p->axis[d];
    const bool row = d == p->naxis - 1;
    inner /= len;
    const int outer = p->ntot / (len * inner);
    int radix[FFT_MAX_STAGES + 1];
    const int ns = fft_radices(len, radix);
    p->axis_tw[d] = p->ntw;
    int done = 1;
    for (int s = 0; s < ns; ++s) {
      FftStage& st = p->st[p->nstage++];
      if (radix[s] == 8) elems = 8;
      st.radix = radix[s];
      st.len = len;
      st.ns = done;
      st.nfft = p->ntot / len;
      st.tw = p->ntw;
      // transforms run over (outer, inner); inner = (middle axis, row) has padded rows
      st.xs = row ? 1 : inner / p->nrow * p->rowlen;
      st.nf2 = row ? 1 : p->nrow;  // f -> (row index, position in the row)
      st.s1 = p->rowlen;
      if (!row && outer > 1) st.s1 = len * st.xs;  // middle axis of three: inner is one row
      st.r_nfft = 1.0f / st.nfft;
      st.r_ns = 1.0f / st.ns;
      st.r_nf2 = 1.0f / st.nf2;
      done *= radix[s];
    }
    p->ntw += len;
  }
  const int need = (p->ntot + elems - 1) / elems;
  p->threads = (need + 63) / 64 * 64;
  return true;
}

// Grids the kernels take: 4096 points, 3840 where an axis has a factor 3 or 5.
inline bool fft_grid_fits(const FftPlan3D& p) {
  const bool pow2 = (p.ntot & (p.ntot - 1)) == 0;
  return p.ntot <= (pow2 ? FFT_MAX_POINTS : 3840);
}

// Threads per block so that every stage of a transform of one grid fits the per-thread butterfly
// budget (a multiple of 64; more threads than that are fine).
inline int fft_block_threads(const FftPlan3D& p) { return p.threads; }

// LDS of one slab and its twiddles.
inline size_t fft_lds_bytes(const FftPlan3D& p) { return (static_cast<size_t>(p.nlds) + p.ntw) * sizeof(double2); }

// Position in the LDS slab of grid point r.
__device__ __forceinline__ int fft_pos(const FftPlan3D& p, int r) {
  return r + fft_div(r, p.r_nrow) * (p.rowlen - p.nrow);
}

// Small DFT kernels on registers; BACK: e^{+i}, else e^{-i}.
template <int R, bool BACK>
__device__ __forceinline__ void dft_small(double2* v) {
  constexpr double sign = BACK ? 1.0 : -1.0;
  auto rot = [](double2 a) { return BACK ? make_double2(-a.y, a.x) : make_double2(a.y, -a.x); };  // (sign i) a
  if constexpr (R == 2) {
    const double2 a = v[0], b = v[1];
    v[0] = cadd(a, b);
    v[1] = csub(a, b);
  } else if constexpr (R == 3) {
    // w = -1/2 + sign i sqrt(3)/2
    constexpr double s3 = 0.86602540378443864676 * sign;
    const double2 t1 = cadd(v[1], v[2]), t2 = csub(v[1], v[2]);
    const double2 m = make_double2(v[0].x - 0.5 * t1.x, v[0].y - 0.5 * t1.y);
    const double2 r = make_double2(-s3 * t2.y, s3 * t2.x);
    v[0] = cadd(v[0], t1);
    v[1] = cadd(m, r);
    v[2] = csub(m, r);
  } else if constexpr (R == 4) {
    const double2 a0 = cadd(v[0], v[2]), a1 = csub(v[0], v[2]);
    const double2 b0 = cadd(v[1], v[3]), b1 = rot(csub(v[1], v[3]));
    v[0] = cadd(a0, b0);
    v[2] = csub(a0, b0);
    v[1] = cadd(a1, b1);
    v[3] = csub(a1, b1);
  } else if constexpr (R == 5) {
    // with t1 = x1 + x4, t2 = x2 + x3, t3 = x1 - x4, t4 = x2 - x3:
    //   X0 = x0 + t1 + t2,  X1,4 = a1 +- i b1,  X2,3 = a2 +- i b2,
    //   a1 = x0 + c1 t1 + c2 t2, a2 = x0 + c2 t1 + c1 t2 (c_k = cos(2 pi k / 5)),
    //   b1 = sign (s1 t3 + s2 t4), b2 = sign (s2 t3 - s1 t4) (s_k = sin(2 pi k / 5))
    constexpr double c1 = 0.30901699437494742410, c2 = -0.80901699437494742410;
    constexpr double s1 = 0.95105651629515357212 * sign, s2 = 0.58778525229247312917 * sign;
    const double2 t1 = cadd(v[1], v[4]), t2 = cadd(v[2], v[3]);
    const double2 t3 = csub(v[1], v[4]), t4 = csub(v[2], v[3]);
    const double2 x0 = v[0];
    const double2 a1 = make_double2(x0.x + c1 * t1.x + c2 * t2.x, x0.y + c1 * t1.y + c2 * t2.y);
    const double2 a2 = make_double2(x0.x + c2 * t1.x + c1 * t2.x, x0.y + c2 * t1.y + c1 * t2.y);
    const double2 b1 = make_double2(s1 * t3.x + s2 * t4.x, s1 * t3.y + s2 * t4.y);
    const double2 b2 = make_double2(s2 * t3.x - s1 * t4.x, s2 * t3.y - s1 * t4.y);
    v[0] = cadd(x0, cadd(t1, t2));
    v[1] = make_double2(a1.x - b1.y, a1.y + b1.x);
    v[4] = make_double2(a1.x + b1.y, a1.y - b1.x);
    v[2] = make_double2(a2.x - b2.y, a2.y + b2.x);
    v[3] = make_double2(a2.x + b2.y, a2.y - b2.x);
  } else if constexpr (R == 6) {
    // prime factors 2 x 3, no twiddles: n = 3 n1 + 2 n2, k = 3 k1 + 4 k2 (mod 6)
    double2 e[3] = {v[0], v[2], v[4]}, o[3] = {v[3], v[5], v[1]};
    dft_small<3, BACK>(e);
    dft_small<3, BACK>(o);
    v[0] = cadd(e[0], o[0]);
    v[3] = csub(e[0], o[0]);
    v[4] = cadd(e[1], o[1]);
    v[1] = csub(e[1], o[1]);
    v[2] = cadd(e[2], o[2]);
    v[5] = csub(e[2], o[2]);
  } else {
    static_assert(R == 8, "radix");
    constexpr double h = 0.70710678118654752440;
    double2 e[4] = {v[0], v[2], v[4], v[6]}, o[4] = {v[1], v[3], v[5], v[7]};
    dft_small<4, BACK>(e);
    dft_small<4, BACK>(o);
    // o_k times exp(sign i pi k / 4)
    const double2 r1 = rot(o[1]), r3 = rot(o[3]);
    o[1] = make_double2(h * (o[1].x + r1.x), h * (o[1].y + r1.y));
    o[2] = rot(o[2]);
    o[3] = make_double2(h * (r3.x - o[3].x), h * (r3.y - o[3].y));
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[k] = cadd(e[k], o[k]);
      v[k + 4] = csub(e[k], o[k]);
    }
  }
}

// One Stockham stage of radix R over all transforms of the slab: reads its inputs into registers
// (FIRST: from the caller's load, else LDS), synchronises and writes LDS. Consecutive threads take
// consecutive transforms. load.begin(f) is called once per butterfly and its result handed to
// load(state, x, f), which returns grid point x * (points behind the first axis) + f.
template <int R, bool BACK, bool FIRST, typename Load>
__device__ __forceinline__ void fft_stage(double2* buf, const FftStage& st, const double2* tw, const Load& load) {
  constexpr int MB = fft_max_bfly(R);
  const int nbf = st.len / R;  // butterflies per transform
  const int total = nbf * st.nfft;
  double2 v[MB][R];
  int dst[MB];
#pragma unroll
  for (int c = 0; c < MB; ++c) {
    const int b = threadIdx.x + c * blockDim.x;
    if (b < total) {
      const int j = fft_div(b, st.r_nfft);
      const int f = b - j * st.nfft;
      const int fq = fft_div(f, st.r_nf2);
      const int base = fq * st.s1 + (f - fq * st.nf2);
      if constexpr (FIRST) {  // ns = 1: no twiddles
        const auto state = load.begin(f);
#pragma unroll
        for (int r = 0; r < R; ++r) v[c][r] = load(state, j + r * nbf, f);
        dst[c] = base + j * R * st.xs;
      } else {
        const int jq = fft_div(j, st.r_ns), k = j - jq * st.ns;
        const double2* src = buf + base + j * st.xs;
#pragma unroll
        for (int r = 0; r < R; ++r) v[c][r] = src[r * nbf * st.xs];
        if (st.ns > 1) {
          const int step = k * (nbf / st.ns);
#pragma unroll
          for (int r = 1; r < R; ++r) v[c][r] = cmul(v[c][r], tw[st.tw + r * step]);  // r step < len
        }
        dst[c] = base + (jq * st.ns * R + k) * st.xs;
      }
      dft_small<R, BACK>(v[c]);
    }
  }
  __syncthreads();
  const int ds = st.ns * st.xs;
#pragma unroll
  for (int c = 0; c < MB; ++c) {
    const int b = threadIdx.x + c * blockDim.x;
    if (b < total) {
#pragma unroll
      for (int r = 0; r < R; ++r) buf[dst[c] + r * ds] = v[c][r];
    }
  }
  __syncthreads();
}

template <bool BACK, bool FIRST, typename Load>
__device__ __forceinline__ void fft_stage_any(double2* buf, const FftStage& st, const double2* tw, const Load& load) {
  switch (st.radix) {
    case 8: fft_stage<8, BACK, FIRST>(buf, st, tw, load); break;
    case 6: fft_stage<6, BACK, FIRST>(buf, st, tw, load); break;
    case 5: fft_stage<5, BACK, FIRST>(buf, st, tw, load); break;
    case 4: fft_stage<4, BACK, FIRST>(buf, st, tw, load); break;
    case 3: fft_stage<3, BACK, FIRST>(buf, st, tw, load); break;
    default: fft_stage<2, BACK, FIRST>(buf, st, tw, load); break;
  }
}

// Twiddle tables exp(+-2 pi i j / n), j < n, of the transformed axes (no barrier).
template <bool BACK>
__device__ __forceinline__ void fft_twiddles(double2* tw, const FftPlan3D& p) {
  for (int d = 0; d < p.naxis; ++d)
    for (int j = threadIdx.x; j < p.axis[d]; j += blockDim.x) {
      double s, c;
      sincospi(2.0 * j / p.axis[d], &s, &c);
      tw[p.axis_tw[d] + j] = make_double2(c, BACK ? s : -s);
    }
}

// 3D FFT of one slab, unnormalised: grid points from load, the result in LDS at fft_pos(r).
// Starts with reads of `load` only: whatever it reads from LDS, the twiddles and the last use of
// buf are ordered against the writes by the stage's own barriers. All threads of the block call it.
template <bool BACK, typename Load>
__device__ __forceinline__ void fft_3d(double2* buf, const FftPlan3D& p, const double2* tw, const Load& load) {
  if (p.nstage == 0) {  // a single point
    if (threadIdx.x == 0) {
      const auto state = load.begin(0);
      buf[0] = load(state, 0, 0);
    }
    __syncthreads();
    return;
  }
  fft_stage_any<BACK, true>(buf, p.st[0], tw, load);
  for (int s = 1; s < p.nstage; ++s) fft_stage_any<BACK, false>(buf, p.st[s], tw, load);
}

// Load of a slab that lies in grid order in memory.
struct FftLoadGrid {
  const double2* src;
  int rest;  // points behind the first transformed axis
  __device__ __forceinline__ int begin(int f) const { return f; }
  __device__ __forceinline__ double2 operator()(int state, int x, int) const { return src[x * rest + state]; }
};

}  // namespace dgami
