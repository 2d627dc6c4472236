// common.h -- complex arithmetic, per-dimension geometry and twiddle access
// shared by every HIP kernel of the hybrid dealiased convolution library.
//
// Conventions (from the reference):
//   * the padded "forward" transform uses the kernel e^{+2 pi i jk/N}
//     (convolve.cc:576-577); the backward transform uses e^{-2 pi i jk/N};
//   * a padded dimension has N = m*q >= M >= L (convolve.cc:403-410,493-509);
//   * data index j in [0,L) carries wavenumber k = j + k0, with k0 = 0 for
//     fftPad and k0 = -floor(L/2) for the centred transforms
//     (fftPadCentered::forward2, convolve.cc:2244-2250);
//   * residue r in [0,q) is the set of padded indices l = q*s + r, s < m.
#pragma once
#include <hip/hip_runtime.h>
#include <stdint.h>
#include <utility>

namespace fftwpp_amd {

template<typename T>
struct cplx {
  T x, y;
};

template<typename T>
__device__ __forceinline__ cplx<T> mk(T a, T b) { cplx<T> c; c.x=a; c.y=b; return c; }
template<typename T>
__device__ __forceinline__ cplx<T> operator+(cplx<T> a, cplx<T> b) { return mk(a.x+b.x,a.y+b.y); }
template<typename T>
__device__ __forceinline__ cplx<T> operator-(cplx<T> a, cplx<T> b) { return mk(a.x-b.x,a.y-b.y); }
template<typename T>
__device__ __forceinline__ cplx<T> operator*(cplx<T> a, cplx<T> b)
{
  return mk(fma(a.x,b.x,-a.y*b.y),fma(a.x,b.y,a.y*b.x));
}
template<typename T>
__device__ __forceinline__ cplx<T> operator*(T s, cplx<T> a) { return mk(s*a.x,s*a.y); }
template<typename T>
__device__ __forceinline__ cplx<T> conjg(cplx<T> a) { return mk(a.x,-a.y); }
// a * conj(b)
template<typename T>
__device__ __forceinline__ cplx<T> mulc(cplx<T> a, cplx<T> b)
{
  return mk(fma(a.x,b.x,a.y*b.y),fma(a.y,b.x,-a.x*b.y));
}
// multiply by +i (sign>0) or -i (sign<0)
template<typename T>
__device__ __forceinline__ cplx<T> muli(cplx<T> a, int sign)
{
  return sign > 0 ? mk(-a.y,a.x) : mk(a.y,-a.x);
}

// The pointwise products of the fused row kernels.  op(F, G, row, l) returns
// the product of the two transformed inputs at padded index l = q s + r of
// row `row` of the row stage; op(u, v, row, l) on two reals is the product of
// one residue of Hermitian rows, whose transforms are real (realMultBinary).
// The kernels bind it (bind_row, below) to rows that exist, once per row and
// residue pass at most; empty slots of a last block take the last row.
// LibMult<MULT>: multNone (0), multBinary (1), multcorrelation (3) fixed at
// compile time; RunMult: the same chosen at run time.  A caller's functor with
// these two members runs in the same kernels (fused user multipliers).
template<int MULT> struct LibMult {
  template<typename T>
  __device__ __forceinline__ cplx<T> operator()(cplx<T> a, cplx<T> b, int64_t, int) const
  {
    if constexpr(MULT == 1) return a*b;
    else if constexpr(MULT == 3) return mulc(a,b);
    else return a;
  }
  template<typename T>
  __device__ __forceinline__ T operator()(T a, T b, int64_t, int) const { return a*b; }
};

// A product functor bound to one row: op.at(row) when Op provides it (the
// functor's work that depends on the row alone), else a
// wrapper that passes the row to every call.  Either way rop(F, G, l).
template<class Op> struct RowBound {
  Op op;
  int64_t row;
  template<typename T>
  __device__ __forceinline__ cplx<T> operator()(cplx<T> a, cplx<T> b, int l) const
  {
    return op(a,b,row,l);
  }
  template<typename T>
  __device__ __forceinline__ T operator()(T a, T b, int l) const { return op(a,b,row,l); }
};

template<class Op, class=void> struct HasAt { static constexpr bool value=false; };
template<class Op>
struct HasAt<Op,decltype((void) std::declval<const Op &>().at((int64_t) 0))> {
  static constexpr bool value=true;
};

template<class Op>
__device__ __forceinline__ auto bind_row(const Op &op, int64_t row)
{
  if constexpr(HasAt<Op>::value) return op.at(row);
  else return RowBound<Op>{op,row};
}

struct RunMult {
  int mult;
  template<typename T>
  __device__ __forceinline__ cplx<T> operator()(cplx<T> a, cplx<T> b, int64_t, int) const
  {
    return mult == 1 ? a*b : (mult == 3 ? mulc(a,b) : a);
  }
  template<typename T>
  __device__ __forceinline__ T operator()(T a, T b, int64_t, int) const { return a*b; }
};

// The library's products: a factor of F times one of G, so that scales of the
// factors may be undone on the product.
template<class Op> struct IsProduct { static constexpr bool value=false; };
template<> struct IsProduct<RunMult> { static constexpr bool value=true; };
template<int MULT> struct IsProduct<LibMult<MULT>> { static constexpr bool value=true; };

// Geometry of one padded dimension as seen by a kernel.
constexpr int MAXSTAGES=24;

struct DimArgs {
  int64_t L;      // input length (full length for Hermitian dimensions)
  int64_t m;      // sub-FFT size
  int64_t q;      // number of residues
  int64_t N;      // padded length m*q
  int64_t k0;     // wavenumber of data index 0
  int64_t H;      // stored modes: L, or ceil(L/2) for a Hermitian dimension
  int nstages;
  int radix[MAXSTAGES];
  const void *zN; // zN[j] = e^{2 pi i j/N}, j < N, in the kernel's precision
  const void *last; // FP64, m = 1024, 2048, 4096: the last stage's twiddles (fftr.h)
};

// Column tile of block x of a grid row of gx blocks.  Blocks are dealt to
// the 8 XCDs round robin by linear id, so block x runs on XCD x mod 8 (when
// gx is a multiple of 8); runs of gx/8 consecutive tiles are given to one
// XCD, so that neighbouring tiles, which share cache lines when a tile row is
// narrower than a line, share that XCD's L2 instead of fetching the line
// twice.  A bijection of [0, gx).
__device__ __forceinline__ int64_t xcd_tile(int64_t x, int64_t gx)
{
  const int64_t per=gx/8;
  return x < 8*per ? (x % 8)*per+x/8 : x;
}

// Up to three arrays transformed by one launch (the inputs of a convolution,
// or the cotangent and both inputs of its adjoint).  Block z of the grid takes
// array z mod n and every gridDim.z/n-th residue from z/n on.
constexpr int MAXARRAYS=3;

struct ColArrays {
  int n;
  const void *in[MAXARRAYS];
  void *out[MAXARRAYS];
};

struct ColBlock {
  const void *in;
  void *out;
  int part, parts;
};

__device__ __forceinline__ ColBlock col_block(const ColArrays &io)
{
  // in scalar registers (a division runs on the vector unit and would take
  // the pointers with it)
  const int z=blockIdx.z, n=io.n;
  const int part=n == 1 ? z : __builtin_amdgcn_readfirstlane(z/n);
  const int a=z-part*n;
  ColBlock b;
  // device memory: as pointers out of a struct they would be taken for
  // generic ones (flat accesses, more registers)
  b.in=(const void *) (const __attribute__((address_space(1))) void *)
    (a == 0 ? io.in[0] : (a == 1 ? io.in[1] : io.in[2]));
  b.out=(void *) (__attribute__((address_space(1))) void *)
    (a == 0 ? io.out[0] : (a == 1 ? io.out[1] : io.out[2]));
  b.part=part;
  b.parts=n == 1 ? (int) gridDim.z : __builtin_amdgcn_readfirstlane((int) gridDim.z/n);
  return b;
}

template<typename T>
__device__ __forceinline__ cplx<T> ztab(const DimArgs &d, int64_t j)
{
  return reinterpret_cast<const cplx<T> *>(d.zN)[j];
}

// e^{2 pi i e/N} for an arbitrary signed exponent e.
template<typename T>
__device__ __forceinline__ cplx<T> zeta(const DimArgs &d, int64_t e)
{
  int64_t r=e % d.N;
  if(r < 0) r += d.N;
  return ztab<T>(d,r);
}

// t as a value that the compiler does not know to be the loop-invariant one:
// without it the LDS addresses and twiddle positions of every stage, which
// depend on t alone, are hoisted out of the caller's loop over rows and
// residues and stay in registers through all of it (30 to 40 of them in a row
// kernel); computed anew per transform they cost one instruction per access.
__device__ __forceinline__ int fresh(int t)
{
  asm volatile("" : "+v"(t));
  return t;
}

// A complex word of a table in LDS whose words are aligned to their size: one
// access with a 64 KB range of immediate offsets (two words of half the size
// reach 2 KB, and the rest of a table costs an addition each).
template<typename T>
__device__ __forceinline__ cplx<T> table_word(const cplx<T> *p)
{
  typedef T pair __attribute__((ext_vector_type(2)));
  const pair v=*reinterpret_cast<const pair *>(p);
  return mk(v.x,v.y);
}

// Buffer access: a complex word at byte offset off (per lane) + soff
// (uniform) of a raw buffer; one offset register serves every load of a
// thread whose words differ by uniform strides.
// Store of one complex word at byte offset off + soff of the buffer r.  The
// 16-byte store takes soff in its vector offset: with a scalar offset register
// the compiler lets the next vector operation overwrite the stored registers,
// and lanes 12..15 of each 16 were then seen to store the new values (rows of
// 256 points differed from run to run).  Without one it keeps the two wait
// states; 8-byte stores read their data at once.
template<typename T>
__device__ __forceinline__ void st_buf(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff,
                                       cplx<T> v);
template<>
__device__ __forceinline__ void st_buf<double>(__amdgpu_buffer_rsrc_t r, unsigned off,
                                               unsigned soff, cplx<double> v)
{
  typedef double d2 __attribute__((ext_vector_type(2)));
  typedef unsigned u4 __attribute__((ext_vector_type(4)));
  d2 w; w.x=v.x; w.y=v.y;
  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(u4,w),r,off+soff,0,0);
}
template<>
__device__ __forceinline__ void st_buf<float>(__amdgpu_buffer_rsrc_t r, unsigned off,
                                              unsigned soff, cplx<float> v)
{
  typedef float f2 __attribute__((ext_vector_type(2)));
  typedef unsigned u2 __attribute__((ext_vector_type(2)));
  f2 w; w.x=v.x; w.y=v.y;
  __builtin_amdgcn_raw_buffer_store_b64(__builtin_bit_cast(u2,w),r,off,soff,0);
}
// Plain (L1-cached) load of one complex word at byte offset off + soff of r.
template<typename T>
__device__ __forceinline__ cplx<T> ld_buf(__amdgpu_buffer_rsrc_t r, unsigned off, unsigned soff);
template<>
__device__ __forceinline__ cplx<double> ld_buf<double>(__amdgpu_buffer_rsrc_t r, unsigned off,
                                                       unsigned soff)
{
  typedef double d2 __attribute__((ext_vector_type(2)));
  const d2 v=__builtin_bit_cast(d2,__builtin_amdgcn_raw_buffer_load_b128(r,off,soff,0));
  return mk(v.x,v.y);
}
template<>
__device__ __forceinline__ cplx<float> ld_buf<float>(__amdgpu_buffer_rsrc_t r, unsigned off,
                                                     unsigned soff)
{
  typedef float f2 __attribute__((ext_vector_type(2)));
  const f2 v=__builtin_bit_cast(f2,__builtin_amdgcn_raw_buffer_load_b64(r,off,soff,0));
  return mk(v.x,v.y);
}

// Raw buffer resource over `words` complex words from base (offsets at or
// beyond the end read 0 and drop stores).  The hardware holds the lane's offset
// against the number of bytes less the scalar offset: where soff may exceed that
// number, all of an access's offset is in off.
template<typename T>
__device__ __forceinline__ __amdgpu_buffer_rsrc_t buf_rsrc(const cplx<T> *base, size_t words)
{
  return __builtin_amdgcn_make_buffer_rsrc((void *) base,0,(int) (words*sizeof(cplx<T>)),
                                           0x00020000);
}

} // namespace fftwpp_amd
