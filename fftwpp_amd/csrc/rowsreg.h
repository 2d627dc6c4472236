// rowsreg.h -- fused row convolutions on the register-resident FFT (fftr.h)
// for a power-of-two sub-FFT size M (16..4096) when one block of M covers the
// row: complex or centred rows with L <= M, Hermitian rows with H <= M.
//
// A slot of TPS = M/V threads owns one row (thread t holds sigma = t + TPS k,
// k < V), loops over the residues with the sums kept in registers and writes
// the row once at the end, so out may equal f.  Rows are contiguous.
//
// Complex rows (Convolution::convolveRaw, convolve.cc:7513-7575, with the
// forward1/backward1 residue transforms, convolve.cc:836-1030, 1468-1613, and
// the centred folds of fftPadCentered): element j has wavenumber k = j + k0
// and sits at sigma = k mod M; residue r is DFT_M[w_N^{k r} f](s).
//
// Hermitian rows (fftPadHermitian, convolve.cc:4309-5447): residues r1, r2 =
// r1 + 1 are packed as W1 + i W2 with W_sigma = sum over k = sigma mod M,
// |k| < H, of w_N^{k r} f(k), f(-k) = conj f(k) (k = sigma and sigma - M),
// multiplied as realMultBinary (real parts, imaginary parts) and unpacked
// after the inverse with the mirror element Z(M - sigma), fetched through the
// slot's LDS exchange area.
#pragma once
#include <limits>
#include <type_traits>
#include "batch.h"

namespace fftwpp_amd {

// e mod N for -N <= e < 2N: the twiddle exponents k r of these kernels have
// |k| < M (rows) or -M <= k < 2M (columns with p <= 2) and 0 <= r < q, so
// they lie in [-N, 2N) with N = M q (kept below 2^30 by the dispatchers).
__device__ __forceinline__ int wrapN(int e, int N)
{
  return e < 0 ? e+N : (e >= N ? e-N : e);
}

// Values per thread: 8 in both precisions (the register sums over residues
// sit beside the two transforms).
struct RowV { static constexpr int V=8; };

// acc of residue lane 0 <- sum of acc over the RP residue lanes of the row,
// through the lanes' exchange areas (2 PAD words each: real parts, then
// imaginary parts).  All threads of the block call it when RP > 1.
template<typename T, int M, int RP>
__device__ __forceinline__ void rowreg_combine(cplx<T> *acc, T *xbase, T *xb,
                                               int rp, int t)
{
  if constexpr(RP > 1) {
    constexpr int V=RowV::V;
    typedef RPlan<M,V> P;
    constexpr int TPS=P::TPS;
    if(rp > 0) {
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int e=xidx<T,M,V>(t+TPS*k);
        xb[e]=acc[k].x;
        xb[P::PAD+e]=acc[k].y;
      }
    }
    __syncthreads();
    if(rp == 0) {
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int e=xidx<T,M,V>(t+TPS*k);
#pragma unroll
        for(int o=1; o < RP; ++o)
          acc[k]=acc[k]+mk(xbase[2*o*P::PAD+e],xbase[(2*o+1)*P::PAD+e]);
      }
    }
    __syncthreads();
  }
}

// Complex or centred rows.  Thread t of a row's slot keeps element sigma =
// t + TPS k at index j = (sigma - k0) mod M of the row (j >= L: zero padding).
//
// Loads go through a buffer over the block's rows (one 32-bit offset per
// thread; zero padding is an offset past the end, which reads 0), all issued
// together.  The host keeps the span of a block's rows below 2^31 bytes.
//
// RP = 1: each slot owns a row (one slot per block when TPS > 64).  RP > 1:
// the block holds one row and its RP slots take every RP-th residue; their
// sums are added through LDS before the row is written.  Dynamic LDS: M
// complex twiddles + slots * 2 RPlan<M,V>::PAD scalar words.
//
// Bound by the chain of LDS exchanges, with two or three waves per SIMD in
// FP64 (166-175 registers: the two transforms and the residue sums alone are
// 96) and four or five in FP32 (about 100).  Branch-free loads, one register
// per exchange instead of one per access, positions computed anew per
// transform (fresh) and the product chosen once per row took 65536 rows of 120
// points (q = 2) from 152 to 113 us in FP64 and from 72 to 55 us in FP32, 8192
// rows of 500 points from 79 to 60 and from 52 to 38 us, 2048 rows of 1000
// points padded to 2048 from 56 to 46 and from 31.5 to 25 us, one such FP64
// row from 10.1 to 9.0 us.  One row of 1500 points with its residues on two
// lanes: FP32 10.7 us with a branch per load, 11.25 with all words loaded and the
// residue twiddles read at each use, 10.1 with them read once; FP64 17.1, 14.5,
// 13.3 us.  (One lane per row has no registers to keep them in.)
// W: waves per SIMD asked of the compiler; three in FP64 where the library's
// own products fit without spills and LDS leaves room for the blocks (113
// against 124 us at M = 128); a caller's functor keeps the registers of two.
template<typename T, int M, int RP, class Op> struct RowCx {
  static constexpr bool MORE=sizeof(T) == 8 && RP == 1 && M >= 128 && M <= 512;
  static constexpr int W=MORE && std::is_same<Op,RunMult>::value ? 3 : 2;
};
template<typename T, int M, int RP, class Op>
__global__ void __launch_bounds__(RP*M/RowV::V > 512 ? 1024 : RP*M/RowV::V > 256 ? 512 : 256,
                                  (RP*M/RowV::V > 512 ? 4 : RowCx<T,M,RP,Op>::W))
rowcx_kernel(DimArgs d, const cplx<T> *f, const cplx<T> *g, int64_t row0, int64_t rows,
             int64_t rs, cplx<T> *out, int64_t os, T scale, Op op)
{
  constexpr int V=RowV::V;
  typedef RPlan<M,V> P;
  constexpr int TPS=P::TPS;
  constexpr unsigned E=sizeof(cplx<T>);
  extern __shared__ char smem_raw[];
  typedef SplitTw<T,M,V> ST;
  cplx<T> *twl=reinterpret_cast<cplx<T> *>(smem_raw);
  const auto tw=stage_table<T,M,V>(twl,d);
  const cplx<T> *zN=(const cplx<T> *) d.zN;
  const int slots=RP > 1 ? 1 : blockDim.x/TPS;      // rows per block
  // a slot of whole waves: its index, and its residue, are uniform over the wave
  int slot=(int) threadIdx.x/TPS;
  if constexpr(TPS >= 64) slot=__builtin_amdgcn_readfirstlane(slot);
  const int t=threadIdx.x-slot*TPS;
  const int rp=RP > 1 ? slot : 0;                     // residue lane
  const int rslot=RP > 1 ? 0 : slot;
  T *xbase=reinterpret_cast<T *>(twl+ST::LDS);
  T *xb=xbase+slot*2*P::PAD;
  const int q=(int) d.q, L=(int) d.L, k0=(int) d.k0;
  cplx<T> a[V], b[V];
  // the words of the slot's row of the block's rows from rb on
  auto load=[&](int64_t rb) {
    const int64_t nr=rows-rb < slots ? rows-rb : slots;
    const size_t words=(size_t) ((nr-1)*rs+L);
    const __amdgpu_buffer_rsrc_t rf=buf_rsrc(f+rb*rs,words), rg=buf_rsrc(g+rb*rs,words);
    const unsigned ro=(unsigned) rslot*(unsigned) rs*E;
#pragma unroll
    for(int k=0; k < V; ++k) {
      const int j=(t+TPS*k-k0) & (M-1);    // k0 <= 0, M a power of two
      const unsigned o=j < L ? ro+(unsigned) j*E : 0x80000000u;   // past the end: reads 0
      a[k]=ld_buf<T>(rf,o,0);
      b[k]=ld_buf<T>(rg,o,0);
    }
  };
  const int64_t step=(int64_t) gridDim.x*slots;
  int64_t rb=(int64_t) blockIdx.x*slots;
  fill_twr<T,M,V,ST::USED>(twl,zN,q,threadIdx.x,blockDim.x);
  __syncthreads();
  for(; rb < rows; rb += step) {
    const int64_t row=rb+rslot;
    cplx<T> acc[V];
#pragma unroll
    for(int k=0; k < V; ++k) acc[k]=mk((T) 0,(T) 0);
    // residue lanes take the same number of passes, as the block's barriers
    // need; one past the last residue repeats residue 0 and adds nothing
    for(int r0=0; r0 < q; r0 += RP) {
      const bool on=RP == 1 || r0+rp < q;
      const int r=on ? r0+rp : 0;
      // w_N^{(j+k0) r}: j + k0 is sigma or sigma - M
      const cplx<T> bt=zN[t*r], zm=conjg(zN[M*r]);
      // w_N^{TPS k r}: of a residue lane read with the row and kept, so that the
      // few blocks of a single row don't wait for them twice
      cplx<T> wk[RP > 1 ? V : 1];
      if constexpr(RP > 1) {
#pragma unroll
        for(int k=0; k < V; ++k) wk[k]=zN[TPS*k*r];
      }
      auto wkr=[&](int k) { return RP > 1 ? wk[RP > 1 ? k : 0] : zN[TPS*k*r]; };
      cplx<T> X[V], Y[V];
      load(rb);
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int sigma=t+TPS*k;
        const int j=(sigma-k0) & (M-1);
        cplx<T> u=a[k], v=b[k];
        if(r) {
          cplx<T> w=bt*wkr(k);
          if(j+k0 < 0) w=w*zm;
          u=w*u;
          v=w*v;
        }
        X[k]=u;
        Y[k]=v;
      }
      fftr_pair<T,M,V,1>(X,Y,xb,tw,t);
      if constexpr(std::is_same<Op,RunMult>::value) {
        // one uniform branch, not a choice per element
        if(op.mult == 1) {
#pragma unroll
          for(int k=0; k < V; ++k) X[k]=X[k]*Y[k];
        } else if(op.mult == 3) {
#pragma unroll
          for(int k=0; k < V; ++k) X[k]=mulc(X[k],Y[k]);
        }
      } else {
        const auto rop=bind_row(op,row0+(row < rows ? row : rows-1));
#pragma unroll
        for(int k=0; k < V; ++k) X[k]=rop(X[k],Y[k],q*(t+TPS*k)+r);
      }
      fftr<T,M,V,-1>(X,xb,tw,t);
#pragma unroll
      for(int k=0; k < V; ++k) {
        if(r) {
          const int sigma=t+TPS*k;
          const int j=(sigma-k0) & (M-1);
          cplx<T> w=bt*wkr(k);
          if(j+k0 < 0) w=w*zm;
          acc[k]=acc[k]+mulc(X[k],w);
        } else if(on)
          acc[k]=acc[k]+X[k];
      }
    }
    rowreg_combine<T,M,RP>(acc,xbase,xb,rp,t);
    if(rp == 0 && row < rows) {
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int sigma=t+TPS*k;
        const int j=(sigma-k0) & (M-1);
        if(j < L) out[row*os+j]=scale*acc[k];
      }
    }
    if(RP > 1) __syncthreads();          // exchange areas are reused by the next row
  }
}

// Hermitian rows (the rows that hrowpk_kernel below leaves: M = 4096, few
// rows).  Dynamic LDS: M complex twiddles + slots * 2 RPlan<M,V>::PAD scalar words
// (each slot's exchange area holds a whole complex sequence, so every
// exchange is one round).
// RP = 1: each slot owns a row (one slot per block when TPS > 64).  RP > 1:
// the block holds one row and its RP slots take every RP-th residue (pair);
// their sums are added through LDS before the row is written.
template<typename T, int M, int RP, class Op>
__global__ void __launch_bounds__(512)
rowreg_kernel(DimArgs d, const cplx<T> *f, const cplx<T> *g, int64_t rows,
              int64_t rs, cplx<T> *out, int64_t os, T scale, Op op)
{
  constexpr int V=RowV::V;
  typedef RPlan<M,V> P;
  constexpr int TPS=P::TPS;
  extern __shared__ char smem_raw[];
  cplx<T> *tw=reinterpret_cast<cplx<T> *>(smem_raw);
  const cplx<T> *zN=(const cplx<T> *) d.zN;
  fill_twr<T,M,V>(tw,zN,(int) d.q,threadIdx.x,blockDim.x);
  __syncthreads();
  const int slots=RP > 1 ? 1 : blockDim.x/TPS;      // rows per block
  const int slot=threadIdx.x/TPS, t=threadIdx.x-slot*TPS;
  const int rp=RP > 1 ? slot : 0;                     // residue lane
  T *xbase=reinterpret_cast<T *>(tw+M);
  T *xb=xbase+slot*2*P::PAD;
  const int q=(int) d.q, H=(int) d.H;
  for(int64_t rb=(int64_t) blockIdx.x*slots; rb < rows; rb += (int64_t) gridDim.x*slots) {
    const int64_t row=rb+(RP > 1 ? 0 : slot);
    if(row >= rows) break;               // uniform over the block when RP > 1
    const cplx<T> *fr=f+row*rs, *gr=g+row*rs;
    cplx<T> acc[V];
#pragma unroll
    for(int k=0; k < V; ++k) acc[k]=mk((T) 0,(T) 0);
    // the same number of passes in every lane, as in rowcx_kernel
    for(int p0=0; p0 < q; p0 += 2*RP) {
      const bool on=RP == 1 || p0+2*rp < q;
      const int r1=on ? p0+2*rp : 0;
      const int r2=r1+1 < q ? r1+1 : -1;
      // w_N^{sigma r} = w_N^{t r} w_N^{TPS k r}; w_N^{(sigma - M) r} adds
      // the factor conj w_N^{M r}
      const cplx<T> zero=mk((T) 0,(T) 0);
      const cplx<T> b1=zN[t*r1], m1=conjg(zN[M*r1]);
      const cplx<T> b2=r2 >= 0 ? zN[t*r2] : zero, m2=r2 >= 0 ? conjg(zN[M*r2]) : zero;
      cplx<T> X[V], Y[V];
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int sigma=t+TPS*k;
        const cplx<T> w1=b1*zN[TPS*k*r1];
        const cplx<T> w2=r2 >= 0 ? b2*zN[TPS*k*r2] : zero;
        cplx<T> a=mk((T) 0,(T) 0), b=a;
        // k = sigma (when < H) and k = sigma - M (when > -H)
        if(sigma < H) {
          const cplx<T> w=w1+muli(w2,1);
          a=w*fr[sigma];
          b=w*gr[sigma];
        }
        if(M-sigma < H) {
          const cplx<T> w=w1*m1+muli(w2*m2,1);
          a=a+w*conjg(fr[M-sigma]);
          b=b+w*conjg(gr[M-sigma]);
        }
        X[k]=a;
        Y[k]=b;
      }
      fftr<T,M,V,1>(X,xb,tw,t);
      fftr<T,M,V,1>(Y,xb,tw,t);
      {
        const auto rop=bind_row(op,row);
#pragma unroll
        for(int k=0; k < V; ++k) {
          const int l=q*(t+TPS*k);
          X[k]=mk(rop(X[k].x,Y[k].x,l+r1),r2 >= 0 ? rop(X[k].y,Y[k].y,l+r2) : (T) 0);
        }
      }
      fftr<T,M,V,-1>(X,xb,tw,t);
      // mirror elements Z(M - sigma) through LDS
      cplx<T> Zm[V];
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int e=xidx<T,M,V>(t+TPS*k);
        xb[e]=X[k].x;
        xb[P::PAD+e]=X[k].y;
      }
      rsync<TPS>();
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int e=xidx<T,M,V>((M-(t+TPS*k)) & (M-1));
        Zm[k]=mk(xb[e],xb[P::PAD+e]);
      }
      rsync<TPS>();
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int sigma=t+TPS*k;
        if(on && sigma < H) {
          const cplx<T> z=X[k], zc=conjg(Zm[k]);
          const cplx<T> y1=(T) 0.5*(z+zc);
          cplx<T> v=mulc(y1,b1*zN[TPS*k*r1]);
          if(r2 >= 0) {
            const cplx<T> y2=muli((T) 0.5*(z-zc),-1);
            v=v+mulc(y2,b2*zN[TPS*k*r2]);
          }
          acc[k]=acc[k]+v;
        }
      }
    }
    rowreg_combine<T,M,RP>(acc,xbase,xb,rp,t);
    if(rp == 0) {
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int sigma=t+TPS*k;
        if(sigma < H) out[row*os+sigma]=scale*acc[k];
      }
    }
    if(RP > 1) __syncthreads();          // exchange areas are reused by the next row
  }
}


// The 32-bit words of a value.
template<int N> struct Words { unsigned w[N]; };

// c over the values of the TPS consecutive lanes of a slot (at most a wave), the
// same bits in each of them; c is a sum or a maximum.  Within 16 lanes by lane
// permutations (lane ^ 1, lane ^ 2, then mirrors, whose groups are uniform by
// then), beyond by swaps of 16 or 32 lanes between two copies of the value.
template<int TPS, typename T, class Combine>
__device__ __forceinline__ T lanes_combine(T v, Combine c)
{
  constexpr int N=sizeof(T)/4;
  auto words=[](T x) { return __builtin_bit_cast(Words<N>,x); };
  auto value=[](Words<N> w) { return __builtin_bit_cast(T,w); };
  auto permuted=[&](auto ctrl) {
    Words<N> w=words(v);
#pragma unroll
    for(int i=0; i < N; ++i)
      w.w[i]=(unsigned) __builtin_amdgcn_update_dpp(0,(int) w.w[i],decltype(ctrl)::value,0xF,0xF,true);
    v=c(v,value(w));
  };
  auto swapped=[&](auto swap) {
    const Words<N> w=words(v);
    Words<N> a, b;
#pragma unroll
    for(int i=0; i < N; ++i) {
      const auto s=swap(w.w[i]);
      a.w[i]=s[0];
      b.w[i]=s[1];
    }
    v=c(value(a),value(b));
  };
  if constexpr(TPS >= 2) permuted(std::integral_constant<int,0xB1>());
  if constexpr(TPS >= 4) permuted(std::integral_constant<int,0x4E>());
  if constexpr(TPS >= 8) permuted(std::integral_constant<int,0x141>());
  if constexpr(TPS >= 16) permuted(std::integral_constant<int,0x140>());
  if constexpr(TPS >= 32)
    swapped([](unsigned u) { return __builtin_amdgcn_permlane16_swap(u,u,false,false); });
  if constexpr(TPS >= 64)
    swapped([](unsigned u) { return __builtin_amdgcn_permlane32_swap(u,u,false,false); });
  return v;
}

// The same over the TPS threads of a slot of whole waves, through red (two
// words for each of the block's waves) when it has several; one block barrier
// then, and the next use takes other words.
template<int TPS, typename T, class Combine>
__device__ __forceinline__ void slot_combine(T &x, T &y, T *red, Combine c)
{
  x=lanes_combine<(TPS < 64 ? TPS : 64)>(x,c);
  y=lanes_combine<(TPS < 64 ? TPS : 64)>(y,c);
  if constexpr(TPS > 64) {
    constexpr int W=TPS/64;
    const int wave=__builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
    if((threadIdx.x & 63) == 0) {
      red[2*wave]=x;
      red[2*wave+1]=y;
    }
    __syncthreads();
    const T *r=red+2*(wave & ~(W-1));
    x=r[0];
    y=r[1];
#pragma unroll
    for(int w=1; w < W; ++w) {
      x=c(x,r[2*w]);
      y=c(y,r[2*w+1]);
    }
  }
}

// The two factors of a Hermitian row share a transform, whose rounding errors
// are relative to the larger one: exact powers of two bring them to one
// magnitude first, 2^-ef F and 2^-eg G, whose norms then differ by at most a
// factor sqrt(2).  near: ef = 0, only G is scaled.  Otherwise (far) both are, to
// norms near 1.  Relative error of a row's product, FP32, H = 128: F of 1e-3 of G's
// magnitude 1e-3 unscaled, 1.6e-7 scaled.  (rowreg_kernel, which transforms the
// factors apart, two residues of one at a time: 1.5e-7 for odd q, whose last
// residue has a transform of its own and drops half of its rounding errors; the
// same as here for even q.)
struct RowScales {
  int ef, eg;
  bool near;     // the same over the wave, or over the block where slots span waves
};
// ef or eg of a factor of zeros: undone, it makes 0 of the other's rounding errors
constexpr int ZEROS=-10000;

// Squares of norms from 2^LO to 2^HI are near: their sums lose nothing that
// matters to underflow, ratios of norms stay normal numbers and the transforms in
// range.  2^-LIM and 2^LIM are normal numbers too.
template<typename T> struct ScaleRange;
template<> struct ScaleRange<double> { static constexpr int LO=-900, HI=900, LIM=1022; };
template<> struct ScaleRange<float> { static constexpr int LO=-120, HI=120, LIM=126; };

__device__ __forceinline__ int exponent(double v) { return __builtin_amdgcn_frexp_exp(v); }
__device__ __forceinline__ int exponent(float v) { return __builtin_amdgcn_frexp_expf(v); }
__device__ __forceinline__ double mantissa(double v) { return __builtin_amdgcn_frexp_mant(v); }
__device__ __forceinline__ float mantissa(float v) { return __builtin_amdgcn_frexp_mantf(v); }
__device__ __forceinline__ double scaled(double v, int e) { return __builtin_amdgcn_ldexp(v,e); }
__device__ __forceinline__ float scaled(float v, int e) { return __builtin_amdgcn_ldexpf(v,e); }

// The scales of a row, given its words a of f and b of g in this thread (each
// word of the row in one thread of the slot).  red: 3 x 2 words per wave of the
// block (slots of several waves).  Far rows take their whole wave along (or the
// block, whose barriers all its threads must reach); their norms are summed
// after a scaling by the largest magnitude.
template<typename T, int M, int SLOTS>
__device__ __forceinline__ RowScales row_scales(const cplx<T> *a, const cplx<T> *b, T *red)
{
  constexpr int V=RowV::V, TPS=M/V, WAVES=(SLOTS*TPS+63)/64;
  typedef ScaleRange<T> SR;
  static_assert(TPS <= 64 || SLOTS <= 2,"every slot of the block is looked at");
  auto add=[](T x, T y) { return x+y; };
  T x=0, y=0;
#pragma unroll
  for(int k=0; k < V; ++k) {
    x=fma(a[k].x,a[k].x,fma(a[k].y,a[k].y,x));
    y=fma(b[k].x,b[k].x,fma(b[k].y,b[k].y,y));
  }
  slot_combine<TPS>(x,y,red,add);
  const T lo=scaled((T) 1,SR::LO), hi=scaled((T) 1,SR::HI);
  auto outside=[&](T u, T v) { return !(u >= lo && u <= hi && v >= lo && v <= hi); };
  bool far=outside(x,y);                 // zeros too: they may be squares that vanished
  if constexpr(TPS > 64 && SLOTS == 2) {
    const int wave=(int) threadIdx.x >> 6;
    const T *r=red+2*((wave & (WAVES/2)) ^ (WAVES/2));    // the other slot
    T u=r[0], v=r[1];
#pragma unroll
    for(int w=1; w < TPS/64; ++w) {
      u=u+r[2*w];
      v=v+r[2*w+1];
    }
    far=far || outside(u,v);
  }
  RowScales s={0,0,true};
  if(__any(far)) {
    const T top=std::numeric_limits<T>::max();
    T mx=0, my=0;
#pragma unroll
    for(int k=0; k < V; ++k) {
      mx=fmax(mx,fmax(fabs(a[k].x),fabs(a[k].y)));
      my=fmax(my,fmax(fabs(b[k].x),fabs(b[k].y)));
    }
    slot_combine<TPS>(mx,my,red+2*WAVES,[](T u, T v) { return fmax(u,v); });
    const int px=mx > 0 && mx <= top ? exponent(mx) : 0, py=my > 0 && my <= top ? exponent(my) : 0;
    x=y=0;
#pragma unroll
    for(int k=0; k < V; ++k) {
      const T fx=scaled(a[k].x,-px), fy=scaled(a[k].y,-px), gx=scaled(b[k].x,-py), gy=scaled(b[k].y,-py);
      x=fma(fx,fx,fma(fy,fy,x));
      y=fma(gx,gx,fma(gy,gy,y));
    }
    slot_combine<TPS>(x,y,red+4*WAVES,add);
    // a factor of zeros, or with Inf or NaN, takes the other's scale
    s.near=false;
    const bool vf=x > 0 && x <= top, vg=y > 0 && y <= top;
    s.ef=vf ? px+(exponent(x) >> 1) : (vg ? py+(exponent(y) >> 1) : 0);
    s.eg=s.ef;
    if(vf && vg) {
      const int d=exponent(y)-exponent(x)+2*(py-px);
      s.eg=s.ef+((d+(mantissa(y) >= mantissa(x) ? 1 : 0)) >> 1);
    }
    s.ef=x == 0 ? ZEROS : min(max(s.ef,-SR::LIM),SR::LIM);
    s.eg=y == 0 ? ZEROS : min(max(s.eg,-SR::LIM),SR::LIM);
  } else
    // log2 of |g|/|f| rounded: half of the difference of the squares'
    // exponents, up where that is odd and the mantissas make up the rest
    s.eg=(exponent(y)-exponent(x)+(mantissa(y) >= mantissa(x) ? 1 : 0)) >> 1;
  if constexpr(TPS >= 64) {              // the same over the wave: scalar registers
    s.ef=__builtin_amdgcn_readfirstlane(s.ef);
    s.eg=__builtin_amdgcn_readfirstlane(s.eg);
  }
  return s;
}

// Residues r1 and r2 of the f + i g pair of a Hermitian row (H <= M), folded
// for the forward transform from one read of the row: X1[k] = U_r1(sigma),
// X2[k] = U_r2(sigma) at sigma = t + TPS k, with
//   U_r(sigma) = w_N^{sigma r} [u(sigma) + w_q^{-r} v(sigma)],
//   u(sigma) = f(sigma) + i g(sigma)                    (sigma < H),
//   v(sigma) = conj f(M - sigma) + i conj g(M - sigma)  (M - sigma < H),
// the wavenumbers k = sigma and sigma - M of the block (f(-k) = conj f(k),
// w_N^{(sigma - M) r} = w_N^{sigma r} w_q^{-r}); f and g stand for the row's
// factors scaled by 2^-ef and 2^-eg (RowScales).  fu, gu: the words sigma, of
// which g's still take the factor su; sf, sg: the factors of the words M - sigma,
// read from rf, rg, the buffers, at byte offset ro; tr[k] = w_N^{TPS k r}, tr[V] =
// w_N^{M r} (LDS); b = w_N^{t r}.  Out-of-range words read zero, past the end of
// the buffers (no branches).
template<typename T, int M>
__device__ __forceinline__ void hpk_fold2(cplx<T> *X1, cplx<T> *X2, const cplx<T> *fu,
                                          const cplx<T> *gu, __amdgpu_buffer_rsrc_t rf,
                                          __amdgpu_buffer_rsrc_t rg, const cplx<T> *tr1,
                                          const cplx<T> *tr2, cplx<T> b1, cplx<T> b2, int t,
                                          int r1, int r2, int H, unsigned ro, T sf, T sg, T su)
{
  constexpr int V=RowV::V, TPS=M/V;
  constexpr unsigned E=sizeof(cplx<T>), END=0x80000000u;
  const cplx<T> c1=conjg(tr1[V]), c2=conjg(tr2[V]);
#pragma unroll
  for(int k=0; k < V; ++k) {
    const int sigma=t+TPS*k;
    const unsigned ov=M-sigma < H ? ro+(unsigned) (M-sigma)*E : END;
    const cplx<T> fv=ld_buf<T>(rf,ov,0), gv=ld_buf<T>(rg,ov,0);
    const cplx<T> u=mk(fma(-su,gu[k].y,fu[k].x),fma(su,gu[k].x,fu[k].y));
    const cplx<T> v=mk(fma(sg,gv.y,sf*fv.x),fma(sg,gv.x,-sf*fv.y));
    cplx<T> a=u+c1*v, b=u+c2*v;
    if(r1) a=(b1*tr1[k])*a;
    if(r2) b=(b2*tr2[k])*b;
    X1[k]=a;
    X2[k]=b;
  }
}

// Hermitian rows with H <= M <= 2048, SLOTS = 256/TPS rows per block of 256
// threads (M = 1024: two rows of two waves; M = 128: sixteen rows, four to a
// wave).  The
// forward transforms of f and g share one complex FFT per residue: the fold
// U_r of f + i g (hpk_fold2) transforms to F_r + i G_r with F_r, G_r real
// (the folds of Hermitian data are Hermitian), so P_r = F_r G_r is
// realMultBinary's product (fftPadHermitian::forward2 and the multiplier,
// convolve.cc:4517-4609, 26-110).  Residues are paired for the inverse,
// P_{r1} + i P_{r2}, and unpacked with the mirror element Z(M - sigma) as in
// rowreg_kernel (backward2, convolve.cc:4749-4843): q forward and ceil(q/2)
// inverse transforms per row instead of 3 ceil(q/2).  Rows are read through
// buffer resources (a 32-bit offset per element; over one row when a slot is
// whole waves, else over the block's rows with the row's offset per lane) and
// the uniform residue twiddles w_N^{TPS k r} come from an LDS table, which keeps
// addresses and twiddles out of the registers that the residue loop carries.
// A row's words sigma are loaded ahead of its pairs: the first loads also give the
// norms by which the factors are scaled (RowScales), which takes 4 to 8% (3072
// rows of H = 1024, q = 3, FP64 80.5 -> 84.2 us, 73728 of 128 182 -> 187 us; with the
// words read again for the first pair 87 and 188 us; both factors scaled at every
// element instead of one 89.5 us).  Slots past the last row run on row rows - 1
// without storing (the block barriers of the transforms need every thread).
// Dynamic LDS: hrowpk_lds().
template<typename T, int M>
struct HRowPk {
  static constexpr int V=RowV::V;
  static constexpr int TPS=M/V;
  static constexpr int SLOTS=256/TPS > 0 ? 256/TPS : 1;
  static constexpr int NT=SLOTS*TPS;
  // waves per SIMD that fit without spills with the library's products (157 to
  // 168 and 90 to 100 registers); a caller's functor keeps the registers of two
  // (the tests' weight 1/(1 + c k^2), 73728 rows of H = 128, FP64: 254 us with three, 246)
  static constexpr int W=sizeof(T) == 4 ? 4 : 3, WF=2;
  typedef SplitTw<T,M,V,2048> ST;           // at 2048 the table leaves two blocks
  static constexpr int RED=TPS > 64 ? 3*2*NT/64 : 0;  // words of row_scales
};

template<typename T, int M>
inline size_t hrowpk_lds(int q)
{
  typedef HRowPk<T,M> K;
  return (size_t) (K::ST::LDS+q*(K::V+1))*sizeof(cplx<T>)+
    ((size_t) K::SLOTS*2*RPlan<M,K::V>::PAD+K::RED)*sizeof(T);
}

template<typename T, int M, class Op>
__global__ void __launch_bounds__((HRowPk<T,M>::NT),(IsProduct<Op>::value ? HRowPk<T,M>::W : HRowPk<T,M>::WF))
hrowpk_kernel(DimArgs d, const cplx<T> *f, const cplx<T> *g, int64_t rows, int64_t rs,
              cplx<T> *out, int64_t os, T scale, Op op)
{
  typedef HRowPk<T,M> K;
  constexpr int V=K::V, TPS=K::TPS, SLOTS=K::SLOTS;
  typedef RPlan<M,V> P;
  constexpr unsigned E=sizeof(cplx<T>);
  extern __shared__ char smem_raw[];
  const int q=(int) d.q, H=(int) d.H;
  cplx<T> *twl=reinterpret_cast<cplx<T> *>(smem_raw);
  const auto tw=stage_table<T,M,V,2048>(twl,d);
  cplx<T> *tq=twl+K::ST::LDS;                 // tq[r (V + 1) + k] = w_N^{TPS k r}
  const cplx<T> *zN=(const cplx<T> *) d.zN;
  fill_twr<T,M,V,K::ST::USED>(twl,zN,q,threadIdx.x,blockDim.x);
  for(int e=threadIdx.x; e < q*(V+1); e += blockDim.x) {
    const int r=e/(V+1), k=e-r*(V+1);
    tq[e]=zN[TPS*k*r];                        // TPS k r <= M r < N
  }
  __syncthreads();
  // a slot of whole waves: its index is uniform over the wave
  int slot=(int) threadIdx.x/TPS;
  if constexpr(TPS >= 64) slot=__builtin_amdgcn_readfirstlane(slot);
  const int t=threadIdx.x-slot*TPS;
  T *xbase=reinterpret_cast<T *>(tq+q*(V+1));
  T *xb=xbase+slot*2*P::PAD;
  for(int64_t rb=(int64_t) blockIdx.x*SLOTS; rb < rows; rb += (int64_t) gridDim.x*SLOTS) {
    const int64_t row=rb+slot;
    const bool live=row < rows;
    // buffers over the row (slots of whole waves), or over the rows of the
    // block with the row's offset per lane
    const int64_t rr=live ? row : rows-1;
    const int64_t b0=TPS >= 64 ? rr : rb;
    const size_t nw=TPS >= 64 ? (size_t) H : (size_t) ((rows-1 < rb+SLOTS-1 ? rows-1-rb : SLOTS-1)*rs+H);
    const unsigned ro=TPS >= 64 ? 0 : (unsigned) ((rr-rb)*rs)*E;
    const __amdgpu_buffer_rsrc_t rf=buf_rsrc(f+b0*rs,nw), rg=buf_rsrc(g+b0*rs,nw);
    // the row's words sigma = t + TPS k
    cplx<T> fu[V], gu[V];
    auto load=[&](int ts) {
#pragma unroll
      for(int k=0; k < V; ++k) {
        const unsigned o=ts+TPS*k < H ? ro+(unsigned) (ts+TPS*k)*E : 0x80000000u;  // past the end: 0
        fu[k]=ld_buf<T>(rf,o,0);
        gu[k]=ld_buf<T>(rg,o,0);
      }
    };
    auto prescale=[&](const RowScales &s) {
      if(s.near) return;                 // hpk_fold2 scales g
#pragma unroll
      for(int k=0; k < V; ++k) {
        fu[k]=mk(scaled(fu[k].x,-s.ef),scaled(fu[k].y,-s.ef));
        gu[k]=mk(scaled(gu[k].x,-s.eg),scaled(gu[k].y,-s.eg));
      }
    };
    load(fresh(t));
    const RowScales sc=row_scales<T,M,SLOTS>(fu,gu,xbase+SLOTS*2*P::PAD);
    prescale(sc);
    cplx<T> acc[V];
#pragma unroll
    for(int k=0; k < V; ++k) acc[k]=mk((T) 0,(T) 0);
    const auto bound=bind_row(op,rr);
    // the product of the unscaled transforms; of far rows, where it is a factor
    // of each, the scales are undone on the results
    auto rop=[&](T F, T G, int l) {
      if constexpr(IsProduct<Op>::value) return bound(F,sc.near ? scaled(G,sc.eg) : G,l);
      else return bound(scaled(F,sc.ef),scaled(G,sc.eg),l);
    };
    for(int r1=0;;) {
      const int r2=r1+1 < q ? r1+1 : -1;
      // the loop's own positions too (see fresh())
      const int ti=fresh(t);
      const cplx<T> b1=zN[ti*r1];
      // both residues folded from one read of the row
      cplx<T> X[V], X2[V];
      T p1[V];
      // (2^-ZEROS is Inf, which a zero must not meet)
      const T sf=scaled((T) 1,-max(fresh(sc.ef),-ScaleRange<T>::LIM));
      const T sg=scaled((T) 1,-max(fresh(sc.eg),-ScaleRange<T>::LIM));
      hpk_fold2<T,M>(X,X2,fu,gu,rf,rg,tq+r1*(V+1),tq+(r2 >= 0 ? r2 : r1)*(V+1),b1,
                     r2 >= 0 ? zN[ti*r2] : b1,ti,r1,r2 >= 0 ? r2 : r1,H,ro,
                     sf,sg,sc.near ? sg : (T) 1);
      if(r2 >= 0) {
        // the two residues' transforms with their butterflies interleaved
        fftr_pair<T,M,V,1>(X,X2,xb,tw,t);
#pragma unroll
        for(int k=0; k < V; ++k) {
          p1[k]=rop(X[k].x,X[k].y,q*(t+TPS*k)+r1);
          X[k]=mk(p1[k],rop(X2[k].x,X2[k].y,q*(t+TPS*k)+r2));
        }
      } else {
        fftr<T,M,V,1>(X,xb,tw,t);
#pragma unroll
        for(int k=0; k < V; ++k) X[k]=mk(rop(X[k].x,X[k].y,q*(t+TPS*k)+r1),(T) 0);
      }
      fftr<T,M,V,-1>(X,xb,tw,t);
      // mirror elements Z(M - sigma) through LDS
      const int tm=fresh(t);
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int e=xidx<T,M,V>(tm+TPS*k);
        xb[e]=X[k].x;
        xb[P::PAD+e]=X[k].y;
      }
      rsync<TPS>();
      const cplx<T> *t1=tq+r1*(V+1), *t2=tq+(r2 >= 0 ? r2 : 0)*(V+1);
      const cplx<T> c1=zN[tm*r1], c2=r2 >= 0 ? zN[tm*r2] : mk((T) 0,(T) 0);
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int e=xidx<T,M,V>((M-(tm+TPS*k)) & (M-1));
        const cplx<T> z=X[k], zc=mk(xb[e],-xb[P::PAD+e]);
        cplx<T> v=mulc((T) 0.5*(z+zc),c1*t1[k]);
        if(r2 >= 0) v=v+mulc(muli((T) 0.5*(z-zc),-1),c2*t2[k]);
        acc[k]=acc[k]+v;
      }
      rsync<TPS>();
      r1 += 2;
      if(r1 >= q) break;
      load(fresh(t));
      prescale(sc);
    }
    if(live) {
      const int to=fresh(t);
#pragma unroll
      for(int k=0; k < V; ++k) acc[k]=scale*acc[k];
      if(IsProduct<Op>::value && !sc.near) {
#pragma unroll
        for(int k=0; k < V; ++k) acc[k]=mk(scaled(acc[k].x,sc.ef+sc.eg),scaled(acc[k].y,sc.ef+sc.eg));
      }
      if constexpr(TPS >= 64) {
        const __amdgpu_buffer_rsrc_t rw=buf_rsrc(out+row*os,H);
#pragma unroll
        for(int k=0; k < V; ++k)
          if(to+TPS*k < H) st_buf<T>(rw,(unsigned) (to+TPS*k)*E,0,acc[k]);
      } else {
        cplx<T> *orow=out+row*os;
#pragma unroll
        for(int k=0; k < V; ++k)
          if(to+TPS*k < H) orow[to+TPS*k]=acc[k];
      }
    }
  }
}


// Hermitian rows longer than one block (H > M): the residue-pair passes of a
// row (fftPadHermitian's D = 2 pairs, convolve.cc:4517-5012) run as
// independent work units (row, pass), each on one slot of TPS threads.  A
// unit folds every block b of the row (wavenumbers k = sigma + b M, |k| < H,
// f(-k) = conj f(k)) into the packed pair W1 + i W2, transforms f and g,
// multiplies as realMultBinary, inverts, unpacks with the mirror element
// Z(M - sigma) and writes its contribution to every stored mode k < H of the
// row into its slice of `part` (slice p = rows x H words); hrows_reduce_kernel
// adds the slices in pass order (deterministic).  Twiddles
// w_N^{(sigma + b M) r} = w_N^{sigma r} w_q^{b r} with w_q^{b r} = zN[(b r mod q) M].
// Dynamic LDS: M complex twiddles + slots * 2 PAD scalar words.
template<typename T, int M>
__global__ void __launch_bounds__(512)
hrows_long_kernel(DimArgs d, const cplx<T> *f, const cplx<T> *g, int64_t rows,
                  int64_t rs, cplx<T> *part)
{
  constexpr int V=RowV::V;
  typedef RPlan<M,V> P;
  constexpr int TPS=P::TPS;
  extern __shared__ char smem_raw[];
  cplx<T> *tw=reinterpret_cast<cplx<T> *>(smem_raw);
  const cplx<T> *zN=(const cplx<T> *) d.zN;
  fill_twr<T,M,V>(tw,zN,(int) d.q,threadIdx.x,blockDim.x);
  __syncthreads();
  const int slots=blockDim.x/TPS;
  const int slot=threadIdx.x/TPS, t=threadIdx.x-slot*TPS;
  T *xb=reinterpret_cast<T *>(tw+M)+slot*2*P::PAD;
  const int q=(int) d.q, H=(int) d.H;
  const int passes=(q+1)/2;
  const int nb=(H-1)/M+1;                 // blocks b in [0, nb) hold the modes k < H
  const int64_t units=rows*passes;
  const cplx<T> zero=mk((T) 0,(T) 0);
  for(int64_t ub=(int64_t) blockIdx.x*slots; ub < units; ub += (int64_t) gridDim.x*slots) {
    const int64_t unit=ub+slot;
    if(unit >= units) break;              // only when slots > 1 (TPS <= 64)
    const int64_t row=unit/passes;
    const int pass=(int) (unit-row*passes);
    const int r1=2*pass, r2=r1+1 < q ? r1+1 : -1;
    const cplx<T> *fr=f+row*rs, *gr=g+row*rs;
    cplx<T> *pr=part+((int64_t) pass*rows+row)*H;
    cplx<T> X[V], Y[V];
#pragma unroll
    for(int k=0; k < V; ++k) X[k]=Y[k]=zero;
    // b r mod q from b = -nb on, advanced by r per block
    int e1=(int) ((q-((int64_t) nb*r1) % q) % q);
    int e2=r2 >= 0 ? (int) ((q-((int64_t) nb*r2) % q) % q) : 0;
    for(int b=-nb; b < nb; ++b) {
      const cplx<T> c1=zN[e1*M], c2=r2 >= 0 ? zN[e2*M] : zero;
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int sigma=t+TPS*k;
        const int kk=sigma+b*M;
        if(kk > -H && kk < H) {
          cplx<T> w=zN[sigma*r1]*c1;
          if(r2 >= 0) w=w+muli(zN[sigma*r2]*c2,1);
          const cplx<T> fv=kk >= 0 ? fr[kk] : conjg(fr[-kk]);
          const cplx<T> gv=kk >= 0 ? gr[kk] : conjg(gr[-kk]);
          X[k]=X[k]+w*fv;
          Y[k]=Y[k]+w*gv;
        }
      }
      e1 += r1;
      if(e1 >= q) e1 -= q;
      if(r2 >= 0) {
        e2 += r2;
        if(e2 >= q) e2 -= q;
      }
    }
    fftr<T,M,V,1>(X,xb,tw,t);
    fftr<T,M,V,1>(Y,xb,tw,t);
#pragma unroll
    for(int k=0; k < V; ++k) X[k]=mk(X[k].x*Y[k].x,X[k].y*Y[k].y);
    fftr<T,M,V,-1>(X,xb,tw,t);
    // mirror elements Z(M - sigma) through LDS
#pragma unroll
    for(int k=0; k < V; ++k) {
      const int e=xidx<T,M,V>(t+TPS*k);
      xb[e]=X[k].x;
      xb[P::PAD+e]=X[k].y;
    }
    rsync<TPS>();
#pragma unroll
    for(int k=0; k < V; ++k) {
      const int e=xidx<T,M,V>((M-(t+TPS*k)) & (M-1));
      const cplx<T> z=X[k], zc=conjg(mk(xb[e],xb[P::PAD+e]));
      // this thread's unpacked pair, with the conjugate twiddles of sigma
      Y[k]=mulc((T) 0.5*(z+zc),zN[(t+TPS*k)*r1]);
      X[k]=r2 >= 0 ? mulc(muli((T) 0.5*(z-zc),-1),zN[(t+TPS*k)*r2]) : zero;
    }
    rsync<TPS>();
    e1=0;
    e2=0;
    for(int b=0; b < nb; ++b) {
      const cplx<T> c1=zN[e1*M], c2=r2 >= 0 ? zN[e2*M] : zero;
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int kk=t+TPS*k+b*M;
        if(kk < H) pr[kk]=mulc(Y[k],c1)+(r2 >= 0 ? mulc(X[k],c2) : zero);
      }
      e1 += r1;
      if(e1 >= q) e1 -= q;
      if(r2 >= 0) {
        e2 += r2;
        if(e2 >= q) e2 -= q;
      }
    }
  }
}

// out[row][k] = scale * sum over passes of part[pass][row][k], k < H, in
// pass order; one block per row (grid-stride).
template<typename T>
__global__ void __launch_bounds__(256)
hrows_reduce_kernel(const cplx<T> *part, int64_t rows, int H, int passes,
                    cplx<T> *out, int64_t os, T scale)
{
  for(int64_t row=blockIdx.x; row < rows; row += gridDim.x)
    for(int k=threadIdx.x; k < H; k += blockDim.x) {
      cplx<T> sum=part[row*H+k];
      for(int p=1; p < passes; ++p) sum=sum+part[((int64_t) p*rows+row)*H+k];
      out[row*os+k]=scale*sum;
    }
}

// ------------------------------------------------------------------------
// Column residue transforms on the register FFT (fftPad forward/backward of
// strided columns, convolve.cc:771-1965) for power-of-two M and at most P2 = 2
// blocks of M per column (p <= 2), complex or centred data.  Lane (c, t) =
// (threadIdx.x % TC, threadIdx.x / TC): consecutive lanes take consecutive
// columns, so every load and store of a wave covers TC adjacent columns; the
// TPS threads of a column span waves and exchange with block barriers, one
// round per stage, through the column's LDS area of CS = 2 PAD + X words
// (real parts, then imaginary parts PAD words on).  Element e of column c
// sits at word base(e) ^ (c BETA mod 32), base being the identity or an XOR
// swizzle (both keep words below M): the (base, X, BETA) of each
// size were found
// by an exhaustive search under the gfx950 LDS bank model (64-bit words:
// writes 16 lanes per pass over 32 banks, reads 32 lanes over 64 banks;
// 32-bit words: 32 lanes over 32 banks) for the lane layout (c, t) above,
// and give conflict-free exchanges (FP32 M = 256: 128 extra passes in 1536).
// Dynamic LDS: M complex twiddles + TC * CS scalar words.
// ------------------------------------------------------------------------
template<typename T, int M> struct ColReg {
  static constexpr int V=8;
  static constexpr int TPS=M/V;
  static constexpr int TC=TPS >= 512 ? 1 : (512/TPS < 64 ? 512/TPS : 64);
  static constexpr int PAD=RPlan<M,V>::PAD;
  static constexpr bool F64=sizeof(T) == 8;
  // base: 0 identity, 2 swizzle
  static constexpr int BASE=M >= 1024 ? 2 : 0;
  static constexpr int X=M == 16 ? 1 : 0;
  static constexpr int BETA=M == 16 || M == 4096 ? 0 : M == 256 ? (F64 ? 17 : 2) : M == 512 ? 9 :
    M == 1024 ? 10 : M == 2048 ? (F64 ? 28 : 20) : 1;
  static constexpr int CS=2*PAD+X;
  static constexpr int NT=TPS*TC;
  typedef SplitTw<T,M,V,2048> ST;
  static __device__ __forceinline__ int at(int e)
  {
    if constexpr(BASE == 2 && F64) return e ^ ((e >> 4) & 7) ^ (((e >> 6) & 1) << 3);
    else if constexpr(BASE == 2) return e ^ ((e >> 5) & 7) ^ (((e >> 6) & 3) << 3);
    else return e;
  }
  // both maps are linear over the bits of e (M >= 1024 swizzles)
  static __device__ __forceinline__ int join(int a, int b) { return a ^ b; }
  // the column's XOR of the word index (M = 16: the words stay below 16)
  static __device__ __forceinline__ int xm(int c) { return (c*BETA) & (M < 32 ? M-1 : 31); }
};

// Waves per SIMD asked of the complex column kernels: four, so that two blocks
// of 512 threads share a CU and one loads while the other transforms, where
// the registers allow it: all FP32 columns (at most 101), FP64 with p = 1 (at
// most 128 forward, 114 backward).  FP64 columns of M >= 2048
// leave room for the second block by reading the last stage's twiddles from
// memory (SplitTw; 2D FP64 2000 x 500: 92 -> 81 us, 4000 x 500: 209 -> 170 us,
// 4000 x 1000: 477 -> 428 us); at 1024 two blocks fit beside the whole table.
template<typename T, int P2> struct ColW {
  static constexpr int W=sizeof(T) == 4 || P2 == 1 ? 4 : 2;
};

// The stage twiddle table of the column kernels (tw) and the residue twiddle
// table they read: zlds = 1 copies the dimension's N twiddles into LDS after
// the exchange areas (the residue twiddles are per-lane gathers, about 10%
// faster from LDS; the host asks for it when the LDS fits without lowering
// occupancy), else the table in global memory.  Ends with a block barrier.
template<typename T, int M> struct ColTwiddles {
  const cplx<T> *zl;      // LDS copy
  const cplx<T> *zN;      // global table
  int zlds;
};

template<typename T, int M>
__device__ __forceinline__ ColTwiddles<T,M> col_twiddles(const DimArgs &d, cplx<T> *tw, int zlds)
{
  typedef ColReg<T,M> CR;
  const cplx<T> *zN=(const cplx<T> *) d.zN;
  fill_twr<T,M,CR::V,CR::ST::USED>(tw,zN,(int) d.q,threadIdx.x,CR::NT);
  cplx<T> *zl=reinterpret_cast<cplx<T> *>(reinterpret_cast<T *>(tw+CR::ST::LDS)+CR::TC*CR::CS);
  if(zlds)
    for(int e=threadIdx.x; e < (int) d.N; e += CR::NT) zl[e]=zN[e];
  __syncthreads();
  return ColTwiddles<T,M>{zl,zN,zlds};
}

// w[i][k] = w_N^{(j0 + M i + k0) r} of the elements kk + k, k < KH, of a
// column, all loaded before the first use (a load per branch made each wait for
// the previous one).  One uniform branch on the table's place: a pointer to
// either would make every load a generic one.  The kernels leave residue 0, whose
// factors are 1, out of it: the only one of a plain FFT (512 x 512 FP64 16.2 us
// with the factors read, 15.5 without).
template<typename T, int M, int P2, int KH>
__device__ __forceinline__ void col_residue(cplx<T> (*w)[KH], const ColTwiddles<T,M> &z,
                                            int t, int kk, int k0, int r, int N)
{
  constexpr int TPS=M/RowV::V;
  typedef const __attribute__((address_space(3))) T *lds_words;
  typedef const __attribute__((address_space(1))) T *global_words;
  auto loads=[&](auto zt) {
#pragma unroll
    for(int k=0; k < KH; ++k) {
      const int j0=(t+TPS*(kk+k)-k0) & (M-1);
#pragma unroll
      for(int i=0; i < P2; ++i) {
        const int e=2*wrapN((j0+M*i+k0)*r,N);
        w[i][k]=mk(zt[e],zt[e+1]);
      }
    }
  };
  if(z.zlds) loads((lds_words) reinterpret_cast<const T *>(z.zl));
  else loads((global_words) reinterpret_cast<const T *>(z.zN));
}

// F[b][(r-r0) M + s][c] = sum_j f[b][j][c] w_N^{(j+k0)(q s + r)}, j < L, for
// each array (f, F) of io;
// column c starts at c*ics of f and c*ocs of F (unit strides for
// interleaved columns, row strides for contiguous rows taken as columns).
template<typename T, int M, int P2>
__global__ void __launch_bounds__(512,(ColW<T,P2>::W))
colfwd_reg_kernel(DimArgs d, ColArrays io, int64_t S, int64_t C,
                  int64_t bsi, int64_t SF, int64_t bso, int64_t r0,
                  int64_t nres, int64_t ics, int64_t ocs, int zlds)
{
  typedef ColReg<T,M> CR;
  constexpr int V=CR::V, TPS=CR::TPS, TC=CR::TC;
  extern __shared__ char smem_raw[];
  cplx<T> *twl=reinterpret_cast<cplx<T> *>(smem_raw);
  const ColTwiddles<T,M> zt=col_twiddles<T,M>(d,twl,zlds);
  const auto tw=stage_table<T,M,V,2048>(twl,d);
  // interleaved columns: consecutive lanes on consecutive columns; rows
  // (column stride ics > 1): a row's threads on consecutive lanes
  const bool rowmap=ics != 1;
  const int c=rowmap ? threadIdx.x/TPS : threadIdx.x % TC;
  const int t=rowmap ? threadIdx.x % TPS : threadIdx.x/TC;
  T *xb=reinterpret_cast<T *>(twl+CR::ST::LDS)+c*CR::CS;
  const int xm=CR::xm(c);
  const int64_t c0=xcd_tile(blockIdx.x,gridDim.x)*TC;
  const bool ok=c0+c < C;
  const ColBlock bk=col_block(io);
  const cplx<T> *fb=(const cplx<T> *) bk.in+(int64_t) blockIdx.y*bsi+(c0+c)*ics;
  cplx<T> *Fb=(cplx<T> *) bk.out+(int64_t) blockIdx.y*bso+(c0+c)*ocs;
  const int N=(int) d.N, L=(int) d.L, k0=(int) d.k0;
  // the column, read once: element j = j0 + M i with j0 = (sigma - k0) mod M
  cplx<T> raw[P2][V];
#pragma unroll
  for(int k=0; k < V; ++k) {
    const int j0=(t+TPS*k-k0) & (M-1);
#pragma unroll
    for(int i=0; i < P2; ++i) {
      const int j=j0+M*i;
      raw[i][k]=ok && j < L ? fb[(int64_t) j*S] : mk((T) 0,(T) 0);
    }
  }
  for(int64_t rr=bk.part; rr < nres; rr += bk.parts) {
    const int r=(int) (r0+rr);
    cplx<T> X[V];
    if(r) {
      cplx<T> w[P2][V];
      col_residue<T,M,P2>(w,zt,fresh(t),0,k0,r,N);
#pragma unroll
      for(int k=0; k < V; ++k) {
        cplx<T> a=raw[0][k]*w[0][k];
#pragma unroll
        for(int i=1; i < P2; ++i) a=a+raw[i][k]*w[i][k];
        X[k]=a;
      }
    } else {
#pragma unroll
      for(int k=0; k < V; ++k) X[k]=P2 == 1 ? raw[0][k] : raw[0][k]+raw[P2-1][k];
    }
    fftr_blkx<T,M,V,1,CR,(sizeof(T) == 8 || P2 == 2)>(X,xb,tw,t,xm);
    if(ok) {
      cplx<T> *Fr=Fb+rr*M*SF;
      const int tf=fresh(t);
#pragma unroll
      for(int k=0; k < V; ++k) Fr[(int64_t) (tf+TPS*k)*SF]=X[k];
    }
  }
}

// f[b][j][c] = scale * ((accumulate ? f : 0) + sum_r w_N^{-(j+k0) r}
// DFT^{-1}[F_r]((j+k0) mod M)), j < L, for each array (F, f) of io.
template<typename T, int M, int P2>
__global__ void __launch_bounds__(512,(ColW<T,P2>::W))
colbwd_reg_kernel(DimArgs d, ColArrays io, int64_t SF, int64_t bsi,
                  int64_t S, int64_t C, int64_t bso, int64_t r0,
                  int64_t nres, int accumulate, T scale, int64_t ics, int64_t ocs,
                  int zlds)
{
  typedef ColReg<T,M> CR;
  constexpr int V=CR::V, TPS=CR::TPS, TC=CR::TC;
  extern __shared__ char smem_raw[];
  cplx<T> *twl=reinterpret_cast<cplx<T> *>(smem_raw);
  const ColTwiddles<T,M> zt=col_twiddles<T,M>(d,twl,zlds);
  const auto tw=stage_table<T,M,V,2048>(twl,d);
  // interleaved columns: consecutive lanes on consecutive columns; rows
  // (column stride ics > 1): a row's threads on consecutive lanes
  const bool rowmap=ics != 1;
  const int c=rowmap ? threadIdx.x/TPS : threadIdx.x % TC;
  const int t=rowmap ? threadIdx.x % TPS : threadIdx.x/TC;
  T *xb=reinterpret_cast<T *>(twl+CR::ST::LDS)+c*CR::CS;
  const int xm=CR::xm(c);
  const int64_t c0=xcd_tile(blockIdx.x,gridDim.x)*TC;
  const bool ok=c0+c < C;
  const ColBlock bk=col_block(io);
  const cplx<T> *Fb=(const cplx<T> *) bk.in+(int64_t) blockIdx.y*bsi+(c0+c)*ics;
  cplx<T> *fb=(cplx<T> *) bk.out+(int64_t) blockIdx.y*bso+(c0+c)*ocs;
  const int N=(int) d.N, L=(int) d.L, k0=(int) d.k0;
  cplx<T> acc[P2][V];
#pragma unroll
  for(int i=0; i < P2; ++i)
#pragma unroll
    for(int k=0; k < V; ++k) acc[i][k]=mk((T) 0,(T) 0);
  for(int64_t rr=0; rr < nres; ++rr) {
    const int r=(int) (r0+rr);
    const cplx<T> *Fr=Fb+rr*M*SF;
    const int tf=fresh(t);
    cplx<T> X[V];
#pragma unroll
    for(int k=0; k < V; ++k) X[k]=ok ? Fr[(int64_t) (tf+TPS*k)*SF] : mk((T) 0,(T) 0);
    fftr_blkx<T,M,V,-1,CR,(sizeof(T) == 8 || P2 == 2)>(X,xb,tw,t,xm);
    // half of the twiddles at a time (all at once costs registers and spills)
    constexpr int KH=V/2;
    if(r == 0) {
#pragma unroll
      for(int k=0; k < V; ++k)
#pragma unroll
        for(int i=0; i < P2; ++i) acc[i][k]=acc[i][k]+X[k];
      continue;
    }
#pragma unroll
    for(int kk=0; kk < V; kk += KH) {
      cplx<T> w[P2][KH];
      col_residue<T,M,P2>(w,zt,tf,kk,k0,r,N);
#pragma unroll
      for(int k=0; k < KH; ++k)
#pragma unroll
        for(int i=0; i < P2; ++i) acc[i][kk+k]=acc[i][kk+k]+mulc(X[kk+k],w[i][k]);
    }
  }
  if(ok) {
    const int tf=fresh(t);
#pragma unroll
    for(int k=0; k < V; ++k) {
      const int j0=(tf+TPS*k-k0) & (M-1);
#pragma unroll
      for(int i=0; i < P2; ++i) {
        const int j=j0+M*i;
        if(j < L) {
          cplx<T> *o=fb+(int64_t) j*S;
          cplx<T> v=acc[i][k];
          if(accumulate) v=v+*o;
          *o=scale*v;
        }
      }
    }
  }
}

// ------------------------------------------------------------------------
// Real columns (fftPadReal, convolve.h:805-980; its forward and backward
// residue transforms, convolve.cc:5449-7483) for power-of-two M and p <= 2.
// For real data the padded transform at l = q s + r and at N - l are complex
// conjugates, so a real dimension keeps K = N/2 + 1 planes, residue-major:
//   r = 0:              s in [0, M/2]  (partner of s: M - s)
//   0 < r < q/2:        s in [0, M)    (partner: residue q - r)
//   r = q/2 (q even):   s in [0, M/2)  (partner of s: M - 1 - s)
// at plane RealKept::base(r) + s.  The planes are complex, so the inner
// dimensions of a real convolution are ordinary complex convolutions over
// K planes; the backward transform folds each kept plane with its partner:
//   f(j) = sum over kept l of c_l Re(F_l w_N^{-j l}),
// c_l = 1 for the self-conjugate planes l = 0 and l = N/2 and 2 for the
// others.  Residues 0 and q/2, which hold their own partners, are inverted
// over all M points with the missing half rebuilt as conjugates of the kept
// half (their real part is then the sum above); the other residues add
// 2 Re(w_N^{-j r} IDFT_M[F_r](j)).  Lanes and LDS as in colfwd_reg_kernel.
// ------------------------------------------------------------------------
struct RealKept {
  __host__ __device__ static int64_t residues(int64_t q) { return q/2+1; }
  __host__ __device__ static int64_t planes(int64_t m, int64_t q) { return m*q/2+1; }
  __host__ __device__ static int64_t base(int64_t m, int64_t r) { return r == 0 ? 0 : m/2+1+(r-1)*m; }
  __host__ __device__ static int64_t count(int64_t m, int64_t q, int64_t r)
  {
    return r == 0 ? m/2+1 : (2*r == q ? m/2 : m);
  }
};

// F[b][base(r) + s][c] = sum_{j < L} f[b][j][c] w_N^{j (q s + r)} for the
// kept (r, s); f real with element stride S and column stride ics (real
// words), F complex with plane stride SF and column stride ocs.
template<typename T, int M, int P2>
__global__ void __launch_bounds__(512,P2 == 1 ? 4 : 2)
colfwd_real_kernel(DimArgs d, ColArrays io, int64_t S, int64_t C, int64_t bsi,
                   int64_t SF, int64_t bso, int64_t ics, int64_t ocs)
{
  typedef ColReg<T,M> CR;
  constexpr int V=CR::V, TPS=CR::TPS, TC=CR::TC;
  extern __shared__ char smem_raw[];
  cplx<T> *twl=reinterpret_cast<cplx<T> *>(smem_raw);
  const auto tw=stage_table<T,M,V,2048>(twl,d);
  const cplx<T> *zN=(const cplx<T> *) d.zN;
  fill_twr<T,M,V,CR::ST::USED>(twl,zN,(int) d.q,threadIdx.x,CR::NT);
  __syncthreads();
  const bool rowmap=ics != 1;
  const int c=rowmap ? threadIdx.x/TPS : threadIdx.x % TC;
  const int t=rowmap ? threadIdx.x % TPS : threadIdx.x/TC;
  T *xb=reinterpret_cast<T *>(twl+CR::ST::LDS)+c*CR::CS;
  const int xm=CR::xm(c);
  const int64_t c0=xcd_tile(blockIdx.x,gridDim.x)*TC;
  const bool ok=c0+c < C;
  const ColBlock bk=col_block(io);
  const T *fb=(const T *) bk.in+(int64_t) blockIdx.y*bsi+(c0+c)*ics;
  cplx<T> *Fb=(cplx<T> *) bk.out+(int64_t) blockIdx.y*bso+(c0+c)*ocs;
  const int N=(int) d.N, L=(int) d.L, q=(int) d.q;
  T raw[P2][V];
#pragma unroll
  for(int k=0; k < V; ++k)
#pragma unroll
    for(int i=0; i < P2; ++i) {
      const int j=t+TPS*k+M*i;
      raw[i][k]=ok && j < L ? fb[(int64_t) j*S] : (T) 0;
    }
  const int R=(int) RealKept::residues(q);
  for(int r=bk.part; r < R; r += bk.parts) {
    // twiddles loaded before the first use (r = 0 reads 1)
    cplx<T> w[P2][V];
#pragma unroll
    for(int k=0; k < V; ++k)
#pragma unroll
      for(int i=0; i < P2; ++i) w[i][k]=zN[wrapN((t+TPS*k+M*i)*r,N)];
    cplx<T> X[V];
#pragma unroll
    for(int k=0; k < V; ++k) {
      cplx<T> a=raw[0][k]*w[0][k];
#pragma unroll
      for(int i=1; i < P2; ++i) a=a+raw[i][k]*w[i][k];
      X[k]=a;
    }
    // fewer registers are live than in the complex columns: on short columns
    // the positions stay in them (256^3 FP64 124 us with fresh ones)
    fftr_blkx<T,M,V,1,CR,(M >= 512)>(X,xb,tw,t,xm);
    if(ok) {
      const int cnt=(int) RealKept::count(M,q,r);
      cplx<T> *Fr=Fb+RealKept::base(M,r)*SF;
#pragma unroll
      for(int k=0; k < V; ++k)
        if(t+TPS*k < cnt) Fr[(int64_t) (t+TPS*k)*SF]=X[k];
    }
  }
}

// f[b][j][c] = scale sum over kept l of c_l Re(F[b][l][c] w_N^{-j l}), j < L.
template<typename T, int M, int P2>
__global__ void __launch_bounds__(512)
colbwd_real_kernel(DimArgs d, const cplx<T> *F, int64_t SF, int64_t bsi,
                   T *f, int64_t S, int64_t C, int64_t bso, T scale,
                   int64_t ics, int64_t ocs)
{
  typedef ColReg<T,M> CR;
  constexpr int V=CR::V, TPS=CR::TPS, TC=CR::TC;
  extern __shared__ char smem_raw[];
  cplx<T> *twl=reinterpret_cast<cplx<T> *>(smem_raw);
  const auto tw=stage_table<T,M,V,2048>(twl,d);
  const cplx<T> *zN=(const cplx<T> *) d.zN;
  fill_twr<T,M,V,CR::ST::USED>(twl,zN,(int) d.q,threadIdx.x,CR::NT);
  __syncthreads();
  const bool rowmap=ics != 1;
  const int c=rowmap ? threadIdx.x/TPS : threadIdx.x % TC;
  const int t=rowmap ? threadIdx.x % TPS : threadIdx.x/TC;
  T *xb=reinterpret_cast<T *>(twl+CR::ST::LDS)+c*CR::CS;
  const int xm=CR::xm(c);
  const int64_t c0=xcd_tile(blockIdx.x,gridDim.x)*TC;
  const bool ok=c0+c < C;
  const cplx<T> *Fb=F+(int64_t) blockIdx.y*bsi+(c0+c)*ics;
  T *fb=f+(int64_t) blockIdx.y*bso+(c0+c)*ocs;
  const int N=(int) d.N, L=(int) d.L, q=(int) d.q;
  T acc[P2][V];
#pragma unroll
  for(int i=0; i < P2; ++i)
#pragma unroll
    for(int k=0; k < V; ++k) acc[i][k]=(T) 0;
  const int R=(int) RealKept::residues(q);
  for(int r=0; r < R; ++r) {
    const cplx<T> *Fr=Fb+RealKept::base(M,r)*SF;
    const bool self=r == 0 || 2*r == q;
    // the full residue: kept s, or the conjugate of the partner's kept word
    const int mirror=r == 0 ? M : M-1;
    cplx<T> X[V];
#pragma unroll
    for(int k=0; k < V; ++k) {
      const int s=t+TPS*k;
      const bool direct=!self || s < (int) RealKept::count(M,q,r);
      cplx<T> v=mk((T) 0,(T) 0);
      if(ok) {
        v=Fr[(int64_t) (direct ? s : mirror-s)*SF];
        if(!direct) v=conjg(v);
      }
      X[k]=v;
    }
    fftr_blkx<T,M,V,-1,CR,(M >= 512)>(X,xb,tw,t,xm);
    const T cr=self ? (T) 1 : (T) 2;
    // twiddles loaded before their use (r = 0 reads 1), half of the values
    // at a time (all at once costs a wave per SIMD)
    constexpr int KH=V/2;
#pragma unroll
    for(int h=0; h < V; h += KH) {
      cplx<T> w[P2][KH];
#pragma unroll
      for(int k=0; k < KH; ++k)
#pragma unroll
        for(int i=0; i < P2; ++i) w[i][k]=zN[wrapN((t+TPS*(h+k)+M*i)*r,N)];
#pragma unroll
      for(int k=0; k < KH; ++k)
#pragma unroll
        for(int i=0; i < P2; ++i)
          acc[i][h+k] += cr*(X[h+k].x*w[i][k].x+X[h+k].y*w[i][k].y);
    }
  }
  if(ok) {
#pragma unroll
    for(int k=0; k < V; ++k)
#pragma unroll
      for(int i=0; i < P2; ++i) {
        const int j=t+TPS*k+M*i;
        if(j < L) fb[(int64_t) j*S]=scale*acc[i][k];
      }
  }
}

} // namespace fftwpp_amd
