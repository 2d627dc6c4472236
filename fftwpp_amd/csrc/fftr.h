// fftr.h -- register-resident Stockham FFT of a compile-time power-of-two
// length M (16 <= M <= 4096): the sub-FFT layer (the role of FFTW's
// mfft1d in the reference, fftw++.h:576-896) for the fused kernels whose
// sub-FFT size is not 256.
//
// TPS = M/V threads hold one sequence, thread t keeping x[t + TPS k] in
// v[k], k < V (V = 16, or 8 to halve the registers of FP64 kernels), before
// and after the transform.  The stages are radix V (and one final smaller
// power of two when log2 M is not a multiple of log2 V); stage s with radix
// R and Ns = (product of the earlier radices) does, for each butterfly
// j = t + TPS b (b < V/R) with k' = j mod Ns,
//     u_t' = v[b + t' V/R] w^{t' k'},   w = e^{S 2 pi i/(Ns R)},
//     out[(j/Ns) Ns R + k' + u Ns] = sum_t' u_t' e^{S 2 pi i u t'/R},
// in place in registers; between stages the outputs go through LDS in one round
// (an area of 2 PAD scalar words: real parts, then imaginary parts PAD words on;
// element e at the word that an index map names, see xidx()) and come back as
// v[k] = out[t + TPS k].  After the last stage v[k] holds X[t + TPS k].
//
// Twiddles: one LDS table of M-1 complex words, stage s at offset off_s
// holding e^{2 pi i t' k'/(Ns R)} at off_s + (t'-1) Ns + k', so the threads
// of a stage read consecutive words; fill_twr() builds it from the
// dimension's FP64-generated table zN (N = M q): e^{2 pi i n/M} = zN[q n].
#pragma once
#include "common.h"
#include "fft_lds.h"
#include "fft256.h"

namespace fftwpp_amd {

template<int M, int V=16> struct RPlan {
  static_assert(M >= 16 && M <= 4096 && (M & (M-1)) == 0, "M must be 2^k, 16..4096");
  static_assert(V == 8 || V == 16, "8 or 16 values per thread");
  static constexpr int TPS=M/V;
  static constexpr int LOG=__builtin_ctz(M);
  static constexpr int LV=__builtin_ctz(V);
  static constexpr int NV=LOG/LV;                       // radix-V stages
  static constexpr int LAST=1 << (LOG-LV*NV);           // remaining factor
  static constexpr int NST=NV+(LAST > 1 ? 1 : 0);
  // exchange words (the swizzled sequences of 512 or more use M of them)
  static constexpr int PAD=M >= 512 ? M : M+M/16;
  __host__ __device__ static constexpr int radix(int s) { return s < NV ? V : LAST; }
  // Stage s writes output u of butterfly j at dest<s>(j) + u ns(s); the bits
  // of j move without mixing, so dest(a + b) = dest(a) + dest(b) for a and b
  // without a bit in common.
  template<int s>
  static __device__ __forceinline__ int dest(int j)
  {
    const int kp=j & (ns(s)-1);
    return (j-kp)*radix(s)+kp;
  }
  // loops rather than recursion, so that calls with a run-time s inline
  __host__ __device__ static constexpr int ns(int s)
  {
    int n=1;
    for(int i=0; i < s; ++i) n *= radix(i);
    return n;
  }
  __host__ __device__ static constexpr int logns(int s) { return s < NV ? LV*s : LV*NV; }
  __host__ __device__ static constexpr int off(int s)
  {
    int o=0;
    for(int i=1; i < s; ++i) o += (radix(i)-1)*ns(i);
    return o;
  }
};

__device__ __forceinline__ int padr(int e) { return e+(e >> 4); }

// Word of sequence element e in each half of an exchange area: an XOR
// swizzle of the low bits by higher bits that makes every exchange of the
// transform conflict-free on gfx950's LDS (64-bit words: writes served 16
// lanes per pass over 32 banks, reads 32 lanes over 64 banks; 32-bit words:
// 32 lanes over 32 banks).  Shorter sequences (V = 8: M < 128 in FP64, M <
// 256 in FP32; V = 16: M < 512) take e + e/16, whose compile-time part is an
// immediate offset of the access: it has conflicts, but needs 10 to 60 fewer
// registers and no instructions (complex rows of M = 64 FP64 98 us against
// 107 swizzled, M = 128 FP32 67 against 91; M = 128 FP64 133 against 126).
// Indices stay below RPlan::PAD.
template<typename T, int M, int V>
__host__ __device__ constexpr bool xswizzled()
{
  return M >= (V == 16 ? 512 : sizeof(T) == 8 ? 128 : 256);
}
template<typename T, int M, int V>
__device__ __forceinline__ int xidx(int e)
{
  if constexpr(V == 8 && xswizzled<T,M,V>()) return e ^ ((e >> 3) & 7) ^ (((e >> 6) & 3) << 3);
  else if constexpr(xswizzled<T,M,V>()) return e ^ ((e >> 4) & 7) ^ (((e >> 7) & 3) << 3);
  else return padr(e);
}

// Twiddle table (M - 1 complex words) from zN of a dimension with N = M q.
template<typename T, int M, int V=16, bool SPLIT=false>
__device__ __forceinline__ void fill_twr(cplx<T> *tw, const cplx<T> *zN, int q,
                                         int tid, int nthreads)
{
  typedef RPlan<M,V> P;
  for(int e=tid; e < (SPLIT ? P::off(P::NST-1) : M-1); e += nthreads) {
    // locate the stage of entry e (constants per unrolled k); Ns and Ns R are
    // powers of two: shifts only
    int ln=P::logns(1), lr=P::logns(1)+__builtin_ctz(P::radix(1)), off=0;
#pragma unroll
    for(int k=2; k < P::NST; ++k)
      if(e >= P::off(k)) { ln=P::logns(k); lr=ln+__builtin_ctz(P::radix(k)); off=P::off(k); }
    const int rel=e-off;
    const int tp=(rel >> ln)+1, kp=rel & ((1 << ln)-1);
    // e^{2 pi i tp kp/(Ns R)} = zN[q tp kp M/(Ns R)]
    tw[e]=zN[(int64_t) q*((tp*kp) << (P::LOG-lr))];
  }
}

// Radix-R butterfly (R = 2, 4, 8, 16) with kernel e^{S 2 pi i ut/R}.
template<typename T, int R, int S>
__device__ __forceinline__ void bfly(cplx<T> *u)
{
  if constexpr(R == 16) dft16<T,S>(u);
  else DFT<T,R>::run(u,S);
}

// Twiddles of a long FP64 transform: those of the last stage, half of the table
// at 1024 points, three quarters at 2048 and seven eighths at 4096, stay in device memory in the table's
// order (DimArgs::last) and are read from there by each transform, consecutive
// lanes consecutive words; LDS holds the others.  These transforms wait on LDS
// and barriers rather than compute (13% of the vector unit's cycles), and with
// all of the table in LDS two waves per SIMD were resident; now three are.
// 2048 rows of 1000 points padded to 2048: 49 -> 41.5 us; 4096 sequences of 64
// to 16384 words, in a process of their own: 632 -> 541 us.
template<typename T, int M, int V, int MIN=1024> struct SplitTw {
  static constexpr bool USED=sizeof(T) == 8 && V == 8 && M >= MIN;
  static constexpr int LDS=USED ? 512 : M;
  const cplx<T> *tw;
  __amdgpu_buffer_rsrc_t last;
};

// The table as the kernels pass it on: split, or all of it in LDS.
template<typename T, int M, int V, int MIN=1024>
__device__ __forceinline__ auto stage_table(const cplx<T> *tw, const DimArgs &d)
{
  if constexpr(SplitTw<T,M,V,MIN>::USED) {
    typedef RPlan<M,V> P;
    return SplitTw<T,M,V,MIN>{tw,buf_rsrc((const cplx<T> *) d.last,(size_t) (M-1-P::off(P::NST-1)))};
  } else return tw;
}

// Twiddle tp of stage s for butterfly j = t + J (J constant): word off(s) +
// (tp - 1) ns(s) + (j mod ns(s)) of the table.
template<typename T, int M, int V, int s>
__device__ __forceinline__ cplx<T> stage_word(const cplx<T> *tw, int t, int J, int tp)
{
  typedef RPlan<M,V> P;
  return table_word(tw+P::off(s)+((t+J) & (P::ns(s)-1))+(tp-1)*P::ns(s));
}
template<typename T, int M, int V, int s, int MIN>
__device__ __forceinline__ cplx<T> stage_word(const SplitTw<T,M,V,MIN> &w, int t, int J, int tp)
{
  typedef RPlan<M,V> P;
  constexpr unsigned E=sizeof(cplx<T>);
  if constexpr(s == P::NST-1) return ld_buf<T>(w.last,(unsigned) t*E,(J+(tp-1)*P::ns(s))*E);
  else return stage_word<T,M,V,s>(w.tw,t,J,tp);
}

// Synchronisation of the threads of a sequence: the wave when a sequence
// does not span waves (its TPS threads are consecutive lanes), else the block.
template<int TPS, bool BLK=false>
__device__ __forceinline__ void rsync()
{
  if constexpr(TPS <= 64 && !BLK) {
    __builtin_amdgcn_fence(__ATOMIC_RELEASE,"wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE,"wavefront");
  } else
    __syncthreads();
}

// Word of element e in each half of an exchange area (the default index map).
// The maps act on disjoint bit fields one by one, so the word of an element
// whose thread part and compile-time part have no bit in common is
// join(at(thread part), at(constant)): one instruction per access and one
// register per stage, where a map evaluated per element took several of each.
template<typename T, int M, int V> struct RowXI {
  static constexpr bool SWIZZLE=xswizzled<T,M,V>();
  static __device__ __forceinline__ int at(int e) { return xidx<T,M,V>(e); }
  static __device__ __forceinline__ int join(int a, int b) { return SWIZZLE ? a ^ b : a+b; }
};

// Stage s of the transform (see the top of this file); recurses into s+1.
// Element e sits at word XI::at(e) ^ xm of each half of the exchange area xb.
template<typename T, int M, int V, int S, int s, bool BLK, class XI=RowXI<T,M,V>, class TW>
__device__ __forceinline__ void fftr_stage(cplx<T> *v, T *xb, const TW &tw,
                                           int t, int xm=0)
{
  typedef RPlan<M,V> P;
  constexpr int TPS=P::TPS;
  constexpr int R=P::radix(s), NB=V/R, Ns=P::ns(s);
  // butterflies in place: slot b + t' NB holds input t' / output u = t'
#pragma unroll
  for(int b=0; b < NB; ++b) {
    cplx<T> u[R];
#pragma unroll
    for(int tp=0; tp < R; ++tp) u[tp]=v[b+tp*NB];
    if constexpr(s > 0) {
#pragma unroll
      for(int tp=1; tp < R; ++tp) {
        const cplx<T> z=stage_word<T,M,V,s>(tw,t,TPS*b,tp);
        u[tp]=S > 0 ? u[tp]*z : mulc(u[tp],z);
      }
    }
    bfly<T,R,S>(u);
#pragma unroll
    for(int tp=0; tp < R; ++tp) v[b+tp*NB]=u[tp];
  }
  if constexpr(s+1 < P::NST) {
    // exchange: output u of butterfly b goes to (j/Ns) Ns R + k' + u Ns
    const int wo=XI::at(P::template dest<s>(t)) ^ xm, ro=XI::at(t) ^ xm;
#pragma unroll
    for(int b=0; b < NB; ++b) {
#pragma unroll
      for(int u=0; u < R; ++u) {
        const int e=XI::join(wo,XI::at(P::template dest<s>(TPS*b)+u*Ns));
        xb[e]=v[b+u*NB].x;
        xb[P::PAD+e]=v[b+u*NB].y;
      }
    }
    rsync<TPS,BLK>();
#pragma unroll
    for(int k=0; k < V; ++k) {
      const int e=XI::join(ro,XI::at(TPS*k));
      v[k]=mk(xb[e],xb[P::PAD+e]);
    }
    rsync<TPS,BLK>();
    fftr_stage<T,M,V,S,s+1,BLK,XI>(v,xb,tw,t,xm);
  }
}

// Stage s of two transforms of the same size and sign at once (one-round
// exchanges, the default index map): the butterflies of both sequences are
// independent work for the same waves, then each is exchanged in turn through
// the one area (the same barriers as two fftr calls).
template<typename T, int M, int V, int S, int s, class TW>
__device__ __forceinline__ void fftr_pair_stage(cplx<T> *X, cplx<T> *Y, T *xb,
                                                const TW &tw, int t)
{
  typedef RPlan<M,V> P;
  typedef RowXI<T,M,V> XI;
  constexpr int TPS=P::TPS;
  constexpr int R=P::radix(s), NB=V/R, Ns=P::ns(s);
#pragma unroll
  for(int b=0; b < NB; ++b) {
    cplx<T> u[R], v[R];
#pragma unroll
    for(int tp=0; tp < R; ++tp) {
      u[tp]=X[b+tp*NB];
      v[tp]=Y[b+tp*NB];
    }
    if constexpr(s > 0) {
#pragma unroll
      for(int tp=1; tp < R; ++tp) {
        const cplx<T> z=stage_word<T,M,V,s>(tw,t,TPS*b,tp);
        u[tp]=S > 0 ? u[tp]*z : mulc(u[tp],z);
        v[tp]=S > 0 ? v[tp]*z : mulc(v[tp],z);
      }
    }
    bfly<T,R,S>(u);
    bfly<T,R,S>(v);
#pragma unroll
    for(int tp=0; tp < R; ++tp) {
      X[b+tp*NB]=u[tp];
      Y[b+tp*NB]=v[tp];
    }
  }
  if constexpr(s+1 < P::NST) {
    const int wo=XI::at(P::template dest<s>(t)), ro=XI::at(t);
#pragma unroll
    for(int pass=0; pass < 2; ++pass) {
      cplx<T> *Z=pass == 0 ? X : Y;
#pragma unroll
      for(int b=0; b < NB; ++b) {
#pragma unroll
        for(int u=0; u < R; ++u) {
          const int e=XI::join(wo,XI::at(P::template dest<s>(TPS*b)+u*Ns));
          xb[e]=Z[b+u*NB].x;
          xb[P::PAD+e]=Z[b+u*NB].y;
        }
      }
      rsync<TPS>();
#pragma unroll
      for(int k=0; k < V; ++k) {
        const int e=XI::join(ro,XI::at(TPS*k));
        Z[k]=mk(xb[e],xb[P::PAD+e]);
      }
      rsync<TPS>();
    }
    fftr_pair_stage<T,M,V,S,s+1>(X,Y,xb,tw,t);
  }
}

// Positions computed anew (see fresh()) with 8 values per thread; with 16 (FP32
// batches) the registers are there, and computing them again per transform took a
// fifth to a third of the time: 2666 items of 3000 words, m = 4096, q = 2, 192 -> 165
// us, 1333 of 6000 words 209 -> 157 us.
template<int V> __device__ __forceinline__ int anew(int t) { return V == 16 ? t : fresh(t); }

// fftr<T,M,V,S> of X and of Y, their butterflies interleaved stage by
// stage; same results, same exchange area and barriers.
template<typename T, int M, int V, int S, class TW>
__device__ __forceinline__ void fftr_pair(cplx<T> *X, cplx<T> *Y, T *xb, const TW &tw,
                                          int t)
{
  fftr_pair_stage<T,M,V,S,0>(X,Y,xb,tw,anew<V>(t));
}

// In-place transform of the sequence held by threads t < TPS (v[V] each)
// with kernel e^{S 2 pi i jk/M}; xb is the sequence's exchange area (2
// RPlan<M,V>::PAD scalar words), tw the twiddle table of RPlan<M,V>.  When
// TPS > 64 every thread of the block must call this.  FRESH: positions computed
// anew (see fresh()).
template<typename T, int M, int V, int S, bool FRESH=true, class TW>
__device__ __forceinline__ void fftr(cplx<T> *v, T *xb, const TW &tw, int t)
{
  fftr_stage<T,M,V,S,0,false>(v,xb,tw,FRESH ? anew<V>(t) : t);
}

// The same transform when the threads of a sequence are not consecutive
// lanes (block barriers; every thread of the block must call it), through the
// index map XI, XORed by xm.  FRESH: positions computed anew (see fresh()).
template<typename T, int M, int V, int S, class XI, bool FRESH=true, class TW>
__device__ __forceinline__ void fftr_blkx(cplx<T> *v, T *xb, const TW &tw,
                                          int t, int xm)
{
  fftr_stage<T,M,V,S,0,true,XI>(v,xb,tw,FRESH ? fresh(t) : t,xm);
}

} // namespace fftwpp_amd
