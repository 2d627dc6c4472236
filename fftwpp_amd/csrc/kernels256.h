// kernels256.h -- residue transforms and fused row convolution for the
// sub-FFT size m = 256 with p = 1 (L <= 256), non-centred data: the shape of
// every dimension of the 256^3 -> 512^3 convolution.  Same contracts as the
// generic kernels in kernels.hip, with the FFT held in registers (fft256.h).
//
// Addressing: element e = j + 16k of a lane lives at
//     (uniform base + 16 k * stride) + (lane offset)
// so each unrolled access uses a scalar base and one 32-bit vector offset
// shared by all k; the host guarantees offsets below 2^31 elements.
#pragma once
#include "fft256.h"


namespace fftwpp_amd {

template<typename T>
__device__ __forceinline__ cplx<T> zero() { return mk((T) 0,(T) 0); }

__device__ __forceinline__ void wsync_rows()
{
  __builtin_amdgcn_fence(__ATOMIC_RELEASE,"wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE,"wavefront");
}

// Column kernels: lane (c, j) = (threadIdx.x % TC, threadIdx.x / TC), so
// consecutive lanes read consecutive columns; the 16 lanes j of column c
// share an exchange area of CS scalar words (block barriers, since they span
// waves).  TC, CS and the swizzle h(c) make every LDS exchange access
// bank-conflict free on gfx950 (64-bit writes are served 16 lanes per pass
// over 32 banks, 64-bit reads 32 lanes per pass over 64 banks, 32-bit
// accesses 32 lanes per pass over 32 banks): FP64 uses 8 columns, areas 276
// words apart and h = 2 for columns 4..7; FP32 uses 16 columns, areas 274
// words apart and no swizzle.
template<typename T> struct Col256 {
  static constexpr int TC=sizeof(T) == 8 ? 8 : 16;
  static constexpr int CS=sizeof(T) == 8 ? 276 : 274;
  __device__ static int swz(int c) { return sizeof(T) == 8 ? ((c >> 1) & 2) : 0; }
};

// Dynamic LDS bytes of the column kernels for nres residues: residue
// twiddles (256 nres complex), stage twiddles (256 complex), exchange areas.
template<typename T>
inline size_t col256_lds(size_t nres)
{
  return (256*nres+256)*sizeof(cplx<T>)+Col256<T>::TC*Col256<T>::CS*sizeof(T);
}

// Dynamic LDS bytes of the row kernel with NR rows per block and q residues.
template<typename T>
inline size_t row256_lds(int NR, size_t q)
{
  return (256*q+256)*sizeof(cplx<T>)+NR*16*17*sizeof(T);
}

// Forward residue transforms of one column: for each residue r = r0 + rr,
// F_r(s) = DFT_256[w_N^{r k} f(k)](s), written at Fb + rr*256*SF; the block
// takes every parts-th rr from part on.
template<typename T>
__device__ __forceinline__ void colfwd_body(const cplx<T> *fb, cplx<T> *Fb,
                                            int64_t S, int64_t SF, bool ok,
                                            int c, int j, int L, int64_t r0,
                                            int64_t nres, int part, int parts,
                                            const cplx<T> *rtab,
                                            const cplx<T> *tw16, T *row, int h)
{
  const unsigned lin=(unsigned) (c+j*S);
  const unsigned lout=(unsigned) (c+j*SF);
  // the column is read once and kept in registers for all residues
  cplx<T> x0[16];
#pragma unroll
  for(int k=0; k < 16; ++k) {
    const cplx<T> *bk=fb+(int64_t) 16*k*S;
    x0[k]=(ok && j+16*k < L) ? bk[lin] : zero<T>();
  }
  for(int64_t rr=part; rr < nres; rr += parts) {
    const int64_t r=r0+rr;
    const cplx<T> *rt=rtab+256*rr;
    cplx<T> v[16];
#pragma unroll
    for(int k=0; k < 16; ++k) {
      v[k]=r == 0 ? x0[k] : x0[k]*table_word(rt+16*k+j);
    }
    fft256s<T,1,0>(v,row,j,h,tw16);
    cplx<T> *Fr=Fb+rr*256*SF;
    if(ok) {
#pragma unroll
      for(int u=0; u < 16; ++u) (Fr+(int64_t) 16*u*SF)[lout]=v[u];
    }
  }
}

// Backward residue transforms of one column, accumulated over the residues:
// f(k) = scale * sum_rr w_N^{-r k} DFT_256^{-1}[F_r](k) (+ f(k) if accumulate).
template<typename T>
__device__ __forceinline__ void colbwd_body(const cplx<T> *Fb, cplx<T> *fb,
                                            int64_t S, int64_t SF, bool ok,
                                            int c, int j, int L, int64_t r0,
                                            int64_t nres, int accumulate,
                                            T scale, const cplx<T> *rtab,
                                            const cplx<T> *tw16, T *row, int h)
{
  const unsigned lin=(unsigned) (c+j*SF);
  const unsigned lout=(unsigned) (c+j*S);
  cplx<T> acc[16];
#pragma unroll
  for(int k=0; k < 16; ++k) acc[k]=zero<T>();
  for(int64_t rr=0; rr < nres; ++rr) {
    const int64_t r=r0+rr;
    const cplx<T> *rt=rtab+256*rr;
    const cplx<T> *Fr=Fb+rr*256*SF;
    cplx<T> v[16];
#pragma unroll
    for(int u=0; u < 16; ++u)
      v[u]=ok ? (Fr+(int64_t) 16*u*SF)[lin] : zero<T>();
    fft256s<T,-1,0>(v,row,j,h,tw16);
#pragma unroll
    for(int k=0; k < 16; ++k)
      acc[k]=acc[k]+(r == 0 ? v[k] : mulc(v[k],table_word(rt+16*k+j)));
  }
  if(ok) {
#pragma unroll
    for(int k=0; k < 16; ++k) {
      if(j+16*k < L) {
        cplx<T> *o=fb+(int64_t) 16*k*S;
        cplx<T> v=acc[k];
        if(accumulate) v=v+o[lout];
        o[lout]=scale*v;
      }
    }
  }
}

template<typename T>
__global__ void __launch_bounds__(16*Col256<T>::TC,sizeof(T) == 4 ? 3 : 2)
colfwd256_kernel(ColArrays io, int64_t S, int64_t C, int64_t bsi,
                 int64_t SF, int64_t bso, int L, int64_t r0,
                 int64_t nres, const cplx<T> *zN, int64_t q)
{
  constexpr int TC=Col256<T>::TC;
  extern __shared__ char smem_raw[];
  cplx<T> *rtab=reinterpret_cast<cplx<T> *>(smem_raw);
  cplx<T> *tw16=rtab+256*nres;
  fill_rtab(rtab,zN,(int) r0,(int) nres,threadIdx.x,16*TC);
  fill_tw16(tw16,zN,(int) q,threadIdx.x,16*TC);
  __syncthreads();
  const int c=threadIdx.x % TC, j=threadIdx.x/TC;
  T *row=reinterpret_cast<T *>(tw16+256)+c*Col256<T>::CS;
  const int64_t c0=xcd_tile(blockIdx.x,gridDim.x)*TC;
  const bool ok=c0+c < C;
  const ColBlock bk=col_block(io);
  const cplx<T> *fb=(const cplx<T> *) bk.in+(int64_t) blockIdx.y*bsi+c0;
  cplx<T> *Fb=(cplx<T> *) bk.out+(int64_t) blockIdx.y*bso+c0;
  colfwd_body<T>(fb,Fb,S,SF,ok,c,j,L,r0,nres,bk.part,bk.parts,rtab,tw16,row,Col256<T>::swz(c));
}

template<typename T>
__global__ void __launch_bounds__(16*Col256<T>::TC,sizeof(T) == 4 ? 3 : 2)
colbwd256_kernel(ColArrays io, int64_t SF, int64_t bsi,
                 int64_t S, int64_t C, int64_t bso, int L, int64_t r0,
                 int64_t nres, int accumulate, T scale, const cplx<T> *zN,
                 int64_t q)
{
  constexpr int TC=Col256<T>::TC;
  extern __shared__ char smem_raw[];
  cplx<T> *rtab=reinterpret_cast<cplx<T> *>(smem_raw);
  cplx<T> *tw16=rtab+256*nres;
  fill_rtab(rtab,zN,(int) r0,(int) nres,threadIdx.x,16*TC);
  fill_tw16(tw16,zN,(int) q,threadIdx.x,16*TC);
  __syncthreads();
  const int c=threadIdx.x % TC, j=threadIdx.x/TC;
  T *row=reinterpret_cast<T *>(tw16+256)+c*Col256<T>::CS;
  const int64_t c0=xcd_tile(blockIdx.x,gridDim.x)*TC;
  const bool ok=c0+c < C;
  const ColBlock bk=col_block(io);
  const cplx<T> *Fb=(const cplx<T> *) bk.in+(int64_t) blockIdx.y*bsi+c0;
  cplx<T> *fb=(cplx<T> *) bk.out+(int64_t) blockIdx.y*bso+c0;
  colbwd_body<T>(Fb,fb,S,SF,ok,c,j,L,r0,nres,accumulate,scale,rtab,tw16,row,
                 Col256<T>::swz(c));
}

// Rows: NR rows per block of 16*NR lanes; lane j of row i = threadIdx.x % 16,
// so the 16 lanes of a row share a wave and exchange through LDS without
// block barriers (row areas 16*17 words apart are conflict free).  The block
// first stages the residue twiddles (256 q) and the stage twiddles (256) in
// LDS.  Dynamic LDS: row256_lds().
// KEEP: the rows of f and g are read once and kept in registers for all
// residues (FP32); otherwise each residue reads them again (FP64, where
// keeping them would leave one wave per SIMD).
template<typename T> struct Row256 {
  static constexpr bool KEEP=sizeof(T) == 4;
  static constexpr int MINW=2;
};
template<typename T, class Op, int NR>
__global__ void __launch_bounds__(16*NR,Row256<T>::MINW)
rowconv256_kernel(const cplx<T> *f, const cplx<T> *g, int64_t rows, int64_t rs,
                  cplx<T> *out, int64_t os, int L, T scale, const cplx<T> *zN,
                  int64_t q, Op op)
{
  extern __shared__ char smem_raw[];
  const int qi=(int) q;
  cplx<T> *rtab=reinterpret_cast<cplx<T> *>(smem_raw);   // 256 q
  cplx<T> *tw16=rtab+256*qi;                              // 256
  T *lds=reinterpret_cast<T *>(tw16+256);
  fill_rtab(rtab,zN,0,qi,threadIdx.x,16*NR);
  fill_tw16(tw16,zN,qi,threadIdx.x,16*NR);
  __syncthreads();
  const int i=threadIdx.x/16, j=threadIdx.x % 16;
  const int64_t row0=(int64_t) blockIdx.x*NR;
  const bool ok=row0+i < rows;
  const cplx<T> *fr=f+row0*rs;
  const cplx<T> *gr=g+row0*rs;
  cplx<T> *orow=out+row0*os;
  const unsigned lin=(unsigned) (i*rs+j);
  const unsigned lo=(unsigned) (i*os+j);
  T *row=lds+i*16*17;
  cplx<T> acc[16];
#pragma unroll
  for(int k=0; k < 16; ++k) acc[k]=zero<T>();
  constexpr bool KEEP=Row256<T>::KEEP;
  cplx<T> a0[KEEP ? 16 : 1], b0[KEEP ? 16 : 1];
  if constexpr(KEEP) {
#pragma unroll
    for(int k=0; k < 16; ++k) {
      bool in=ok && j+16*k < L;
      a0[k]=in ? (fr+16*k)[lin] : zero<T>();
      b0[k]=in ? (gr+16*k)[lin] : zero<T>();
    }
  }
  for(int r=0; r < qi; ++r) {
    const cplx<T> *rt=rtab+256*r;
    cplx<T> a[16], b[16];
#pragma unroll
    for(int k=0; k < 16; ++k) {
      cplx<T> x, y;
      if constexpr(KEEP) {
        x=a0[k];
        y=b0[k];
      } else {
        bool in=ok && j+16*k < L;
        x=in ? (fr+16*k)[lin] : zero<T>();
        y=in ? (gr+16*k)[lin] : zero<T>();
      }
      if(r != 0) {
        cplx<T> w=table_word(rt+16*k+j);
        x=x*w;
        y=y*w;
      }
      a[k]=x;
      b[k]=y;
    }
    fft256s<T,1,1>(a,row,j,0,tw16);
    fft256s<T,1,1>(b,row,j,0,tw16);
    {
      const auto rop=bind_row(op,ok ? row0+i : rows-1);
#pragma unroll
      for(int k=0; k < 16; ++k) a[k]=rop(a[k],b[k],qi*(j+16*k)+r);
    }
    fft256s<T,-1,1>(a,row,j,0,tw16);
#pragma unroll
    for(int k=0; k < 16; ++k)
      acc[k]=acc[k]+(r == 0 ? a[k] : mulc(a[k],table_word(rt+16*k+j)));
  }
  if(ok) {
#pragma unroll
    for(int k=0; k < 16; ++k)
      if(j+16*k < L) (orow+16*k)[lo]=scale*acc[k];
  }
}

// Reduce-scatter over the two 16-lane groups of each 32-lane half of the wave
// (groups 0 and 1): lanes of group 0 get the sum over the groups of x, lanes
// of group 1 that of y.  v_permlane16_swap exchanges the odd 16-lane rows of
// its first operand with the even rows of its second, so its results are
// (x of group 0, y of group 0) and (x of group 1, y of group 1) on the lanes of
// (group 0, group 1).
__device__ __forceinline__ float pair16_scatter(float x, float y)
{
  auto s=__builtin_amdgcn_permlane16_swap(__float_as_uint(x),__float_as_uint(y),false,false);
  return __uint_as_float(s[0])+__uint_as_float(s[1]);
}
__device__ __forceinline__ double pair16_scatter(double x, double y)
{
  const unsigned long long u=(unsigned long long) __double_as_longlong(x);
  const unsigned long long v=(unsigned long long) __double_as_longlong(y);
  auto lo=__builtin_amdgcn_permlane16_swap((unsigned) u,(unsigned) v,false,false);
  auto hi=__builtin_amdgcn_permlane16_swap((unsigned) (u >> 32),(unsigned) (v >> 32),
                                           false,false);
  const double a=__longlong_as_double((long long) (((unsigned long long) hi[0] << 32) | lo[0]));
  const double b=__longlong_as_double((long long) (((unsigned long long) hi[1] << 32) | lo[1]));
  return a+b;
}

// Rows with q = 2 (N = 512): a wave holds 2 rows x 2 residues x 16 lanes,
// lane = j + 16 (2 i + r) for row i of the wave and residue r.  The two
// residue groups of a row load the same elements in the same instruction, so
// f and g are read from memory once; each group transforms its residue, and a
// reduce-scatter across the group pair leaves lane j of group r with the
// outputs j + 16 k, k in [8 r, 8 r + 8).  The grid is persistent: each block
// fills its twiddle tables once and its waves, which exchange only within
// themselves, loop over row pairs independently.  Rows are read and written
// through buffers over the pair: one offset per lane, past the end (read as 0,
// not stored) for padding and for a missing second row.
//
// Bound by the vector unit in FP64 (the loop issues 1765 -> 1591 vector
// instructions per row pair, at four cycles each on one of 1024 SIMDs): the
// branches around every load and store and the sum of all sixteen outputs in
// both groups were an eighth of them.  262144 rows of 256: FP64 778 -> 705 us,
// FP32 392 -> 376 us (four waves per SIMD with the library's products; a caller's
// functor keeps the registers of two: the tests' weight 1/(1 + c k^2) spilled 284
// bytes at four and took 666 to 712 us, 525 us at two).
// Dynamic LDS: row256_lds(4 WPB, 2).
template<typename T, class Op, int WPB>
__global__ void __launch_bounds__(64*WPB,(sizeof(T) == 4 && IsProduct<Op>::value ? 4 : 2))
rowconv256p_kernel(const cplx<T> *f, const cplx<T> *g, int64_t rows,
                   int64_t rs, cplx<T> *out, int64_t os, int L, T scale,
                   const cplx<T> *zN, Op op)
{
  extern __shared__ char smem_raw[];
  cplx<T> *rtab=reinterpret_cast<cplx<T> *>(smem_raw);   // 2 x 256
  cplx<T> *tw16=rtab+512;                                 // 256
  T *lds=reinterpret_cast<T *>(tw16+256);
  fill_rtab(rtab,zN,0,2,threadIdx.x,64*WPB);
  fill_tw16(tw16,zN,2,threadIdx.x,64*WPB);
  __syncthreads();
  constexpr unsigned E=sizeof(cplx<T>), END=0x80000000u;
  const int j=threadIdx.x & 15;
  const int grp=threadIdx.x >> 4;          // 4 groups per wave
  const int r=grp & 1, i=(grp & 3) >> 1;   // residue and row of the wave
  const int wave=__builtin_amdgcn_readfirstlane((int) threadIdx.x >> 6);
  const cplx<T> *rt=rtab+256*r;
  constexpr int RS=17;                     // row stride of the exchange areas
  T *xrow=lds+grp*16*RS;
  const int64_t pairs=(rows+1)/2;
  for(int64_t pr=(int64_t) blockIdx.x*WPB+wave; pr < pairs; pr += (int64_t) gridDim.x*WPB) {
    const int64_t row=2*pr+i;
    const bool ok=row < rows;
    const size_t two=2*pr+1 < rows;        // the pair's second row exists
    const __amdgpu_buffer_rsrc_t rf=buf_rsrc(f+2*pr*rs,two*rs+L), rg=buf_rsrc(g+2*pr*rs,two*rs+L);
    const unsigned in=ok ? (unsigned) (i*(int) rs+j)*E : END;
    cplx<T> a[16], b[16];
    if(L == 256) {                         // the buffers hold every scalar offset
#pragma unroll
      for(int k=0; k < 16; ++k) {
        a[k]=ld_buf<T>(rf,in,16*k*E);
        b[k]=ld_buf<T>(rg,in,16*k*E);
      }
    } else {
      const int jf=fresh(j);
#pragma unroll
      for(int k=0; k < 16; ++k) {
        const unsigned o=jf+16*k < L ? in : END;
        a[k]=ld_buf<T>(rf,o+16*k*E,0);
        b[k]=ld_buf<T>(rg,o+16*k*E,0);
      }
    }
#pragma unroll
    for(int k=0; k < 16; ++k) {
      const cplx<T> w=table_word(rt+16*k+j); // w_512^{r (j + 16 k)}
      a[k]=a[k]*w;
      b[k]=b[k]*w;
    }
    fft256s_pair<T,1,1,RS>(a,b,xrow,j,0,tw16);
    {
      const auto rop=bind_row(op,ok ? row : rows-1);
#pragma unroll
      for(int k=0; k < 16; ++k) a[k]=rop(a[k],b[k],2*(j+16*k)+r);
    }
    fft256s<T,-1,1,RS>(a,xrow,j,0,tw16);
#pragma unroll
    for(int k=0; k < 16; ++k) a[k]=mulc(a[k],table_word(rt+16*k+j));
    const __amdgpu_buffer_rsrc_t ro=buf_rsrc(out+2*pr*os,two*os+L);
    const int j0=fresh(j)+128*r;           // this group's first output
    const unsigned to=ok ? (unsigned) (i*(int) os+j0)*E : END;
#pragma unroll
    for(int k=0; k < 8; ++k) {
      const cplx<T> v=mk(pair16_scatter(a[k].x,a[k+8].x),pair16_scatter(a[k].y,a[k+8].y));
      st_buf<T>(ro,(j0+16*k < L ? to : END)+16*k*E,0,scale*v);
    }
  }
}

} // namespace fftwpp_amd
