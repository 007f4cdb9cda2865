// kernels_svwide.hpp -- the level-by-level sweeps for blocks of 4, 16 or 32
// right-hand sides on the matrix cores (reference kernels/solve_ztrsmsp.c:
// 300-424 forward, :449-625 backward).
//
// The sweeps of kernels_svsolve.hpp carry at most 8 right-hand sides per
// pass over the factor, so a block of 32 streamed it four times, and each
// level's launches took their 10 to 20 us of dependent memory trips four
// times.  Here a pass carries NR = 4, 16 or 32: a factor entry is one operand
// of a 16 x 16 x 4 product instead of 8 multiply-adds with 8 LDS reads.  The
// vectors are held by rows, NR values of a row next to each other (V[row *
// NR + q]), so that every operand row, result and atomic is one contiguous
// run of min(NR, 16) values; the columns q >= nq of a pass hold zeros.  With NR
// = 4 the lanes 4 .. 15 of a product's columns repeat the last one and their
// results are dropped: a quarter of the product counts, which a pass over a
// double factor can afford and one over a large single factor cannot
// (wide_from in engine.hip).
//
// Bound: the factor's bytes on the wide levels (each entry once per sweep),
// the three or four dependent trips of a level's two launches at the top.
// 60^3 nodes x 3, 32 right-hand sides, float factor: 22.26 ms in narrow passes,
// 6.78 ms in one wide pass.
#pragma once
#include "kernels_svsolve.hpp"

// Rows [row0, row0 + nrows) (records) against columns [c0, min(c0 + 64, n))
// of one cblk: a workgroup of the backward sweep.
struct sv_block {
    int32_t n;
    int32_t fcolnum;
    int32_t c0;
    int32_t nrows;
    int64_t row0;
};
// Backward blocks take up to this many rows: the 64 x NR sums of a block go
// to Y by atomics once, so more rows mean fewer atomics; a level with few
// blocks takes fewer rows to keep the chip full.
#define PXD_SVW_ROWS   256
#define PXD_SVW_BLOCKS 1024

// a where c, else zero (selected by parts: the complex types stay in registers)
template <typename T>
__device__ inline T
svw_where( bool c, T a )
{
    if constexpr ( std::is_same<T, typename px_real<T>::type>::value ) {
        return c ? a : (T)0;
    }
    else {
        return T( c ? a.re : 0, c ? a.im : 0 );
    }
}

// columns of a forward batch (4 per step), by the registers they take
template <typename T> struct svw_steps { static constexpr int value = sizeof( T ) == 4 ? 6 : sizeof( T ) == 8 ? 4 : 2; };

// v (column-major, ld) <-> rows of NR values
template <typename T, typename TV, int NR>
__global__ void __launch_bounds__( PXD_THREADS )
k_svw_pack( int64_t n, const TV *__restrict__ v, int64_t ld, int nq, T *__restrict__ out )
{
    __shared__ T  s[64][NR + 1];
    const int64_t i0 = (int64_t)blockIdx.x * 64;
    const int     r = threadIdx.x & 63;
    for ( int q = threadIdx.x >> 6; q < NR; q += PXD_THREADS / 64 ) {
        s[r][q] = ( q < nq && i0 + r < n ) ? px_from_any<T>( v[i0 + r + q * ld] ) : (T)0;
    }
    __syncthreads();
    for ( int e = threadIdx.x; e < 64 * NR; e += PXD_THREADS ) {
        if ( i0 + e / NR < n ) out[i0 * NR + e] = s[e / NR][e % NR];
    }
}
template <typename T, typename TV, int NR>
__global__ void __launch_bounds__( PXD_THREADS )
k_svw_unpack( int64_t n, const T *__restrict__ in, int nq, TV *__restrict__ v, int64_t ld )
{
    __shared__ T  s[64][NR + 1];
    const int64_t i0 = (int64_t)blockIdx.x * 64;
    const int     r = threadIdx.x & 63;
    for ( int e = threadIdx.x; e < 64 * NR; e += PXD_THREADS ) {
        if ( i0 + e / NR < n ) s[e / NR][e % NR] = in[i0 * NR + e];
    }
    __syncthreads();
    for ( int q = threadIdx.x >> 6; q < nq; q += PXD_THREADS / 64 ) {
        if ( i0 + r < n ) v[i0 + r + q * ld] = px_from_any<TV>( s[r][q] );
    }
}

// y_i <- y_i / D_i (LDL^T, between the sweeps)
template <typename T, int NR>
__global__ void
k_svw_dscale( int64_t n, const int32_t *__restrict__ col2cblk, const dcblk *__restrict__ cb, const T *__restrict__ L,
              T *__restrict__ Y )
{
    const int64_t e = (int64_t)blockIdx.x * blockDim.x + threadIdx.x, i = e / NR;
    if ( i >= n ) return;
    const dcblk   c  = cb[col2cblk[i]];
    const int32_t nk = c.lcolnum - c.fcolnum + 1;
    Y[e] = px_div( Y[e], L[c.coefoff + (int64_t)( i - c.fcolnum ) * ( nk + 1 )] );
}

// Forward tile: X[g(s)] -= A(s, :) y_k for its 64 rows; the waves share its
// columns (and `split` workgroups, on launches with few tiles).
template <typename T, int NR>
__global__ void __launch_bounds__( PXD_THREADS )
k_svw_fwd( const sv_tile *__restrict__ tiles, const sv_row *__restrict__ rows, const T *__restrict__ L, T *X,
           const T *__restrict__ Y, int nq, int split )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    constexpr int NB = ( NR + 15 ) / 16, NT = 4, US = svw_steps<T>::value;
    __shared__ T       red[2][64][NR + 1];
    __shared__ int32_t sg[64];
    const int     idx = xcd_task( blockIdx.x, gridDim.x );
    const sv_tile t   = tiles[idx / split];
    const int     ps  = idx % split;
    const int     tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int     lr = lane & 15, lg = lane >> 4, lq = min( lr, NR - 1 );
    const int     nr = min( 64, t.stride - t.r0 );
    const int32_t cs0 = ( t.n * ps ) / split, cw = ( t.n * ( ps + 1 ) ) / split - cs0;
    const int32_t c0 = cs0 + ( cw * w ) / 4, c1 = cs0 + ( cw * ( w + 1 ) ) / 4;
    if ( tid < nr ) {
        sg[tid] = rows[t.row0 + tid].g;
    }
    // rows past the tile repeat its last one
    const T *pa[NT];
    int32_t  la[NT];
#pragma unroll
    for ( int i = 0; i < NT; i++ ) {
        const sv_row ri = rows[t.row0 + min( 16 * i + lr, nr - 1 )];
        pa[i] = L + ri.base;
        la[i] = ri.ld;
    }
    const T *y = Y + (int64_t)t.fcolnum * NR + lq;
    acc_t    acc[NT][NB];
#pragma unroll
    for ( int i = 0; i < NT; i++ )
#pragma unroll
        for ( int b = 0; b < NB; b++ ) acc[i][b] = M::zero();
    for ( int32_t cb = c0; cb < c1; cb += 4 * US ) {
        T a[NT][US], v[NB][US];
#pragma unroll
        for ( int u = 0; u < US; u++ ) {
            const int32_t col = cb + 4 * u + lg, cc = min( col, c1 - 1 );
#pragma unroll
            for ( int i = 0; i < NT; i++ ) a[i][u] = pa[i][(int64_t)cc * la[i]];
#pragma unroll
            for ( int b = 0; b < NB; b++ ) v[b][u] = y[(int64_t)cc * NR + 16 * b];
        }
#pragma unroll
        for ( int u = 0; u < US; u++ ) {
            const bool ok = cb + 4 * u + lg < c1;
#pragma unroll
            for ( int b = 0; b < NB; b++ ) {
                const T yv = svw_where( ok, v[b][u] );
#pragma unroll
                for ( int i = 0; i < NT; i++ ) acc[i][b] = M::mma( a[i][u], yv, acc[i][b] );
            }
        }
    }
    // the waves' sums: two and two, then everyone adds the pair
    if ( w >= 2 && lr < NR ) {
#pragma unroll
        for ( int i = 0; i < NT; i++ )
#pragma unroll
            for ( int b = 0; b < NB; b++ )
#pragma unroll
                for ( int e = 0; e < 4; e++ ) red[w - 2][16 * i + M::row( lane, e )][16 * b + lr] = M::get( acc[i][b], e );
    }
    __syncthreads();
    if ( w < 2 && lr < NR ) {
#pragma unroll
        for ( int i = 0; i < NT; i++ )
#pragma unroll
            for ( int b = 0; b < NB; b++ )
#pragma unroll
                for ( int e = 0; e < 4; e++ ) red[w][16 * i + M::row( lane, e )][16 * b + lr] += M::get( acc[i][b], e );
    }
    __syncthreads();
    for ( int e = tid; e < nr * NR; e += PXD_THREADS ) {
        const int r = e / NR, q = e % NR;
        if ( q < nq ) {
            px_atomic_add( X + (int64_t)sg[r] * NR + q, -( red[0][r][q] + red[1][r][q] ) );
        }
    }
}

// Backward block: Y[fcolnum + j] -= sum over its rows s of A(s, j) X[g(s)] for
// 64 columns j.  Each 64-row step passes through LDS (loads along the rows,
// operands along the columns); wave w sums columns 16 w .. 16 w + 15.
template <typename T, int NR>
__global__ void __launch_bounds__( PXD_THREADS )
k_svw_bwd( const sv_block *__restrict__ blocks, const sv_row *__restrict__ rows, const T *__restrict__ L,
           const T *__restrict__ X, T *Y, int nq )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    constexpr int NB = ( NR + 15 ) / 16, NU = 64 * 64 / PXD_THREADS;
    // complex double takes 32 rows at a time
    constexpr int RS = sizeof( T ) > 8 ? 32 : 64, CSTEP = PXD_THREADS / RS, NA = NU * RS / 64;
    constexpr int NXR = ( RS * NR + PXD_THREADS - 1 ) / PXD_THREADS;
    __shared__ T       sA[64][RS + 1];    // [col][row]
    __shared__ T       sx[RS][NR];
    __shared__ int32_t sg[PXD_SVW_ROWS];
    const sv_block t   = blocks[xcd_task( blockIdx.x, gridDim.x )];
    const int      tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int      lr = lane & 15, lg = lane >> 4, lq = min( lr, NR - 1 );
    const int      nc = min( 64, t.n - t.c0 );
    const int      ar = tid % RS, ac = tid / RS;
    for ( int r = tid; r < t.nrows; r += PXD_THREADS ) sg[r] = rows[t.row0 + r].g;
    __syncthreads();
    acc_t acc[NB];
#pragma unroll
    for ( int b = 0; b < NB; b++ ) acc[b] = M::zero();
    T    a[NA], x[NXR];
    auto load = [&]( int r0 ) {
        // rows past the block repeat its last one against zeros of X; columns
        // past the cblk repeat the last one, and their sums are dropped
        const sv_row ri = rows[t.row0 + min( r0 + ar, t.nrows - 1 )];
        const T     *p  = L + ri.base + (int64_t)t.c0 * ri.ld;
#pragma unroll
        for ( int u = 0; u < NA; u++ ) a[u] = p[(int64_t)min( ac + CSTEP * u, nc - 1 ) * ri.ld];
#pragma unroll
        for ( int u = 0; u < NXR; u++ ) {
            const int e = tid + PXD_THREADS * u, r = r0 + e / NR;
            if ( RS * NR < PXD_THREADS && e >= RS * NR ) break;
            const T v = X[(int64_t)sg[min( r, t.nrows - 1 )] * NR + e % NR];
            x[u] = svw_where( r < t.nrows, v );
        }
    };
    load( 0 );
    for ( int r0 = 0; r0 < t.nrows; r0 += RS ) {
#pragma unroll
        for ( int u = 0; u < NA; u++ ) sA[ac + CSTEP * u][ar] = a[u];
#pragma unroll
        for ( int u = 0; u < NXR; u++ ) {
            const int e = tid + PXD_THREADS * u;
            if ( RS * NR >= PXD_THREADS || e < RS * NR ) sx[e / NR][e % NR] = x[u];
        }
        __syncthreads();
        if ( r0 + RS < t.nrows ) {
            load( r0 + RS );
        }
#pragma unroll
        for ( int s = 0; s < RS / 4; s++ ) {
            const T av = sA[16 * w + lr][4 * s + lg];
#pragma unroll
            for ( int b = 0; b < NB; b++ ) acc[b] = M::mma( av, sx[4 * s + lg][16 * b + lq], acc[b] );
        }
        __syncthreads();
    }
#pragma unroll
    for ( int e = 0; e < 4; e++ ) {
        const int j = 16 * w + M::row( lane, e );
#pragma unroll
        for ( int b = 0; b < NB; b++ ) {
            if ( j < nc && 16 * b + lr < nq ) {
                px_atomic_add( Y + (int64_t)( t.fcolnum + t.c0 + j ) * NR + 16 * b + lr, -M::get( acc[b], e ) );
            }
        }
    }
}

// Rows R0 .. R0 + 15 of out = Linv in (forward) or Linv^T in (backward).  The
// waves take the 16-column groups of the triangle's part in turn; Linv holds
// zeros in its other triangle.
template <typename T, int NR>
__global__ void __launch_bounds__( PXD_THREADS )
k_svw_diag( const sv_chunk *__restrict__ chunks, const T *__restrict__ Linv, const T *__restrict__ Xin,
            T *__restrict__ Yout, int trans )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    constexpr int CR = PXD_DIAG_ROWS, NB = ( NR + 15 ) / 16, GU = sizeof( T ) == 4 ? 3 : sizeof( T ) == 8 ? 2 : 1;
    static_assert( CR == 16, "a chunk is one row block of the products" );
    __shared__ T   red[4][CR][NR + 1];
    const sv_chunk ch  = chunks[xcd_task( blockIdx.x, gridDim.x )];
    const int32_t  n   = ch.n;
    const int      tid = threadIdx.x, lane = tid & 63, w = tid >> 6;
    const int      lr = lane & 15, lg = lane >> 4, lq = min( lr, NR - 1 );
    const T       *LI  = Linv + ch.dinvoff;
    const int32_t  i   = min( ch.R0 + lr, n - 1 );
    // element (i, k) of the operand
    const T      *p  = trans ? LI + (int64_t)i * n : LI + i;
    const int64_t sk = trans ? 1 : n;
    const int32_t k0 = trans ? ch.R0 : 0, k1 = trans ? n : min( n, ch.R0 + CR );
    const T      *x  = Xin + (int64_t)ch.fcolnum * NR + lq;
    acc_t         acc[NB];
#pragma unroll
    for ( int b = 0; b < NB; b++ ) acc[b] = M::zero();
    for ( int32_t kb = k0 + 16 * w; kb < k1; kb += 64 * GU ) {
        T a[GU][4], v[GU][NB][4];
#pragma unroll
        for ( int u = 0; u < GU; u++ )
#pragma unroll
            for ( int s = 0; s < 4; s++ ) {
                // step s takes k = 4 lg + s: 4 consecutive values per lane of a column of Linv
                const int32_t k = min( kb + 64 * u + 4 * lg + s, k1 - 1 );
                a[u][s] = p[k * sk];
#pragma unroll
                for ( int b = 0; b < NB; b++ ) v[u][b][s] = x[(int64_t)k * NR + 16 * b];
            }
#pragma unroll
        for ( int u = 0; u < GU; u++ )
#pragma unroll
            for ( int s = 0; s < 4; s++ ) {
                const bool ok = kb + 64 * u + 4 * lg + s < k1;
#pragma unroll
                for ( int b = 0; b < NB; b++ ) acc[b] = M::mma( a[u][s], svw_where( ok, v[u][b][s] ), acc[b] );
            }
    }
#pragma unroll
    for ( int b = 0; b < NB; b++ )
#pragma unroll
        for ( int e = 0; e < 4; e++ ) {
            if ( lr < NR ) red[w][M::row( lane, e )][16 * b + lr] = M::get( acc[b], e );
        }
    __syncthreads();
    for ( int e = tid; e < CR * NR; e += PXD_THREADS ) {
        const int r = e / NR, q = e % NR;
        if ( ch.R0 + r < n ) {
            Yout[(int64_t)( ch.fcolnum + ch.R0 + r ) * NR + q] =
                ( red[0][r][q] + red[1][r][q] ) + ( red[2][r][q] + red[3][r][q] );
        }
    }
}

// Levels whose cblks all fit one chunk: one wavefront per cblk, diagonal and
// off-diagonal rows in one launch.  A product's result holds, in lane (lr,
// lg), rows row(lane, 0..3) of column lr, which is the next product's second
// operand when its step s takes k = row(lane, s): nothing passes through LDS.
template <typename T, int NR>
__global__ void __launch_bounds__( PXD_THREADS )
k_svw_small_fwd( const sv_small *__restrict__ tasks, int64_t ntasks, const sv_row *__restrict__ rows,
                 const T *__restrict__ L, const T *__restrict__ Linv, T *X, T *__restrict__ Y, int nq )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    constexpr int NB = ( NR + 15 ) / 16;
    const int     lane = threadIdx.x & 63, lr = lane & 15, lq = min( lr, NR - 1 );
    const int64_t ti = (int64_t)xcd_task( blockIdx.x, gridDim.x ) * 4 + ( threadIdx.x >> 6 );
    if ( ti >= ntasks ) {
        return;
    }
    const sv_small t  = tasks[ti];
    const T       *LI = Linv + t.dinvoff;
    acc_t          y[NB];
    {
        T a[4], v[NB][4];
#pragma unroll
        for ( int s = 0; s < 4; s++ ) {
            const int k = M::row( lane, s ), kk = min( k, t.n - 1 );
            a[s] = LI[min( lr, t.n - 1 ) + (int64_t)kk * t.n];
            a[s] = svw_where( lr < t.n && k < t.n, a[s] );
#pragma unroll
            for ( int b = 0; b < NB; b++ ) {
                const T x = X[(int64_t)( t.fcolnum + kk ) * NR + 16 * b + lq];
                v[b][s] = svw_where( k < t.n, x );
            }
        }
#pragma unroll
        for ( int b = 0; b < NB; b++ ) {
            y[b] = M::zero();
#pragma unroll
            for ( int s = 0; s < 4; s++ ) y[b] = M::mma( a[s], v[b][s], y[b] );
        }
    }
#pragma unroll
    for ( int e = 0; e < 4; e++ ) {
        const int r = M::row( lane, e );
        if ( r < t.n && lr < NR ) {
#pragma unroll
            for ( int b = 0; b < NB; b++ ) Y[(int64_t)( t.fcolnum + r ) * NR + 16 * b + lr] = M::get( y[b], e );
        }
    }
    for ( int32_t r0 = 0; r0 < t.nrows; r0 += 16 ) {
        const sv_row ri = rows[t.row0 + min( r0 + lr, t.nrows - 1 )];
        T            a[4];
#pragma unroll
        for ( int s = 0; s < 4; s++ ) a[s] = L[ri.base + (int64_t)min( M::row( lane, s ), t.n - 1 ) * ri.ld];
        acc_t d[NB];
#pragma unroll
        for ( int b = 0; b < NB; b++ ) {
            d[b] = M::zero();
            // rows of y past the cblk are zero
#pragma unroll
            for ( int s = 0; s < 4; s++ ) d[b] = M::mma( a[s], M::get( y[b], s ), d[b] );
        }
#pragma unroll
        for ( int e = 0; e < 4; e++ ) {
            const int     r = M::row( lane, e );
            const int32_t g = __shfl( ri.g, r );
#pragma unroll
            for ( int b = 0; b < NB; b++ ) {
                if ( r0 + r < t.nrows && 16 * b + lr < nq ) {
                    px_atomic_add( X + (int64_t)g * NR + 16 * b + lr, -M::get( d[b], e ) );
                }
            }
        }
    }
}

template <typename T, int NR>
__global__ void __launch_bounds__( PXD_THREADS )
k_svw_small_bwd( const sv_small *__restrict__ tasks, int64_t ntasks, const sv_row *__restrict__ rows,
                 const T *__restrict__ L, const T *__restrict__ Linv, T *X, const T *__restrict__ Y )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    constexpr int NB = ( NR + 15 ) / 16;
    const int     lane = threadIdx.x & 63, lr = lane & 15, lq = min( lr, NR - 1 );
    const int64_t ti = (int64_t)xcd_task( blockIdx.x, gridDim.x ) * 4 + ( threadIdx.x >> 6 );
    if ( ti >= ntasks ) {
        return;
    }
    const sv_small t  = tasks[ti];
    const T       *LI = Linv + t.dinvoff;
    const int      j  = min( lr, t.n - 1 );
    acc_t          acc[NB];
#pragma unroll
    for ( int b = 0; b < NB; b++ ) acc[b] = M::zero();
    for ( int32_t r0 = 0; r0 < t.nrows; r0 += 16 ) {
        T a[4], v[NB][4];
#pragma unroll
        for ( int s = 0; s < 4; s++ ) {
            const int    r  = r0 + M::row( lane, s );
            const sv_row ri = rows[t.row0 + min( r, t.nrows - 1 )];
            a[s] = L[ri.base + (int64_t)j * ri.ld];
#pragma unroll
            for ( int b = 0; b < NB; b++ ) {
                const T x = X[(int64_t)ri.g * NR + 16 * b + lq];
                v[b][s] = svw_where( r < t.nrows, x );
            }
        }
#pragma unroll
        for ( int b = 0; b < NB; b++ )
#pragma unroll
            for ( int s = 0; s < 4; s++ ) acc[b] = M::mma( a[s], v[b][s], acc[b] );
    }
    T a[4], z[NB][4];
#pragma unroll
    for ( int s = 0; s < 4; s++ ) {
        const int k = M::row( lane, s ), kk = min( k, t.n - 1 );
        a[s] = LI[kk + (int64_t)j * t.n];
        a[s] = svw_where( lr < t.n && k < t.n, a[s] );
#pragma unroll
        for ( int b = 0; b < NB; b++ ) {
            const T y = Y[(int64_t)( t.fcolnum + kk ) * NR + 16 * b + lq] - M::get( acc[b], s );
            z[b][s] = svw_where( k < t.n, y );
        }
    }
#pragma unroll
    for ( int b = 0; b < NB; b++ ) {
        acc[b] = M::zero();
#pragma unroll
        for ( int s = 0; s < 4; s++ ) acc[b] = M::mma( a[s], z[b][s], acc[b] );
#pragma unroll
        for ( int e = 0; e < 4; e++ ) {
            const int r = M::row( lane, e );
            if ( r < t.n && lr < NR ) X[(int64_t)( t.fcolnum + r ) * NR + 16 * b + lr] = M::get( acc[b], e );
        }
    }
}
