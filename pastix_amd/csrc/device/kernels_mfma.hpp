// kernels_mfma.hpp -- matrix-core factorization kernels and the inverse-based
// solve kernels of the MI355X engine.
//
// The diagonal block L_kk of every cblk is inverted explicitly (Linv, n x n,
// column major, upper part zero): the off-diagonal TRSM of the reference
// (core_ztrsmsp.c:148-183, L_off <- L_off L_kk^{-T}) becomes the product
// L_off Linv^T on the matrix cores, and the diagonal solves of the sweeps
// (solve_ztrsmsp.c:74-108) become Linv b and Linv^T b.
#pragma once
#include "kernels_fact.hpp"
#include "kernels_solve.hpp"
#include <type_traits>
#include "kernels_elim.hpp"

// tasks of the block-column inversion: cblk and first column of the block
struct inv_task {
    int32_t cblk;
    int32_t J;
};

// Waves of a kernel on the critical path of the factorization (panels,
// inverses, TRSM and the updates that the next level waits for) raise their
// instruction-issue priority, so that they keep their pace on CUs that they
// share with the bulk update kernels of the other stream.
__device__ inline void
wave_priority( int prio )
{
    if ( prio ) {
        __builtin_amdgcn_s_setprio( 3 );
    }
}

// Row i >= column j of entry idx of a row-major packed lower triangle.
__device__ inline void
tri_index( int idx, int &i, int &j )
{
    i = (int)( ( sqrtf( 8.f * (float)idx + 1.f ) - 1.f ) * 0.5f );
    if ( ( i + 1 ) * ( i + 2 ) / 2 <= idx ) i++;
    if ( i * ( i + 1 ) / 2 > idx ) i--;
    j = idx - i * ( i + 1 ) / 2;
}

// Per-workgroup timing for the kernel timing log: when stamps is not null,
// task i of the launch writes its start and end times (constant-rate wall
// clock ticks) to stamps[2i] and stamps[2i+1].
__device__ inline uint64_t
stamp_begin( const uint64_t *stamps )
{
    return stamps ? (uint64_t)wall_clock64() : 0;
}
__device__ inline void
stamp_end( uint64_t *stamps, int64_t i, uint64_t t0 )
{
    if ( stamps ) {
        __syncthreads();
        if ( threadIdx.x == 0 ) {
            stamps[2 * i]     = t0;
            stamps[2 * i + 1] = (uint64_t)wall_clock64();
        }
    }
}

// Keys of the row searches of an update tile, staged in LDS with one parallel
// load: stacked row offsets of the source bloks [b, lb) and first rows of the
// facing cblk's bloks [ffb, flb).  Lists longer than PXD_SEARCH_CAP are
// searched in global memory instead.
#define PXD_SEARCH_CAP 512
struct search_keys {
    int32_t row[PXD_SEARCH_CAP];
    int32_t frow[PXD_SEARCH_CAP];
};

__device__ inline void
stage_search_keys( search_keys &sk, const dblok *__restrict__ bk, int32_t b, int32_t lb, int32_t ffb,
                   int32_t flb, int tid )
{
    const int32_t ns = min( lb - b, PXD_SEARCH_CAP ), nf = min( flb - ffb, PXD_SEARCH_CAP );
    for ( int32_t i = tid; i < ns; i += PXD_THREADS ) sk.row[i] = bk[b + i].rowoff;
    for ( int32_t i = tid; i < nf; i += PXD_THREADS ) sk.frow[i] = bk[ffb + i].frownum;
}

// Source blok (in [b, lb)) holding stacked row s, and facing blok (in
// [ffb, flb)) holding global row g, from the staged keys.
__device__ inline int32_t
search_row( const search_keys &sk, const dblok *__restrict__ bk, int32_t b, int32_t lb, int32_t s )
{
    return ( lb - b <= PXD_SEARCH_CAP ) ? b + lds_search_le( sk.row, lb - b, s ) : find_blok_by_row( bk, b, lb, s );
}
__device__ inline int32_t
search_grow( const search_keys &sk, const dblok *__restrict__ bk, int32_t ffb, int32_t flb, int32_t g )
{
    return ( flb - ffb <= PXD_SEARCH_CAP ) ? ffb + lds_search_le( sk.frow, flb - ffb, g )
                                           : find_blok_by_grow( bk, ffb, flb, g );
}


// ---------------------------------------------------------------------------
// Panel: Cholesky of the diagonal tile with static pivoting, right looking by
// PXD_NB columns; the unblocked step updates with unscaled columns so that it
// needs one barrier per column.  The inverses of the PXD_NB x PXD_NB diagonal
// sub-blocks go to the diagonal blocks of Linv.  The first pcap rows of the
// current block's L21 are kept in dynamic LDS; rows beyond pcap (a strip that
// would not fit the CU's LDS) are read back from the copy just written to A.
// Option panel_mw = 0: one workgroup per cblk, where k_panel takes one per
// 32-row block.
template <typename T>
__global__ void __launch_bounds__( PXD_THREADS )
k_potrf2( const int32_t *__restrict__ list, const dcblk *__restrict__ cb, T *__restrict__ L,
          T *__restrict__ Linv, double thresh, int *__restrict__ npiv,
          uint64_t *__restrict__ stamps, int prio, int32_t pcap )
{
    __shared__ T sA[PXD_NB][PXD_NB + 1];   // sA[col][row]
    __shared__ T sI[PXD_NB][PXD_NB + 1];   // inverse, sI[col][row]
    __shared__ T sD[PXD_NB];
    // L21 of the current block, sP[row][k]: dynamic LDS for the widest cblk of the launch
    extern __shared__ unsigned char smem_raw[];
    T ( *sP )[PXD_NB + 1] = reinterpret_cast<T ( * )[PXD_NB + 1]>( smem_raw );

    const int32_t k   = list[blockIdx.x];
    const uint64_t t_stamp = stamp_begin( stamps );
    wave_priority( prio );
    const dcblk   c   = cb[k];
    const int32_t n   = c.lcolnum - c.fcolnum + 1;
    const int     tid = threadIdx.x;
    T *A  = L + c.coefoff;            // n x n, ld n
    T *LI = Linv + c.dinvoff;         // n x n, ld n
    int piv = 0;
    typedef typename px_real<T>::type R;
    const R tau = (R)thresh;

    for ( int32_t kb = 0; kb < n; kb += PXD_NB ) {
        const int32_t bs = min( PXD_NB, n - kb );

        {
            constexpr int NU = PXD_NB * PXD_NB / PXD_THREADS;
            T v[NU];
#pragma unroll
            for ( int u = 0; u < NU; u++ ) {
                const int idx = tid + u * PXD_THREADS, r = idx % PXD_NB, cc = idx / PXD_NB;
                v[u] = ( r < bs && cc < bs && r >= cc ) ? A[( kb + r ) + (int64_t)( kb + cc ) * n] : (T)0;
            }
#pragma unroll
            for ( int u = 0; u < NU; u++ ) {
                const int idx = tid + u * PXD_THREADS, r = idx % PXD_NB, cc = idx / PXD_NB;
                sA[cc][r] = v[u];
                sI[cc][r] = ( r == cc && r < bs ) ? (T)1 : (T)0;   // W = I
            }
        }
        __syncthreads();

        // unblocked elimination A = U D U^T, W = U^{-1} alongside
        if ( tid < 64 ) {
            piv += elim32<T, false, false>( sA, sI, nullptr, sD, bs, tau, tid );
        }
        __syncthreads();
        // Cholesky: L = U D^{1/2}, the columns scaled by 1/sqrt(pivot), and
        // L^{-1} = D^{-1/2} U^{-1}, the rows of W scaled likewise.
        for ( int idx = tid; idx < PXD_NB * PXD_NB; idx += PXD_THREADS ) {
            const int rr = idx % PXD_NB, cc = idx / PXD_NB;
            if ( rr >= bs || cc >= bs ) continue;
            if ( rr > cc ) {
                sA[cc][rr] = sA[cc][rr] / px_sqrt( sD[cc] );
            }
            if ( rr >= cc ) {
                sI[cc][rr] = sI[cc][rr] / px_sqrt( sD[rr] );
            }
        }
        __syncthreads();
        if ( tid < bs ) {
            sA[tid][tid] = px_sqrt( sD[tid] );
        }
        __syncthreads();

        for ( int idx = tid; idx < PXD_NB * PXD_NB; idx += PXD_THREADS ) {
            const int rr = idx % PXD_NB, cc = idx / PXD_NB;
            if ( rr >= bs || cc >= bs ) continue;
            if ( rr >= cc ) {
                A[( kb + rr ) + (int64_t)( kb + cc ) * n] = sA[cc][rr];
            }
            LI[( kb + rr ) + (int64_t)( kb + cc ) * n] = sI[cc][rr];
        }

        // rows below the block inside the tile: A21 <- A21 * L11^{-T} on the
        // matrix cores, one wave per 16-row block (two 16 x 16 output tiles,
        // the inverse's transpose read from LDS); the result goes to A and to
        // sP for the trailing update
        typedef mfma16<T>         M;
        typedef typename M::acc_t acc_t;
        const int     lane = tid & 63, w = tid >> 6;
        const int32_t m0   = kb + bs;
        const int32_t m    = n - m0;
        for ( int32_t rb = 16 * w; rb < m; rb += 64 ) {
            T             a[PXD_NB / 4];
            const int32_t ra = m0 + rb + ( lane & 15 );
#pragma unroll
            for ( int s4 = 0; s4 < PXD_NB / 4; s4++ ) {
                const int l = 4 * s4 + ( lane >> 4 );
                a[s4] = ( ra < n && l < bs ) ? A[ra + (int64_t)( kb + l ) * n] : (T)0;
            }
            acc_t acc0 = M::zero(), acc1 = M::zero();
#pragma unroll
            for ( int s4 = 0; s4 < PXD_NB / 4; s4++ ) {
                const int l = 4 * s4 + ( lane >> 4 );
                acc0 = M::mma( a[s4], sI[l][( lane & 15 )], acc0 );
                acc1 = M::mma( a[s4], sI[l][16 + ( lane & 15 )], acc1 );
            }
#pragma unroll
            for ( int v = 0; v < 4; v++ ) {
                const int32_t rr = rb + M::row( lane, v );
                const int     c0 = lane & 15, c1 = 16 + ( lane & 15 );
                if ( rr < m ) {
                    if ( rr < pcap ) {
                        sP[rr][c0] = M::get( acc0, v );   // zero beyond bs: sI is zero there
                        sP[rr][c1] = M::get( acc1, v );
                    }
                    if ( c0 < bs ) A[( m0 + rr ) + (int64_t)( kb + c0 ) * n] = M::get( acc0, v );
                    if ( c1 < bs ) A[( m0 + rr ) + (int64_t)( kb + c1 ) * n] = M::get( acc1, v );
                }
            }
        }
        __syncthreads();

        // trailing update A22 -= L21 L21^T (lower part) on the matrix cores
        // from sP: 32 x 32 tiles, wave w takes every fourth tile, two at a
        // time, with the tiles' loads of A22 issued before their products.
        // Row ri of the product beyond pcap comes from A.
        auto prow = [&]( int32_t ri, int l ) -> T {
            if ( ri < pcap ) {
                return sP[ri][l];
            }
            if ( l >= bs ) {
                return (T)0;
            }
            return A[( m0 + ri ) + (int64_t)( kb + l ) * n];
        };
        {
            const int32_t nt = ( m + 31 ) / 32;
            const int32_t ntile = nt * ( nt + 1 ) / 2;
            for ( int32_t t0 = 2 * w; t0 < ntile; t0 += 8 ) {
                int32_t ti[2], tj[2];
                bool    tv[2];
#pragma unroll
                for ( int g = 0; g < 2; g++ ) {
                    // tile t0 + g in row-wise order of the lower triangle
                    int32_t tt = t0 + g, r = 0;
                    while ( ( r + 1 ) * ( r + 2 ) / 2 <= tt ) r++;
                    ti[g] = r;
                    tj[g] = tt - r * ( r + 1 ) / 2;
                    tv[g] = tt < ntile;
                }
                T old[2][2][2][4];
#pragma unroll
                for ( int g = 0; g < 2; g++ )
#pragma unroll
                    for ( int a = 0; a < 2; a++ )
#pragma unroll
                        for ( int b = 0; b < 2; b++ )
#pragma unroll
                            for ( int v = 0; v < 4; v++ ) {
                                const int32_t r  = 32 * ti[g] + 16 * a + M::row( lane, v );
                                const int32_t cc = 32 * tj[g] + 16 * b + ( lane & 15 );
                                const bool    ok = tv[g] && r < m && cc < m && r >= cc;
                                old[g][a][b][v] = ok ? A[( m0 + r ) + (int64_t)( m0 + cc ) * n] : (T)0;
                            }
                acc_t acc[2][2][2];
#pragma unroll
                for ( int g = 0; g < 2; g++ )
#pragma unroll
                    for ( int a = 0; a < 2; a++ )
#pragma unroll
                        for ( int b = 0; b < 2; b++ ) acc[g][a][b] = M::zero();
#pragma unroll
                for ( int s4 = 0; s4 < PXD_NB / 4; s4++ ) {
                    const int l = 4 * s4 + ( lane >> 4 );
#pragma unroll
                    for ( int g = 0; g < 2; g++ ) {
                        T af[2], bf[2];
#pragma unroll
                        for ( int a = 0; a < 2; a++ ) {
                            const int32_t ri = 32 * ti[g] + 16 * a + ( lane & 15 );
                            const int32_t rj = 32 * tj[g] + 16 * a + ( lane & 15 );
                            af[a] = ( ri < m ) ? prow( ri, l ) : (T)0;
                            bf[a] = ( rj < m ) ? prow( rj, l ) : (T)0;
                        }
#pragma unroll
                        for ( int a = 0; a < 2; a++ )
#pragma unroll
                            for ( int b = 0; b < 2; b++ ) acc[g][a][b] = M::mma( af[a], bf[b], acc[g][a][b] );
                    }
                }
#pragma unroll
                for ( int g = 0; g < 2; g++ )
#pragma unroll
                    for ( int a = 0; a < 2; a++ )
#pragma unroll
                        for ( int b = 0; b < 2; b++ )
#pragma unroll
                            for ( int v = 0; v < 4; v++ ) {
                                const int32_t r  = 32 * ti[g] + 16 * a + M::row( lane, v );
                                const int32_t cc = 32 * tj[g] + 16 * b + ( lane & 15 );
                                if ( tv[g] && r < m && cc < m && r >= cc ) {
                                    A[( m0 + r ) + (int64_t)( m0 + cc ) * n] = old[g][a][b][v] - M::get( acc[g][a][b], v );
                                }
                            }
            }
        }
        __syncthreads();
    }
    if ( tid == 0 && piv > 0 ) {
        atomicAdd( npiv, piv );
    }
    stamp_end( stamps, blockIdx.x, t_stamp );
}

// ---------------------------------------------------------------------------
// Inverse of the lower-triangular L_kk by block columns, one workgroup per
// (cblk, block column J).  The diagonal blocks D_K = L[K,K]^{-1} were written
// to Linv by the panel.  Column sweep: R = -L[J+1:, J] D_J, then for K = J+1,
// J+2, ...: X[K,J] = D_K R[K], R[K+1:] -= L[K+1:, K] X[K,J].  The first rcap
// rows of R stay in LDS, rows that would not fit in place in
// Linv, where X[K,J] later overwrites them; both products run on the matrix
// cores.
template <typename T>
__global__ void __launch_bounds__( PXD_THREADS )
k_trtri( const inv_task *__restrict__ tasks, const dcblk *__restrict__ cb, const T *__restrict__ L,
         T *__restrict__ Linv, uint64_t *__restrict__ stamps, int prio, int32_t rcap )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    __shared__ T sX[PXD_NB][PXD_NB + 1];   // the current X[K,J] (or D_J), sX[row][col]
    __shared__ T sD[PXD_NB][PXD_NB + 1];   // D_K, sD[row][col]
    extern __shared__ unsigned char smem_raw[];
    T ( *sR )[PXD_NB + 1] = reinterpret_cast<T ( * )[PXD_NB + 1]>( smem_raw );   // rows below block J

    const inv_task t    = tasks[blockIdx.x];
    const uint64_t t_stamp = stamp_begin( stamps );
    wave_priority( prio );
    const dcblk    c    = cb[t.cblk];
    const int32_t  n    = c.lcolnum - c.fcolnum + 1;
    const int      tid  = threadIdx.x;
    const int      lane = tid & 63, w = tid >> 6;
    const T       *A    = L + c.coefoff;
    T             *LI   = Linv + c.dinvoff;
    const int32_t  J    = t.J;                 // first column of the block column
    const int32_t  r0   = J + PXD_NB;          // first row of R
    const int32_t  nr   = n - r0;
    const int32_t  bj   = min( PXD_NB, n - J );
    // R(row, col): rows below rcap in LDS, the others at their place in Linv
    // (nr > 0 implies bj == PXD_NB, so every column is inside the tile)
    auto rget = [&]( int32_t rr, int cc ) -> T {
        return ( rr < rcap ) ? sR[rr][cc] : LI[( r0 + rr ) + (int64_t)( J + cc ) * n];
    };
    auto rset = [&]( int32_t rr, int cc, T v ) {
        if ( rr < rcap ) {
            sR[rr][cc] = v;
        }
        else {
            LI[( r0 + rr ) + (int64_t)( J + cc ) * n] = v;
        }
    };

    // load a 32 x 32 block of Linv (rows R0, cols C0) into dst[row][col]
    auto load_block = [&]( T ( *dst )[PXD_NB + 1], int32_t R0, int32_t C0, int32_t nrow, int32_t ncol ) {
        constexpr int NU = PXD_NB * PXD_NB / PXD_THREADS;
        T v[NU];
#pragma unroll
        for ( int u = 0; u < NU; u++ ) {
            const int idx = tid + u * PXD_THREADS, r = idx % PXD_NB, cc = idx / PXD_NB;
            v[u] = ( r < nrow && cc < ncol ) ? LI[( R0 + r ) + (int64_t)( C0 + cc ) * n] : (T)0;
        }
#pragma unroll
        for ( int u = 0; u < NU; u++ ) {
            const int idx = tid + u * PXD_THREADS, r = idx % PXD_NB, cc = idx / PXD_NB;
            dst[r][cc] = v[u];
        }
    };
    // R[rows >= rfirst] -= L[r0 + rows, K .. K+31] * sX  (16-row blocks per wave)
    auto sweep = [&]( int32_t rfirst, int32_t K, int32_t bk ) {
        for ( int32_t rb = rfirst + 16 * w; rb < nr; rb += 64 ) {
            T             a[PXD_NB / 4];
            const int32_t ra = rb + ( lane & 15 );
#pragma unroll
            for ( int s4 = 0; s4 < PXD_NB / 4; s4++ ) {
                const int l = 4 * s4 + ( lane >> 4 );
                a[s4] = ( ra < nr && l < bk ) ? -A[( r0 + ra ) + (int64_t)( K + l ) * n] : (T)0;
            }
            acc_t acc0, acc1;
#pragma unroll
            for ( int v = 0; v < 4; v++ ) {
                const int32_t rr = rb + M::row( lane, v );
                M::set( acc0, v, ( rr < nr ) ? rget( rr, lane & 15 ) : (T)0 );
                M::set( acc1, v, ( rr < nr ) ? rget( rr, 16 + ( lane & 15 ) ) : (T)0 );
            }
#pragma unroll
            for ( int s4 = 0; s4 < PXD_NB / 4; s4++ ) {
                const int l = 4 * s4 + ( lane >> 4 );
                acc0 = M::mma( a[s4], sX[l][lane & 15], acc0 );
                acc1 = M::mma( a[s4], sX[l][16 + ( lane & 15 )], acc1 );
            }
#pragma unroll
            for ( int v = 0; v < 4; v++ ) {
                const int32_t rr = rb + M::row( lane, v );
                if ( rr < nr ) {
                    rset( rr, lane & 15, M::get( acc0, v ) );
                    rset( rr, 16 + ( lane & 15 ), M::get( acc1, v ) );
                }
            }
        }
    };

    for ( int idx = tid; idx < min( nr, rcap ) * ( PXD_NB + 1 ); idx += PXD_THREADS ) {
        ( &sR[0][0] )[idx] = (T)0;
    }
    for ( int idx = tid; idx < ( nr - rcap ) * PXD_NB; idx += PXD_THREADS ) {
        rset( rcap + idx % ( nr - rcap ), idx / ( nr - rcap ), (T)0 );
    }
    load_block( sX, J, J, bj, bj );   // D_J
    __syncthreads();
    sweep( 0, J, bj );                // R = -L[r0:, J] D_J
    for ( int32_t K = r0; K < n; K += PXD_NB ) {
        const int32_t bk = min( PXD_NB, n - K );
        load_block( sD, K, K, bk, bk );
        __syncthreads();
        // X[K,J] = D_K R[K - r0 .. +31]: wave w computes the 16 x 16 block
        // (w >> 1, w & 1) of the 32 x 32 product
        {
            const int32_t bi = w >> 1, bc = w & 1;
            acc_t         acc = M::zero();
#pragma unroll
            for ( int s4 = 0; s4 < PXD_NB / 4; s4++ ) {
                const int l = 4 * s4 + ( lane >> 4 );
                const T   a = sD[16 * bi + ( lane & 15 )][l];
                const T   b = ( K - r0 + l < nr ) ? rget( K - r0 + l, 16 * bc + ( lane & 15 ) ) : (T)0;
                acc = M::mma( a, b, acc );
            }
            __syncthreads();   // every wave has read sX (previous step) and sR[K block]
#pragma unroll
            for ( int v = 0; v < 4; v++ ) {
                const int r = 16 * bi + M::row( lane, v ), cc = 16 * bc + ( lane & 15 );
                sX[r][cc] = M::get( acc, v );
                if ( r < bk && cc < bj ) LI[( K + r ) + (int64_t)( J + cc ) * n] = M::get( acc, v );
            }
        }
        __syncthreads();
        if ( K + PXD_NB < n ) {
            sweep( K + PXD_NB - r0, K, bk );
        }
    }
    stamp_end( stamps, blockIdx.x, t_stamp );
}

// ---------------------------------------------------------------------------
// Off-diagonal TRSM on the matrix cores: X = B * Linv^T for a tile of 64
// off-diagonal rows and all n columns of the cblk, in place (the workgroup
// owns complete rows, so every read of B precedes every write of X).
// Columns go in passes of NTP = 4 * CPW 16-column tiles, the highest pass
// first: Linv is lower triangular, so a pass reads only B columns up to its
// own last one and may overwrite its columns before the lower passes run.
// In a pass every wave covers all 64 rows against CPW column tiles (tiles
// w, w+4, ...), so each LDS fragment feeds 4 or CPW products; the k values
// of an MFMA step are permuted (lane group g takes k = KV*g + s) so that
// every fragment is one 16-byte read.  Stages whose k range lies above a
// column tile (Linv zero there) are skipped for that tile.
// LU takes its two sides (L with the inverses of the U_kk^T, U^T with those of
// the L_kk) in one launch: one after the other, each left most of the chip idle
// at the top of the tree. TRSM launches alone, 64^3 float 4.87 ->
// 3.49 ms, 41^3 double 1.93 -> 1.14 ms.
template <typename T> struct trsm_cpw;
template <> struct trsm_cpw<float>  { static constexpr int value = 2; };
template <> struct trsm_cpw<double> { static constexpr int value = 2; };
template <> struct trsm_cpw<pxcf>   { static constexpr int value = 2; };
template <> struct trsm_cpw<pxcd>   { static constexpr int value = 1; };

template <typename T>
__global__ void __launch_bounds__( PXD_THREADS, 2 )
k_trsm_mfma( const row_task *__restrict__ tasks, int32_t ntasks, const dcblk *__restrict__ cb,
             const dblok *__restrict__ bk, T *__restrict__ L0, const T *__restrict__ Linv0, T *__restrict__ L1,
             const T *__restrict__ Linv1, int ldlt, uint64_t *__restrict__ stamps0, uint64_t *__restrict__ stamps1,
             int prio )
{
    typedef mfma16<T>                 M;
    typedef typename M::acc_t         acc_t;
    typedef typename lds_vec<T>::type vec_t;
    constexpr int KV  = lds_vec<T>::n;
    constexpr int BK  = 4 * KV;                      // k values per stage
    constexpr int LDK = BK + KV;
    constexpr int CPW = trsm_cpw<T>::value;          // column tiles per wave
    constexpr int NTP = 4 * CPW;                     // column tiles per pass
    constexpr int CPT = NTP * 16;                    // columns per pass
    constexpr int TPC = PXD_THREADS / CPT;           // Linv loader threads per column
    constexpr int KPC = BK / TPC;                    // k values per Linv loader thread
    __shared__ __align__( 16 ) T sB[64 * LDK];       // B rows, k contiguous
    __shared__ __align__( 16 ) T sLi[CPT * LDK];     // Linv columns of the pass, k contiguous
    __shared__ int64_t sBase[64];
    __shared__ int32_t sLd[64];
    __shared__ T       sDi[PXD_TRSM_NT * 16];        // LDL^T: 1 / D of the cblk

    // LU: the tiles of both sides in one launch
    int32_t        ti = xcd_task( blockIdx.x, gridDim.x );
    const bool     u  = ti >= ntasks;
    T *__restrict__ L = u ? L1 : L0;
    const T *__restrict__ Linv = u ? Linv1 : Linv0;
    uint64_t *stamps  = u ? stamps1 : stamps0;
    ti -= u ? ntasks : 0;
    const row_task t = tasks[ti];
    const uint64_t t_stamp = stamp_begin( stamps );
    wave_priority( prio );
    const dcblk    c    = cb[t.cblk];
    const int32_t  n    = c.lcolnum - c.fcolnum + 1;
    const int32_t  lb   = cb[t.cblk + 1].fblok;
    const int      tid  = threadIdx.x;
    const int      lane = tid & 63, w = tid >> 6;
    const int      lr   = lane & 15, lg = lane >> 4;
    const T       *LI   = Linv + c.dinvoff;
    const int      nt   = ( n + 15 ) >> 4;

    if ( ldlt ) {
        for ( int32_t i = tid; i < n; i += PXD_THREADS ) sDi[i] = (T)1 / L[c.coefoff + (int64_t)i * ( n + 1 )];
    }
    __shared__ int32_t skeys[PXD_ROWKEY_CAP];
    stage_row_keys( skeys, bk, c.fblok, lb );
    __syncthreads();
    if ( tid < 64 ) {
        int32_t s = t.r0 + tid;
        if ( s < c.stride ) {
            int32_t b  = search_row_keys( skeys, bk, c.fblok, lb, s );
            dblok   bb = bk[b];
            sBase[tid] = c.coefoff + (int64_t)bb.rowoff * n + ( s - bb.rowoff );
            sLd[tid]   = bb.lrownum - bb.frownum + 1;
        }
        else {
            sBase[tid] = -1;
            sLd[tid]   = 0;
        }
    }
    __syncthreads();

    // B loader: row br, k values [bq * KV, bq * KV + KV) of a stage
    const int     br    = tid & 63, bq = tid >> 6;
    const int64_t lbase = sBase[br];
    const int32_t lld   = sLd[br];
    // Linv loader: column lc of the pass, k values [lq * KPC, lq * KPC + KPC)
    const int     lc = tid % CPT, lq = tid / CPT;

    const int npass = ( nt + NTP - 1 ) / NTP;
    for ( int pass = npass - 1; pass >= 0; pass-- ) {
        const int32_t cb0  = pass * CPT;                       // first column of the pass
        const int32_t lend = min( n, cb0 + CPT );              // Linv[c][l] = 0 for l > c
        acc_t acc[4][CPW];
#pragma unroll
        for ( int i = 0; i < 4; i++ )
#pragma unroll
            for ( int j = 0; j < CPW; j++ ) acc[i][j] = M::zero();

        // the next stage's loads are issued before the current stage's products
        T    rb[KV], rl[KPC];
        auto load = [&]( int32_t l0 ) {
#pragma unroll
            for ( int q = 0; q < KV; q++ ) {
                const int32_t l = l0 + bq * KV + q;
                rb[q] = ( lbase >= 0 && l < lend ) ? L[lbase + (int64_t)l * lld] : (T)0;
            }
#pragma unroll
            for ( int q = 0; q < KPC; q++ ) {
                const int32_t cc = cb0 + lc, l = l0 + lq * KPC + q;
                rl[q] = ( cc < n && l <= cc ) ? LI[cc + (int64_t)l * n] : (T)0;
            }
        };
        load( 0 );
        for ( int32_t l0 = 0; l0 < lend; l0 += BK ) {
            {
                vec_t v;
#pragma unroll
                for ( int e = 0; e < KV; e++ ) v[e] = rb[e];
                *(vec_t *)&sB[br * LDK + bq * KV] = v;
            }
#pragma unroll
            for ( int q = 0; q < KPC; q += KV ) {
                vec_t v;
#pragma unroll
                for ( int e = 0; e < KV; e++ ) v[e] = rl[q + e];
                *(vec_t *)&sLi[lc * LDK + lq * KPC + q] = v;
            }
            __syncthreads();
            if ( l0 + BK < lend ) {
                load( l0 + BK );
            }
            vec_t av[4], bv[CPW];
#pragma unroll
            for ( int i = 0; i < 4; i++ ) av[i] = *(const vec_t *)&sB[( 16 * i + lr ) * LDK + KV * lg];
#pragma unroll
            for ( int j = 0; j < CPW; j++ ) bv[j] = *(const vec_t *)&sLi[( 16 * ( w + 4 * j ) + lr ) * LDK + KV * lg];
#pragma unroll
            for ( int j = 0; j < CPW; j++ ) {
                const int32_t c0 = cb0 + 16 * ( w + 4 * j );   // first column of the tile
                if ( c0 < n && c0 + 15 >= l0 ) {
#pragma unroll
                    for ( int e = 0; e < KV; e++ )
#pragma unroll
                        for ( int i = 0; i < 4; i++ ) acc[i][j] = M::mma( av[i][e], bv[j][e], acc[i][j] );
                }
            }
            __syncthreads();
        }
#pragma unroll
        for ( int j = 0; j < CPW; j++ ) {
            const int cc = cb0 + 16 * ( w + 4 * j ) + lr;
#pragma unroll
            for ( int i = 0; i < 4; i++ )
#pragma unroll
                for ( int v = 0; v < 4; v++ ) {
                    const int r = 16 * i + M::row( lane, v );
                    if ( sBase[r] >= 0 && cc < n ) {
                        // LDL^T: L_off = B L_kk^{-T} D^{-1}
                        L[sBase[r] + (int64_t)cc * sLd[r]] = ldlt ? M::get( acc[i][j], v ) * sDi[cc] : M::get( acc[i][j], v );
                    }
                }
        }
        __syncthreads();   // the pass's stores precede the next pass's loads
    }
    stamp_end( stamps, ti, t_stamp );
}


// ---------------------------------------------------------------------------
// Supernodal update on the matrix cores: C[f(i)] -= A_i * A_b^T for one
// 64 x 64 output tile (four waves of 32 x 32), fused row remap into the
// facing cblk in the epilogue (atomic adds when another source of the same
// level may hit the same columns).
template <typename T>
__global__ void __launch_bounds__( PXD_THREADS )
k_update_mfma( const upd_task *__restrict__ tasks, const dcblk *__restrict__ cb,
               const dblok *__restrict__ bk, T *L, T *U, int ldlt,
               uint64_t *__restrict__ stamps, int prio )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    constexpr int BK = 16;
    __shared__ T       sA[BK][64 + 4];
    __shared__ T       sB[BK][64 + 4];
    __shared__ int64_t sSrc[64];
    __shared__ int32_t sSrcLd[64];
    __shared__ int64_t sDst[64];
    __shared__ int32_t sDstLd[64];
    __shared__ search_keys sk;
    __shared__ T           sDk[PXD_TRSM_NT * 16];   // LDL^T: D of the source cblk

    const int32_t  ti   = xcd_task( blockIdx.x, gridDim.x );
    const upd_task t    = tasks[ti];
    const uint64_t t_stamp = stamp_begin( stamps );
    wave_priority( prio );
    const int      tid  = threadIdx.x;
    const int      lane = tid & 63, w = tid >> 6;
    const dcblk    c    = cb[t.cblk];
    const int32_t  K    = c.lcolnum - c.fcolnum + 1;
    const int32_t  lb   = cb[t.cblk + 1].fblok;
    const dblok    bb   = bk[t.blok];
    const int32_t  N    = bb.lrownum - bb.frownum + 1;
    // U-side tile (LU): A = U^T rows after blok b, B = L rows of blok b, C = U
    const bool     uside = ( t.flags & 2 ) != 0;
    const T       *LA   = uside ? U : L;
    const T       *LB   = uside ? L : U;
    T             *LC   = uside ? U : L;
    const int32_t  r0   = bb.rowoff + ( uside ? N : 0 );
    const int32_t  Mr   = c.stride - r0;
    const int32_t  F    = bb.fcblknm;
    const dcblk    cf   = cb[F];
    const int32_t  Fn   = cf.lcolnum - cf.fcolnum + 1;
    const int32_t  flb  = cb[F + 1].fblok;
    const int32_t  colF0 = bb.frownum - cf.fcolnum + t.tn * 64;
    const int64_t  bbase = c.coefoff + (int64_t)bb.rowoff * K + t.tn * 64;
    if ( bb.frownum < cf.fcolnum || bb.lrownum > cf.lcolnum ) {
        return;   // inconsistent structure: the host checks prevent this
    }

    stage_search_keys( sk, bk, t.blok, lb, cf.fblok, flb, tid );
    if ( ldlt ) {
        // LDL^T: C -= A_i (A_b D)^T (the reference's DL^T workspace, formed on the fly)
        for ( int32_t i = tid; i < K; i += PXD_THREADS ) sDk[i] = L[c.coefoff + (int64_t)i * ( K + 1 )];
    }
    __syncthreads();
    if ( tid < 64 ) {
        int32_t r = t.tm * 64 + tid;
        if ( r < Mr ) {
            int32_t s  = r0 + r;
            int32_t bi = search_row( sk, bk, t.blok, lb, s );
            dblok   ib = bk[bi];
            int32_t g  = ib.frownum + ( s - ib.rowoff );
            sSrc[tid]   = c.coefoff + (int64_t)ib.rowoff * K + ( s - ib.rowoff );
            sSrcLd[tid] = ib.lrownum - ib.frownum + 1;
            int32_t fi  = search_grow( sk, bk, cf.fblok, flb, g );
            dblok   fb  = bk[fi];
            bool    ok  = ( g >= fb.frownum && g <= fb.lrownum );
            sDst[tid]   = ok ? cf.coefoff + (int64_t)fb.rowoff * Fn + ( g - fb.frownum ) : -1;
            sDstLd[tid] = fb.lrownum - fb.frownum + 1;
        }
        else {
            sSrc[tid]   = -1;
            sSrcLd[tid] = 0;
            sDst[tid]   = -1;
            sDstLd[tid] = 0;
        }
    }
    __syncthreads();

    const int     lr     = tid & 63;
    const int64_t src    = sSrc[lr];
    const int32_t srcld  = sSrcLd[lr];
    const int32_t nvalid = min( 64, N - t.tn * 64 );

    acc_t acc[2][2];
#pragma unroll
    for ( int i = 0; i < 2; i++ )
#pragma unroll
        for ( int j = 0; j < 2; j++ ) acc[i][j] = M::zero();
    const int wr = 32 * ( w >> 1 ), wc = 32 * ( w & 1 );

    for ( int32_t k0 = 0; k0 < K; k0 += BK ) {
        T va[BK / 4], vb[BK / 4];
#pragma unroll
        for ( int u = 0; u < BK / 4; u++ ) {
            const int32_t kg = k0 + ( tid >> 6 ) + 4 * u;
            va[u] = ( kg < K && src >= 0 ) ? LA[src + (int64_t)kg * srcld] : (T)0;
            vb[u] = ( kg < K && lr < nvalid ) ? LB[bbase + lr + (int64_t)kg * N] : (T)0;
        }
#pragma unroll
        for ( int u = 0; u < BK / 4; u++ ) {
            const int32_t kg = k0 + ( tid >> 6 ) + 4 * u;
            sA[( tid >> 6 ) + 4 * u][lr] = va[u];
            sB[( tid >> 6 ) + 4 * u][lr] = ( ldlt && kg < K ) ? vb[u] * sDk[kg] : vb[u];
        }
        __syncthreads();
#pragma unroll
        for ( int k4 = 0; k4 < BK; k4 += 4 ) {
            const int kr = k4 + ( lane >> 4 );
            T a0 = sA[kr][wr + ( lane & 15 )];
            T a1 = sA[kr][wr + 16 + ( lane & 15 )];
            T b0 = sB[kr][wc + ( lane & 15 )];
            T b1 = sB[kr][wc + 16 + ( lane & 15 )];
            acc[0][0] = M::mma( a0, b0, acc[0][0] );
            acc[0][1] = M::mma( a0, b1, acc[0][1] );
            acc[1][0] = M::mma( a1, b0, acc[1][0] );
            acc[1][1] = M::mma( a1, b1, acc[1][1] );
        }
        __syncthreads();
    }

    // scatter into F: all loads of the read-modify-writes first, then the stores
    const bool atomic = ( t.flags & 1 );
    T         *p[2][4];
    bool       pv[2][2][4];
#pragma unroll
    for ( int i = 0; i < 2; i++ ) {
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
            const int r = wr + 16 * i + M::row( lane, v );
            p[i][v]     = LC + ( sDst[r] >= 0 ? sDst[r] : 0 ) + (int64_t)colF0 * sDstLd[r];
#pragma unroll
            for ( int j = 0; j < 2; j++ ) pv[i][j][v] = sDst[r] >= 0 && wc + 16 * j + ( lane & 15 ) < nvalid;
        }
    }
    T old[2][2][4];
#pragma unroll
    for ( int i = 0; i < 2; i++ )
#pragma unroll
        for ( int j = 0; j < 2; j++ )
#pragma unroll
            for ( int v = 0; v < 4; v++ ) {
                const int r  = wr + 16 * i + M::row( lane, v );
                const int cc = wc + 16 * j + ( lane & 15 );
                T *dst = p[i][v] + (int64_t)cc * sDstLd[r];
                if ( atomic ) {
                    if ( pv[i][j][v] ) px_atomic_add( dst, -M::get( acc[i][j], v ) );
                }
                else {
                    old[i][j][v] = pv[i][j][v] ? *dst : (T)0;
                }
            }
    if ( !atomic ) {
#pragma unroll
        for ( int i = 0; i < 2; i++ )
#pragma unroll
            for ( int j = 0; j < 2; j++ )
#pragma unroll
                for ( int v = 0; v < 4; v++ ) {
                    const int r  = wr + 16 * i + M::row( lane, v );
                    const int cc = wc + 16 * j + ( lane & 15 );
                    if ( pv[i][j][v] ) p[i][v][(int64_t)cc * sDstLd[r]] = old[i][j][v] - M::get( acc[i][j], v );
                }
    }
    stamp_end( stamps, ti, t_stamp );
}

// ---------------------------------------------------------------------------
// Small supernodal updates, one wavefront per 64 stacked rows of a blok
// update (the lower tree has hundreds of thousands of them with a few rows
// and columns): task {cblk, blok, tm, flags} covers the stacked rows
// [64 tm, 64 tm + 64) of an update with at most PXD_SMALL_M stacked rows
// (Mr), PXD_SMALL_N facing columns (N) and PXD_SMALL_K source columns (K).
// Lane r owns stacked row 64 tm + r and keeps its K values of A in
// registers; the facing columns go by chunks of PXD_SMALL_NC: the chunk of
// B (the rows of blok b, D-scaled for LDL^T) is staged in the wavefront's
// LDS area, C[f(r), chunk] -= A_r B_chunk^T, plain read-modify-write or
// atomic adds when the task is flagged.  The four wavefronts of a workgroup
// are independent (no workgroup barrier).
#define PXD_SMALL_M  256
#define PXD_SMALL_N  64
#define PXD_SMALL_NC 16
#define PXD_SMALL_K  32
template <typename T>
__global__ void __launch_bounds__( PXD_THREADS )
k_update_small( const upd_task *__restrict__ tasks, int32_t ntasks, const dcblk *__restrict__ cb,
                const dblok *__restrict__ bk, T *L, T *U, int ldlt, uint64_t *__restrict__ stamps, int prio )
{
    constexpr int NC = PXD_SMALL_NC;
    __shared__ T sB[PXD_THREADS / 64][PXD_SMALL_K][NC + 1];
    const uint64_t t_stamp = stamp_begin( stamps );
    wave_priority( prio );
    const int     lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int32_t ti   = blockIdx.x * ( PXD_THREADS / 64 ) + w;
    if ( ti < ntasks ) {
        const upd_task t  = tasks[ti];
        const dcblk    c  = cb[t.cblk];
        const int32_t  K  = c.lcolnum - c.fcolnum + 1;
        const int32_t  lb = cb[t.cblk + 1].fblok;
        const dblok    bb = bk[t.blok];
        const int32_t  N  = bb.lrownum - bb.frownum + 1;
        const bool     uside = ( t.flags & 2 ) != 0;
        const T       *LA = uside ? U : L;
        const T       *LB = uside ? L : U;
        T             *LC = uside ? U : L;
        const int32_t  r0 = bb.rowoff + ( uside ? N : 0 );
        const int32_t  Mr = c.stride - r0;
        const int32_t  F  = bb.fcblknm;
        const dcblk    cf = cb[F];
        const int32_t  Fn = cf.lcolnum - cf.fcolnum + 1;
        const int32_t  flb = cb[F + 1].fblok;
        const int32_t  colF0 = bb.frownum - cf.fcolnum;
        const int64_t  bbase = c.coefoff + (int64_t)bb.rowoff * K;
        const int32_t  row   = 64 * t.tm + lane;   // stacked row of the lane, from r0
        // the lane's row: its K values of A and its place in F
        T       a[PXD_SMALL_K];
        T      *dst = nullptr;
        int32_t dld = 0;
        if ( row < Mr ) {
            const int32_t s   = r0 + row;
            const int32_t bi  = find_blok_by_row( bk, t.blok, lb, s );
            const dblok   ib  = bk[bi];
            const int64_t src = c.coefoff + (int64_t)ib.rowoff * K + ( s - ib.rowoff );
            const int32_t sld = ib.lrownum - ib.frownum + 1;
            const int32_t g   = ib.frownum + ( s - ib.rowoff );
#pragma unroll
            for ( int kk = 0; kk < PXD_SMALL_K; kk++ ) a[kk] = ( kk < K ) ? LA[src + (int64_t)kk * sld] : (T)0;
            const int32_t fi = find_blok_by_grow( bk, cf.fblok, flb, g );
            const dblok   fb = bk[fi];
            if ( g >= fb.frownum && g <= fb.lrownum ) {
                dld = fb.lrownum - fb.frownum + 1;
                dst = LC + cf.coefoff + (int64_t)fb.rowoff * Fn + ( g - fb.frownum ) + (int64_t)colF0 * dld;
            }
        }
        for ( int32_t j0 = 0; j0 < N; j0 += NC ) {
            const int32_t nc = min( NC, N - j0 );
            // B[j][k] = LB[bbase + j + k N] for the chunk's columns, times D_k for LDL^T
            for ( int idx = lane; idx < nc * K; idx += 64 ) {
                const int j = idx % nc, kk = idx / nc;
                const T   v = LB[bbase + j0 + j + (int64_t)kk * N];
                sB[w][kk][j] = ldlt ? v * L[c.coefoff + (int64_t)kk * ( K + 1 )] : v;
            }
            __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
            if ( dst != nullptr ) {
                T acc[NC];
#pragma unroll
                for ( int j = 0; j < NC; j++ ) acc[j] = (T)0;
#pragma unroll
                for ( int kk = 0; kk < PXD_SMALL_K; kk++ ) {
                    if ( kk < K ) {
#pragma unroll
                        for ( int j = 0; j < NC; j++ ) acc[j] += a[kk] * sB[w][kk][j];
                    }
                }
                T *d0 = dst + (int64_t)j0 * dld;
                if ( t.flags & 1 ) {
#pragma unroll
                    for ( int j = 0; j < NC; j++ ) {
                        if ( j < nc ) px_atomic_add( d0 + (int64_t)j * dld, -acc[j] );
                    }
                }
                else {
                    T old[NC];
#pragma unroll
                    for ( int j = 0; j < NC; j++ ) old[j] = ( j < nc ) ? d0[(int64_t)j * dld] : (T)0;
#pragma unroll
                    for ( int j = 0; j < NC; j++ ) {
                        if ( j < nc ) d0[(int64_t)j * dld] = old[j] - acc[j];
                    }
                }
            }
            // every lane has read the chunk before the next one is staged
            __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
            __builtin_amdgcn_wave_barrier();
            __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
        }
    }
    stamp_end( stamps, blockIdx.x, t_stamp );
}

// ---------------------------------------------------------------------------
// Supernodal update for tall tiles: C[f(i)] -= A_i * A_b^T for upd_rows<T>
// stacked rows x PXD_UPD_BN facing columns, wave w owning rows
// [w*BM/4, (w+1)*BM/4).  The next k-stage is loaded into registers while the
// current one is on the matrix cores.  LDS holds each row's k values
// contiguously, and the k values of one MFMA step are permuted (lane group g
// takes k = KV*g + s in step s) so that every fragment is one 16-byte read.
// C[rows, cols] -= acc for one 16 x 64 row block of an update tile: row r of
// the block goes to L + dst[r] + col * ld[r], columns colF0 + [0, nvalid).
template <typename T>
__device__ inline void
update_scatter( T *L, const typename mfma16<T>::acc_t ( &acc )[4], int r0, int lane,
                const int64_t *dst, const int32_t *ld, int32_t colF0, int32_t nvalid, bool atomic )
{
    typedef mfma16<T> M;
    T      *p[4];
    int32_t pl[4];
    bool    pv[4];
#pragma unroll
    for ( int v = 0; v < 4; v++ ) {
        const int r = r0 + M::row( lane, v );
        pv[v]       = dst[r] >= 0;
        pl[v]       = ld[r];
        p[v]        = L + ( pv[v] ? dst[r] : 0 ) + (int64_t)colF0 * pl[v];
    }
    if ( atomic ) {
#pragma unroll
        for ( int j = 0; j < 4; j++ ) {
            const int cc = 16 * j + ( lane & 15 );
#pragma unroll
            for ( int v = 0; v < 4; v++ ) {
                if ( pv[v] && cc < nvalid ) px_atomic_add( p[v] + (int64_t)cc * pl[v], -M::get( acc[j], v ) );
            }
        }
        return;
    }
    T old[4][4];
#pragma unroll
    for ( int j = 0; j < 4; j++ ) {
        const int cc = 16 * j + ( lane & 15 );
#pragma unroll
        for ( int v = 0; v < 4; v++ ) old[j][v] = ( pv[v] && cc < nvalid ) ? p[v][(int64_t)cc * pl[v]] : (T)0;
    }
#pragma unroll
    for ( int j = 0; j < 4; j++ ) {
        const int cc = 16 * j + ( lane & 15 );
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
            if ( pv[v] && cc < nvalid ) p[v][(int64_t)cc * pl[v]] = old[j][v] - M::get( acc[j], v );
        }
    }
}

#define PXD_UPD_BN 64
template <typename T> struct upd_rows;
template <> struct upd_rows<float>  { static constexpr int value = 256; };
template <> struct upd_rows<double> { static constexpr int value = 128; };
template <> struct upd_rows<pxcf>   { static constexpr int value = 128; };
template <> struct upd_rows<pxcd>   { static constexpr int value = 64; };

template <typename T, int NH>
__global__ void __launch_bounds__( PXD_THREADS, ( NH == 1 ) ? 3 : 2 )
k_update_big( const upd_task *__restrict__ tasks, int32_t ntasks, const dcblk *__restrict__ cb,
              const dblok *__restrict__ bk, T *L, T *U, int ldlt,
              uint64_t *__restrict__ stamps, int prio )
{
    typedef mfma16<T>          M;
    typedef typename M::acc_t  acc_t;
    typedef typename lds_vec<T>::type vec_t;
    constexpr int BM  = upd_rows<T>::value;
    constexpr int KV  = lds_vec<T>::n;    // k values per fragment
    constexpr int BK  = NH * 4 * KV;      // k values per stage (NH MFMA k-groups of 4*KV)
    constexpr int LDK = BK + KV;          // row stride of the staged tiles
    constexpr int TPR = PXD_THREADS / BM; // loader threads per row
    constexpr int KPT = BK / TPR;         // k values loaded per thread
    constexpr int RB  = BM / 64;          // 16-row blocks per wave
    constexpr uint32_t ES = sizeof( T );
    constexpr int WR  = 16 * RB;          // rows per wave
    constexpr int SE  = ( BM * LDK > 4 * WR * 17 ) ? BM * LDK : 4 * WR * 17;
    __shared__ __align__( 16 ) T sA[SE];  // staged A tile; after the k loop, the epilogue's transposes
    __shared__ __align__( 16 ) T sB[PXD_UPD_BN * LDK];
    __shared__ uint32_t sDst[BM];         // byte offset of the row in F (PXD_OOB: none)
    __shared__ uint32_t sDstLd[BM];       // byte stride between F's columns for the row
    __shared__ search_keys sk;
    __shared__ T           sDk[PXD_TRSM_NT * 16];   // LDL^T: D of the source cblk

    const int32_t  ti   = xcd_task( blockIdx.x, ntasks );
    const upd_task t    = tasks[ti];
    const uint64_t t_stamp = stamp_begin( stamps );
    wave_priority( prio );
    const int      tid  = threadIdx.x;
    const int      lane = tid & 63, w = tid >> 6;
    const dcblk    c    = cb[t.cblk];
    const int32_t  K    = c.lcolnum - c.fcolnum + 1;
    const int32_t  lb   = cb[t.cblk + 1].fblok;
    const dblok    bb   = bk[t.blok];
    const int32_t  N    = bb.lrownum - bb.frownum + 1;
    // U-side tile (LU): A = U^T rows after blok b, B = L rows of blok b, C = U
    const bool     uside = ( t.flags & 2 ) != 0;
    const T       *LA   = uside ? U : L;
    const T       *LB   = uside ? L : U;
    T             *LC   = uside ? U : L;
    const int32_t  r0   = bb.rowoff + ( uside ? N : 0 );
    const int32_t  Mr   = c.stride - r0;
    const int32_t  F    = bb.fcblknm;
    const dcblk    cf   = cb[F];
    const int32_t  Fn   = cf.lcolnum - cf.fcolnum + 1;
    const int32_t  flb  = cb[F + 1].fblok;
    const int32_t  colF0 = bb.frownum - cf.fcolnum + t.tn * PXD_UPD_BN;
    if ( bb.frownum < cf.fcolnum || bb.lrownum > cf.lcolnum ) {
        return;   // inconsistent structure: the host checks prevent this
    }
    const __amdgpu_buffer_rsrc_t rA = make_rsrc( LA + c.coefoff, (uint32_t)( (int64_t)c.stride * K * ES ) );
    const __amdgpu_buffer_rsrc_t rB = make_rsrc( LB + c.coefoff, (uint32_t)( (int64_t)c.stride * K * ES ) );
    const __amdgpu_buffer_rsrc_t rC = make_rsrc( LC + cf.coefoff, (uint32_t)( (int64_t)cf.stride * Fn * ES ) );

    stage_search_keys( sk, bk, t.blok, lb, cf.fblok, flb, tid );
    if ( ldlt ) {
        // LDL^T: C -= A_i (A_b D)^T (the reference's DL^T workspace, formed on the fly)
        for ( int32_t i = tid; i < K; i += PXD_THREADS ) sDk[i] = L[c.coefoff + (int64_t)i * ( K + 1 )];
    }
    __syncthreads();

    // loader row ar (k values [ap*KPT, ap*KPT+KPT) of each stage): byte
    // offset of its first element and byte stride between its columns; the
    // threads with ap == 0 also map the row into F
    const int ar = tid % BM, ap = tid / BM;
    uint32_t  abase = PXD_OOB, astep = 0;
    {
        const int32_t r   = t.tm * BM + ar;
        uint32_t      dst = PXD_OOB, dld = 0;
        if ( r < Mr ) {
            const int32_t s  = r0 + r;
            const dblok   ib = bk[search_row( sk, bk, t.blok, lb, s )];
            const int32_t g  = ib.frownum + ( s - ib.rowoff );
            abase = (uint32_t)( ib.rowoff * K + ( s - ib.rowoff ) ) * ES;
            astep = (uint32_t)( ib.lrownum - ib.frownum + 1 ) * ES;
            if ( ap == 0 ) {
                const dblok fb = bk[search_grow( sk, bk, cf.fblok, flb, g )];
                if ( g >= fb.frownum && g <= fb.lrownum ) {
                    dst = (uint32_t)( fb.rowoff * Fn + ( g - fb.frownum ) ) * ES;
                    dld = (uint32_t)( fb.lrownum - fb.frownum + 1 ) * ES;
                }
            }
        }
        if ( ap == 0 ) {
            sDst[ar]   = dst;
            sDstLd[ar] = dld;
        }
    }
    // B loader: facing column bc, k group bq
    const int      bc     = tid & ( PXD_UPD_BN - 1 ), bq = tid / PXD_UPD_BN;
    const int32_t  nvalid = min( PXD_UPD_BN, N - t.tn * PXD_UPD_BN );
    const uint32_t bbase  = ( bc < nvalid ) ? (uint32_t)( bb.rowoff * K + t.tn * PXD_UPD_BN + bc ) * ES : PXD_OOB;
    const uint32_t bstep  = ( bc < nvalid ) ? (uint32_t)N * ES : 0;

    T ra[KPT], rb[NH * KV];
    auto load = [&]( int32_t k0 ) {
#pragma unroll
        for ( int q = 0; q < KPT; q++ ) {
            const int32_t kg = k0 + ap * KPT + q;
            ra[q] = bufio<T>::load( rA, ( kg < K ) ? abase + (uint32_t)kg * astep : PXD_OOB );
        }
#pragma unroll
        for ( int q = 0; q < NH * KV; q++ ) {
            const int32_t kg = k0 + bq * NH * KV + q;
            rb[q] = bufio<T>::load( rB, ( kg < K ) ? bbase + (uint32_t)kg * bstep : PXD_OOB );
        }
    };

    acc_t acc[RB][4];
#pragma unroll
    for ( int i = 0; i < RB; i++ )
#pragma unroll
        for ( int j = 0; j < 4; j++ ) acc[i][j] = M::zero();

    const int lr = lane & 15, lg = lane >> 4;
    load( 0 );
    for ( int32_t k0 = 0; k0 < K; k0 += BK ) {
#pragma unroll
        for ( int q = 0; q < KPT; q += KV ) {
            vec_t v;
#pragma unroll
            for ( int e = 0; e < KV; e++ ) v[e] = ra[q + e];
            *(vec_t *)&sA[ar * LDK + ap * KPT + q] = v;
        }
#pragma unroll
        for ( int h = 0; h < NH; h++ ) {
            vec_t v;
#pragma unroll
            for ( int e = 0; e < KV; e++ ) {
                const int32_t kg = k0 + bq * NH * KV + h * KV + e;
                v[e] = ( ldlt && kg < K ) ? rb[h * KV + e] * sDk[kg] : rb[h * KV + e];
            }
            *(vec_t *)&sB[bc * LDK + bq * NH * KV + h * KV] = v;
        }
        __syncthreads();
        if ( k0 + BK < K ) {
            load( k0 + BK );
        }
#pragma unroll
        for ( int h = 0; h < NH; h++ ) {
            vec_t av[RB], bv[4];
#pragma unroll
            for ( int i = 0; i < RB; i++ )
                av[i] = *(const vec_t *)&sA[( 16 * ( RB * w + i ) + lr ) * LDK + 4 * KV * h + KV * lg];
#pragma unroll
            for ( int j = 0; j < 4; j++ ) bv[j] = *(const vec_t *)&sB[( 16 * j + lr ) * LDK + 4 * KV * h + KV * lg];
#pragma unroll
            for ( int s = 0; s < KV; s++ )
#pragma unroll
                for ( int i = 0; i < RB; i++ )
#pragma unroll
                    for ( int j = 0; j < 4; j++ ) acc[i][j] = M::mma( av[i][s], bv[j][s], acc[i][j] );
        }
        __syncthreads();
    }

    // scatter into F, one 16-column slab at a time: each wave transposes its
    // WR x 16 block through LDS so that a lane owns one row and every memory
    // instruction covers WR consecutive rows of one column (coalesced, as F is
    // column major).  Plain tiles issue all loads of a slab, then the stores
    // (out-of-range rows and columns read 0 and drop their stores); tiles
    // flagged atomic use atomic adds.
    const bool    atomic = ( t.flags & 1 );
    T            *sE     = sA + w * ( WR * 17 );
    constexpr int LPR    = 64 / WR;        // lanes per row
    constexpr int CPL    = 16 / LPR;       // columns per lane
    const int     erow   = lane % WR, epart = lane / WR;
    const uint32_t rowoff = sDst[WR * w + erow];
    const uint32_t rowld  = sDstLd[WR * w + erow];
#pragma unroll
    for ( int j = 0; j < 4; j++ ) {
#pragma unroll
        for ( int i = 0; i < RB; i++ )
#pragma unroll
            for ( int v = 0; v < 4; v++ ) sE[( 16 * i + M::row( lane, v ) ) * 17 + lr] = M::get( acc[i][j], v );
        __syncthreads();
        uint32_t off[CPL];
        T        val[CPL];
#pragma unroll
        for ( int c = 0; c < CPL; c++ ) {
            const int col = epart * CPL + c, cc = 16 * j + col;
            off[c] = ( rowoff != PXD_OOB && cc < nvalid ) ? rowoff + (uint32_t)( colF0 + cc ) * rowld : PXD_OOB;
            val[c] = sE[erow * 17 + col];
        }
        if ( atomic ) {
#pragma unroll
            for ( int c = 0; c < CPL; c++ ) {
                if ( off[c] != PXD_OOB ) px_atomic_add( LC + cf.coefoff + off[c] / ES, -val[c] );
            }
        }
        else {
            T old[CPL];
#pragma unroll
            for ( int c = 0; c < CPL; c++ ) old[c] = bufio<T>::load( rC, off[c] );
#pragma unroll
            for ( int c = 0; c < CPL; c++ ) bufio<T>::store( old[c] - val[c], rC, off[c] );
        }
        __syncthreads();
    }
    stamp_end( stamps, ti, t_stamp );
}


// ---------------------------------------------------------------------------
// Tall-tile update with its operands moved from HBM straight into LDS by
// buffer loads that write LDS (no register staging), in a ring of NBUF buffers
// of BK k values: while a stage's products run, the loads of the next NBUF - 1
// stages are in flight, and each stage ends with one barrier.
//
// Every lane of a load instruction writes LDS at its own consecutive place, 4
// or 16 bytes; the staged tiles are k major.  Wave w loads and computes the rows
// [w BM/4, (w+1) BM/4) of A, and the waves share the k values of B.
//   float: 4 bytes per lane, one k value of the wave's 64 rows (of the 64
//     columns of B).
//   8-byte types: where the wave's 32 rows lie in one blok, 16 bytes per lane,
//     4 k values of all of them (A[wave][k][32 rows]); else 4 bytes per lane,
//     one k value.  B, whose 64 columns always lie in one blok, 16 bytes per
//     lane (columns past the update are other values of the cblk, and their
//     results are dropped).  100^3 double, update launches: 133.6 ms with 4
//     bytes per lane throughout, 126.1 ms; 80^3 complex64 72.2 -> 70.2 ms.  In
//     float the same gained nothing (65.4 against 68.0 ms).
//   complex double: 16 bytes per lane, an element; each wave loads all 64 rows
//     at its own k value.
//
// C -= acc goes a 16-column slab at a time through LDS, each wave for itself,
// so that a memory instruction covers the wave's 16 to 64 consecutive rows of
// one column.  The runs matter more than the barriers: straight from the
// accumulators (runs of 16 rows) the 100^3 float updates took 73.6 ms, by
// slabs 65.3 ms.  The rows' places in the facing cblk are in the registers of
// the lanes that loaded them.
//
// What bounds it: the matrix cores (busy 0.71 of the time in float, 0.73 in
// double), and the movement of the operands beside them.  100^3 double, update
// launches alone, 126 ms: timing-only copies without the loop's loads 108.9,
// without the C part 121.4, without both 101.2; the products alone take 96 at
// the rate of a large matrix product.  Several pieces of a supernode updating
// C together, which halves the bytes of C, gained nothing.  Float 66.7 -> 65.3
// ms against the same scheme with two workgroup barriers per slab and no load
// in flight across a stage's barrier, double 136.2 -> 133.2 ms and 80^3
// complex64 LDL^T 73.0 -> 71.8 ms against k_update_big (factorizations 155.8
// -> 150.7 and 88.0 -> 84.9 ms).
//
// LDL^T scales A by D (kept in LDS), the reference's D L^T workspace.

// 4 or 16 bytes per lane from r + off to LDS, at the lane's place from dst on
template <int BYTES>
__device__ inline void
load_lds( __amdgpu_buffer_rsrc_t r, void *dst, uint32_t off )
{
    typedef __attribute__( ( address_space( 3 ) ) ) void lds_t;
    if constexpr ( BYTES == 16 ) {
        __builtin_amdgcn_raw_ptr_buffer_load_lds( r, (lds_t *)dst, 16, off, 0, 0, 0 );
    }
    else {
        __builtin_amdgcn_raw_ptr_buffer_load_lds( r, (lds_t *)dst, 4, off, 0, 0, 0 );
    }
}
// Barrier of the workgroup alone: no wait for memory, and no memory access of
// the wave moves across it (wavefront fences order the compiler only).
__device__ inline void
bare_barrier()
{
    __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
}
// k values per stage, and dynamic LDS that leaves CU room to the panels of the
// other stream (float: option upd_dma_pad; complex double 19.1 -> 18.3 ms at
// 50^3 with three workgroups per CU instead of four; in double and complex
// float fewer than four cost more than they give: 150.7 -> 155.6 and 84.9 ->
// 86.9 ms)
template <typename T> struct dma_shape;
template <> struct dma_shape<float>  { static constexpr int bk = 8, pad = -1; };
template <> struct dma_shape<double> { static constexpr int bk = 8, pad = 0; };
template <> struct dma_shape<pxcf>   { static constexpr int bk = 8, pad = 0; };
template <> struct dma_shape<pxcd>   { static constexpr int bk = 4, pad = 10240; };

template <typename T, bool LDLT>
__global__ void __launch_bounds__( PXD_THREADS, 4 )
k_update_dma( const upd_task *__restrict__ tasks, int32_t ntasks, const dcblk *__restrict__ cb,
              const dblok *__restrict__ bk, T *L, T *U, uint64_t *__restrict__ stamps, int prio )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    constexpr int      BK = dma_shape<T>::bk, NBUF = 3;
    constexpr int      BM = upd_rows<T>::value, BN = PXD_UPD_BN;
    constexpr uint32_t ES = sizeof( T );
    constexpr int      LPE = ( ES == 8 ) ? 2 : 1;            // lanes per element of a load of one row per lane
    constexpr int      WR  = BM / 4, RB = WR / 16;           // rows and 16-row blocks per wave
    constexpr bool     OWN = ( ES < 16 );                    // a wave loads its own rows (else all rows of its k)
    constexpr bool     W16 = ( ES == 8 );                    // 16 bytes per lane where the rows allow it
    constexpr int      QW  = BK / 4;                         // ... loads of A per stage and wave
    constexpr int      QN  = OWN ? BK : BK / 4;              // and one row per lane (pair)
    constexpr int      AST = W16 ? WR : BM + ( ES == 4 ? 16 : 0 );   // elements between the k values of A
                                                             // (float: 64 bytes more, else two meet in a bank)
    constexpr int      SA0 = W16 ? BK * WR : WR;             // ... and between the waves' rows
    constexpr int      ASZ = W16 ? BK * BM : BK * AST;       // elements of A in a stage
    constexpr int      BL  = ( ES == 4 ) ? 4 : 16;           // bytes per lane of a load of B
    constexpr int      BE  = BL / (int)ES, KB = 64 * BE / BN;   // elements per lane, k values per load
    constexpr int      QB  = BK / KB / 4;                    // loads of B per stage and wave
    static_assert( BK % 4 == 0 && QB * KB * 4 == BK, "stages of whole 4-k products" );
    static_assert( !W16 || WR * ES == 256, "16 lanes hold a wave's rows in 16 bytes each" );
    static_assert( sizeof( search_keys ) <= ASZ * ES, "search keys fit in one A buffer" );
    constexpr int DN = PXD_TRSM_NT * 16 + BK;
    constexpr int SE = ASZ + BK * BN;   // elements of a stage
    // one variable per stage (A, then B): the compiler tells loads into one
    // from reads of another only by the variable, and waits for all of them
    // where it cannot
    __shared__ __align__( 16 ) T stage0[SE];
    __shared__ __align__( 16 ) T stage1[SE];
    __shared__ __align__( 16 ) T stage2[SE];
    T *sD = nullptr;
    if constexpr ( LDLT ) {
        __shared__ T sDk[DN];
        sD = sDk;
    }
    auto buffer = [&]( auto bc ) -> T * {
        constexpr int b = decltype( bc )::value;
        if constexpr ( b == 0 ) return stage0;
        else if constexpr ( b == 1 ) return stage1;
        else return stage2;
    };
    search_keys &sk = *reinterpret_cast<search_keys *>( stage2 );

    const int32_t  ti      = xcd_task( blockIdx.x, ntasks );
    const upd_task t       = tasks[ti];
    const uint64_t t_stamp = stamp_begin( stamps );
    wave_priority( prio );
    const int     tid = threadIdx.x;
    const int     lane = tid & 63, w = __builtin_amdgcn_readfirstlane( tid >> 6 );
    const dcblk   c   = cb[t.cblk];
    const int32_t K   = c.lcolnum - c.fcolnum + 1;
    const int32_t lb  = cb[t.cblk + 1].fblok;
    const dblok   bb  = bk[t.blok];
    const int32_t N   = bb.lrownum - bb.frownum + 1;
    // U-side tile (LU): A = U^T rows after blok b, B = L rows of blok b, C = U
    const bool    uside = ( t.flags & 2 ) != 0;
    const T      *LA    = uside ? U : L;
    const T      *LB    = uside ? L : U;
    T            *LC    = uside ? U : L;
    const int32_t r0    = bb.rowoff + ( uside ? N : 0 );
    const int32_t Mr    = c.stride - r0;
    const int32_t F     = bb.fcblknm;
    const dcblk   cf    = cb[F];
    const int32_t Fn    = cf.lcolnum - cf.fcolnum + 1;
    const int32_t flb   = cb[F + 1].fblok;
    const int32_t colF0 = bb.frownum - cf.fcolnum + t.tn * BN;
    if ( bb.frownum < cf.fcolnum || bb.lrownum > cf.lcolnum ) {
        return;   // inconsistent structure: the host checks prevent this
    }
    const __amdgpu_buffer_rsrc_t rA = make_rsrc( LA + c.coefoff, (uint32_t)( (int64_t)c.stride * K * ES ) );
    const __amdgpu_buffer_rsrc_t rB = make_rsrc( LB + c.coefoff, (uint32_t)( (int64_t)c.stride * K * ES ) );
    const __amdgpu_buffer_rsrc_t rC = make_rsrc( LC + cf.coefoff, (uint32_t)( (int64_t)cf.stride * Fn * ES ) );

    stage_search_keys( sk, bk, t.blok, lb, cf.fblok, flb, tid );
    if constexpr ( LDLT ) {
        for ( int32_t i = tid; i < DN; i += PXD_THREADS ) {
            sD[i] = ( i < K ) ? L[c.coefoff + (int64_t)i * ( K + 1 )] : (T)0;
        }
    }
    __syncthreads();

    // the lane's row of the tile (complex double: every wave all rows, its own
    // the same place): its blok's stacked offset, its place in the blok and
    // the byte stride between its columns in the source, its place in F
    const int r0w   = t.tm * BM + ( OWN ? WR * w : 0 );
    int32_t   boff = 0, ain = 0;
    uint32_t  astep = 0, dst = PXD_OOB, dld = 0;
    {
        const int32_t r = r0w + lane / LPE;
        if ( r < Mr ) {
            const int32_t s  = r0 + r;
            const dblok   ib = bk[search_row( sk, bk, t.blok, lb, s )];
            const int32_t g  = ib.frownum + ( s - ib.rowoff );
            boff  = ib.rowoff;
            ain   = s - ib.rowoff;
            astep = (uint32_t)( ib.lrownum - ib.frownum + 1 ) * ES;
            const dblok fb = bk[search_grow( sk, bk, cf.fblok, flb, g )];
            if ( g >= fb.frownum && g <= fb.lrownum ) {
                dst = (uint32_t)( fb.rowoff * Fn + ( g - fb.frownum ) ) * ES;
                dld = (uint32_t)( fb.lrownum - fb.frownum + 1 ) * ES;
            }
        }
    }
    // the wave's rows in one blok: the row of lane 0 and the last one inside
    // the update (rows past it read what follows, and are dropped)
    const int  lastl = LPE * min( WR - 1, Mr - 1 - r0w );
    const bool wide  = W16 && lastl >= 0 &&
                      __builtin_amdgcn_readfirstlane( boff ) == __builtin_amdgcn_readlane( boff, max( 0, lastl ) );
    uint32_t ao = PXD_OOB;
    int      ak0 = OWN ? 0 : w;   // the lane's first k value of a stage
    if ( wide ) {
        ak0   = lane >> 4;
        astep = __builtin_amdgcn_readfirstlane( astep );
        ao    = (uint32_t)( __builtin_amdgcn_readfirstlane( boff ) * K + __builtin_amdgcn_readfirstlane( ain ) ) * ES +
             16 * ( lane & 15 ) + ak0 * astep;
        astep *= 4;
    }
    else if ( r0w + lane / LPE < Mr ) {
        ao = (uint32_t)( boff * K + ain ) * ES + 4 * ( lane % LPE ) + ak0 * astep;
        if constexpr ( !OWN ) astep *= 4;
    }
    // the lane's columns of B, at the k values KB (w + 4 q) + lane / (lanes per k)
    const int32_t  nvalid = min( BN, N - t.tn * BN );
    const int      bcol   = BE * ( lane % ( BN / BE ) ), bk0 = KB * w + lane / ( BN / BE );
    const uint32_t bstep  = (uint32_t)( 4 * KB * N ) * ES;
    uint32_t       bo     = (uint32_t)( bb.rowoff * K + t.tn * BN + bcol + bk0 * N ) * ES;

    // stage k0 into buffer b; the offsets advance from load to load, so that
    // no per-k products stay live across the loop
    auto dma = [&]( auto bc, int32_t k0 ) {
        T         *dA   = buffer( bc ) + ( OWN ? SA0 * w : AST * w );
        T         *dB   = buffer( bc ) + ASZ + KB * BN * w;
        const bool full = ( k0 + BK <= K );
        if ( W16 && wide ) {
#pragma unroll
            for ( int q = 0; q < QW; q++ ) {
                load_lds<16>( rA, dA + 4 * q * AST, ( full || k0 + 4 * q + ak0 < K ) ? ao : PXD_OOB );
                ao += astep;
            }
        }
        else {
#pragma unroll
            for ( int q = 0; q < QN; q++ ) {
                constexpr int KS = OWN ? 1 : 4;
                load_lds<OWN ? 4 : 16>( rA, dA + KS * q * AST, ( full || k0 + KS * q + ak0 < K ) ? ao : PXD_OOB );
                ao += astep;
            }
        }
#pragma unroll
        for ( int q = 0; q < QB; q++ ) {
            load_lds<BL>( rB, dB + 4 * KB * BN * q, ( full || k0 + 4 * KB * q + bk0 < K ) ? bo : PXD_OOB );
            bo += bstep;
        }
    };

    acc_t acc[RB][4];
#pragma unroll
    for ( int i = 0; i < RB; i++ )
#pragma unroll
        for ( int j = 0; j < 4; j++ ) acc[i][j] = M::zero();

    // End of a stage: this wave's loads of the next stage are in LDS (those of
    // the one after, issued since, may be in flight), and after the barrier
    // every wave's are.  The products stay ahead of it, so every LDS read of
    // the stage has returned.  Not __syncthreads(): its fence waits for the
    // loads in flight too (vmcnt 0), which leaves no stage ahead of the
    // products.
    auto next_stage = [&]() {
        __builtin_amdgcn_sched_barrier( 0 );
        static_assert( QN + QB < 16, "4 bits of vmcnt" );
        if ( W16 && wide ) {
            __builtin_amdgcn_s_waitcnt( 0x0F70 | ( QW + QB ) );   // vmcnt: the loads of one stage
        }
        else {
            __builtin_amdgcn_s_waitcnt( 0x0F70 | ( QN + QB ) );
        }
        bare_barrier();
        __builtin_amdgcn_sched_barrier( 0 );
    };

    // 16-byte reads of B: VB columns next to each other feed VB of the four
    // column tiles (tile j holds the columns 16 VB (j / VB) + VB r + j % VB),
    // and of A in the 8-byte types: block i holds the rows 2 r + i of the
    // wave's (elsewhere 16 i + r)
    constexpr int VB = 16 / ES;
    struct __align__( 16 ) bvec { T e[VB]; };
    static_assert( RB == VB, "a lane's rows fill 16 bytes" );
    const int     lr = lane & 15, lg = lane >> 4;
    const int32_t ns = ( K + BK - 1 ) / BK;
    // stage s from buffer b = s % NBUF, with the loads of stage s + NBUF - 1
    // into the buffer that stage s - 1 read (issued past the last stage too,
    // as out-of-range loads, so that every stage leaves the same count)
    auto stage = [&]( auto bc, int32_t s ) {
        constexpr int b  = decltype( bc )::value;
        const T      *SA = buffer( bc ) + SA0 * w + ( W16 ? VB : 1 ) * lr;
        const T      *SB = buffer( bc ) + ASZ + VB * lr;
        bvec          av[BK / 4], bv[BK / 4][4 / VB];
#pragma unroll
        for ( int ks = 0; ks < BK / 4; ks++ ) {
            if constexpr ( W16 ) {
                av[ks] = *(const bvec *)&SA[( 4 * ks + lg ) * AST];
            }
            else {
#pragma unroll
                for ( int i = 0; i < RB; i++ ) av[ks].e[i] = SA[( 4 * ks + lg ) * AST + 16 * i];
            }
#pragma unroll
            for ( int j = 0; j < 4 / VB; j++ ) bv[ks][j] = *(const bvec *)&SB[( 4 * ks + lg ) * BN + 16 * VB * j];
        }
        if constexpr ( LDLT ) {
#pragma unroll
            for ( int ks = 0; ks < BK / 4; ks++ ) {
                const T d = sD[s * BK + 4 * ks + lg];
#pragma unroll
                for ( int i = 0; i < RB; i++ ) av[ks].e[i] = av[ks].e[i] * d;
            }
        }
        dma( std::integral_constant<int, ( b + NBUF - 1 ) % NBUF>{}, ( s + NBUF - 1 ) * BK );
#pragma unroll
        for ( int ks = 0; ks < BK / 4; ks++ )
#pragma unroll
            for ( int i = 0; i < RB; i++ )
#pragma unroll
                for ( int j = 0; j < 4; j++ ) acc[i][j] = M::mma( bv[ks][j / VB].e[j % VB], av[ks].e[i], acc[i][j] );
        next_stage();
    };
    dma( std::integral_constant<int, 0>{}, 0 );
    dma( std::integral_constant<int, 1>{}, BK );
    next_stage();
    for ( int32_t s = 0; s < ns; s += NBUF ) {
        stage( std::integral_constant<int, 0>{}, s );
        if ( s + 1 < ns ) stage( std::integral_constant<int, 1>{}, s + 1 );
        if ( s + 2 < ns ) stage( std::integral_constant<int, 2>{}, s + 2 );
    }
    // the loads past the last stage land before the workgroup's LDS is given up
    __builtin_amdgcn_s_waitcnt( 0x0F70 );

    // C -= acc, a slab of 16 columns at a time through the wave's own part of
    // the stage buffers, so that a lane owns a row (LPR lanes to a row) and a
    // memory instruction covers WR consecutive rows of one column
    const bool    atomic = ( t.flags & 1 );
    constexpr int LPR = 64 / WR, CPL = 16 / LPR;             // lanes per row, columns per lane
    constexpr int CH  = ( CPL < 8 ) ? CPL : 8;               // columns in flight
    static_assert( WR * 17 <= SE, "a wave's slab fits in a stage buffer" );
    T *sE = ( w == 0 ) ? stage0 : ( w == 1 ) ? stage1 : stage2;
    bare_barrier();
    if constexpr ( 2 * WR * 17 <= SE ) {
        sE = ( w == 3 ) ? stage2 + WR * 17 : sE;
    }
    else {
        __shared__ T slab3[WR * 17];
        sE = ( w == 3 ) ? slab3 : sE;
    }
    const int      erow = lane / LPR, epart = lane % LPR;
    const uint32_t ro = __shfl( dst, ( OWN ? 0 : WR * w ) + ( OWN ? LPE : 1 ) * erow );
    const uint32_t rl = __shfl( dld, ( OWN ? 0 : WR * w ) + ( OWN ? LPE : 1 ) * erow );
#pragma unroll
    for ( int j = 0; j < 4; j++ ) {
#pragma unroll
        for ( int i = 0; i < RB; i++ )
#pragma unroll
            for ( int v = 0; v < 4; v++ ) sE[( W16 ? VB * lr + i : 16 * i + lr ) * 17 + M::row( lane, v )] = M::get( acc[i][j], v );
        __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
#pragma unroll
        for ( int h = 0; h < CPL; h += CH ) {
            uint32_t off[CH];
            T        val[CH];
#pragma unroll
            for ( int q = 0; q < CH; q++ ) {
                const int m  = CPL * epart + h + q;
                const int cc = 16 * VB * ( j / VB ) + VB * m + j % VB;
                off[q] = ( ro != PXD_OOB && cc < nvalid ) ? ro + (uint32_t)( colF0 + cc ) * rl : PXD_OOB;
                val[q] = sE[erow * 17 + m];
            }
            if ( atomic ) {
#pragma unroll
                for ( int q = 0; q < CH; q++ ) {
                    if ( off[q] != PXD_OOB ) px_atomic_add( LC + cf.coefoff + off[q] / ES, -val[q] );
                }
            }
            else {
                T old[CH];
#pragma unroll
                for ( int q = 0; q < CH; q++ ) old[q] = bufio<T>::load( rC, off[q] );
#pragma unroll
                for ( int q = 0; q < CH; q++ ) bufio<T>::store( old[q] - val[q], rC, off[q] );
            }
        }
        __builtin_amdgcn_fence( __ATOMIC_RELEASE, "wavefront" );
        __builtin_amdgcn_wave_barrier();
        __builtin_amdgcn_fence( __ATOMIC_ACQUIRE, "wavefront" );
    }
    stamp_end( stamps, ti, t_stamp );
}
