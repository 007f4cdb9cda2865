// kernels_panel.hpp -- the diagonal tiles of a level: factorization and
// explicit inverse, several workgroups per cblk, for the three
// factorizations and the four arithmetics.
//
// One launch per level holds two kinds of tasks:
//
//   rows      one per 32-row block p of a cblk's n x n diagonal tile.  For
//             j = 0 .. p-1 it forms X(p,j) = (T(p,j) - sum_{k<j} X(p,k)
//             L(j,k)^T) D_j^T with D_j the inverse of diagonal block j, then
//             it eliminates its own diagonal block and publishes D_p.  LU
//             runs the same recurrence twice, on L and on U^T (the other
//             side's blocks in the sum, both inverses of a diagonal block).
//   columns   one per 32-column block J but the last (and per side for LU)
//             of the inverse: X(K,J) = -D_K sum_{i=J}^{K-1} L(K,i) X(i,J) for
//             K = J+1, J+2, ..., each as soon as row K has it.
//
// What bounds it: latency.  A tile is a chain of its diagonal blocks, and
// each link is the exchange of D_j between two workgroups (a store and two
// loads that cross the XCDs), three 32 x 32 products and the 32 elimination
// steps.  So the rows work ahead: while row p waits for D_j it sums column
// j+1 over k < j, and the diagonal block's own sum is kept up to date with
// every X(p,j).  A column ends one product after the last row.  Operands go
// from memory to the matrix cores without LDS (a fragment load covers 16
// consecutive rows of 4 columns), and the only tiles in LDS are the two or
// three that the step transposes or eliminates, so that a task fits next to
// the update workgroups of the other stream (9 KiB in float, 18 KiB in
// double, against 8.4 KiB per block row before: a ten-block tile in double
// took 101 KiB and waited for a CU almost free of updates).
//
// Exchange between the workgroups: blocks that others read are stored and
// loaded with agent-scope relaxed atomics (panel_st, panel_ld), which are
// coherent across the XCDs by themselves.  flag[p] counts the blocks of row
// p that are out: j + 1 after X(p,j), p + 1 after D_p.  A task waits only for
// rows before it in the list, and workgroups start in list order, so the
// first unfinished one can always run; every wait is also bounded
// (panel_wait).  A row's own earlier blocks are read back with plain loads:
// they were stored by the same workgroup before a barrier.
#pragma once
#include "kernels_mfma.hpp"

// A row block (J < 0) or a column of the inverse (J >= 0) of cblk's tile;
// flag0 is the place of the cblk's first row in the flags, nblk its rows.
struct pan_task {
    int32_t cblk;
    int32_t p;       // row block; column tasks: J, plus PXD_PAN_COL (U side: and PXD_PAN_USIDE)
    int32_t flag0;
    int32_t nblk;
};
#define PXD_PAN_COL   ( 1 << 16 )
#define PXD_PAN_USIDE ( 1 << 17 )

// Start of a factorization: counters, the pivot threshold (in memory, so that a
// captured factorization serves every matrix of the structure) and the flags.
__global__ void
k_fact_begin( int *scratch, double *dthresh, double thresh, int *flags, int64_t nflags )
{
    const int64_t i = (int64_t)blockIdx.x * blockDim.x + threadIdx.x;
    if ( i < nflags ) flags[i] = 0;
    if ( i < 4 ) scratch[i] = 0;
    if ( i == 0 ) *dthresh = thresh;
}

enum { PAN_LLT = 0, PAN_LDLT = 1, PAN_LU = 2 };

// Bound of one wait in ticks of the constant clock (wall_clock64), set on
// every device from its clock rate when an engine context is created (2 s
// by default, engine option "wait_ms").
__constant__ uint64_t pxd_wait_ticks = 200000000ull;

// Every wave waits for itself (no barrier): *f >= target, or the bound, or a
// bound that expired elsewhere (*err), after which every wait falls through.
__device__ inline void
panel_wait( const int *f, int target, int *err )
{
    auto get = [&]( const int *q ) {
        return __builtin_amdgcn_readfirstlane( __hip_atomic_load( q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT ) );
    };
    if ( get( f ) < target ) {
        const uint64_t t0 = (uint64_t)wall_clock64();
        while ( get( f ) < target && get( err ) == 0 ) {
            if ( (uint64_t)wall_clock64() - t0 > pxd_wait_ticks ) {
                __hip_atomic_store( err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
                break;
            }
            __builtin_amdgcn_s_sleep( 1 );
        }
    }
    __atomic_signal_fence( __ATOMIC_SEQ_CST );   // the loads of the block stay after the wait
}

// Every thread's panel_st are complete (vmcnt 0) before the barrier, so the
// flag is stored after all of them.
__device__ inline void
panel_publish( int *f, int value, int tid )
{
    __atomic_signal_fence( __ATOMIC_SEQ_CST );
    __builtin_amdgcn_s_waitcnt( 0 );
    __syncthreads();
    if ( tid == 0 ) {
        __hip_atomic_store( f, value, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
    }
}

template <typename T>
__device__ inline T
panel_ld( const T *p )
{
    if constexpr ( std::is_same<T, pxcf>::value ) {
        return __builtin_bit_cast( pxcf, __hip_atomic_load( (const unsigned long long *)p, __ATOMIC_RELAXED,
                                                            __HIP_MEMORY_SCOPE_AGENT ) );
    }
    else if constexpr ( std::is_same<T, pxcd>::value ) {
        return pxcd( __hip_atomic_load( &p->re, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT ),
                     __hip_atomic_load( &p->im, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT ) );
    }
    else {
        return __hip_atomic_load( p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
    }
}
template <typename T>
__device__ inline void
panel_st( T *p, T v )
{
    if constexpr ( std::is_same<T, pxcf>::value ) {
        __hip_atomic_store( (unsigned long long *)p, __builtin_bit_cast( unsigned long long, v ), __ATOMIC_RELAXED,
                            __HIP_MEMORY_SCOPE_AGENT );
    }
    else if constexpr ( std::is_same<T, pxcd>::value ) {
        __hip_atomic_store( &p->re, v.re, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
        __hip_atomic_store( &p->im, v.im, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
    }
    else {
        __hip_atomic_store( p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT );
    }
}

// One operand of a 32 x 32 product: f[s] = element (row, 4 s + lane / 16) of
// a block whose element (i, l) is at base[i * rs + l * cs].  The result of
// the product of rows X and rows Y is sum_l X(i, l) Y(j, l).
template <typename T, bool AGENT>
__device__ inline void
pan_frag( T ( &f )[PXD_NB / 4], const T *base, int64_t rs, int64_t cs, int row, int lane )
{
    const T *p = base + row * rs + ( lane >> 4 ) * cs;
#pragma unroll
    for ( int s = 0; s < PXD_NB / 4; s++ ) {
        f[s] = AGENT ? panel_ld( p + 4 * s * cs ) : p[4 * s * cs];
    }
}
// the same from a tile in LDS, s[col][row]
template <typename T>
__device__ inline void
pan_frag_lds( T ( &f )[PXD_NB / 4], const T ( *s )[PXD_NB + 1], int row, int lane )
{
#pragma unroll
    for ( int s4 = 0; s4 < PXD_NB / 4; s4++ ) f[s4] = s[4 * s4 + ( lane >> 4 )][row];
}
// acc +- X Y^T
template <typename T, bool SUB>
__device__ inline void
pan_mma( typename mfma16<T>::acc_t &acc, const T ( &a )[PXD_NB / 4], const T ( &b )[PXD_NB / 4] )
{
#pragma unroll
    for ( int s = 0; s < PXD_NB / 4; s++ ) acc = mfma16<T>::mma( SUB ? -a[s] : a[s], b[s], acc );
}

// Column J of the inverse of a cblk's lower triangle A (U side: of U_kk^T).
template <typename T>
__device__ inline void
panel_inverse_column( const T *A, T *LI, int32_t n, int J, int nblk, const int *flag, int *err, T ( *sS )[PXD_NB + 1],
                      int tid )
{
    typedef mfma16<T>         M;
    typedef typename M::acc_t acc_t;
    constexpr int NB = PXD_NB;
    const int     lane = tid & 63, w = tid >> 6, lr = lane & 15;
    const int     qr = w >> 1, qc = w & 1;
    const int64_t ld = n;
    panel_wait( flag + J, J + 1, err );
    for ( int K = J + 1; K < nblk; K++ ) {
        const int bk = min( NB, n - NB * K );
        const int ra = min( 16 * qr + lr, bk - 1 );   // rows past the tile repeat the last one
        panel_wait( flag + K, K, err );
        acc_t acc = M::zero();
        {
            T a[NB / 4], b[NB / 4];
            pan_frag<T, true>( a, A + NB * K + (int64_t)( NB * J ) * ld, 1, ld, ra, lane );
            pan_frag<T, true>( b, LI + NB * J + (int64_t)( NB * J ) * ld, ld, 1, 16 * qc + lr, lane );
            pan_mma<T, true>( acc, a, b );
        }
        for ( int i = J + 1; i < K; i++ ) {
            T a[NB / 4], b[NB / 4];
            pan_frag<T, true>( a, A + NB * K + (int64_t)( NB * i ) * ld, 1, ld, ra, lane );
            pan_frag<T, false>( b, LI + NB * i + (int64_t)( NB * J ) * ld, ld, 1, 16 * qc + lr, lane );
            pan_mma<T, true>( acc, a, b );
        }
        __syncthreads();   // every wave has read the previous sS
#pragma unroll
        for ( int v = 0; v < 4; v++ ) sS[16 * qr + M::row( lane, v )][16 * qc + lr] = M::get( acc, v );
        __syncthreads();
        panel_wait( flag + K, K + 1, err );
        // X(K,J) = D_K S; sS holds S by rows, so its columns are the second operand's rows
        T d[NB / 4], b[NB / 4];
#pragma unroll
        for ( int s = 0; s < NB / 4; s++ ) {
            const int l = 4 * s + ( lane >> 4 );
            const T   x = panel_ld( LI + NB * K + ra + (int64_t)( NB * K + min( l, bk - 1 ) ) * ld );
            d[s] = ( l < bk ) ? x : (T)0;
        }
        pan_frag_lds<T>( b, sS, 16 * qc + lr, lane );
        acc = M::zero();
        pan_mma<T, false>( acc, d, b );
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
            const int r = 16 * qr + M::row( lane, v );
            if ( r < bk ) LI[NB * K + r + (int64_t)( NB * J + 16 * qc + lr ) * ld] = M::get( acc, v );
        }
        __syncthreads();   // X(K,J) is there for the next rows
    }
}

template <typename T, int KIND>
__global__ void __launch_bounds__( PXD_THREADS )
k_panel( const pan_task *__restrict__ tasks, const dcblk *__restrict__ cb, T *L, T *U, T *DL, T *DU,
         const double *__restrict__ thresh,
         int *__restrict__ npiv, int *flags, int *err, uint64_t *__restrict__ stamps, int prio )
{
    typedef mfma16<T>                 M;
    typedef typename M::acc_t         acc_t;
    typedef typename px_real<T>::type R;
    constexpr int  NB = PXD_NB;
    constexpr bool LU = ( KIND == PAN_LU );
    constexpr int  NS = LU ? 2 : 1;      // sides
    constexpr int  NU = NB * NB / PXD_THREADS;
    typedef T tile_t[NB][NB + 1];        // [col][row]
    __shared__ tile_t sX;                // X(p,j); the diagonal block
    __shared__ tile_t sY;                // LDL^T: X(p,j) D^{-1}; LU: the U side's X(p,j); the diagonal block's inverse
    T( *sZ )[NB + 1] = nullptr;          // LU: the second inverse
    if constexpr ( LU ) {
        __shared__ tile_t sZ_lu;
        sZ = sZ_lu;
    }
    __shared__ T      sD[NB];

    const pan_task tk      = tasks[blockIdx.x];
    const uint64_t t_stamp = stamp_begin( stamps );
    wave_priority( prio );
    const dcblk   c   = cb[tk.cblk];
    const int32_t n   = c.lcolnum - c.fcolnum + 1;
    const int64_t ld  = n;
    const int     tid = threadIdx.x;
    T            *A   = L + c.coefoff;    // n x n, ld n
    T            *AU  = LU ? U + c.coefoff : nullptr;
    T            *IL  = DL + c.dinvoff;
    T            *IU  = LU ? DU + c.dinvoff : IL;
    int          *flag = flags + tk.flag0;

    if ( tk.p & PXD_PAN_COL ) {
        const bool us = LU && ( tk.p & PXD_PAN_USIDE );
        panel_inverse_column<T>( us ? AU : A, us ? IU : IL, n, tk.p & ( PXD_PAN_COL - 1 ), tk.nblk, flag, err, sX, tid );
        stamp_end( stamps, blockIdx.x, t_stamp );
        return;
    }

    const int     lane = tid & 63, w = tid >> 6, lr = lane & 15;
    const int     qr = w >> 1, qc = w & 1;       // the wave's 16 x 16 quadrant of every product
    const int     p  = tk.p;
    const int32_t R0 = NB * p;
    const int32_t bs = min( NB, n - R0 );
    const int     ra = min( 16 * qr + lr, bs - 1 );   // operand rows past the tile repeat the last one
    const int     rb = min( 16 * qc + lr, bs - 1 );

    // T(p,j) (LU: L side, and U^T side = the upper part of the L tile plus the
    // U tile).  The products are summed from zero and subtracted from it once:
    // subtracted one by one they would be rounded at the size of T.
    T    t[NS][4];
    auto load_tile = [&]( int j ) {
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
            const int     r  = min( 16 * qr + M::row( lane, v ), bs - 1 );
            const int64_t cc = NB * j + 16 * qc + lr;
            t[0][v] = A[R0 + r + cc * ld];
            if constexpr ( LU ) {
                t[NS - 1][v] = A[cc + ( R0 + r ) * ld] + AU[R0 + r + cc * ld];
            }
        }
    };
    // acc += X(p,k) L(j,k)^T for one k: own blocks by plain loads (LDL^T: X
    // is the transpose above the diagonal), row j's across the XCDs
    auto sub_block = [&]( acc_t ( &acc )[NS], int j, int k ) {
        T a[NB / 4], b[NB / 4];
        if constexpr ( KIND == PAN_LDLT ) {
            pan_frag<T, false>( a, A + NB * k + R0 * ld, ld, 1, ra, lane );
        }
        else {
            pan_frag<T, false>( a, A + R0 + (int64_t)( NB * k ) * ld, 1, ld, ra, lane );
        }
        pan_frag<T, true>( b, ( LU ? AU : A ) + NB * j + (int64_t)( NB * k ) * ld, 1, ld, 16 * qc + lr, lane );
        if constexpr ( LU ) {
            T a2[NB / 4], b2[NB / 4];
            pan_frag<T, false>( a2, AU + R0 + (int64_t)( NB * k ) * ld, 1, ld, ra, lane );
            pan_frag<T, true>( b2, A + NB * j + (int64_t)( NB * k ) * ld, 1, ld, 16 * qc + lr, lane );
            pan_mma<T, false>( acc[NS - 1], a2, b2 );
        }
        pan_mma<T, false>( acc[0], a, b );
    };

    // the diagonal block's sum (symmetric forms: the lower part counts)
    acc_t accd = M::zero();
    T     td[4];
#pragma unroll
    for ( int v = 0; v < 4; v++ ) {
        const int r = min( 16 * qr + M::row( lane, v ), bs - 1 ), cc = rb;
        T         x = A[R0 + r + ( R0 + cc ) * ld];
        if constexpr ( LU ) {
            const T y = AU[R0 + cc + ( R0 + r ) * ld];
            x = ( r < cc ) ? x + y : x;
        }
        td[v] = x;
    }
    acc_t acc[NS];
#pragma unroll
    for ( int s = 0; s < NS; s++ ) acc[s] = M::zero();
    if ( p > 0 ) {
        load_tile( 0 );
    }
    for ( int j = 0; j < p; j++ ) {
        if ( j > 0 ) {
            // the k = j - 1 term: X(p,j-1) is still in LDS
            panel_wait( flag + j, j, err );
            T a[NB / 4], b[NB / 4];
            pan_frag<T, true>( b, ( LU ? AU : A ) + NB * j + (int64_t)( NB * ( j - 1 ) ) * ld, 1, ld, 16 * qc + lr, lane );
            pan_frag_lds<T>( a, sX, 16 * qr + lr, lane );
            if constexpr ( LU ) {
                T a2[NB / 4], b2[NB / 4];
                pan_frag<T, true>( b2, A + NB * j + (int64_t)( NB * ( j - 1 ) ) * ld, 1, ld, 16 * qc + lr, lane );
                pan_frag_lds<T>( a2, sY, 16 * qr + lr, lane );
                pan_mma<T, false>( acc[NS - 1], a2, b2 );
            }
            pan_mma<T, false>( acc[0], a, b );
        }
        __syncthreads();   // every wave has read sX and sY
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
            const int r = 16 * qr + M::row( lane, v ), cc = 16 * qc + lr;
            sX[cc][r] = t[0][v] - M::get( acc[0], v );
            if constexpr ( LU ) sY[cc][r] = t[NS - 1][v] - M::get( acc[NS - 1], v );
        }
        // ahead of D_j: the next column's terms up to k = j - 1
        if ( j + 1 < p ) {
            load_tile( j + 1 );
#pragma unroll
            for ( int s = 0; s < NS; s++ ) acc[s] = M::zero();
            panel_wait( flag + j + 1, j, err );
            for ( int k = 0; k < j; k++ ) sub_block( acc, j + 1, k );
        }
        __syncthreads();   // the sums are in sX and sY
        panel_wait( flag + j, j + 1, err );
        acc_t x[NS];
        T     dinv = (T)1;
        {
            T a[NB / 4], b[NB / 4];
            pan_frag<T, true>( b, ( LU ? IU : IL ) + NB * j + (int64_t)( NB * j ) * ld, 1, ld, 16 * qc + lr, lane );
            if constexpr ( KIND == PAN_LDLT ) {
                dinv = (T)1 / panel_ld( A + ( NB * j + 16 * qc + lr ) * ( ld + 1 ) );
            }
            pan_frag_lds<T>( a, sX, 16 * qr + lr, lane );
            x[0] = M::zero();
            pan_mma<T, false>( x[0], a, b );
            if constexpr ( LU ) {
                pan_frag<T, true>( b, IL + NB * j + (int64_t)( NB * j ) * ld, 1, ld, 16 * qc + lr, lane );
                pan_frag_lds<T>( a, sY, 16 * qr + lr, lane );
                x[NS - 1] = M::zero();
                pan_mma<T, false>( x[NS - 1], a, b );
            }
        }
        __syncthreads();   // every wave has read the sums
#pragma unroll
        for ( int v = 0; v < 4; v++ ) {
            const int r = 16 * qr + M::row( lane, v ), cc = 16 * qc + lr;
            sX[cc][r] = M::get( x[0], v );
            if constexpr ( KIND == PAN_LDLT ) sY[cc][r] = M::get( x[0], v ) * dinv;
            if constexpr ( LU ) sY[cc][r] = M::get( x[NS - 1], v );
        }
        __syncthreads();
        // rows of L (and of U^T) for the others and the factor; the
        // transposes above the diagonal (D L^T, and LU's packed tiles) for
        // the factor alone
#pragma unroll
        for ( int u = 0; u < NU; u++ ) {
            const int r = tid % NB, cc = tid / NB + u * ( PXD_THREADS / NB );
            if ( r < bs ) {
                panel_st( A + R0 + r + ( NB * j + cc ) * ld, ( KIND == PAN_LDLT ) ? sY[cc][r] : sX[cc][r] );
                if constexpr ( LU ) panel_st( AU + R0 + r + ( NB * j + cc ) * ld, sY[cc][r] );
            }
            if constexpr ( KIND != PAN_LLT ) {
                if ( cc < bs ) {
                    A[NB * j + r + ( R0 + cc ) * ld] = LU ? sY[r][cc] : sX[r][cc];
                    if constexpr ( LU ) AU[NB * j + r + ( R0 + cc ) * ld] = sX[r][cc];
                }
            }
        }
        {
            T a[NB / 4], b[NB / 4];
            pan_frag_lds<T>( a, sX, 16 * qr + lr, lane );
            pan_frag_lds<T>( b, ( KIND == PAN_LLT ) ? sX : sY, 16 * qc + lr, lane );
            pan_mma<T, false>( accd, a, b );
        }
        panel_publish( flag + p, j + 1, tid );
    }

    // the diagonal block: elimination with the inverses built alongside
    T( *sA )[NB + 1] = sX;
    T( *sI )[NB + 1] = sY;
    __syncthreads();
#pragma unroll
    for ( int v = 0; v < 4; v++ ) {
        const int r = 16 * qr + M::row( lane, v ), cc = 16 * qc + lr;
        sA[cc][r] = ( r < bs && cc < bs && ( LU || r >= cc ) ) ? td[v] - M::get( accd, v ) : (T)0;
    }
#pragma unroll
    for ( int u = 0; u < NU; u++ ) {
        const int r = tid % NB, cc = tid / NB + u * ( PXD_THREADS / NB );
        sI[cc][r] = ( r == cc && r < bs ) ? (T)1 : (T)0;
        if constexpr ( LU ) sZ[cc][r] = ( r == cc && r < bs ) ? (T)1 : (T)0;
    }
    __syncthreads();
    const R tau = (R)*thresh;
    int     piv = 0;
    if ( w == 0 ) {
        piv = elim32<T, KIND != PAN_LLT, LU>( sA, sI, sZ, sD, bs, tau, lane );
    }
    __syncthreads();
    // Cholesky: L = U D^{1/2}, L^{-1} = D^{-1/2} U^{-1}.  LDL^T: L = U, the
    // diagonal holds D, the upper part D L^T (the unscaled columns).  LU: the
    // multipliers are scaled by the pivots, and (U^T)^{-1} = D^{-1} W_U; the
    // U tile gets the transpose of the packed block.
#pragma unroll
    for ( int u = 0; u < NU; u++ ) {
        const int     r = tid % NB, cc = tid / NB + u * ( PXD_THREADS / NB );
        const int64_t at = R0 + r + ( R0 + cc ) * ld, ta = R0 + cc + ( R0 + r ) * ld;
        if ( r >= bs || cc >= bs ) {
            continue;
        }
        if constexpr ( KIND == PAN_LLT ) {
            if ( r >= cc ) {
                const T sr = px_sqrt( sD[r] );
                A[at] = ( r == cc ) ? sr : sA[cc][r] / px_sqrt( sD[cc] );
                panel_st( IL + at, sI[cc][r] / sr );
            }
        }
        else if constexpr ( KIND == PAN_LDLT ) {
            if ( r > cc ) {
                A[at] = sA[cc][r] / sD[cc];
                A[ta] = sA[cc][r];
            }
            else if ( r == cc ) {
                panel_st( A + at, sD[cc] );
            }
            panel_st( IL + at, sI[cc][r] );
        }
        else {
            const T x = ( r > cc ) ? sA[cc][r] / sD[cc] : ( r == cc ) ? sD[cc] : sA[cc][r];
            A[at]  = x;
            AU[ta] = x;
            panel_st( IL + at, sI[cc][r] );
            panel_st( IU + at, ( r >= cc ) ? sZ[cc][r] / sD[r] : sZ[cc][r] );
        }
    }
    if ( tk.nblk > 1 ) {
        panel_publish( flag + p, p + 1, tid );
    }
    if ( tid == 0 && piv > 0 ) {
        atomicAdd( npiv, piv );
    }
    stamp_end( stamps, blockIdx.x, t_stamp );
}
