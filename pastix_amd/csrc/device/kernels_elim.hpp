// kernels_elim.hpp -- elimination of a 32 x 32 diagonal block, with the
// inverses of its triangular factors, by one wavefront in registers.
//
// The chain of diagonal blocks bounds the panels, and 32 elimination steps are
// most of a link.  With the block spread over four waves (one LDS round
// trip and one workgroup barrier per step) they took 10 to 13 us.
// Here the block is two 16-column halves, eliminated one after the other, and
// the products between them run on the matrix cores:
//
//   lane (r, g) holds row r of a 16 x 16 matrix at the columns M::row(lane, 0..3)
//   ("by rows").  The value of a row's pivot lane is a DPP broadcast within 16
//   lanes, the pivot column one across the four groups (two permlane swaps):
//   a step is register arithmetic alone.
//   A matrix held so is both operands of a product whose step s takes k =
//   M::row(lane, s), and the result of sum_s mma(x[s], y[s]) is Y X^T by rows.
//
// A step is the in-place one: column c of the matrix is done when its
// multipliers are out, and takes column c of the inverse from there on, so
// that one update serves the columns of both.
//
// Panel launches alone, four waves with a barrier per step against this: 100^3
// float 11.9 -> 8.4 ms, double 13.2 -> 10.1 ms; 64^3 LU float 6.3 -> 4.2 ms;
// 80^3 complex64 LDL^T 12.4 -> 8.7 ms; 50^3 complex128 LDL^T 7.0 -> 5.1 ms.
#pragma once
#include "mfma.hpp"

template <int G>
__device__ inline unsigned
group_word( unsigned x )
{
    // rows of 16 lanes (0 1 2 3) -> (a b a b) -> all G
    const auto p = __builtin_amdgcn_permlane32_swap( x, x, false, false );
    const unsigned h = ( G >> 1 ) ? p[1] : p[0];
    const auto q = __builtin_amdgcn_permlane16_swap( h, h, false, false );
    return ( G & 1 ) ? q[1] : q[0];
}
template <int C>
__device__ inline unsigned
lane_word( unsigned x )
{
    return (unsigned)__builtin_amdgcn_update_dpp( 0, (int)x, 0x150 + C, 0xf, 0xf, true );   // row_newbcast
}
template <typename T> struct word_array { unsigned w[sizeof( T ) / 4]; };

// the values of lane group G in every group
template <int G, typename T>
__device__ inline T
group_bcast( T x )
{
    word_array<T> a = __builtin_bit_cast( word_array<T>, x );
#pragma unroll
    for ( unsigned i = 0; i < sizeof( T ) / 4; i++ ) a.w[i] = group_word<G>( a.w[i] );
    return __builtin_bit_cast( T, a );
}
// the value of lane C of the 16 in all of them
template <int C, typename T>
__device__ inline T
lane_bcast( T x )
{
    word_array<T> a = __builtin_bit_cast( word_array<T>, x );
#pragma unroll
    for ( unsigned i = 0; i < sizeof( T ) / 4; i++ ) a.w[i] = lane_word<C>( a.w[i] );
    return __builtin_bit_cast( T, a );
}
template <typename T>
__device__ inline T
elim_sel( bool c, T a, T b )
{
    if constexpr ( std::is_same<T, typename px_real<T>::type>::value ) {
        return c ? a : b;
    }
    else {
        return T( c ? a.re : b.re, c ? a.im : b.im );
    }
}

// Y X^T by rows
template <typename T>
__device__ inline void
elim_prod( T ( &p )[4], const T ( &x )[4], const T ( &y )[4] )
{
    typedef mfma16<T> M;
    auto acc = M::zero();
#pragma unroll
    for ( int s = 0; s < 4; s++ ) acc = M::mma( x[s], y[s], acc );
#pragma unroll
    for ( int s = 0; s < 4; s++ ) p[s] = M::get( acc, s );
}

// Steps C .. 15 of the elimination of a 16 x 16 matrix of bs columns: x by
// rows (LU: y its transpose).  On return x holds the inverse of the unit lower
// factor up to the diagonal (LU: U above it; y: the inverse of U~, U11^T = U~
// D), m (n) the multipliers times their pivots below the diagonal, di the
// reciprocal pivots of the lane's columns.  A pivot below tau becomes tau
// (Cholesky) or tau with the sign of its real part.
template <typename T, bool SIGN, bool LU, int C>
__device__ inline void
elim16( T ( &x )[4], T ( &m )[4], T ( &y )[4], T ( &n )[4], T ( &di )[4], T *sD, int bs,
        typename px_real<T>::type tau, int lane, int &piv )
{
    typedef mfma16<T>                 M;
    typedef typename px_real<T>::type R;
    if constexpr ( C < 16 ) {
        if ( C >= bs ) {
            return;
        }
        constexpr bool F32 = sizeof( R ) == 4;               // column C's group and register
        constexpr int  G = F32 ? C >> 2 : C & 3, V = F32 ? C & 3 : C >> 2;
        const int  r   = lane & 15;
        const bool act = r > C, own = ( lane >> 4 ) == G;
        const T    col = group_bcast<G>( x[V] );
        T          d   = lane_bcast<C>( col );
        if ( px_abs( d ) < tau ) {
            d = ( SIGN && px_re( d ) < (R)0 ) ? (T)-tau : (T)tau;
            piv++;
        }
        if ( lane == 0 ) {
            sD[C] = d;
        }
        const T rinv = (T)1 / d, t = col * rinv;
        // column C of the inverse starts as the identity's
        const bool inv = own && r >= C;
        const T    unit = elim_sel( r == C, (T)1, (T)0 );
        m[V]  = elim_sel( own && act, x[V], m[V] );
        di[V] = elim_sel( own, rinv, di[V] );
        x[V]  = elim_sel( inv, unit, x[V] );
#pragma unroll
        for ( int u = 0; u < 4; u++ ) x[u] = elim_sel( act, x[u] - t * lane_bcast<C>( x[u] ), x[u] );
        if constexpr ( LU ) {
            const T tu = group_bcast<G>( y[V] ) * rinv;
            n[V] = elim_sel( own && act, y[V], n[V] );
            y[V] = elim_sel( inv, unit, y[V] );
#pragma unroll
            for ( int u = 0; u < 4; u++ ) y[u] = elim_sel( act, y[u] - tu * lane_bcast<C>( y[u] ), y[u] );
        }
        elim16<T, SIGN, LU, C + 1>( x, m, y, n, di, sD, bs, tau, lane, piv );
    }
}

// The block in LDS (s[col][row], zero beyond bs rows and columns; symmetric
// forms: the lower part counts) by the 64 lanes of one wave.  On return sA
// holds the multipliers times their pivots below the diagonal and (LU) U
// above it, sI the inverse of the unit lower factor, sZ (LU) that of U~, sD
// the pivots; the result counts the replaced ones.
template <typename T, bool SIGN, bool LU>
__device__ inline int
elim32( T ( *sA )[PXD_NB + 1], T ( *sI )[PXD_NB + 1], T ( *sZ )[PXD_NB + 1], T *sD, int bs,
        typename px_real<T>::type tau, int lane )
{
    typedef mfma16<T> M;
    const int r = lane & 15;
    int       piv = 0;
    auto at = [&]( int i, int j ) { return ( LU || i >= j ) ? sA[j][i] : sA[i][j]; };
    T x1[4], m1[4], y1[4], n1[4], d1[4];
#pragma unroll
    for ( int u = 0; u < 4; u++ ) {
        const int c = M::row( lane, u );
        x1[u] = at( r, c );
        y1[u] = LU ? at( c, r ) : (T)0;
        m1[u] = n1[u] = d1[u] = (T)0;
    }
    elim16<T, SIGN, LU, 0>( x1, m1, y1, n1, d1, sD, bs, tau, lane, piv );
    T w1[4], z1[4];
#pragma unroll
    for ( int u = 0; u < 4; u++ ) {
        const int  c  = M::row( lane, u );
        const bool in = c <= r && r < bs;   // rows past the block are zero
        w1[u] = elim_sel( in, x1[u], (T)0 );
        z1[u] = LU ? elim_sel( in, y1[u], (T)0 ) : (T)0;
        sI[c][r] = w1[u];
        if constexpr ( LU ) sZ[c][r] = z1[u];
        if ( c < r ) sA[c][r] = m1[u];
        if ( LU && c > r ) sA[c][r] = x1[u];
    }
    if ( bs > 16 ) {
        T a[4], b[4], x21[4], u21[4], y21[4], v21[4], p[4], x2[4], m2[4], y2[4], n2[4], d2[4];
#pragma unroll
        for ( int u = 0; u < 4; u++ ) {
            const int c = M::row( lane, u );
            a[u]  = sA[c][16 + r];
            b[u]  = LU ? sA[16 + r][c] : (T)0;
            x2[u] = at( 16 + r, 16 + c );
            y2[u] = LU ? at( 16 + c, 16 + r ) : (T)0;
            m2[u] = n2[u] = d2[u] = (T)0;
        }
        // X21 = L21 D1 = A21 W^T (W the inverse of U~, in the symmetric forms
        // of L11), U12^T = A12^T L11^{-T}
        elim_prod<T>( x21, LU ? z1 : w1, a );
        if constexpr ( LU ) elim_prod<T>( y21, w1, b );
#pragma unroll
        for ( int u = 0; u < 4; u++ ) {
            const int c = M::row( lane, u );
            u21[u] = x21[u] * d1[u];
            sA[c][16 + r] = x21[u];
            if constexpr ( LU ) {
                v21[u] = y21[u] * d1[u];
                sA[16 + r][c] = y21[u];
            }
        }
        // A22 - L21 U12 (and its transpose)
        elim_prod<T>( p, LU ? v21 : u21, x21 );
#pragma unroll
        for ( int u = 0; u < 4; u++ ) x2[u] = x2[u] - p[u];
        if constexpr ( LU ) {
            elim_prod<T>( p, u21, y21 );
#pragma unroll
            for ( int u = 0; u < 4; u++ ) y2[u] = y2[u] - p[u];
        }
        elim16<T, SIGN, LU, 0>( x2, m2, y2, n2, d2, sD + 16, bs - 16, tau, lane, piv );
        T w2[4], e[4], q[4], id[4];
#pragma unroll
        for ( int u = 0; u < 4; u++ ) {
            const int  c  = M::row( lane, u );
            const bool in = c <= r && 16 + r < bs;
            id[u] = elim_sel( c == r, (T)1, (T)0 );
            w2[u] = elim_sel( in, x2[u], (T)0 );
            sI[16 + c][16 + r] = w2[u];
            sI[16 + c][r]      = (T)0;
            if ( c < r ) sA[16 + c][16 + r] = m2[u];
            if ( LU && c > r ) sA[16 + c][16 + r] = x2[u];
        }
        // W21 = -W22 (L21 W11): E = W11^T, Q = (L21 W11)^T
        elim_prod<T>( e, w1, id );
        elim_prod<T>( q, u21, e );
        elim_prod<T>( p, q, w2 );
#pragma unroll
        for ( int u = 0; u < 4; u++ ) sI[M::row( lane, u )][16 + r] = -p[u];
        if constexpr ( LU ) {
            T z2[4];
#pragma unroll
            for ( int u = 0; u < 4; u++ ) {
                const int  c  = M::row( lane, u );
                const bool in = c <= r && 16 + r < bs;
                z2[u] = elim_sel( in, y2[u], (T)0 );
                sZ[16 + c][16 + r] = z2[u];
                sZ[16 + c][r]      = (T)0;
            }
            elim_prod<T>( e, z1, id );
            elim_prod<T>( q, v21, e );
            elim_prod<T>( p, q, z2 );
#pragma unroll
            for ( int u = 0; u < 4; u++ ) sZ[M::row( lane, u )][16 + r] = -p[u];
        }
    }
    return piv;
}
