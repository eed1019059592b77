// ocean_device.hpp -- device functions shared by the single-ocean kernels
// (ocean_kernels.hip) and the batched kernels (ocean_batch.hip): noise and the
// Phillips spectrum, the dispersion phase, the Hermitian fold, the XCD-aware
// block order, the LDS-staged column transform of one strip and the fused
// row + normal-map + Jacobian walk of one band.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include <type_traits>

#include "fft_core.hpp"
#include "ocean_kernels.h"

namespace ocn {

// ------------------------------------------------------------------ output stores

// The frame's outputs are written once and never read back by these kernels:
// non-temporal stores keep them from displacing the intermediates (still to be
// read by other blocks of the row pass) in L2 and the Infinity Cache.
__device__ __forceinline__ void st_out(float* p, float v) { __builtin_nontemporal_store(v, p); }
__device__ __forceinline__ void st_out(float4* p, float4 v)
{
    typedef float f32x4 __attribute__((ext_vector_type(4)));
    const f32x4 w = {v.x, v.y, v.z, v.w};
    __builtin_nontemporal_store(w, reinterpret_cast<f32x4*>(p));
}

// ------------------------------------------------------------------ noise

// Philox4x32-10 (Salmon et al., SC'11).  Whole 64-bit products: one
// quarter-rate multiply each instead of two for the halves.
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint2 k)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        if (r) { k.x += 0x9E3779B9u; k.y += 0xBB67AE85u; }
        const uint64_t p0 = (uint64_t)0xD2511F53u * c.x, p1 = (uint64_t)0xCD9E8D57u * c.z;
        c = make_uint4((uint32_t)(p1 >> 32) ^ c.y ^ k.x, (uint32_t)p1, (uint32_t)(p0 >> 32) ^ c.w ^ k.y, (uint32_t)p0);
    }
    return c;
}

// (m + 1/2) * 2^-23 from the top 23 bits: exact in FP32.
__device__ __forceinline__ float u01(uint32_t x) { return ((float)(x >> 9) + 0.5f) * (1.0f / 8388608.0f); }

// gauss_rnd (tilde_h0_k_cs.glsl:51-68): clamp to [0.001, 1], two Box-Muller pairs.
__device__ __forceinline__ float4 box_muller(float n0, float n1, float n2, float n3)
{
    n0 = fminf(fmaxf(n0, 0.001f), 1.0f);
    n1 = fminf(fmaxf(n1, 0.001f), 1.0f);
    n2 = fminf(fmaxf(n2, 0.001f), 1.0f);
    n3 = fminf(fmaxf(n3, 0.001f), 1.0f);
    float s0, c0, s1, c1;
    sincospif(2.0f * n0, &s0, &c0);
    sincospif(2.0f * n2, &s1, &c1);
    const float r0 = sqrtf(-2.0f * logf(n1));
    const float r1 = sqrtf(-2.0f * logf(n3));
    return make_float4(r0 * c0, r0 * s0, r1 * c1, r1 * s1);
}

// sqrt(P(k))/sqrt(2) before the clamp (tilde_h0_k_cs.glsl:35-45, 76-88).
// k_hat = k / |k|_clamped: equal to normalize(k) for k != 0, and 0 at DC where
// normalize(0) is undefined.  pow(d, 2.0) is d*d.
__device__ __forceinline__ float phillips_amp_raw(const SpecConst& sc, int tx, int ty)
{
    const float kx = sc.kscale * (float)(tx - sc.N / 2);
    const float ky = sc.kscale * (float)(ty - sc.N / 2);
    float kmag = sqrtf(kx * kx + ky * ky);
    if (kmag < 0.00001f) kmag = 0.00001f;
    const float k2  = kmag * kmag;
    const float sup = expf(-k2 * sc.l2);
    const float d   = (kx * sc.wx + ky * sc.wy) / kmag;
    const float P   = sc.A * expf(-1.0f / (k2 * sc.Lp2)) * (d * d) * sup / (k2 * k2);
    return sqrtf(P) * 0.70710678118654752f;
}

// clamp(sqrt(P(k))/sqrt(2), -4000, 4000) (tilde_h0_k_cs.glsl:87-88); P >= 0.
__device__ __forceinline__ float phillips_amp(const SpecConst& sc, int tx, int ty)
{
    return fminf(phillips_amp_raw(sc, tx, ty), 4000.0f);
}

// ------------------------------------------------------------------ A4 time evolution

// Dispersion phase w t / (2 pi) with w = sqrt(g |k|_clamped) (tilde_h0_t_cs.glsl:77-79),
// as a fraction of a turn in [-1/2, 1/2].  w t reaches hundreds of radians,
// where FP32 rounding of w alone would cost ~1e-5 rad, so w is refined in FP64:
// an FP32 estimate w0 plus one Newton step on w^4 = g^2 |k|^2 (|k|^2 is exact
// from the integer wave numbers), then the product with t / (2 pi) is reduced
// to one turn before the FP32 sincos.  m = nx^2 + ny^2.  kinv receives
// kscale / |k|_clamped, the factor of the choppy spectra (-i k/|k| = -i n kinv).
// Two reciprocal square roots give the FP32 parts: 1/sqrt(m) is kinv itself,
// and s = 1/sqrt(g |k|) gives w0 = g |k| s and the Newton step's 1/w0^3 = s^3.
__device__ __forceinline__ double omega_fp64(const SpecConst& sc, int m, float& kinv)
{
    const float mf = (float)m;
    const float r  = __builtin_amdgcn_rsqf(mf);  // +inf at m = 0
    const float kr = sc.kscale * (mf * r);       // |k|; NaN at m = 0
    const bool  lo = !(kr >= 0.00001f);          // |k| below the 1e-5 clamp (or DC)
    const float kf = lo ? 0.00001f : kr;
    kinv = lo ? sc.kscale * 100000.0f : r;
    const float  gk = sc.g * kf;
    const float  s  = __builtin_amdgcn_rsqf(gk);
    const float  w0 = gk * s;
    const double Q  = fmax(sc.k2_d * (double)m, 1e-10) * sc.g2_d;  // g^2 |k|_clamped^2
    const double w  = (double)w0;
    const double w2 = w * w;
    return w - (w2 * w2 - Q) * (double)(0.25f * s * s * s);
}

// w t / (2 pi) reduced to [-1/2, 1/2] turns, w from omega_fp64.
__device__ __forceinline__ float turns(double w, double t_rev)
{
    const double rev = w * t_rev;
    return (float)(rev - rint(rev));
}

__device__ __forceinline__ float phase_turns(const SpecConst& sc, int m, double t_rev, float& kinv)
{
    return turns(omega_fp64(sc, m, kinv), t_rev);
}

// sin and cos of 2 pi fr for fr in [-1/2, 1/2]: reduction by quarter turns
// q = rint(4 fr) (the remainder r = fr - q/4 is exact), Taylor polynomials of
// sin and cos on |2 pi r| <= pi/4 to degree 9 and 10 (truncation < 2e-9),
// then rotation by q quarter turns.
__device__ __forceinline__ void sincos_turns(float fr, float& s, float& c)
{
    const float q  = rintf(4.0f * fr);
    const float th = (fr - 0.25f * q) * 6.28318530717958647692f;
    const float t2 = th * th;
    const float sp = th * fmaf(t2, fmaf(t2, fmaf(t2, fmaf(t2, 2.75573192239858907e-6f, -1.98412698412698413e-4f),
                                                 8.33333333333333333e-3f), -1.66666666666666667e-1f), 1.0f);
    const float cp = fmaf(t2, fmaf(t2, fmaf(t2, fmaf(t2, fmaf(t2, -2.75573192239858907e-7f, 2.48015873015873016e-5f),
                                                       -1.38888888888888889e-3f), 4.16666666666666667e-2f), -0.5f),
                          1.0f);
    // quarter turn qi: (s, c) = (sp, cp), (cp, -sp), (-sp, -cp), (-cp, sp),
    // as a select and two sign-bit flips (no divergent branches)
    const int   qi = (int)q & 3;
    const float a  = (qi & 1) ? cp : sp;
    const float b  = (qi & 1) ? sp : cp;
    s = __int_as_float(__float_as_int(a) ^ ((qi & 2) << 30));
    c = __int_as_float(__float_as_int(b) ^ (((qi + 1) & 2) << 30));
}

// a e^{i th} + C(b) e^{-i th} for h = (a, b) = (h0k, h0mk) (tilde_h0_t_cs.glsl:94-110).
__device__ __forceinline__ float2 evolve_amp(const SpecConst& sc, float4 h, float s, float c)
{
    const float bi = sc.conj_mode ? -h.w : h.w;
    return make_float2(fmaf(h.x, c, -h.y * s) + fmaf(h.z, c, bi * s), fmaf(h.x, s, h.y * c) + fmaf(bi, c, -h.z * s));
}

// -i m * H  (tilde_h0_t_cs.glsl:113-126).  Its products stay out of the sums
// they go into (no fused multiply-add), so that every kernel instance that
// folds a texel gives the transform the same input, bit for bit.
__device__ __forceinline__ float2 choppy(float m, float2 h)
{
#pragma clang fp contract(off)
    return make_float2(m * h.y, -m * h.x);
}

// ------------------------------------------------------------------ folded spectrum

// The column pass needs, per texel u of the half plane tx <= N/2, only the
// Hermitian parts A = (H(u) + conj H(-u))/2 of the height spectrum and, on the
// edges, B = (H(u) - conj H(-u))/2.  With a, b = h0k, h0mk at u and a', b' at
// the mirror -u, H(u) = a e + C(b) conj(e) (e = e^{i w t}, |k| and so w shared by
// u and -u), hence A = P e + Q conj(e) = U cos + V sin with
//   P = (a + conj C(b'))/2, Q = (C(b) + conj a')/2, U = P + Q, V = i (P - Q):
// four real coefficients per half-plane texel, made with h0 (k_tilde_h0_k),
// that are half of what h0 itself holds for the pair, and one multiply-add per
// component and frame.  The choppy spectra follow: -i k/|k| changes sign with
// k, so their Hermitian parts are -i (n kinv) A, except where the centred index
// n of the mirror is not -n: column tx = 0 for Dx and row ty = 0 for Dz (index
// -N/2), where they are -i (n kinv) B, with B = U' cos + V' sin from
// P' = (a - conj C(b'))/2 and Q' = (C(b) - conj a')/2.
//
// Layout, float4 (U.re, U.im, V.re, V.im): column tx of the half plane at
// tx*N + ty (a column is one contiguous run: a wave that transforms a column
// reads 1 KB per load), then the N entries of B in column 0 (by ty), then the
// N/2 + 1 of B in row 0 (by tx).
__host__ __device__ constexpr size_t uv_bcol(int N) { return (size_t)N * (N / 2 + 1); }
__host__ __device__ constexpr size_t uv_brow(int N) { return uv_bcol(N) + N; }

// (U, V) of A (sign = 1) or B (sign = -1) from h0 at u (p) and at -u (q).
__device__ __forceinline__ float4 fold_coeffs(float4 p, float4 q, int conj_mode, float sign)
{
    const float bi = conj_mode ? -p.w : p.w, qi = conj_mode ? -q.w : q.w;  // Im C(b), Im C(b')
    const float Px = 0.5f * (p.x + sign * q.z), Py = 0.5f * (p.y - sign * qi);
    const float Qx = 0.5f * (p.z + sign * q.x), Qy = 0.5f * (bi - sign * q.y);
    return make_float4(Px + Qx, Py + Qy, Qy - Py, Px - Qx);
}

// U cos + V sin.
__device__ __forceinline__ float2 fold_at(float4 uv, float s, float c)
{
    return make_float2(fmaf(uv.x, c, uv.z * s), fmaf(uv.y, c, uv.w * s));
}

// ------------------------------------------------------------------ intermediate column order

// Position of column x in a row of the column-pass intermediates (Z1, Z2):
// columns 0..N/2 in place, columns N/2+1..N-1 reversed after them (column
// N - u at N/2 + u).  A strip of half-plane columns tx and its mirror columns
// N - tx then occupy two aligned runs of equal length, so neighbouring strips
// complete whole cache lines instead of splitting the mirror run across lines
// written by different strips.
template <int N>
__device__ __forceinline__ int zpos(int x)
{
    return x <= N / 2 ? x : 3 * N / 2 - x;
}

// zpos of element r of a row transform held as x = j + r*T (T = N/E, j < T),
// with the half the element falls in known at compile time.
template <int N, int E>
__device__ __forceinline__ int zpos_elem(int j, int r)
{
    constexpr int T = N / E;
    if (2 * r < E) return j + r * T;
    if (2 * r > E) return 3 * N / 2 - (j + r * T);
    return j == 0 ? N / 2 : N - j;
}

// Z1 and Z2 are stored in tiles of two rows: element (row y, position p) sits
// at float2 index (y/2 * N + p) * 2 + y%2, the two rows of a tile interleaved.
// A column strip of C columns then writes runs of 2C values (one 16-byte store
// per column and tile) instead of runs of C per row, which halves the write
// requests of the column pass, and the row pass reads both rows of a tile with
// one 16-byte load per position.  Tiles start 16-byte aligned when the buffer
// does.
template <int N>
__device__ __forceinline__ size_t zidx(int y, int p)
{
    return ((size_t)(y >> 1) * N + p) * 2 + (y & 1);
}
template <int N>
__device__ __forceinline__ float4* ztile(float2* z, int m)
{
    return reinterpret_cast<float4*>(z) + (size_t)m * N;
}
template <int N>
__device__ __forceinline__ const float4* ztile(const float2* z, int m)
{
    return reinterpret_cast<const float4*>(z) + (size_t)m * N;
}

// ------------------------------------------------------------------ XCD-aware block order

// MI355X spreads the workgroups of a launch round-robin over its 8 XCDs
// (workgroup b runs on XCD b % 8), and each XCD has its own L2.  This maps the
// hardware block index to a logical index such that XCD x processes the
// contiguous logical range [x*q + min(x, r), ...) in order (q = n / 8,
// r = n % 8): consecutive logical blocks share an L2.  It is a bijection on
// [0, n) for any n.
__device__ __forceinline__ int xcd_logical(int b, int n)
{
    constexpr int X = 8;
    const int q = n / X, r = n % X, x = b % X;
    return x * q + (x < r ? x : r) + b / X;
}

// Column strips per block group (consecutive blocks on one XCD): G strips of
// C columns cover 32 columns of every Z tile row from N = 256 on (four whole
// 128-byte lines), 16 below.  Wider groups complete more lines in one L2
// before they are written back: at N = 1024 the column pass writes 14.5
// instead of 16.7 B/texel and the frame drops from 17.3 to 16.6 us; groups
// of 64 or 128 columns were slower again, and at N = 128 the wider group
// cost 1%.
template <int N, int C>
__host__ __device__ constexpr int strip_group()
{
    constexpr int W = N >= 256 ? 32 : 16;
    return C >= W ? 1 : W / C;
}


// ------------------------------------------------------------------ column pass: one strip

// Column strips per frame: the N/2 + 1 half-plane columns
// 0 .. N/2 in strips of C, with the two self-mirror columns 0 and N/2 sharing
// one transform (below), i.e. N/2 column slots.
template <int N, int C>
__host__ __device__ constexpr int lds_strips()
{
    return (N / 2) / C;
}

// Stride (float2) of the per-(field, column) LDS buffers of cols_lds_strip:
// lds_len(N) plus a few elements.  The fold writes of 16 lanes (4 columns by
// 4 consecutive rows, then their partner rows N - ty) and the store reads
// then fall on distinct banks more often: with a stride of 1 mod 32 the 32
// banks of a 16-lane b64 access saw up to 4 lanes per bank in the fold
// writes.  A bank model of the strip's accesses gives 1536 instead of 2979
// fold-write cycles per block at N = 1024 and C = 4 (7424 instead of 8960
// over folds, transforms and store reads with one fold per texel pair), and
// no width C in 1..8 more.
__host__ __device__ constexpr int strip_len(int N)
{
    return N == 1024 ? 1091 : N == 512 ? 547 : N == 256 ? 275 : N == 128 ? 152 : N == 64 ? 76 : lds_len(N);
}

// Z1 of rows 2m and 2m+1 at column tx, and at its mirror N - tx: G_h + i G_dx
// with G(-tx) = conj G(tx).  (y, x) = (G_h, G_dx).
__device__ __forceinline__ float4 zpack(float2 y0, float2 x0, float2 y1, float2 x1)
{
    return make_float4(y0.x - x0.y, y0.y + x0.x, y1.x - x1.y, y1.y + x1.x);
}
__device__ __forceinline__ float4 zpack_mirror(float2 y0, float2 x0, float2 y1, float2 x1)
{
    return make_float4(y0.x + x0.y, x0.x - y0.y, y1.x + x1.y, x1.x - y1.y);
}

// Z2 tile m (Z2 rows 2m, 2m+1; Z2 row q pairs G_dz rows 2q and 2q+1) of column
// tx and its mirror, from the column's G_dz in its LDS buffer.  The mirror's
// position is N/2 + tx (zpos); in slot 0 the real parts are column 0's and the
// imaginary parts column N/2's.
template <int N>
__device__ __forceinline__ void z2_store(float2* __restrict__ z2, int m, int tx, const float2* buf)
{
    const float2 a = buf[lds_pad(4 * m)], b = buf[lds_pad(4 * m + 1)];
    const float2 d = buf[lds_pad(4 * m + 2)], e = buf[lds_pad(4 * m + 3)];
    float4*      t2 = ztile<N>(z2, m) + tx;
    t2[0]     = tx == 0 ? make_float4(a.x, b.x, d.x, e.x) : zpack(a, b, d, e);
    t2[N / 2] = tx == 0 ? make_float4(a.y, b.y, d.y, e.y) : zpack_mirror(a, b, d, e);
}

// LDS-staged column transforms of one strip, for single frames: the C
// half-plane columns tx = strip*C + c, block of NB >= 3*C*T threads (T = N/16,
// a transform inside one wave); lds holds 3*C*strip_len(N), z1/z2 point at the
// frame's intermediate.
// Phase A: all NB threads fold the spectrum into per-(field, column) LDS
// buffers, consecutive threads down a column, two rows ty and N - ty per
// task: they share |k| and so one dispersion phase.  Phase B: each of the 3C
// transforms runs inside one T-thread group and leaves its result in natural
// order in its buffer.  Phase C: every thread stores Z1 = G_h + i G_dx (at tx
// and its mirror N - tx) and Z2 = G_dz(2p) + i G_dz(2p+1), in two-row tiles
// (zidx).
// The three fields' transforms run side by side and the folds are spread over
// the whole block: with about one block per CU (a single frame) that is the
// shorter chain; with many blocks cols_strip does less work per column.
// The self-mirror columns 0 and N/2 have Hermitian folded spectra,
// A(-ty) = conj A(ty), so their column transforms are real: column slot 0 of
// strip 0 transforms A_0 + i A_{N/2} and its result holds column 0 in the real
// parts and column N/2 in the imaginary parts.  That leaves N/2 column slots, a
// whole number of strips (at N = 1024 and C = 2, exactly one block per CU for a
// single frame instead of 257 blocks on 256 CUs).
template <int N, int C, int NB>
__device__ __forceinline__ void cols_lds_strip(const float4* __restrict__ uv, float2* __restrict__ z1,
                                               float2* __restrict__ z2, const float2* __restrict__ tw,
                                               const SpecConst& sc, double t_rev, int strip, float2* lds)
{
    constexpr int E = 16, T = N / E, NT = 3 * C * T, LEN = strip_len(N), H = N / 2 + 1;
    constexpr int ITERS = (C * H + NB - 1) / NB;  // row-pair tasks per thread
    static_assert(NB >= NT && T <= 64 && 64 % T == 0, "transforms inside one wave");
    static_assert((N / 2) % C == 0, "strips of C columns tile the half plane");
    // Row 0 and, in strip 0 (FIRST), column 0 take their B coefficients by the load's
    // address: a load in a branch is another trip to memory, and every column has a row 0.
    auto folds = [&](auto first) {
        constexpr bool FIRST = decltype(first)::value;
#pragma unroll
        for (int it = 0; it < ITERS; ++it) {
            const int k = threadIdx.x + it * NB;
            if (k < C * H) {
                const int    c = k / H, ra = k % H, rb = (N - ra) & (N - 1);
                const int    tx = strip * C + c, nx = tx - N / 2, ny = ra - N / 2;
                const size_t col = (size_t)tx * N;
                const float4 qa = uv[col + ra], qb = uv[col + rb];
                const float4 qz = uv[ra == 0 ? uv_brow(N) + tx : col + ra];
                const size_t bx = FIRST && tx == 0 ? uv_bcol(N) : col;
                const float4 xa = FIRST ? uv[bx + ra] : qa, xb = FIRST ? uv[bx + rb] : qb;
                float        kinv, s, cs;
                sincos_turns(turns(omega_fp64(sc, nx * nx + ny * ny, kinv), t_rev), s, cs);
                const float2 B = fold_at(qb, s, cs);
                const float  mx = (float)nx * kinv, mz = (float)ny * kinv;
                lds[(0 * C + c) * LEN + lds_pad(ra)] = fold_at(qa, s, cs);
                lds[(1 * C + c) * LEN + lds_pad(ra)] = choppy(mx, fold_at(xa, s, cs));
                lds[(2 * C + c) * LEN + lds_pad(ra)] = choppy(mz, fold_at(qz, s, cs));
                if (rb != ra) {  // rows 0 and N/2 are their own partners
                    lds[(0 * C + c) * LEN + lds_pad(rb)] = B;
                    lds[(1 * C + c) * LEN + lds_pad(rb)] = choppy(mx, fold_at(xb, s, cs));
                    lds[(2 * C + c) * LEN + lds_pad(rb)] = choppy(-mz, B);
                }
            }
        }
    };
    if (strip == 0) {
        // column slot 0 += i * (the Nyquist column's folds), its rows spread
        // over the whole block; its Dx spectrum is 0 (nx = 0).  They are made first, so
        // that only the sums are left behind the barrier.
        constexpr int NI = (N + NB - 1) / NB;
        float2        h[NI], z[NI];
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int    ty = (threadIdx.x + i * NB) & (N - 1), ny = ty - N / 2;
            const float4 q  = uv[(size_t)(N / 2) * N + ty];
            const float4 qz = uv[ty == 0 ? uv_brow(N) + N / 2 : (size_t)(N / 2) * N + ty];
            float        kinv, s, cs;
            sincos_turns(phase_turns(sc, ny * ny, t_rev, kinv), s, cs);
            h[i] = fold_at(q, s, cs);
            z[i] = choppy((float)ny * kinv, fold_at(qz, s, cs));
        }
        folds(std::true_type{});
        __syncthreads();
#pragma unroll
        for (int i = 0; i < NI; ++i) {
            const int ty = threadIdx.x + i * NB;
            if (ty < N) {
                float2& ah = lds[0 * C * LEN + lds_pad(ty)];
                float2& az = lds[2 * C * LEN + lds_pad(ty)];
                ah = make_float2(ah.x - h[i].y, ah.y + h[i].x);
                az = make_float2(az.x - z[i].y, az.y + z[i].x);
            }
        }
    } else {
        folds(std::false_type{});
    }
    __syncthreads();
    if (NB == NT || (int)threadIdx.x < NT) {
        const int g = threadIdx.x / T, j = threadIdx.x % T;
        float2*   buf = lds + g * LEN;
        float2    v[E];
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = buf[lds_pad(j + r * T)];
        fft_inverse<N, E>(v, j, buf, tw, WaveSync{});
        WaveSync{}();
#pragma unroll
        for (int r = 0; r < E; ++r) buf[lds_pad(j + r * T)] = v[r];
    }
    __syncthreads();
    // thread k stores Z1 tile m = k / C (rows 2m, 2m+1) and, for m < N/4, Z2
    // tile m (Z2 rows 2m, 2m+1, i.e. G_dz rows 4m..4m+3) of column c = k % C
    constexpr int ITZ = (C * N / 2 + NB - 1) / NB;
#pragma unroll
    for (int it = 0; it < ITZ; ++it) {
        const int k = threadIdx.x + it * NB;
        if (k < C * N / 2) {
            const int    c = k % C, m = k / C, tx = strip * C + c;
            const float2 y0 = lds[(0 * C + c) * LEN + lds_pad(2 * m)];
            const float2 x0 = lds[(1 * C + c) * LEN + lds_pad(2 * m)];
            const float2 y1 = lds[(0 * C + c) * LEN + lds_pad(2 * m + 1)];
            const float2 x1 = lds[(1 * C + c) * LEN + lds_pad(2 * m + 1)];
            float4*      t1 = ztile<N>(z1, m) + tx;
            t1[0]     = tx == 0 ? make_float4(y0.x, x0.x, y1.x, x1.x) : zpack(y0, x0, y1, x1);
            t1[N / 2] = tx == 0 ? make_float4(y0.y, x0.y, y1.y, x1.y) : zpack_mirror(y0, x0, y1, x1);
            if (m < N / 4) z2_store<N>(z2, m, tx, lds + (2 * C + c) * LEN);
        }
    }
}

// Column transforms of one strip in registers: the C half-plane columns
// tx = strip*C + c, one group of T = N/E threads per column (NB >= C*T threads
// in the block, the rest only store); lds holds C*strip_len(N).
// A group folds its column straight into registers (thread j rows j + r*T, each
// load one contiguous run of the column), since the three folded spectra are
// real multiples of one another (-i n kinv A): it runs the three transforms one
// after another in its one LDS buffer and keeps the results in registers until
// they are staged, so the strip needs a third of the LDS of cols_lds_strip
// (35 KB at N = 1024 and C = 4).  Registers (127 a thread, four waves per SIMD) leave
// two blocks of eight waves per CU there, instead of one of twelve, and one block's
// loads, arithmetic and stores overlap the other's; at N = 4096 a block of 16 waves
// is alone.
// Dz goes first: its result leaves the registers before the height's and Dx's,
// which meet in Z1, are made.  Stores go through the buffers so that C lanes
// write C adjacent columns of a tile (16 bytes each).
// Column slot 0 packs columns 0 and N/2 as in cols_lds_strip.  Its folds, two
// columns' for each transform, are spread over the whole block (slot0_fold):
// left to the slot's own group, strip 0 took several times a strip's time, and
// launches of few blocks waited for it.
template <int N, int NB>
__device__ __forceinline__ void slot0_fold(const float4* __restrict__ uv, const SpecConst& sc, double t_rev,
                                           int field, float2* buf)
{
#pragma unroll 1
    for (int ty = threadIdx.x; ty < N; ty += NB) {
        const int    ny   = ty - N / 2;
        const bool   edge = field == 2 && ty == 0;
        const float4 qa = uv[field == 1 ? uv_bcol(N) + ty : edge ? uv_brow(N) : (size_t)ty];
        const float4 qb = uv[edge ? uv_brow(N) + N / 2 : (size_t)(N / 2) * N + ty];
        float        k0, kN, s, c;
        sincos_turns(phase_turns(sc, (N / 2) * (N / 2) + ny * ny, t_rev, k0), s, c);
        float2 a = fold_at(qa, s, c), b = make_float2(0.0f, 0.0f);  // Dx is 0 in column N/2 (nx = 0)
        if (field != 1) {
            sincos_turns(phase_turns(sc, ny * ny, t_rev, kN), s, c);
            b = fold_at(qb, s, c);
            if (field == 2) {
                a = choppy((float)ny * k0, a);
                b = choppy((float)ny * kN, b);
            }
        } else {
            a = choppy((float)(-N / 2) * k0, a);
        }
        buf[lds_pad(ty)] = make_float2(a.x - b.y, a.y + b.x);
    }
}

template <int N, int E, int C, int NB>
__device__ __forceinline__ void cols_strip(const float4* __restrict__ uv, float2* __restrict__ z1,
                                           float2* __restrict__ z2, const float2* __restrict__ tw,
                                           const SpecConst& sc, double t_rev, int strip, float2* lds)
{
    constexpr int T = N / E, NT = C * T, LEN = strip_len(N);
    using Sync = typename std::conditional<(T <= 64), WaveSync, BlockSync>::type;
    static_assert((N / 2) % C == 0, "strips of C columns tile the half plane");
    static_assert(NB >= NT && NB % T == 0, "whole groups");
    // Threads past the strip's groups only store; where the transforms meet
    // block barriers (T > 64) they transform a column of their own for nothing
    // (lds then holds NB/T buffers).
    const bool active = NB == NT || T > 64 || (int)threadIdx.x < NT;
    const int  g = threadIdx.x / T, j = threadIdx.x % T;
    const int  tx = g < C ? strip * C + g : N / 2 - 1;
    float2*    buf = lds + g * LEN;
    float2     A[E], v[E];
    auto put = [&](float2 (&x)[E]) {
#pragma unroll
        for (int r = 0; r < E; ++r) buf[lds_pad(j + r * T)] = x[r];
    };
    auto get = [&](float2 (&x)[E]) {
#pragma unroll
        for (int r = 0; r < E; ++r) x[r] = buf[lds_pad(j + r * T)];
    };
    // strip is the same for every thread of the block
    if (strip == 0) {
        slot0_fold<N, NB>(uv, sc, t_rev, 2, lds);
        __syncthreads();
    }
    if (active) {
        const float4* col = uv + (size_t)tx * N;
        const int     nx  = tx - N / 2;
        float         kinv[E];
        float4        q[E];
#pragma unroll
        for (int r = 0; r < E; ++r) q[r] = col[j + r * T];
        // row 0's coefficients for Dz: one column to a wave from N = 512 on
        const float4 row0 = uv[uv_brow(N) + (T >= 64 ? __builtin_amdgcn_readfirstlane(tx) : tx)];
        // Every load before the first phase: left to the scheduler, each came just
        // before its use with one other in flight, eight trips to memory in a row
        // (64-ocean batch 1209 -> 1187 us, N = 1024 sequence 748 -> 740)
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int ny = j + r * T - N / 2;
            float     s, c;
            sincos_turns(phase_turns(sc, nx * nx + ny * ny, t_rev, kinv[r]), s, c);
            A[r] = fold_at(q[r], s, c);
            v[r] = choppy((float)ny * kinv[r], r == 0 && j == 0 ? fold_at(row0, s, c) : A[r]);
        }
        if (tx == 0) get(v);
        fft_inverse<N, E>(v, j, buf, tw, Sync{});
        Sync{}();
        put(v);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            v[r] = A[r];
            A[r] = choppy((float)nx * kinv[r], A[r]);
        }
    }
    __syncthreads();
    for (int k = threadIdx.x; k < C * N / 4; k += NB) z2_store<N>(z2, k / C, strip * C + k % C, lds + (k % C) * LEN);
    __syncthreads();
    if (strip == 0) {
        slot0_fold<N, NB>(uv, sc, t_rev, 0, lds);
        __syncthreads();
    }
    if (active) {
        if (tx == 0) get(v);
        fft_inverse<N, E>(v, j, buf, tw, Sync{});
    }
    if (strip == 0) {
        __syncthreads();
        slot0_fold<N, NB>(uv, sc, t_rev, 1, lds);
        __syncthreads();
    }
    if (active) {
        if (tx == 0) get(A);
        fft_inverse<N, E>(A, j, buf, tw, Sync{});
        // Z1 at tx and its mirror (slot 0: the real and the imaginary parts)
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const float2 y = v[r], x = A[r];
            v[r] = tx == 0 ? make_float2(y.x, x.x) : make_float2(y.x - x.y, y.y + x.x);
            A[r] = tx == 0 ? make_float2(y.y, x.y) : make_float2(y.x + x.y, x.x - y.y);
        }
        Sync{}();
        put(v);
    }
    auto store = [&](int side) {
        for (int k = threadIdx.x; k < C * N / 2; k += NB) {
            const int    c = k % C, m = k / C;
            const float2 a = lds[c * LEN + lds_pad(2 * m)], b = lds[c * LEN + lds_pad(2 * m + 1)];
            ztile<N>(z1, m)[strip * C + c + side * (N / 2)] = make_float4(a.x, a.y, b.x, b.y);
        }
    };
    __syncthreads();
    store(0);
    __syncthreads();
    if (active) put(A);
    __syncthreads();
    store(1);
}

// ------------------------------------------------------------------ row pass + normals + Jacobian: one band

// Row transforms fused with the normal map (nearest taps) and the Jacobian
// for one band of R rows [y0, y0 + R), y0 = band*R even (R even, dividing N;
// the caller checks).  A group of T = N/E
// threads (thread j holds x = j + r*T) walks the band with a three-row window
// in registers: for each new row it transforms Z1 (height + i Dx) and, on
// even rows, the Z2 row holding Dz of that row and the next, then applies
// (-1)^(x+y) / N^2 (inversion_cs.glsl:35-41).  The x-neighbours of the stencil
// pass through the group's LDS buffer buf (lds_len(N) entries); halo rows
// y0-1 and y0+R are transformed too (periodic).  Sobel taps as
// normal_map_cs.glsl:37-53; J = (1 - l dDx/dx)(1 - l dDz/dz) - l^2 dDx/dz dDz/dx
// for the render displacement (-l Dx, -l Dz) (grid_tes.glsl:60-62), central
// differences with spacing L/N.  All pointers are at the frame's data;
// normals or jac may be null.  RENDER adds the render export (disp, rnorm,
// either may be null): (-l Dx, s h, -l Dz, J) and the unit normal of the
// displaced surface, dP/dv x dP/du.
template <int N, int E, class Sync, bool RENDER = false, bool PAIR2 = false, bool ALT = false>
__device__ __forceinline__ void rows_nrm_band(const float2* __restrict__ z1, const float2* __restrict__ z2,
                                              float* __restrict__ height, float* __restrict__ dx,
                                              float* __restrict__ dz, float4* __restrict__ normals,
                                              float* __restrict__ jac, const float2* __restrict__ tw, float2* buf,
                                              int j, int band, int R, float lambda, float inv2d,
                                              float4* __restrict__ disp = nullptr, float4* __restrict__ rnorm = nullptr,
                                              float dscale = 0.0f)
{
    constexpr int T = N / E;
    constexpr float scale = 1.0f / ((float)N * (float)N);
    // With ALT, odd bands walk their rows upwards, so that the halo tiles two
    // neighbouring bands share are read by both near the same time (both
    // walks end at their common boundary and start at the band boundaries
    // they share with the other neighbours) and come from one L2 fetch.
    // The walk runs over walk rows w = y0 .. y0+R-1 in its own order: walk row
    // w is grid row arow(w) = w, or N-1-w on an upward walk; both take the
    // unwrapped -1 .. N.  The flip maps a two-row tile onto a two-row tile
    // with its halves exchanged (N-1 is odd), and a Z2 row (rows 2u, 2u+1 in
    // its real and imaginary parts) onto a Z2 row with the parts exchanged, so
    // the walk below reads tiles and Z2 parts in walk order.  Signs, output
    // rows and stencils use grid rows, with the neighbours named by grid
    // position, so that every row's arithmetic is that of a downward walk
    // (frames are bit-identical either way).  N=1024 / 2048 frames -0.9%; below
    // that the selects cost more than the halo reads (N=512 +2%).
    const bool flip = ALT && (band & 1) != 0;
    const int  fm   = flip ? -1 : 0;
    const int  y0   = flip ? N - (band + 1) * R : band * R;
    auto arow  = [&](int w) { return (w ^ fm) & (N - 1); };
    auto arow2 = [&](int u) { return (u ^ fm) & (N / 2 - 1); };  // Z2 rows

    // Rows are read from the two-row tiles of Z1 / Z2: load_row takes one grid
    // row (8 bytes of every 16), load_pair the tile holding walk rows w, w+1
    // (w even; the caller passes the tile index arow(w) >> 1) -- walk row w
    // into v, w+1 into w -- with one 16-byte load per position.  Thread j
    // holds x = j + r*T (natural order after the transform).
    auto load_row = [&](const float2* z, int y, float2 (&v)[E]) {
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = z[zidx<N>(y, zpos_elem<N, E>(j, r))];
    };
    auto load_pair = [&](const float2* z, int tile, float2 (&v)[E], float2 (&w)[E]) {
        const float4* t = ztile<N>(z, tile);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const float4 q  = t[zpos_elem<N, E>(j, r)];
            const float2 lo = make_float2(q.x, q.y), hi = make_float2(q.z, q.w);
            v[r] = flip ? hi : lo;
            w[r] = flip ? lo : hi;
        }
    };
    auto fft = [&](float2 (&v)[E]) { fft_inverse<N, E>(v, j, buf, tw, Sync{}); };
    // a transformed Z2 row in walk order: even walk row in .x, odd in .y
    auto fft2 = [&](float2 (&v)[E]) {
        fft(v);
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = flip ? make_float2(v[r].y, v[r].x) : v[r];
    };
    // (-1)^(x+y) / N^2 of grid row y; x = j + r*T and T is even, so the parity is that of j + y
    auto sgn = [&](int y) { return ((j + y) & 1) ? -scale : scale; };
    // d/dz by central differences: walk neighbours (next - previous) times this
    const float vinv = flip ? -inv2d : inv2d;

    // The band reads walk rows y0-1 .. y0+R of Z1 and Z2 rows (y0-1)/2 .. (y0+R)/2
    // (row N wraps to 0), counted unwrapped: an even Z1 row y >= y0 other
    // than the last is loaded together with row y+1, which waits in p1 for
    // the next step.  With PAIR2 the Z2 rows b2 .. e2 are paired the same way
    // (pending row in p2); without it they are read one at a time, which saves
    // the registers of p2.
    const int b2 = y0 >> 1, e2 = b2 + R / 2;
    float hA[E], xA[E], zA[E], hB[E], xB[E], zB[E], zN[E];
    float2 v[E], p1[E], p2[E];
    {
        const int yA = (y0 - 1) & (N - 1);  // odd: Dz from the odd part of Z2 row yA >> 1
        load_row(z2, arow2(yA >> 1), v);
        fft2(v);
        const float sa = sgn(arow(yA));
#pragma unroll
        for (int r = 0; r < E; ++r) zA[r] = sa * v[r].y;
        load_row(z1, arow(yA), v);
        fft(v);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            hA[r] = sa * v[r].x;
            xA[r] = sa * v[r].y;
        }
        const float sb = sgn(arow(y0));
        if (PAIR2 && (b2 & 1) == 0) load_pair(z2, arow2(b2) >> 1, v, p2);
        else load_row(z2, arow2(b2), v);
        fft2(v);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            zB[r] = sb * v[r].x;
            zN[r] = -sb * v[r].y;  // Dz of walk row y0 + 1 (opposite sign)
        }
        load_pair(z1, arow(y0) >> 1, v, p1);  // R >= 2: walk row y0 + 1 is in the band
        fft(v);
#pragma unroll
        for (int r = 0; r < E; ++r) {
            hB[r] = sb * v[r].x;
            xB[r] = sb * v[r].y;
        }
    }

#pragma unroll 1
    for (int k = 0; k < R; ++k) {
        const int   y  = y0 + k;                 // walk row
        const int   yu = y + 1;                  // unwrapped, <= N
        const int   yC = yu & (N - 1);
        const float sc = sgn(arow(yu));
        float zC[E];
        if ((yC & 1) == 0) {
            const int u = yu >> 1;  // Z2 walk row, unwrapped
            if (PAIR2 && (u & 1)) {
#pragma unroll
                for (int r = 0; r < E; ++r) v[r] = p2[r];
            } else if (PAIR2 && u < e2) {
                load_pair(z2, arow2(u) >> 1, v, p2);
            } else {
                load_row(z2, arow2(yC >> 1), v);
            }
            fft2(v);
#pragma unroll
            for (int r = 0; r < E; ++r) {
                zC[r] = sc * v[r].x;
                zN[r] = -sc * v[r].y;
            }
        } else {
#pragma unroll
            for (int r = 0; r < E; ++r) zC[r] = zN[r];
        }
        if (yu & 1) {
#pragma unroll
            for (int r = 0; r < E; ++r) v[r] = p1[r];
        } else if (yu < y0 + R) {
            load_pair(z1, arow(yC) >> 1, v, p1);
        } else {
            load_row(z1, arow(yC), v);
        }
        fft(v);  // v = height + i Dx of walk row yC (unsigned)

        const size_t row = (size_t)arow(y) * N;
        if (normals) {
            // v_s = h(y-1) + 2 h(y) + h(y+1), d_s = h(y-1) - h(y+1); nx = v_s(x-1) - v_s(x+1),
            // nz = d_s(x-1) + 2 d_s(x) + d_s(x+1)  (normal_map_cs.glsl:49-51); up / dn are the
            // grid rows y-1 / y+1 (walk rows y+1 / y-1 on an upward walk)
            Sync{}();
#pragma unroll
            for (int r = 0; r < E; ++r) {
                const float hC = sc * v[r].x;
                const float up = flip ? hC : hA[r], dn = flip ? hA[r] : hC;
                buf[lds_pad(j + r * T)] = make_float2(up + 2.0f * hB[r] + dn, up - dn);
            }
            Sync{}();
#pragma unroll
            for (int r = 0; r < E; ++r) {
                const int    x  = j + r * T;
                const float2 lf = buf[lds_pad((x - 1) & (N - 1))];
                const float2 rt = buf[lds_pad((x + 1) & (N - 1))];
                const float2 md = buf[lds_pad(x)];
                const float  nx = lf.x - rt.x;
                const float  nz = lf.y + 2.0f * md.y + rt.y;
                const float  inv = rsqrtf(fmaf(nx, nx, fmaf(nz, nz, 1.0f)));
                st_out(&normals[row + x], make_float4(nx * inv, inv, nz * inv, 1.0f));
            }
        }
        if (jac || (RENDER && (disp || rnorm))) {
            float dhdx[E];
            if (RENDER && rnorm) {  // x-derivative of the height for the displaced-surface normal
                Sync{}();
#pragma unroll
                for (int r = 0; r < E; ++r) buf[lds_pad(j + r * T)] = make_float2(hB[r], 0.0f);
                Sync{}();
#pragma unroll
                for (int r = 0; r < E; ++r) {
                    const int x = j + r * T;
                    dhdx[r] = (buf[lds_pad((x + 1) & (N - 1))].x - buf[lds_pad((x - 1) & (N - 1))].x) * inv2d;
                }
            }
            Sync{}();
#pragma unroll
            for (int r = 0; r < E; ++r) buf[lds_pad(j + r * T)] = make_float2(xB[r], zB[r]);
            Sync{}();
#pragma unroll
            for (int r = 0; r < E; ++r) {
                const int    x    = j + r * T;
                const float2 lf   = buf[lds_pad((x - 1) & (N - 1))];
                const float2 rt   = buf[lds_pad((x + 1) & (N - 1))];
                const float  dxdx = (rt.x - lf.x) * inv2d;
                const float  dzdx = (rt.y - lf.y) * inv2d;
                const float  dxdz = (sc * v[r].y - xA[r]) * vinv;
                const float  dzdz = (zC[r] - zA[r]) * vinv;
                const float  J = (1.0f - lambda * dxdx) * (1.0f - lambda * dzdz) - lambda * lambda * dxdz * dzdx;
                if (jac) st_out(&jac[row + x], J);
                if (!RENDER) continue;
                if (disp) st_out(&disp[row + x], make_float4(-lambda * xB[r], dscale * hB[r], -lambda * zB[r], J));
                if (rnorm) {
                    // n = dP/dv x dP/du with dP/du = (1 - l dDx/dx, s dh/dx, -l dDz/dx),
                    // dP/dv = (-l dDx/dz, s dh/dz, 1 - l dDz/dz); its y component is J
                    const float dhdz = (sc * v[r].x - hA[r]) * vinv;
                    const float nx = -dscale * (lambda * dhdz * dzdx + (1.0f - lambda * dzdz) * dhdx[r]);
                    const float nz = -dscale * (lambda * dxdz * dhdx[r] + dhdz * (1.0f - lambda * dxdx));
                    const float inv = rsqrtf(fmaf(nx, nx, fmaf(J, J, nz * nz)));
                    st_out(&rnorm[row + x], make_float4(nx * inv, J * inv, nz * inv, 1.0f));
                }
            }
        }
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int x = j + r * T;
            st_out(&height[row + x], hB[r]);
            st_out(&dx[row + x], xB[r]);
            st_out(&dz[row + x], zB[r]);
            hA[r] = hB[r];
            xA[r] = xB[r];
            zA[r] = zB[r];
            hB[r] = sc * v[r].x;
            xB[r] = sc * v[r].y;
            zB[r] = zC[r];
        }
    }
}

}  // namespace ocn
