// ocean_kernels.hip -- gfx950 kernels of the Tessendorf ocean path.
//
// Reference passes (diharaw/fft-ocean-waves) and their kernels here:
//   tilde_h0_k         (main.cpp:553-583, tilde_h0_k_cs.glsl)   -> k_tilde_h0_k, k_tilde_h0_k_noise
//   tilde_h0_t         (main.cpp:587-608, tilde_h0_t_cs.glsl)   -> k_tilde_h0_t            (pass API)
//   butterfly_fft      (main.cpp:612-683, butterfly_cs.glsl,
//                       inversion_cs.glsl)                      -> k_ifft2_rows + k_ifft2_cols_inv (pass API)
//   generate_normal_map(main.cpp:687-707, normal_map_cs.glsl)   -> k_normals
//   update() frame     (main.cpp:240-244)                       -> k_cols / k_cols_lds + k_rows_nrm /
//                                                                  k_rows_nrm_par / k_rows + k_normals
//
// Fused frame data flow (per texel, FP32):
//   folded spectrum (float4 per half-plane texel) --columns--> Z1 (N x N float2), Z2 (N/2 x N float2)
//                          --rows--> height, dx, dz (float), normals (float4), Jacobian (float)
// The column pass evaluates each field's Hermitian part (whose inverse DFT is Re
// of the field's inverse DFT, which is all inversion_cs.glsl keeps) from the
// folded spectrum (ocean_device.hpp) and runs the column (ty) transforms for the
// half plane tx in [0, N/2].  It stores the packed rows Z1 = G_h + i G_dx (full
// width via G(-tx) = conj G(tx)) and Z2 = G_dz(2p) + i G_dz(2p + 1).  The row pass
// runs the row (tx) transforms: Re/Im of each result are two real outputs at once.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <mutex>
#include <type_traits>

#include "fft_core.hpp"
#include "ocean_device.hpp"
#include "ocean_kernels.h"

namespace ocn {

// ------------------------------------------------------------------ A3 tilde_h0_k

// tilde_h0_k_cs.glsl:74-94 with Philox uniforms (counter = (texel, ocean,
// cascade, 0), key = seed), or NOISE: the reference's four 256x256 8-bit noise
// images sampled NEAREST + CLAMP_TO_EDGE at gid/N (tilde_h0_k_cs.glsl:53-58,
// main.cpp:1102-1116).  Output: h0, float4 (h0k.re, h0k.im, h0mk.re, h0mk.im),
// and the folded spectrum uv that the column pass reads (fold_coeffs).
// One thread per pair (texel of the half plane, its mirror), tiles of 16 x 16
// pairs, which go through LDS to uv's columns in runs of 256 bytes.  The noise's
// integer products bound the kernel at N <= 512, so the pairs are cut to fill
// the grid exactly (512 blocks, two per CU, at N = 512) and share the amplitude,
// which is even in k off the edges: the columns 0 and N/2, whose mirrors lie in
// themselves, hold N + 2 pairs, and the N threads of column 0 take them all.
// Against drawing h0 alone (and, from N = 2048, transposing it): N=512 3.9 -> 4.7
// us, 1024 11.1 -> 12.6, 2048 57.8 -> 37.5.
// SRC kStored takes h0 as it stands and makes uv alone.
constexpr int kH0Tile = 16;
enum H0Source { kPhilox, kNoiseImages, kStored };
template <H0Source SRC>
__device__ __forceinline__ void h0_tile(float4* __restrict__ h0, float4* __restrict__ uv,
                                        const uint8_t* __restrict__ noise, const SpecConst& sc)
{
    __shared__ float4 tile[kH0Tile][kH0Tile + 1];  // [tx][ty]
    const int N = sc.N, lx = threadIdx.x % kH0Tile, ly = threadIdx.x / kH0Tile;
    const int x0 = blockIdx.x * kH0Tile, y0 = blockIdx.y * kH0Tile;
    const int tx = x0 + lx, ty = y0 + ly;
    // Column 0's threads: rows 0 and N/2, their own mirrors, take that row of
    // both columns; a row below N/2 takes its pair of column 0, one above that
    // of column N/2.
    const bool self = tx == 0 && (ty & (N / 2 - 1)) == 0;
    const int  my   = (N - ty) & (N - 1);
    const int  px = tx == 0 && ty > N / 2 ? N / 2 : tx, py = ty;
    const int  qx = self ? N / 2 : (N - px) & (N - 1), qy = self ? ty : my;
    auto texel = [&](int x, int y, float s) {
        if constexpr (SRC == kStored) return h0[(size_t)y * N + x];
        float4 xi;
        if constexpr (SRC == kNoiseImages) {
            const int o = min((y * 256) / N, 255) * 256 + min((x * 256) / N, 255);
            xi = box_muller(noise[o] / 255.0f, noise[65536 + o] / 255.0f, noise[131072 + o] / 255.0f,
                            noise[196608 + o] / 255.0f);
        } else {
            const uint4 r = philox4x32_10(make_uint4((uint32_t)y * (uint32_t)N + (uint32_t)x, sc.ocean_id,
                                                     sc.cascade_id, 0u), make_uint2(sc.key0, sc.key1));
            xi = box_muller(u01(r.x), u01(r.y), u01(r.z), u01(r.w));
        }
        return make_float4(s * xi.x, s * xi.y, s * xi.z, s * xi.w);
    };
    const float  s = phillips_amp(sc, px, py);
    const float  t = tx != 0 && ty != 0 ? s : phillips_amp(sc, qx, qy);
    const float4 p = texel(px, py, s), q = texel(qx, qy, t);
    if constexpr (SRC != kStored) {
        h0[(size_t)py * N + px] = p;
        h0[(size_t)qy * N + qx] = q;
    }
    const int cm = sc.conj_mode;
    if (tx != 0) {
        tile[lx][ly] = fold_coeffs(p, q, cm, 1.0f);
        if (ty == 0) uv[uv_brow(N) + tx] = fold_coeffs(p, q, cm, -1.0f);
    } else {
        const float4 pm = self ? p : q, qm = self ? q : p;  // h0 at the mirrors
        uv[(size_t)px * N + py] = fold_coeffs(p, pm, cm, 1.0f);
        uv[(size_t)qx * N + qy] = fold_coeffs(q, qm, cm, 1.0f);
        if (px == 0) uv[uv_bcol(N) + py] = fold_coeffs(p, pm, cm, -1.0f);
        if (qx == 0) uv[uv_bcol(N) + qy] = fold_coeffs(q, qm, cm, -1.0f);
        if (ty == 0) {
            uv[uv_brow(N)]         = fold_coeffs(p, pm, cm, -1.0f);
            uv[uv_brow(N) + N / 2] = fold_coeffs(q, qm, cm, -1.0f);
        }
    }
    __syncthreads();
    if (x0 + ly != 0) uv[(size_t)(x0 + ly) * N + y0 + lx] = tile[ly][lx];
}

template <H0Source SRC>
__global__ __launch_bounds__(kH0Tile* kH0Tile) void k_tilde_h0_k(float4* __restrict__ h0, float4* __restrict__ uv,
                                                                 const uint8_t* __restrict__ noise, SpecConst sc)
{
    h0_tile<SRC>(h0, uv, noise, sc);
}

// uv of the spectra of a list (blockIdx.z), all of size N, as they stand.
__global__ __launch_bounds__(kH0Tile* kH0Tile) void k_fold(FoldList list, int N)
{
    SpecConst sc{};
    sc.N         = N;
    sc.conj_mode = list.conj_mode[blockIdx.z];
    h0_tile<kStored>(list.h0[blockIdx.z], list.uv[blockIdx.z], nullptr, sc);
}

// Pass API: the three spectrum textures of tilde_h0_t (dy, dx, dz), float2 each.
__global__ __launch_bounds__(256) void k_tilde_h0_t(const float4* __restrict__ h0, float2* __restrict__ hy,
                                                    float2* __restrict__ hx, float2* __restrict__ hz, SpecConst sc,
                                                    double t_rev)
{
    const int tx = blockIdx.x * blockDim.x + threadIdx.x;
    const int ty = blockIdx.y;
    if (tx >= sc.N) return;
    const size_t i  = (size_t)ty * sc.N + tx;
    const int    nx = tx - sc.N / 2, ny = ty - sc.N / 2;
    float kinv, s, c;
    sincos_turns(phase_turns(sc, nx * nx + ny * ny, t_rev, kinv), s, c);
    const float2 h = evolve_amp(sc, h0[i], s, c);
    hy[i] = h;
    hx[i] = choppy((float)nx * kinv, h);
    hz[i] = choppy((float)ny * kinv, h);
}

// ------------------------------------------------------------------ fused frame, pass 1

// Column pass: 1-D grid of (strip groups x frames x G) blocks, one strip of one
// frame each.  Block order (after the XCD remap): group-major, then frame, then
// strip, so a group's columns of the folded spectrum (the same for every frame)
// and the Z lines its G strips fill together are served by one XCD's L2.
template <int N, int C>
__device__ __forceinline__ void cols_block(const FrameBatch& fb, int& f, int& strip)
{
    constexpr int G = strip_group<N, C>();
    const int L    = xcd_logical(blockIdx.x, gridDim.x);
    const int rest = L / G;
    f     = rest % fb.nframes;
    strip = (rest / fb.nframes) * G + L % G;
}

// Register strips (cols_strip): C columns x T = N/8 threads, four waves per SIMD.
// Radix 8: a thread holds its column's three fields in 128 registers; at radix 16
// they take 190-210 (two waves per SIMD; capped at three, they spill).  Against
// the strips it replaced, us per frame (column pass alone): N=1024, 16 frames per
// launch 4.56 -> 3.6 (4 columns); N=2048, 4 frames 26.8 -> 17.6; N=4096, 4 frames
// 179 -> 151; the 192-cascade batch 627 -> 430 us.  It writes 12 B/texel at 3.5 TB/s
// (N=1024): bound by the chain of each block's phases, two blocks of eight waves per
// CU deep.
template <int N, int C>
__global__ __launch_bounds__(C*(N / 8), 4) void k_cols(const float4* __restrict__ uv, float2* __restrict__ z1,
                                                       float2* __restrict__ z2, const float2* __restrict__ tw,
                                                       SpecConst sc, FrameBatch fb)
{
    __shared__ float2 lds[C * strip_len(N)];
    int f, strip;
    cols_block<N, C>(fb, f, strip);
    if (strip >= lds_strips<N, C>()) return;  // padding of the last group (whole block)
    cols_strip<N, 8, C, C*(N / 8)>(uv, z1 + (size_t)f * fb.z1_stride, z2 + (size_t)f * fb.z2_stride, tw, sc,
                                   fb.t_rev[f], strip, lds);
}

// LDS-staged strips (cols_lds_strip), for launches of few frames: a short chain from
// the first load to the last store.  Threads for the strip's C (N/2 + 1) row pairs, and
// with them its stores, in one round where a block of 1024 holds them, else twice the
// transforms' 3C x T; those past the transforms fold and store only.  A second round
// puts another trip to memory and another dispersion phase behind the first: with
// twice the transforms' threads at every size, single frames (us) N=64 8.5 -> 7.6, 128
// 8.8 -> 8.0, 256 9.5 -> 8.8, 512 12.9 -> 12.6, 1024 27.0 -> 26.6.
template <int N, int C>
constexpr int cols_lds_threads()
{
    constexpr int one = (C * (N / 2 + 1) + 63) / 64 * 64;
    return one <= 1024 ? one : 2 * 3 * C * (N / 16);
}
template <int N, int C>
__global__ __launch_bounds__((cols_lds_threads<N, C>())) void k_cols_lds(const float4* __restrict__ uv,
                                                                        float2* __restrict__ z1,
                                                                        float2* __restrict__ z2,
                                                                        const float2* __restrict__ tw, SpecConst sc,
                                                                        FrameBatch fb)
{
    __shared__ float2 lds[3 * C * strip_len(N)];
    int f, strip;
    cols_block<N, C>(fb, f, strip);
    if (strip >= lds_strips<N, C>()) return;  // padding of the last group (whole block)
    cols_lds_strip<N, C, cols_lds_threads<N, C>()>(uv, z1 + (size_t)f * fb.z1_stride, z2 + (size_t)f * fb.z2_stride,
                                                   tw, sc, fb.t_rev[f], strip, lds);
}

// ------------------------------------------------------------------ fused frame, pass 2

// Row pass.  Grid = (N/2, frames).  Block p handles rows 2p and 2p+1: group 0
// transforms Z1 row 2p, group 1 Z1 row 2p+1, group 2 Z2 row p (whose real and
// imaginary parts are Dz of rows 2p and 2p+1), then applies the inversion step
// (-1)^(x+y) / N^2 (inversion_cs.glsl:35-41).
template <int N, int E>
__global__ __launch_bounds__(3 * (N / E)) void k_rows(const float2* __restrict__ z1, const float2* __restrict__ z2,
                                                      float* __restrict__ height, float* __restrict__ dx,
                                                      float* __restrict__ dz, const float2* __restrict__ tw,
                                                      FrameBatch fb)
{
    constexpr int T = N / E;
    __shared__ float2 lds[3 * lds_len(N)];
    const int f = blockIdx.y;
    z1 += (size_t)f * fb.z1_stride;
    z2 += (size_t)f * fb.z2_stride;
    const size_t o = (size_t)f * fb.out_stride;
    height += o;
    dx += o;
    dz += o;
    const int g = threadIdx.x / T;
    const int j = threadIdx.x % T;
    const int p = blockIdx.x;
    // Z1 rows 2p, 2p+1 form one two-row tile (zidx); Z2 row p is read alone
    const float2* src = g == 2 ? z2 : z1;
    const int     y   = g == 2 ? p : 2 * p + g;
    float2 v[E];
#pragma unroll
    for (int r = 0; r < E; ++r) v[r] = src[zidx<N>(y, zpos_elem<N, E>(j, r))];
    fft_inverse<N, E>(v, j, lds + g * lds_len(N), tw, BlockSync{});
    constexpr float scale = 1.0f / ((float)N * (float)N);
    const size_t row0 = (size_t)(2 * p) * N, row1 = row0 + N;
#pragma unroll
    for (int r = 0; r < E; ++r) {
        const int   x = j + r * T;
        const float s = (x & 1) ? -scale : scale;  // sign of row 2p; row 2p+1 has the opposite sign
        if (g == 0) {
            height[row0 + x] = s * v[r].x;
            dx[row0 + x]     = s * v[r].y;
        } else if (g == 1) {
            height[row1 + x] = -s * v[r].x;
            dx[row1 + x]     = -s * v[r].y;
        } else {
            dz[row0 + x] = s * v[r].x;
            dz[row1 + x] = -s * v[r].y;
        }
    }
}

// ------------------------------------------------------------------ fused row pass + normals + Jacobian

// Row pass fused with the normal map (nearest taps) and the Jacobian: each
// group of T = N/E threads walks one band of R rows (rows_nrm_band).  Groups
// lie in one wave when T <= 64 (wave-level ordering), otherwise a block is one
// group.  1-D grid of ceil(bands*frames / groups per block) blocks; after the
// XCD remap, neighbouring bands (which share halo rows) run on the same XCD.
// At least two waves per SIMD: the band walk holds about 260 registers a lane
// when left unbounded, and one wave per SIMD cannot hide its load latency (the
// bound trades that for a few spilled registers; N=1024 frames 18.7 -> 17.6 us).
template <int N, int E, int R, bool RENDER>
__global__ __launch_bounds__(N / E >= 64 ? N / E : 64, 2) void k_rows_nrm(
    const float2* __restrict__ z1, const float2* __restrict__ z2, float* __restrict__ height,
    float* __restrict__ dx, float* __restrict__ dz, float4* __restrict__ normals, float* __restrict__ jac,
    const float2* __restrict__ tw, FrameBatch fb, float lambda, float inv2d, float4* __restrict__ disp,
    float4* __restrict__ rnorm, float dscale)
{
    constexpr int T   = N / E;
    constexpr int GPB = T >= 64 ? 1 : 64 / T;  // groups per block
    constexpr int NB  = N / R;                  // bands per frame
    using Sync = typename std::conditional<(T <= 64), WaveSync, BlockSync>::type;
    __shared__ float2 lds[GPB * lds_len(N)];
    // With one group per block (block = T threads) g is 0: stated at compile
    // time so that the frame and its buffer offsets stay scalar.
    const int g    = GPB == 1 ? 0 : (int)threadIdx.x / T;
    const int j    = GPB == 1 ? (int)threadIdx.x : (int)threadIdx.x % T;
    const int L    = xcd_logical(blockIdx.x, gridDim.x) * GPB + g;
    const int band = L % NB;
    const int f    = L / NB;
    if (f >= fb.nframes) return;  // whole group (a wave part when T <= 64): padding of the last block
    const size_t fo = (size_t)f * fb.out_stride;
    // Z2 rows paired up to N=1024 (N=512 frames -4%, N=1024 -1%), and at N=2048
    // without the render export (247 registers with the upward walk, N=2048
    // frames -0.4%; the render variant would spill).  Odd bands walk upwards
    // from N=1024 (halo tiles shared in time with the neighbours)
    static_assert(R % 2 == 0 && N % R == 0, "bands of an even number of rows");
    constexpr bool PAIR2 = N <= 1024 || (N <= 2048 && !RENDER);
    rows_nrm_band<N, E, Sync, RENDER, PAIR2, (N >= 1024)>(
        z1 + (size_t)f * fb.z1_stride, z2 + (size_t)f * fb.z2_stride, height + fo, dx + fo, dz + fo,
        normals ? normals + fo : nullptr, jac ? jac + fo : nullptr, tw, lds + g * lds_len(N), j, band, R, lambda,
        inv2d, disp ? disp + fo : nullptr, rnorm ? rnorm + fo : nullptr, dscale);
}

// ------------------------------------------------------------------ fused row pass, parallel bands

// Row pass fused with the normal map and the Jacobian for launches of few
// frames: where the band walk of k_rows_nrm runs its rows one after another
// (long bands, few groups), here one block owns a band of R output rows
// [y0, y0 + R) and transforms all the rows its stencils need at once: Z1 rows
// y0 - 1 .. y0 + R and Z2 rows y0/2 - 1 .. y0/2 + R/2, one T-thread group
// (radix E) each.  The results stay in the groups' LDS buffers in natural
// order; after one block barrier every thread takes texels of the band, applies
// (-1)^(x+y) / N^2 (inversion_cs.glsl:35-41) to each value it reads and computes
// the Sobel normal (normal_map_cs.glsl:37-53) and the Jacobian of the render
// displacement (grid_tes.glsl:60-62) with the band walk's arithmetic.  1-D grid
// of (N/R) x frames blocks; after the XCD remap neighbouring bands, which read
// the same halo tiles, run on one XCD.
//
// RENDER adds the render export (disp, rnorm, either may be null), as in the walk.
// Launches of 2^19 to 2^22 texels write it by plain stores: an export of 134 MB, half
// of the Infinity Cache, stays there.  With all outputs non-temporal, frames written
// to the same buffers over and over were slower than the unfused passes (N=512, 8
// frames, us per frame: unfused 5.8, non-temporal 6.3, plain 5.5; into buffers that
// change 6.4, 5.4, 5.1; N=1024, 2 frames 24.3, 25.2, 23.4).  Larger exports do not stay
// in the cache (N=512, 32 frames: non-temporal 4.13, plain 4.34); smaller ones would
// stay in the L2s and be written back at the launch's end (N=512, single frames 13.5,
// 14.2).
// BIL takes the height taps bilinearly at texel corners (OCN_NORMALS_BILINEAR):
// the 2x2 box folded into the Sobel weights is [1 3 3 1] along one axis and
// [1 1 -1 -1] along the other over x-2..x+1, y-2..y+1, so one more Z1 row is
// transformed above the band.  Both used to take the unfused row pass and the
// normal-map kernel, which read height, Dx and Dz back: 12 bytes a texel and a
// launch more.  Whole frames, unfused -> here (us per frame): render export N=256
// 17.0 -> 10.2 (single), 2.09 -> 1.66 (16 per launch), N=512 20.9 -> 13.5, N=1024
// 38.4 -> 32.0; bilinear N=256 17.5 -> 9.2, N=512 21.5 -> 12.6 and 5.2 -> 3.9
// (8 per launch), N=1024 33.4 -> 25.7 and 18.9 -> 13.0 (16), N=2048 88 -> 66 (4).
template <int N, int E, int R, bool BIL = false>
constexpr int par_groups()
{
    return (R + 2 + (BIL ? 1 : 0)) + (R / 2 + 2);
}

template <int N, int E, int R, int W, bool BIL, bool RENDER>
__global__ __launch_bounds__((W * par_groups<N, E, R, BIL>() * (N / E))) void k_rows_nrm_par(
    const float2* __restrict__ z1, const float2* __restrict__ z2, float* __restrict__ height,
    float* __restrict__ dx, float* __restrict__ dz, float4* __restrict__ normals, float* __restrict__ jac,
    const float2* __restrict__ tw, FrameBatch fb, float lambda, float inv2d, float4* __restrict__ disp,
    float4* __restrict__ rnorm, float dscale, bool plain)
{
    // W = 2: twice the threads, the extra ones (after the G transform groups)
    // taking part in the stencils only
    constexpr int UP = BIL ? 2 : 1;  // rows above the band
    constexpr int T = N / E, G1 = R + UP + 1, G = par_groups<N, E, R, BIL>(), LEN = lds_len(N), NT = W * G * T;
    static_assert(R % 2 == 0 && N % R == 0, "bands of an even number of rows");
    static_assert(T % 64 == 0 || 64 % T == 0, "transform groups of whole waves or within one wave");
    static_assert(W == 1 || T <= 64, "extra threads only beside wave-local transforms");
    using Sync = typename std::conditional<(T <= 64), WaveSync, BlockSync>::type;
    constexpr float scale = 1.0f / ((float)N * (float)N);
    __shared__ float2 lds[G * LEN];
    const int L    = xcd_logical(blockIdx.x, gridDim.x);
    const int band = L % (N / R);
    const int f    = L / (N / R);
    const int y0   = band * R;
    z1 += (size_t)f * fb.z1_stride;
    z2 += (size_t)f * fb.z2_stride;
    const size_t fo = (size_t)f * fb.out_stride;
    height += fo;
    dx += fo;
    dz += fo;
    if (normals) normals += fo;
    if (jac) jac += fo;
    if (RENDER && disp) disp += fo;
    if (RENDER && rnorm) rnorm += fo;

    if (W == 1 || (int)threadIdx.x < G * T) {
        const int g = threadIdx.x / T, j = threadIdx.x % T;
        // group g < G1: Z1 row y0 - UP + g; else Z2 row y0/2 - 1 + (g - G1) (periodic)
        const bool    is1 = g < G1;
        const float2* src = is1 ? z1 : z2;
        const int     row = is1 ? (y0 - UP + g) & (N - 1) : ((y0 >> 1) - 1 + (g - G1)) & (N / 2 - 1);
        float2        v[E];
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = src[zidx<N>(row, zpos_elem<N, E>(j, r))];
        float2* buf = lds + g * LEN;
        fft_inverse<N, E>(v, j, buf, tw, Sync{});
        Sync{}();
#pragma unroll
        for (int r = 0; r < E; ++r) buf[lds_pad(j + r * T)] = v[r];
    }
    __syncthreads();

    auto put = [&](float4* p, float4 v) {
        if (plain) *p = v;
        else st_out(p, v);
    };
    // Stencils: each thread walks whole columns x of the band, keeping the
    // signed values of x-1, x, x+1 for all band and halo rows in registers
    // (each LDS value is read once per column).  The sign (-1)^(x+y) / N^2 of
    // texel (x, y): rows y0 - UP + g alternate starting from that of
    // (x, y0 - UP) (y0 is even); columns x +- 1 have the opposite sign of x.
    constexpr int G2 = G - G1;
    for (int x = threadIdx.x; x < N; x += NT) {
        const int   pl = lds_pad((x - 1) & (N - 1)), pm = lds_pad(x), pr = lds_pad((x + 1) & (N - 1));
        const float s0 = ((x + UP) & 1) ? -scale : scale;  // (x, y0 - UP)
        float2 hl[G1], hm[G1], hr[G1];  // (height, Dx) of rows y0 - UP .. y0 + R at x - 1, x, x + 1
        float  hll[BIL ? G1 : 1];       // height at x - 2
#pragma unroll
        for (int g = 0; g < G1; ++g) {
            const float  sm = (g & 1) ? -s0 : s0;
            const float2 l = lds[g * LEN + pl], m = lds[g * LEN + pm], r = lds[g * LEN + pr];
            hl[g] = make_float2(-sm * l.x, -sm * l.y);
            hm[g] = make_float2(sm * m.x, sm * m.y);
            hr[g] = make_float2(-sm * r.x, -sm * r.y);
            if constexpr (BIL) hll[g] = sm * lds[g * LEN + lds_pad((x - 2) & (N - 1))].x;
        }
        // Dz of rows y0 - 1 .. y0 + R (index 0 .. R + 1): Z2 row y0/2 - 1 + q holds
        // rows y0 - 2 + 2q (re) and y0 - 1 + 2q (im), i.e. indices 2q - 1, 2q
        const float z0 = ((x + 1) & 1) ? -scale : scale;  // (x, y0 - 1)
        float zl[R + 2], zm[R + 2], zr[R + 2];
#pragma unroll
        for (int q = 0; q < G2; ++q) {
            const float2 l = lds[(G1 + q) * LEN + pl], m = lds[(G1 + q) * LEN + pm], r = lds[(G1 + q) * LEN + pr];
#pragma unroll
            for (int part = 0; part < 2; ++part) {
                const int i = 2 * q - 1 + part;
                if (i < 0 || i >= R + 2) continue;
                const float sm = (i & 1) ? -z0 : z0;
                zl[i] = -sm * (part ? l.y : l.x);
                zm[i] = sm * (part ? m.y : m.x);
                zr[i] = -sm * (part ? r.y : r.x);
            }
        }
#pragma unroll
        for (int k = 0; k < R; ++k) {
            const int    g = k + UP, i = k + 1;  // grid row y0 + k
            const size_t o = (size_t)(y0 + k) * N + x;
            if (normals) {
                float nx, nz;
                if constexpr (BIL) {
                    auto vs = [&](float a, float b, float c, float d) { return a + 3.0f * (b + c) + d; };
                    auto ds = [&](float a, float b, float c, float d) { return (a + b) - (c + d); };
                    const float v0 = vs(hll[g - 2], hll[g - 1], hll[g], hll[g + 1]);
                    const float v1 = vs(hl[g - 2].x, hl[g - 1].x, hl[g].x, hl[g + 1].x);
                    const float v2 = vs(hm[g - 2].x, hm[g - 1].x, hm[g].x, hm[g + 1].x);
                    const float v3 = vs(hr[g - 2].x, hr[g - 1].x, hr[g].x, hr[g + 1].x);
                    const float d0 = ds(hll[g - 2], hll[g - 1], hll[g], hll[g + 1]);
                    const float d1 = ds(hl[g - 2].x, hl[g - 1].x, hl[g].x, hl[g + 1].x);
                    const float d2 = ds(hm[g - 2].x, hm[g - 1].x, hm[g].x, hm[g + 1].x);
                    const float d3 = ds(hr[g - 2].x, hr[g - 1].x, hr[g].x, hr[g + 1].x);
                    nx = 0.25f * ds(v0, v1, v2, v3);
                    nz = 0.25f * vs(d0, d1, d2, d3);
                } else {
                    // v_s = h(y-1) + 2 h(y) + h(y+1), d_s = h(y-1) - h(y+1) at x-1, x, x+1;
                    // nx = v_s(x-1) - v_s(x+1), nz = d_s(x-1) + 2 d_s(x) + d_s(x+1)
                    const float vl  = hl[g - 1].x + 2.0f * hl[g].x + hl[g + 1].x;
                    const float vr  = hr[g - 1].x + 2.0f * hr[g].x + hr[g + 1].x;
                    nx = vl - vr;
                    nz = (hl[g - 1].x - hl[g + 1].x) + 2.0f * (hm[g - 1].x - hm[g + 1].x) +
                         (hr[g - 1].x - hr[g + 1].x);
                }
                const float inv = rsqrtf(fmaf(nx, nx, fmaf(nz, nz, 1.0f)));
                st_out(&normals[o], make_float4(nx * inv, inv, nz * inv, 1.0f));
            }
            if (jac || (RENDER && (disp || rnorm))) {
                const float dxdx = (hr[g].y - hl[g].y) * inv2d;
                const float dzdx = (zr[i] - zl[i]) * inv2d;
                const float dxdz = (hm[g + 1].y - hm[g - 1].y) * inv2d;
                const float dzdz = (zm[i + 1] - zm[i - 1]) * inv2d;
                const float J = (1.0f - lambda * dxdx) * (1.0f - lambda * dzdz) - lambda * lambda * dxdz * dzdx;
                if (jac) st_out(&jac[o], J);
                if (RENDER && disp) put(&disp[o], make_float4(-lambda * hm[g].y, dscale * hm[g].x, -lambda * zm[i], J));
                if (RENDER && rnorm) {
                    // n = dP/dv x dP/du (rows_nrm_band); its y component is J
                    const float dhdx = (hr[g].x - hl[g].x) * inv2d, dhdz = (hm[g + 1].x - hm[g - 1].x) * inv2d;
                    const float nx  = -dscale * (lambda * dhdz * dzdx + (1.0f - lambda * dzdz) * dhdx);
                    const float nz  = -dscale * (lambda * dxdz * dhdx + dhdz * (1.0f - lambda * dxdx));
                    const float inv = rsqrtf(fmaf(nx, nx, fmaf(J, J, nz * nz)));
                    put(&rnorm[o], make_float4(nx * inv, J * inv, nz * inv, 1.0f));
                }
            }
            st_out(&height[o], hm[g].x);
            st_out(&dx[o], hm[g].y);
            st_out(&dz[o], zm[i]);
        }
    }
}

// ------------------------------------------------------------------ A7 normals (+ Jacobian)

// normal_map_cs.glsl:24-54 (Sobel on the height, ny = 1, normalize, w = 1),
// and optionally the Jacobian J = (1 - l dDx/dx)(1 - l dDz/dz) - l^2 dDx/dz dDz/dx
// of the render displacement (-l Dx, -l Dz) (grid_tes.glsl:60-62), by periodic
// central differences with spacing L/N.
//
// Tiled: a block owns a 64 x H texel tile and first stages height/dx/dz for
// the tile plus a 2-texel periodic halo in LDS with coalesced row loads (the
// bilinear taps reach two texels down/left, the others one), then every tap
// comes from LDS.  1-D grid of (N/64) x (N/H) x frames blocks; frame f reads
// and writes at offset f*stride.  After the XCD remap, tiles of neighbouring
// rows run on the same XCD, so the halo rows are L2 hits.
constexpr int kNrmW = 64, kNrmHalo = 2;
constexpr int kNrmLW = kNrmW + 2 * kNrmHalo;
// H = 16 reads 1.25 rows per row kept and is what memory wants where the grid
// fills the chip (N = 4096: 131 us, H = 4 196; N = 2048: 24 against 32).  A grid
// below four blocks per CU waits for the chain of one block instead, seven
// staging loads and four texels in each thread; H = 4 cuts it to three and one:
// back to back N = 64 5.7 -> 3.2 us, N = 256 6.0 -> 3.4, N = 512 6.5 -> 4.8 (H = 8:
// 4.1, 4.3, 5.2).  N = 1024 sits at four blocks: 9.3 with 16, 10.5 with 4.
constexpr int normals_tile_rows(int N, int nframes) { return (N / kNrmW) * (N / 16) * nframes >= 1024 ? 16 : 4; }

// texture() of the staged tile under NEAREST + REPEAT (s[y][x], halo-offset
// coordinates) or LINEAR + REPEAT at a texel corner: 2x2 box over (x-1..x, y-1..y).
__device__ __forceinline__ float stap(const float (*s)[kNrmLW], int y, int x, int mode)
{
    return mode ? 0.25f * (s[y - 1][x - 1] + s[y - 1][x] + s[y][x - 1] + s[y][x]) : s[y][x];
}

template <int H>
__global__ __launch_bounds__(256) void k_normals(const float* __restrict__ height, const float* __restrict__ dx,
                                                 const float* __restrict__ dz, float4* __restrict__ normals,
                                                 float* __restrict__ jac, int N, int mode, float lambda,
                                                 float inv2d, size_t stride, float4* __restrict__ disp,
                                                 float4* __restrict__ rnorm, float dscale)
{
    constexpr int LH = H + 2 * kNrmHalo;
    __shared__ float sh[LH][kNrmLW], sx[LH][kNrmLW], sz[LH][kNrmLW];
    const int tiles_x = N / kNrmW, tiles_y = N / H;
    const int L  = xcd_logical(blockIdx.x, gridDim.x);
    const int bx = L % tiles_x;
    const int by = (L / tiles_x) % tiles_y;
    const int f  = L / (tiles_x * tiles_y);
    const size_t fo = (size_t)f * stride;
    height += fo;
    dx += fo;
    dz += fo;
    if (normals) normals += fo;
    if (jac) jac += fo;
    if (disp) disp += fo;
    if (rnorm) rnorm += fo;
    const bool need_h = normals || disp || rnorm, need_xz = jac || disp || rnorm;
    const int x0 = bx * kNrmW, y0 = by * H;
    for (int k = threadIdx.x; k < LH * kNrmLW; k += 256) {
        const int ly = k / kNrmLW, lx = k % kNrmLW;
        const size_t gi = (size_t)((y0 + ly - kNrmHalo) & (N - 1)) * N + ((x0 + lx - kNrmHalo) & (N - 1));
        if (need_h) sh[ly][lx] = height[gi];
        if (need_xz) {
            sx[ly][lx] = dx[gi];
            sz[ly][lx] = dz[gi];
        }
    }
    __syncthreads();
    const int cx = (threadIdx.x & 63) + kNrmHalo;
#pragma unroll
    for (int k = 0; k < H / 4; ++k) {
        const int ly = (threadIdx.x >> 6) + 4 * k;
        const int cy = ly + kNrmHalo;
        const size_t i = (size_t)(y0 + ly) * N + x0 + (threadIdx.x & 63);
        if (normals) {
            // z0..z7 at (x-1,y-1) (x,y-1) (x+1,y-1) (x-1,y) (x+1,y) (x-1,y+1) (x,y+1) (x+1,y+1)
            const float z0 = stap(sh, cy - 1, cx - 1, mode), z1 = stap(sh, cy - 1, cx, mode);
            const float z2 = stap(sh, cy - 1, cx + 1, mode), z3 = stap(sh, cy, cx - 1, mode);
            const float z4 = stap(sh, cy, cx + 1, mode), z5 = stap(sh, cy + 1, cx - 1, mode);
            const float z6 = stap(sh, cy + 1, cx, mode), z7 = stap(sh, cy + 1, cx + 1, mode);
            const float nz  = z0 + 2.0f * z1 + z2 - z5 - 2.0f * z6 - z7;
            const float nx  = z0 + 2.0f * z3 + z5 - z2 - 2.0f * z4 - z7;
            const float inv = rsqrtf(fmaf(nx, nx, fmaf(nz, nz, 1.0f)));
            normals[i] = make_float4(nx * inv, inv, nz * inv, 1.0f);
        }
        if (need_xz) {
            const float dxdx = (sx[cy][cx + 1] - sx[cy][cx - 1]) * inv2d;
            const float dxdz = (sx[cy + 1][cx] - sx[cy - 1][cx]) * inv2d;
            const float dzdx = (sz[cy][cx + 1] - sz[cy][cx - 1]) * inv2d;
            const float dzdz = (sz[cy + 1][cx] - sz[cy - 1][cx]) * inv2d;
            const float J    = (1.0f - lambda * dxdx) * (1.0f - lambda * dzdz) - lambda * lambda * dxdz * dzdx;
            if (jac) jac[i] = J;
            if (disp) disp[i] = make_float4(-lambda * sx[cy][cx], dscale * sh[cy][cx], -lambda * sz[cy][cx], J);
            if (rnorm) {
                // n = dP/dv x dP/du of P = (u - l Dx, s h, v - l Dz); its y component is J
                const float dhdx = (sh[cy][cx + 1] - sh[cy][cx - 1]) * inv2d;
                const float dhdz = (sh[cy + 1][cx] - sh[cy - 1][cx]) * inv2d;
                const float nx   = -dscale * (lambda * dhdz * dzdx + (1.0f - lambda * dzdz) * dhdx);
                const float nz   = -dscale * (lambda * dxdz * dhdx + dhdz * (1.0f - lambda * dxdx));
                const float inv  = rsqrtf(fmaf(nx, nx, fmaf(J, J, nz * nz)));
                rnorm[i] = make_float4(nx * inv, J * inv, nz * inv, 1.0f);
            }
        }
    }
}

static void normals_pass(int N, int nframes, const float* height, const float* dx, const float* dz, float4* normals,
                         float* jac, int mode, float lambda, float inv2d, size_t stride, float4* disp, float4* rnorm,
                         float dscale, hipStream_t s)
{
    const int H = normals_tile_rows(N, nframes);
    hipLaunchKernelGGL(H == 16 ? k_normals<16> : k_normals<4>, dim3((N / kNrmW) * (N / H) * nframes), dim3(256), 0, s,
                       height, dx, dz, normals, jac, N, mode, lambda, inv2d, stride, disp, rnorm, dscale);
}

// ------------------------------------------------------------------ A5+A6 pass API (general complex input)

// The inversion pass keeps Re of the inverse DFT of F, which is the inverse DFT
// of F's Hermitian part A(y, x) = (F(y, x) + conj F(-y, -x))/2.  So:
//   rows     A's rows 0..N/2 only (row N-y of the result is the conjugate of row
//            y's); rows 0 and N/2 have real results and share one transform;
//   columns  the results are real: two columns share one transform.
// Half the transforms and half the intermediate (4 instead of 8 bytes a texel)
// of transforming F itself: 20 instead of 28 bytes a texel cross the kernels.
// Both calls' time against whole complex transforms (us): N=256 6.2 -> 6.2 (two
// launches), 512 9.1 -> 6.4, 1024 16.0 -> 10.9, 2048 48.9 -> 22.9, 4096 302 ->
// 74; at N=2048 84 MB move at 3.7 TB/s, one block of 16 waves per CU and kernel.
//
// Rows: a group of T = N/E threads per row y < N/2, which reads rows y and N-y of
// src.  mid row y: the row's transform; row 0: that of row 0 in the real parts,
// of row N/2 in the imaginary parts.
template <int N, int E, int NB>
__global__ __launch_bounds__(NB) void k_ifft2_rows(const float2* __restrict__ src, float2* __restrict__ mid,
                                                   const float2* __restrict__ tw)
{
    constexpr int T = N / E, GPB = NB / T;
    using Sync = typename std::conditional<(T <= 64), WaveSync, BlockSync>::type;
    static_assert(NB % T == 0 && (T <= 64 || GPB == 1), "groups inside a wave, or one per block");
    __shared__ float2 lds[GPB * lds_len(N)];
    const int g = threadIdx.x / T, j = threadIdx.x % T;
    const int y = blockIdx.x * GPB + g;
    // the Hermitian part of src's row a (mirror row b)
    auto fold = [&](int a, int b, float2 (&v)[E]) {
        float2 m[E];
#pragma unroll
        for (int r = 0; r < E; ++r) {
            const int x = j + r * T;
            v[r] = src[(size_t)a * N + x];
            m[r] = src[(size_t)b * N + ((N - x) & (N - 1))];
        }
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = make_float2(0.5f * (v[r].x + m[r].x), 0.5f * (v[r].y - m[r].y));
    };
    float2 v[E];
    fold(y, (N - y) & (N - 1), v);
    if (y == 0) {
        float2 w[E];
        fold(N / 2, N / 2, w);
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = make_float2(v[r].x - w[r].y, v[r].y + w[r].x);
    }
    fft_inverse<N, E>(v, j, lds + g * lds_len(N), tw, Sync{});
#pragma unroll
    for (int r = 0; r < E; ++r) mid[(size_t)y * N + j + r * T] = v[r];
}

// Columns + inversion, out = (-1)^(x+y) (.) / N^2: C column pairs (2p, 2p + 1) per
// block, a group of T = N/E threads each; Z = R(., 2p) + i R(., 2p+1), whose rows
// above N/2 follow from mid's by conjugation.  Both ways go through LDS, where
// C lanes read 16C contiguous bytes of a mid row and write 8C of an output row.
// V2: out is 8-byte aligned.
template <int N, int E, int C, bool V2>
__global__ __launch_bounds__(C*(N / E)) void k_ifft2_cols_inv(const float2* __restrict__ mid, float* __restrict__ out,
                                                              const float2* __restrict__ tw)
{
    constexpr int T = N / E, NB = C * T, LEN = strip_len(N);
    using Sync = typename std::conditional<(T <= 64), WaveSync, BlockSync>::type;
    constexpr float scale = 1.0f / ((float)N * (float)N);
    __shared__ float2 lds[C * LEN];
    const int p0 = xcd_logical(blockIdx.x, gridDim.x) * C;
#pragma unroll
    for (int it = 0; it < E / 2; ++it) {
        const int    k = threadIdx.x + it * NB, c = k % C, y = k / C;
        const float4 q = reinterpret_cast<const float4*>(mid + (size_t)y * N)[p0 + c];
        float2*      buf = lds + c * LEN;
        buf[lds_pad(y)]                       = y == 0 ? make_float2(q.x, q.z) : make_float2(q.x - q.w, q.y + q.z);
        buf[lds_pad(y == 0 ? N / 2 : N - y)] = y == 0 ? make_float2(q.y, q.w) : make_float2(q.x + q.w, q.z - q.y);
    }
    __syncthreads();
    {
        const int j = threadIdx.x % T;
        float2*   buf = lds + (threadIdx.x / T) * LEN;
        float2    v[E];
#pragma unroll
        for (int r = 0; r < E; ++r) v[r] = buf[lds_pad(j + r * T)];
        fft_inverse<N, E>(v, j, buf, tw, Sync{});
        Sync{}();
#pragma unroll
        for (int r = 0; r < E; ++r) buf[lds_pad(j + r * T)] = v[r];
    }
    __syncthreads();
#pragma unroll
    for (int it = 0; it < E; ++it) {
        const int    k = threadIdx.x + it * NB, c = k % C, y = k / C;
        const float2 q = lds[c * LEN + lds_pad(y)];
        const float  s = (y & 1) ? -scale : scale;  // of the even column
        float*       o = out + (size_t)y * N + 2 * (p0 + c);
        if constexpr (V2) {
            *reinterpret_cast<float2*>(o) = make_float2(s * q.x, -s * q.y);
        } else {
            o[0] = s * q.x;
            o[1] = -s * q.y;
        }
    }
}

// ------------------------------------------------------------------ launchers

// Column-pass schedules: columns per block C of k_cols (radix 8), or lds: of
// k_cols_lds (radix 16; the three transforms of a column side by side, folds
// staged in LDS).  The numbers of earlier builds, which had a kernel for most
// of them, stay valid for the sizes [min_N, max_N] that took them, in calls and
// in saved autotune files; several now name one kernel.  A strip is at most
// 1024 threads wide (cols_width).
struct ColsVariant {
    int  C;
    bool lds;
    int  min_N, max_N;
};
constexpr ColsVariant kColsVariants[kNumColsVariants] = {
    {1, false, 64, 4096},   {2, false, 64, 4096},   {4, false, 64, 4096},   {8, false, 64, 2048},
    {2, false, 64, 4096},   {4, false, 64, 2048},   {8, false, 64, 1024},   {1, false, 64, 1024},
    {2, false, 64, 1024},   {4, false, 64, 1024},   {2, false, 64, 1024},   {4, false, 64, 1024},
    {8, false, 64, 1024},   {1, true, 64, 1024},    {2, true, 64, 1024},    {2, false, 2048, 4096},
    {2, false, 2048, 2048}, {2, false, 2048, 4096}, {4, false, 2048, 2048}, {4, false, 64, 512},
    {8, false, 64, 256},    {4, true, 64, 512}};
constexpr int cols_width(int N, int C) { return C * (N / 8) <= 1024 ? C : 1024 / (N / 8); }
// Row-pass schedules: band 0 = k_rows (radix E) followed by k_normals;
// band R > 0 = k_rows_nrm with bands of R rows (radix E), normals fused;
// par = k_rows_nrm_par (bands of R rows whose rows are transformed at once).
struct RowsVariant {
    int  E, band;
    bool par;
    int  W;  // parallel bands: threads per transform-group thread
};
constexpr RowsVariant kRowsVariants[kNumRowsVariants] = {{16, 0, false, 1}, {8, 0, false, 1},  {8, 4, false, 1},
                                                         {8, 8, false, 1},  {8, 16, false, 1}, {8, 32, false, 1},
                                                         {16, 4, true, 1},  {16, 2, true, 1},  {16, 2, true, 2}};

constexpr bool cols_fits(int N, int v) { return N >= kColsVariants[v].min_N && N <= kColsVariants[v].max_N; }
template <int N, int E, int B, bool PAR = false, int W = 1, bool BIL = false>
constexpr bool rows_fits()
{
    if constexpr (PAR) {
        constexpr int T = N / E, G = par_groups<N, E, B, BIL>();
        return N >= 2 * E && N % B == 0 && (T % 64 == 0 || 64 % T == 0) && (W == 1 || T <= 64) &&
               W * G * T <= 1024 && G * lds_len(N) * 8 <= 160 * 1024;
    } else if constexpr (B == 0) {
        return N >= 2 * E && 3 * (N / E) <= 1024;
    } else {
        return N >= 2 * E && N % B == 0 && N / E <= 1024;
    }
}

constexpr int radix_slot(int E) { return E == 16 ? 1 : 0; }

template <int N, int V>
static hipError_t launch_cols_v(const FrameArgs& a, hipStream_t s)
{
    if constexpr (!cols_fits(N, V)) {
        return hipErrorInvalidValue;
    } else {
        constexpr int C = cols_width(N, kColsVariants[V].C);
        constexpr int G = strip_group<N, C>(), groups = (lds_strips<N, C>() + G - 1) / G;
        const dim3    grid(groups * G * a.nframes);
        if constexpr (kColsVariants[V].lds)
            hipLaunchKernelGGL((k_cols_lds<N, C>), grid, dim3(cols_lds_threads<N, C>()), 0, s, a.uv, a.z1, a.z2,
                               a.tw[radix_slot(16)], a.sc, a.fb);
        else
            hipLaunchKernelGGL((k_cols<N, C>), grid, dim3(C * (N / 8)), 0, s, a.uv, a.z1, a.z2, a.tw[radix_slot(8)],
                               a.sc, a.fb);
        return hipGetLastError();
    }
}

template <int N, int V>
static hipError_t launch_rows_v(const FrameArgs& a, hipStream_t s)
{
    constexpr int  E = kRowsVariants[V].E, B = kRowsVariants[V].band, W = kRowsVariants[V].W;
    constexpr bool P = kRowsVariants[V].par;
    if constexpr (!rows_fits<N, E, B, P, W>()) {
        return hipErrorInvalidValue;
    } else if constexpr (P) {
        auto launch = [&](auto bil, auto ren) {
            constexpr bool BIL = decltype(bil)::value, REN = decltype(ren)::value;
            const int      texels = a.nframes * N * N;
            if constexpr (!rows_fits<N, E, B, true, W, BIL>()) {
                return hipErrorInvalidValue;
            } else {
                hipLaunchKernelGGL((k_rows_nrm_par<N, E, B, W, BIL, REN>), dim3((N / B) * a.nframes),
                                   dim3(W * par_groups<N, E, B, BIL>() * (N / E)), 0, s, a.z1, a.z2, a.height, a.dx,
                                   a.dz, a.normals, a.jacobian, a.tw[radix_slot(E)], a.fb, a.lambda, a.inv2d, a.disp,
                                   a.rnorm, a.dscale, texels > (1 << 19) && texels <= (1 << 22));
                return hipGetLastError();
            }
        };
        const bool ren = a.disp || a.rnorm;
        if (a.normal_mode != 0) return ren ? launch(std::true_type{}, std::true_type{}) : launch(std::true_type{}, std::false_type{});
        return ren ? launch(std::false_type{}, std::true_type{}) : launch(std::false_type{}, std::false_type{});
    } else if constexpr (B == 0) {
        hipLaunchKernelGGL((k_rows<N, E>), dim3(N / 2, a.nframes), dim3(3 * (N / E)), 0, s, a.z1, a.z2, a.height,
                           a.dx, a.dz, a.tw[radix_slot(E)], a.fb);
        return hipGetLastError();
    } else {
        constexpr int T = N / E, GPB = T >= 64 ? 1 : 64 / T;
        const int groups = (N / B) * a.nframes;
        if (a.disp || a.rnorm)
            hipLaunchKernelGGL((k_rows_nrm<N, E, B, true>), dim3((groups + GPB - 1) / GPB), dim3(GPB * T), 0, s,
                               a.z1, a.z2, a.height, a.dx, a.dz, a.normals, a.jacobian, a.tw[radix_slot(E)], a.fb,
                               a.lambda, a.inv2d, a.disp, a.rnorm, a.dscale);
        else
            hipLaunchKernelGGL((k_rows_nrm<N, E, B, false>), dim3((groups + GPB - 1) / GPB), dim3(GPB * T), 0, s,
                               a.z1, a.z2, a.height, a.dx, a.dz, a.normals, a.jacobian, a.tw[radix_slot(E)], a.fb,
                               a.lambda, a.inv2d, nullptr, nullptr, 0.0f);
        return hipGetLastError();
    }
}

// The row variant that a frame with bilinear normals takes for rv: the walks
// read nearest taps only, so the parallel bands of 2 rows stand in for them; an
// N whose bands do not fit a block with the extra row (4096) runs the unfused
// radix-16 pass, and so does a single N = 2048 frame, whose textures the
// normal-map kernel reads back from the Infinity Cache (75 us against 78 with
// the bands, one block per CU; from 2 frames on 82 against 71).
template <int N>
constexpr int bilinear_rows(int rv, int nframes)
{
#define OCN_BFITS(v) \
    (rows_fits<N, kRowsVariants[v].E, kRowsVariants[v].band, kRowsVariants[v].par, kRowsVariants[v].W, true>())
    if (kRowsVariants[rv].band == 0) return rv;
    if (!kRowsVariants[rv].par) {
        if (N == 2048 && nframes == 1) return 0;
        rv = 7;
    }
    return (rv == 6 ? OCN_BFITS(6) : rv == 7 ? OCN_BFITS(7) : OCN_BFITS(8)) ? rv : 0;
#undef OCN_BFITS
}

template <int N>
static hipError_t launch_frame_n(const FrameArgs& a, int stages, hipStream_t s)
{
    hipError_t e = hipSuccess;
    if (stages & 1) {
        switch (a.cols_variant) {
        case 0: e = launch_cols_v<N, 0>(a, s); break;
        case 1: e = launch_cols_v<N, 1>(a, s); break;
        case 2: e = launch_cols_v<N, 2>(a, s); break;
        case 3: e = launch_cols_v<N, 3>(a, s); break;
        case 4: e = launch_cols_v<N, 4>(a, s); break;
        case 5: e = launch_cols_v<N, 5>(a, s); break;
        case 6: e = launch_cols_v<N, 6>(a, s); break;
        case 7: e = launch_cols_v<N, 7>(a, s); break;
        case 8: e = launch_cols_v<N, 8>(a, s); break;
        case 9: e = launch_cols_v<N, 9>(a, s); break;
        case 10: e = launch_cols_v<N, 10>(a, s); break;
        case 11: e = launch_cols_v<N, 11>(a, s); break;
        case 12: e = launch_cols_v<N, 12>(a, s); break;
        case 13: e = launch_cols_v<N, 13>(a, s); break;
        case 14: e = launch_cols_v<N, 14>(a, s); break;
        case 15: e = launch_cols_v<N, 15>(a, s); break;
        case 16: e = launch_cols_v<N, 16>(a, s); break;
        case 17: e = launch_cols_v<N, 17>(a, s); break;
        case 18: e = launch_cols_v<N, 18>(a, s); break;
        case 19: e = launch_cols_v<N, 19>(a, s); break;
        case 20: e = launch_cols_v<N, 20>(a, s); break;
        case 21: e = launch_cols_v<N, 21>(a, s); break;
        default: e = hipErrorInvalidValue;
        }
        if (e != hipSuccess) return e;
    }
    // Bilinear normals and the parallel bands' render export are fused into the
    // row pass of a whole frame only: the row or the normal-map stage by itself
    // is the unfused kernel, which works from and on the output textures.
    int        rv  = a.rows_variant;
    const bool bil = a.normal_mode != 0, ren = a.disp || a.rnorm, whole = (stages & 6) == 6;
    if (rv >= 0 && rv < kNumRowsVariants && bil) rv = whole ? bilinear_rows<N>(rv, a.nframes) : kRowsVariants[rv].band > 0 ? 0 : rv;
    if (rv >= 0 && rv < kNumRowsVariants && kRowsVariants[rv].par && ren && !whole) rv = 1;
    const bool fused = rv >= 0 && rv < kNumRowsVariants && kRowsVariants[rv].band > 0;
    if (stages & 2) {
        switch (rv) {
        case 0: e = launch_rows_v<N, 0>(a, s); break;
        case 1: e = launch_rows_v<N, 1>(a, s); break;
        case 2: e = launch_rows_v<N, 2>(a, s); break;
        case 3: e = launch_rows_v<N, 3>(a, s); break;
        case 4: e = launch_rows_v<N, 4>(a, s); break;
        case 5: e = launch_rows_v<N, 5>(a, s); break;
        case 6: e = launch_rows_v<N, 6>(a, s); break;
        case 7: e = launch_rows_v<N, 7>(a, s); break;
        case 8: e = launch_rows_v<N, 8>(a, s); break;
        default: e = hipErrorInvalidValue;
        }
        if (e != hipSuccess) return e;
    }
    if ((stages & 4) && !fused && (a.normals || a.jacobian || a.disp || a.rnorm)) {
        normals_pass(N, a.nframes, a.height, a.dx, a.dz, a.normals, a.jacobian, a.normal_mode, a.lambda, a.inv2d,
                     a.fb.out_stride, a.disp, a.rnorm, a.dscale, s);
        e = hipGetLastError();
    }
    return e;
}

template <int N>
static bool variant_ok_n(int cols_v, int rows_v)
{
    constexpr bool c[kNumColsVariants] = {
#define OCN_FITS(v) cols_fits(N, v)
        OCN_FITS(0), OCN_FITS(1), OCN_FITS(2), OCN_FITS(3), OCN_FITS(4),
        OCN_FITS(5), OCN_FITS(6), OCN_FITS(7), OCN_FITS(8), OCN_FITS(9),
        OCN_FITS(10), OCN_FITS(11), OCN_FITS(12), OCN_FITS(13), OCN_FITS(14), OCN_FITS(15), OCN_FITS(16),
        OCN_FITS(17), OCN_FITS(18), OCN_FITS(19), OCN_FITS(20), OCN_FITS(21)};
#undef OCN_FITS
#define OCN_RFITS(v) \
    rows_fits<N, kRowsVariants[v].E, kRowsVariants[v].band, kRowsVariants[v].par, kRowsVariants[v].W>()
    constexpr bool r[kNumRowsVariants] = {OCN_RFITS(0), OCN_RFITS(1), OCN_RFITS(2), OCN_RFITS(3), OCN_RFITS(4),
                                          OCN_RFITS(5), OCN_RFITS(6), OCN_RFITS(7), OCN_RFITS(8)};
#undef OCN_RFITS
    return cols_v >= 0 && cols_v < kNumColsVariants && rows_v >= 0 && rows_v < kNumRowsVariants && c[cols_v] &&
           r[rows_v];
}

template <int N>
static hipError_t launch_ifft2_n(const float2* src, float2* mid, float* out, const float2* const* tw, hipStream_t s)
{
    // Radix 8: at radix 16 a thread's 30 loads and longer chain cost the small
    // sizes (N=256 6.2 -> 6.8 us) and gain nothing at the large ones.  4 column
    // pairs per block (64-byte runs read, 32 written), 2 at N = 4096, whose four
    // would be 2048 threads; 2 or 8 at N = 512..2048 are within 4% or slower.
    constexpr int T = N / 8, NB = T < 64 ? 64 : T, C = N <= 2048 ? 4 : 2;
    hipLaunchKernelGGL((k_ifft2_rows<N, 8, NB>), dim3(N / 2 / (NB / T)), dim3(NB), 0, s, src, mid, tw[radix_slot(8)]);
    const dim3 grid(N / 2 / C), block(C * T);
    if (reinterpret_cast<uintptr_t>(out) & 7)
        hipLaunchKernelGGL((k_ifft2_cols_inv<N, 8, C, false>), grid, block, 0, s, mid, out, tw[radix_slot(8)]);
    else
        hipLaunchKernelGGL((k_ifft2_cols_inv<N, 8, C, true>), grid, block, 0, s, mid, out, tw[radix_slot(8)]);
    return hipGetLastError();
}

#define OCN_DISPATCH_N(N, CALL, BAD)                \
    switch (N) {                                    \
    case 64: return CALL(64);                       \
    case 128: return CALL(128);                     \
    case 256: return CALL(256);                     \
    case 512: return CALL(512);                     \
    case 1024: return CALL(1024);                   \
    case 2048: return CALL(2048);                   \
    case 4096: return CALL(4096);                   \
    default: return BAD;                            \
    }

hipError_t launch_frame(int N, const FrameArgs& a, int stages, hipStream_t s)
{
    if (a.nframes < 1 || a.nframes > kMaxFrames) return hipErrorInvalidValue;
#define CALL(n) launch_frame_n<n>(a, stages, s)
    OCN_DISPATCH_N(N, CALL, hipErrorInvalidValue)
#undef CALL
}

bool schedule_valid(int N, int cols_variant, int rows_variant)
{
#define CALL(n) variant_ok_n<n>(cols_variant, rows_variant)
    OCN_DISPATCH_N(N, CALL, false)
#undef CALL
}

void cols_variant_shape(int N, int v, int* E, int* C)
{
    *E = kColsVariants[v].lds ? 16 : 8;
    *C = cols_width(N, kColsVariants[v].C);
}

int rows_variant_radix(int v) { return kRowsVariants[v].E; }

int rows_variant_band(int v) { return kRowsVariants[v].band; }

bool rows_variant_walk(int v) { return kRowsVariants[v].band > 0 && !kRowsVariants[v].par; }

hipError_t launch_ifft2(int N, const float2* src, float2* tmp, float* out, const float2* const* tw, hipStream_t s)
{
#define CALL(n) launch_ifft2_n<n>(src, tmp, out, tw, s)
    OCN_DISPATCH_N(N, CALL, hipErrorInvalidValue)
#undef CALL
}

// ------------------------------------------------------------------ static scratch

// Z1 and Z2 of ocn_update_frames_noalloc, for callers that cannot allocate
// device memory.  Each GPU the library runs on holds its own copy of this
// array until the process ends.  Host code never passes `scratch` itself to a
// kernel (in host code the name is a host-side stand-in, not a device
// address): static_scratch_resolve looks up the device address once per
// device with hipGetSymbolAddress, and the frame launches take that pointer.
// Nothing in it needs clearing: the column pass writes every element of Z1
// and Z2 before the row pass of the same launch reads them.
static __device__ __align__(256) unsigned char scratch[kStaticScratchBytes];

namespace {
std::mutex g_scratch_mu;
void*      g_scratch_addr[kMaxScratchDevices] = {};
}  // namespace

hipError_t static_scratch_resolve(int device)
{
    if (device < 0 || device >= kMaxScratchDevices) return hipErrorInvalidDevice;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    if (g_scratch_addr[device]) return hipSuccess;
    void*      p = nullptr;
    hipError_t e = hipGetSymbolAddress(&p, HIP_SYMBOL(scratch));
    if (e != hipSuccess) return e;
    g_scratch_addr[device] = p;
    return hipSuccess;
}

void* static_scratch_ptr(int device)
{
    if (device < 0 || device >= kMaxScratchDevices) return nullptr;
    std::lock_guard<std::mutex> lk(g_scratch_mu);
    return g_scratch_addr[device];
}

hipError_t launch_h0(int N, float4* h0, float4* uv, const uint8_t* noise, const SpecConst& sc, hipStream_t s)
{
    const dim3 grid(N / 2 / kH0Tile, N / kH0Tile), block(kH0Tile * kH0Tile);
    if (noise) hipLaunchKernelGGL(k_tilde_h0_k<kNoiseImages>, grid, block, 0, s, h0, uv, noise, sc);
    else hipLaunchKernelGGL(k_tilde_h0_k<kPhilox>, grid, block, 0, s, h0, uv, noise, sc);
    return hipGetLastError();
}

hipError_t launch_fold(int N, const FoldList& list, int count, hipStream_t s)
{
    hipLaunchKernelGGL(k_fold, dim3(N / 2 / kH0Tile, N / kH0Tile, count), dim3(kH0Tile * kH0Tile), 0, s, list, N);
    return hipGetLastError();
}

hipError_t launch_spectrum_t(int N, const float4* h0, float2* hy, float2* hx, float2* hz, const SpecConst& sc,
                             double t_rev, hipStream_t s)
{
    hipLaunchKernelGGL(k_tilde_h0_t, dim3((N + 255) / 256, N), dim3(256), 0, s, h0, hy, hx, hz, sc, t_rev);
    return hipGetLastError();
}

hipError_t launch_normals(int N, const float* height, const float* dx, const float* dz, float4* normals,
                          float* jacobian, int mode, float lambda, float inv2d, hipStream_t s)
{
    normals_pass(N, 1, height, dx, dz, normals, jacobian, mode, lambda, inv2d, 0, nullptr, nullptr, 0.0f, s);
    return hipGetLastError();
}

}  // namespace ocn
