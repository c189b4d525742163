// Kernels of the learned warm start: a 3-level 3D convolutional U-Net
// trained on the GPU.  No reference counterpart.
//
// Layout: activations are channels-last, [N][D][H][W][C] with C a multiple
// of 8, stored as BF16 (raw 16-bit words); gradients and master weights are
// FP32.  A 3x3x3 convolution (zero padding 1) is an implicit GEMM
//     out[p][co] = sum_{k = tap*Ci + ci} W[co][k] * in[p + off(tap)][ci]
// computed with gfx950's v_mfma_f32_16x16x32_bf16 (BF16 operands, FP32
// accumulation): the weights are the A operand (rows = output channels),
// the gathered activations the B operand (columns = 16 positions), so each
// lane ends with 4 consecutive output channels of one position and stores
// them as one 8-byte word.  Weights are [Co][Kpad] with Kpad = 27*Ci rounded
// up to 32 (zero-filled).
//
// The backward data pass is the same kernel applied to the gradient with
// the weights transposed and the taps mirrored (conv_wt_transpose); the
// weight gradient is a second MFMA GEMM reducing over positions.  Both take
// their operands from tiles staged in LDS (k_conv3_tile, k_conv3_wgrad_tile);
// k_conv3, k_conv3_wgrad and k_conv3_wgrad_t, which load every operand from
// global memory, serve the shapes whose tile does not fit or is mostly
// padding.
#include <hip/hip_runtime.h>
#include <stdint.h>

#include <algorithm>

#include "../../include/stencil_nn.h"
#include "st_device.hpp"
#include "st_internal.hpp"

namespace st {

typedef uint16_t bf16_t;
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef unsigned int u32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ bf16_t f2bf(float f)
{
    uint32_t x = __float_as_uint(f);
    if ((x & 0x7fffffffu) > 0x7f800000u) return (bf16_t)((x >> 16) | 0x40);
    x += 0x7fffu + ((x >> 16) & 1u);
    return (bf16_t)(x >> 16);
}

// two values rounded to BF16, low word first (v_cvt_pk_bf16_f32: round to
// nearest even, the same words as f2bf)
__device__ __forceinline__ uint32_t pack_bf(float a, float b)
{
    typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
    const bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
}

__device__ __forceinline__ float bf2f(bf16_t h) { return __uint_as_float((uint32_t)h << 16); }

__device__ __forceinline__ bf16x8 load8(const bf16_t *p)
{
    const u32x4 v = *reinterpret_cast<const u32x4 *>(p);
    return __builtin_bit_cast(bf16x8, v);
}

__device__ __forceinline__ bf16x8 zero8()
{
    const u32x4 z = {0u, 0u, 0u, 0u};
    return __builtin_bit_cast(bf16x8, z);
}

struct ConvGeom {
    int N, D, H, W;
    int Ci, Co;
    int Kpad;       // row length of the weight matrix
    int P;          // N*D*H*W (below 2^31)
};

__device__ __forceinline__ void decode(const ConvGeom &g, int p, int &n, int &z, int &y, int &x)
{
    x = p % g.W;
    int t = p / g.W;
    y = t % g.H;
    t /= g.H;
    z = t % g.D;
    n = t / g.D;
}

__device__ __forceinline__ bf16x8 pack8(const unsigned short (&v)[8])
{
    u32x4 w;
    w[0] = (uint32_t)v[0] | ((uint32_t)v[1] << 16);
    w[1] = (uint32_t)v[2] | ((uint32_t)v[3] << 16);
    w[2] = (uint32_t)v[4] | ((uint32_t)v[5] << 16);
    w[3] = (uint32_t)v[6] | ((uint32_t)v[7] << 16);
    return __builtin_bit_cast(bf16x8, w);
}

// ---------------------------------------------------------------- conv forward / backward data

// Wave tile: MB blocks of 16 positions x NB blocks of 16 output channels.
template <int NB, int MB>
__global__ __launch_bounds__(256) void k_conv3(const bf16_t *__restrict__ act,
                                               const bf16_t *__restrict__ wt,
                                               const float *__restrict__ bias,
                                               bf16_t *__restrict__ out_bf,
                                               float *__restrict__ out_f, ConvGeom g, int relu,
                                               int accumulate)
{
    const int lane = threadIdx.x & 63;
    const int j = lane & 15, grp = lane >> 4;
    const long long wave = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int nct = (g.Co + 16 * NB - 1) / (16 * NB);
    const long long pt = wave / nct;
    const int ct = (int)(wave % nct);
    const int p0 = (int)(pt * 16 * MB);
    const int c0 = ct * 16 * NB;
    if (pt * 16 * MB >= g.P) return;

    int pn[MB], pz[MB], py[MB], px[MB];
    bool pv[MB];
#pragma unroll
    for (int mb = 0; mb < MB; ++mb) {
        const int p = p0 + mb * 16 + j;
        pv[mb] = p < g.P;
        decode(g, pv[mb] ? p : 0, pn[mb], pz[mb], py[mb], px[mb]);
    }
    f32x4 acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) acc[nb][mb] = f32x4{0.f, 0.f, 0.f, 0.f};

    const int nk = g.Kpad / 32;
    for (int kc = 0; kc < nk; ++kc) {
        const int k = kc * 32 + grp * 8;
        const int tap = k / g.Ci;
        const int ci = k - tap * g.Ci;
        bf16x8 a[NB], b[MB];
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int co = c0 + nb * 16 + j;
            a[nb] = co < g.Co ? load8(wt + (long long)co * g.Kpad + k) : zero8();
        }
        const int dz = tap / 9 - 1, dy = (tap / 3) % 3 - 1, dx = tap % 3 - 1;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            const int zz = pz[mb] + dz, yy = py[mb] + dy, xx = px[mb] + dx;
            const bool ok = pv[mb] && tap < 27 && zz >= 0 && zz < g.D && yy >= 0 && yy < g.H &&
                            xx >= 0 && xx < g.W;
            const long long q = (((long long)pn[mb] * g.D + zz) * g.H + yy) * g.W + xx;
            b[mb] = ok ? load8(act + q * g.Ci + ci) : zero8();
        }
#pragma unroll
        for (int nb = 0; nb < NB; ++nb)
#pragma unroll
            for (int mb = 0; mb < MB; ++mb)
                acc[nb][mb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[nb], b[mb], acc[nb][mb], 0, 0, 0);
    }
    // lane holds D[co = 4*grp + v][position j] of each (nb, mb) block
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        const int cb = c0 + nb * 16 + 4 * grp;
#pragma unroll
        for (int mb = 0; mb < MB; ++mb) {
            if (!pv[mb]) continue;
            const long long p = (long long)p0 + mb * 16 + j;
            float v[4];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                float t = acc[nb][mb][e];
                if (bias && cb + e < g.Co) t += bias[cb + e];
                if (relu) t = t > 0.f ? t : 0.f;
                v[e] = t;
            }
            if (out_f) {
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    if (cb + e < g.Co) {
                        float *o = out_f + p * g.Co + cb + e;
                        *o = accumulate ? *o + v[e] : v[e];
                    }
            }
            if (out_bf) {
                if (cb + 3 < g.Co) {
                    const uint32_t lo = (uint32_t)f2bf(v[0]) | ((uint32_t)f2bf(v[1]) << 16);
                    const uint32_t hi = (uint32_t)f2bf(v[2]) | ((uint32_t)f2bf(v[3]) << 16);
                    *reinterpret_cast<uint2 *>(out_bf + p * g.Co + cb) = make_uint2(lo, hi);
                } else {
#pragma unroll
                    for (int e = 0; e < 4; ++e)
                        if (cb + e < g.Co) out_bf[p * g.Co + cb + e] = f2bf(v[e]);
                }
            }
        }
    }
}

// ---------------------------------------------------------------- conv forward / backward data, LDS tiles

// The same sums in the same order (chunks of 32 weight columns, one MFMA
// each), with the activations read from LDS: a workgroup of four waves stages
// the 18 x 6 x (TZ+2) neighbourhood of a tile of 16 x 4 x TZ positions once
// and takes all 27 taps from it, where k_conv3 loads every operand of every
// tap from global memory (16 bytes per lane and MFMA: the L2 and its address
// arithmetic held it at 180 TFLOP/s).  A wave computes MB rows of 16
// positions and 16*NB output channels.
//
// Bound: LDS reads (1 KiB per wave and MFMA at NB = 1; a CU reads 128 bytes
// a cycle and starts an MFMA every 4) and the staging of the tiles, which two
// workgroups per CU overlap in part.  8 x 64^3 positions, k_conv3 and now:
// 48 -> 16 channels 453 -> 272 us, 16 -> 48 FP32 489 -> 266, 16 -> 16 159 ->
// 92; 8 x 16^3, 64 -> 64 64 -> 31.  Weights straight from L2 (16 rows of 64
// bytes per load) instead of through LDS: 16 -> 48 370 us.  The position
// stride in LDS carries 16 bytes of padding where Ci is a multiple
// of 32, else eight lanes of a read would meet in the same banks.
constexpr int kTx = 16, kTy = 4;

// LDS bytes from one position of a tile to the next
__host__ __device__ constexpr int tile_stride(int ci) { return 2 * (ci % 32 == 0 ? ci + 8 : ci); }
__host__ __device__ constexpr int tile_positions(int tz) { return (kTx + 2) * (kTy + 2) * (tz + 2); }

struct TileGeom {
    ConvGeom g;
    int tx, ty, tz;  // tiles per axis (of one sample)
};

// Tile `t`: sample and first position.
__device__ __forceinline__ void tile_origin(const TileGeom &q, int t, int depth, int &n, int &z, int &y, int &x)
{
    x = t % q.tx * kTx;
    t /= q.tx;
    y = t % q.ty * kTy;
    t /= q.ty;
    z = t % q.tz * depth;
    n = t / q.tz;
}

// Stage the neighbourhood of a tile of depth TZ (positions -1 .. +1 around
// it; zero outside the sample): all Ci channels, position stride S bytes.
// A row of 18 positions is one run of memory; a wave takes a row at a time in
// 16-byte words, so the words' places are computed once per wave (computing
// them per word took as many instructions as the products).
template <int TZ, int WAVES>
__device__ __forceinline__ void tile_stage(const bf16_t *__restrict__ act, const ConvGeom &g, int n, int z0, int y0,
                                           int x0, char *lds, int S)
{
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int nc8 = g.Ci >> 3, words = (kTx + 2) * nc8;
    const long long sample = (long long)n * g.D * g.H * g.W;
    constexpr int ROWS = (kTy + 2) * (TZ + 2);
    for (int i0 = 0; i0 < words; i0 += 64) {
        const int i = i0 + lane, px = i / nc8, c8 = i - px * nc8;
        const bool have = i < words, xin = have && (unsigned)(x0 + px - 1) < (unsigned)g.W;
        const unsigned go = (unsigned)i * 16u;  // byte offset in the row, from position x0 - 1
        char *const to = lds + px * S + c8 * 16;
#pragma unroll 5
        for (int r = w; r < ROWS; r += WAVES) {
            const int py = r % (kTy + 2), pz = r / (kTy + 2), y = y0 + py - 1, z = z0 + pz - 1;
            const bool rin = (unsigned)y < (unsigned)g.H && (unsigned)z < (unsigned)g.D;
            u32x4 v = {0u, 0u, 0u, 0u};
            if (rin && xin) {
                const char *row = reinterpret_cast<const char *>(act + (sample + ((long long)z * g.H + y) * g.W + x0 - 1) * g.Ci);
                v = *reinterpret_cast<const u32x4 *>(row + go);
            }
            if (have) *reinterpret_cast<u32x4 *>(to + r * (kTx + 2) * S) = v;
        }
    }
}

// LDS offset of tap `tap`, channel `ci`, from a position's first neighbour
__device__ __forceinline__ int tap_offset(int tap, int ci, int S)
{
    return ((tap / 9 * (kTy + 2) + tap / 3 % 3) * (kTx + 2) + tap % 3) * S + 2 * ci;
}

// weight chunks staged at a time
__host__ __device__ constexpr int conv_chunks(int nb) { return nb == 1 ? 8 : 4; }

template <int NB, int MB>
__global__ __launch_bounds__(256) void k_conv3_tile(const bf16_t *__restrict__ act, const bf16_t *__restrict__ wt,
                                                    const float *__restrict__ bias, bf16_t *__restrict__ out_bf,
                                                    float *__restrict__ out_f, TileGeom q, int nct, int relu,
                                                    int accumulate)
{
    constexpr int TZ = MB;  // 4*MB rows of 16 positions, MB per wave
    constexpr int KC = conv_chunks(NB), WR = KC * NB / 4;
    extern __shared__ __align__(16) char lds[];
    const ConvGeom &g = q.g;
    const int S = tile_stride(g.Ci), nk = g.Kpad / 32;
    int *tab = reinterpret_cast<int *>(lds + tile_positions(TZ) * S);  // offset of chunk kc, lane group grp
    const unsigned id = xcd_remap(blockIdx.x, gridDim.x);
    const int ct = (int)(id % (unsigned)nct), c0 = ct * 16 * NB;
    int n, z0, y0, x0;
    tile_origin(q, (int)(id / (unsigned)nct), TZ, n, z0, y0, x0);
    for (int i = threadIdx.x; i < 4 * nk; i += 256) {
        const int k = i * 8, tap = k / g.Ci;
        tab[i] = tap < 27 ? tap_offset(tap, k - tap * g.Ci, S) : 0;
    }
    // weights: KC chunks at a time in LDS, in operand order (16 bytes of lane
    // l of chunk u, block nb at ((u*NB + nb)*64 + l)*16), double buffered
    char *const wlds = reinterpret_cast<char *>(tab + 4 * ((nk + 3) / 4 * 4));
    u32x4 wreg[WR];
    auto weights = [&](int st) {
#pragma unroll
        for (int u = 0; u < WR; ++u) {
            const int i = threadIdx.x + 256 * u, row = i / (KC * 4), kq = st * KC * 4 + i % (KC * 4);
            wreg[u] = u32x4{0u, 0u, 0u, 0u};
            if (c0 + row < g.Co && kq < nk * 4)
                wreg[u] = *reinterpret_cast<const u32x4 *>(wt + (long long)(c0 + row) * g.Kpad + kq * 8);
        }
    };
    auto put = [&](int st) {
        char *const to = wlds + (st & 1) * (KC * NB * 1024);
#pragma unroll
        for (int u = 0; u < WR; ++u) {
            const int i = threadIdx.x + 256 * u, row = i / (KC * 4), kq = i % (KC * 4);
            *reinterpret_cast<u32x4 *>(to + (((kq >> 2) * NB + (row >> 4)) * 64 + (kq & 3) * 16 + (row & 15)) * 16) = wreg[u];
        }
    };
    weights(0);
    tile_stage<TZ, 4>(act, g, n, z0, y0, x0, lds, S);
    put(0);
    __syncthreads();

    const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
    const int j = lane & 15, grp = lane >> 4;
    const char *base[MB];
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const int row = w * MB + m;
        base[m] = lds + ((row / kTy * (kTy + 2) + row % kTy) * (kTx + 2) + j) * S;
    }
    f32x4 acc[NB][MB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb)
#pragma unroll
        for (int m = 0; m < MB; ++m) acc[nb][m] = f32x4{0.f, 0.f, 0.f, 0.f};

    // activations of a chunk are fetched while the one before is multiplied
    auto taps = [&](int kc, bf16x8 (&b)[MB]) {
        const int off = tab[min(kc, nk - 1) * 4 + grp];
#pragma unroll
        for (int m = 0; m < MB; ++m) b[m] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(base[m] + off));
    };
    // the last chunk's columns beyond 27*Ci multiply zeros
    const bool pad = (nk - 1) * 32 + grp * 8 >= 27 * g.Ci;
    bf16x8 b[2][MB];
    taps(0, b[0]);
    const int stages = (nk + KC - 1) / KC;
    for (int st = 0; st < stages; ++st) {
        if (st + 1 < stages) weights(st + 1);
        const char *wl = wlds + (st & 1) * (KC * NB * 1024) + lane * 16;
        bf16x8 a[2][NB];
        auto wfetch = [&](int u, bf16x8 (&d)[NB]) {
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
                d[nb] = __builtin_bit_cast(bf16x8, *reinterpret_cast<const u32x4 *>(wl + (u * NB + nb) * 1024));
        };
        wfetch(0, a[0]);
#pragma unroll
        for (int u = 0; u < KC; ++u) {
            const int kc = st * KC + u;
            if (kc >= nk) break;
            if (u + 1 < KC) wfetch(u + 1, a[(u + 1) & 1]);
            taps(kc + 1, b[(u + 1) & 1]);
            if (kc == nk - 1 && pad) {
#pragma unroll
                for (int m = 0; m < MB; ++m) b[u & 1][m] = zero8();
            }
#pragma unroll
            for (int nb = 0; nb < NB; ++nb)
#pragma unroll
                for (int m = 0; m < MB; ++m)
                    acc[nb][m] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[u & 1][nb], b[u & 1][m], acc[nb][m], 0, 0, 0);
        }
        if (st + 1 < stages) {
            put(st + 1);
            __syncthreads();
        }
    }

    // lane holds D[co = 4*grp + v][position j] of each (nb, m) block
    const long long sample = (long long)n * g.D * g.H * g.W;
#pragma unroll
    for (int m = 0; m < MB; ++m) {
        const int row = w * MB + m, z = z0 + row / kTy, y = y0 + row % kTy, x = x0 + j;
        if (z >= g.D || y >= g.H || x >= g.W) continue;
        const long long p = sample + ((long long)z * g.H + y) * g.W + x;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int cb = c0 + nb * 16 + 4 * grp;
            if (cb >= g.Co) continue;  // Co is a multiple of 4
            f32x4 v = acc[nb][m];
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                if (bias) v[e] += bias[cb + e];
                if (relu) v[e] = v[e] > 0.f ? v[e] : 0.f;
            }
            if (out_f) {
                f32x4 *o = reinterpret_cast<f32x4 *>(out_f + p * g.Co + cb);
                if (accumulate) {
                    const f32x4 t = *o;
#pragma unroll
                    for (int e = 0; e < 4; ++e) (*o)[e] = t[e] + v[e];
                } else {
                    *o = v;
                }
            }
            if (out_bf) {
                *reinterpret_cast<uint2 *>(out_bf + p * g.Co + cb) = make_uint2(pack_bf(v[0], v[1]), pack_bf(v[2], v[3]));
            }
        }
    }
}

// ---------------------------------------------------------------- weight gradient

// dW[co][k] += sum_p dY[p][co] * X[p + off(tap(k))][ci(k)]
// MFMA rows = output channels (A = dY^T), columns = 16 weight columns k
// (B = shifted X), reduction over 32 positions per instruction; each wave
// covers `pchunk` positions and adds its partial sums atomically.
template <int NB>
__global__ __launch_bounds__(256) void k_conv3_wgrad(const bf16_t *__restrict__ X,
                                                     const bf16_t *__restrict__ dY,
                                                     float *__restrict__ dW, ConvGeom g,
                                                     int pchunk)
{
    const int lane = threadIdx.x & 63;
    const int j = lane & 15, grp = lane >> 4;
    const long long wave = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int K = 27 * g.Ci;
    const int nkt = (K + 16 * NB - 1) / (16 * NB);
    const int nct = (g.Co + 15) / 16;
    const long long nchunks = ((long long)g.P + pchunk - 1) / pchunk;
    const long long total = nchunks * nkt * nct;
    if (wave >= total) return;
    const int kt = (int)(wave % nkt);
    const long long r2 = wave / nkt;
    const int ct = (int)(r2 % nct);
    const int pc = (int)(r2 / nct);
    const int co = ct * 16 + j;  // A-operand row of this lane
    int ci[NB], kk[NB], dz[NB], dy[NB], dx[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        kk[nb] = kt * 16 * NB + nb * 16 + j;  // B-operand column of this lane
        const int kc = kk[nb] < K ? kk[nb] : 0;
        const int tap = kc / g.Ci;
        ci[nb] = kc - tap * g.Ci;
        dz[nb] = tap / 9 - 1;
        dy[nb] = (tap / 3) % 3 - 1;
        dx[nb] = tap % 3 - 1;
    }
    f32x4 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int pbeg = pc * pchunk, pend = min(pbeg + pchunk, g.P);
    for (int ps = pbeg; ps < pend; ps += 32) {
        // the 8 positions of this lane group, walked from one decode
        int n0, z0, y0, x0;
        const int pfirst = ps + grp * 8;
        decode(g, min(pfirst, g.P - 1), n0, z0, y0, x0);
        int pn[8], pz[8], py[8], px[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            pn[e] = n0; pz[e] = z0; py[e] = y0; px[e] = x0;
            if (++x0 == g.W) {
                x0 = 0;
                if (++y0 == g.H) {
                    y0 = 0;
                    if (++z0 == g.D) { z0 = 0; ++n0; }
                }
            }
        }
        unsigned short av[8];
#pragma unroll
        for (int e = 0; e < 8; ++e) {
            const int p = pfirst + e;
            av[e] = (p < pend && co < g.Co) ? dY[(long long)p * g.Co + co] : (unsigned short)0;
        }
        const bf16x8 a = pack8(av);
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            unsigned short bv[8];
#pragma unroll
            for (int e = 0; e < 8; ++e) {
                const int zz = pz[e] + dz[nb], yy = py[e] + dy[nb], xx = px[e] + dx[nb];
                const bool ok = pfirst + e < pend && kk[nb] < K && zz >= 0 && zz < g.D && yy >= 0 &&
                                yy < g.H && xx >= 0 && xx < g.W;
                bv[e] = ok ? X[((((long long)pn[e] * g.D + zz) * g.H + yy) * g.W + xx) * g.Ci + ci[nb]]
                           : (unsigned short)0;
            }
            acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a, pack8(bv), acc[nb], 0, 0, 0);
        }
    }
    // lane holds D[row co = ct*16 + 4*grp + v][column k = kt*16*NB + nb*16 + j]
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (kk[nb] >= K) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = ct * 16 + 4 * grp + e;
            if (c < g.Co) atomicAdd(dW + (long long)c * g.Kpad + kk[nb], acc[nb][e]);
        }
    }
}

// ---------------------------------------------------------------- weight gradient, channel-major operands

// The MFMA operands of the weight gradient run along positions (8
// consecutive positions of one channel per lane), which channels-last
// activations hold Ci values apart: the gather above issues one 2-byte load
// per value.  When rows are a multiple of 8 positions, both operands are
// first transposed to channel-major [C][P] copies, and then every operand is
// one 16-byte load: the dY rows directly, the X rows of a tap with dx = -1
// or +1 from two aligned loads joined by a 16-bit funnel shift (a group of 8
// positions never crosses a row, so only its first or last value can fall
// outside the row, and it is zeroed).

// [P][C] -> [C][P] (16-bit words) through LDS, 64 positions per workgroup.
constexpr int kTrMaxC = 128;
__global__ __launch_bounds__(256) void k_pc_transpose(const bf16_t *__restrict__ src, bf16_t *__restrict__ dst,
                                                      int P, int C)
{
    __shared__ bf16_t t[kTrMaxC * 66];
    const long long p0 = (long long)blockIdx.x * 64;
    const int np = (int)min(64LL, (long long)P - p0);
    for (int i = threadIdx.x; i < np * C; i += 256) {
        const int pp = i / C, c = i - pp * C;
        t[c * 66 + pp] = src[p0 * C + i];
    }
    __syncthreads();
    for (int i = threadIdx.x; i < 64 * C; i += 256) {
        const int c = i >> 6, pp = i & 63;
        if (pp < np) dst[(long long)c * P + p0 + pp] = t[c * 66 + pp];
    }
}

__device__ __forceinline__ u32x4 load8u(const bf16_t *p) { return *reinterpret_cast<const u32x4 *>(p); }

// dW[co][k] += sum_p dYt[co][p] * Xt[ci(k)][p + off(tap(k))]; the same
// tiling as k_conv3_wgrad (rows = output channels, 16*NB weight columns,
// 32 positions per MFMA, `pchunk` positions per wave, atomics at the end).
// Requires W % 8 == 0 and pchunk % 32 == 0.
template <int NB>
__global__ __launch_bounds__(256) void k_conv3_wgrad_t(const bf16_t *__restrict__ Xt,
                                                       const bf16_t *__restrict__ dYt,
                                                       float *__restrict__ dW, ConvGeom g, int pchunk)
{
    const int lane = threadIdx.x & 63;
    const int j = lane & 15, grp = lane >> 4;
    const long long wave = (long long)blockIdx.x * (blockDim.x >> 6) + (threadIdx.x >> 6);
    const int K = 27 * g.Ci;
    const int nkt = (K + 16 * NB - 1) / (16 * NB);
    const int nct = (g.Co + 15) / 16;
    const long long nchunks = ((long long)g.P + pchunk - 1) / pchunk;
    const long long total = nchunks * nkt * nct;
    if (wave >= total) return;
    const int kt = (int)(wave % nkt);
    const long long r2 = wave / nkt;
    const int ct = (int)(r2 % nct);
    const int pc = (int)(r2 / nct);
    const int co = ct * 16 + j;  // A-operand row of this lane
    const long long HW = (long long)g.H * g.W;
    const bf16_t *arow = dYt + (long long)min(co, g.Co - 1) * g.P;
    int kk[NB], dz[NB], dy[NB], dx[NB];
    const bf16_t *brow[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        kk[nb] = kt * 16 * NB + nb * 16 + j;  // B-operand column of this lane
        const int kc = kk[nb] < K ? kk[nb] : 0;
        const int tap = kc / g.Ci;
        const int ci = kc - tap * g.Ci;
        dz[nb] = tap / 9 - 1;
        dy[nb] = (tap / 3) % 3 - 1;
        dx[nb] = tap % 3 - 1;
        brow[nb] = Xt + (long long)ci * g.P;
    }
    f32x4 acc[NB];
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) acc[nb] = f32x4{0.f, 0.f, 0.f, 0.f};
    const int pbeg = pc * pchunk, pend = min(pbeg + pchunk, g.P);
    const u32x4 zero = {0u, 0u, 0u, 0u};
    for (int ps = pbeg; ps < pend; ps += 32) {
        // this lane group's 8 positions: one row segment (W % 8 == 0)
        const int pf = ps + grp * 8;
        const bool pin = pf < pend;
        int n0, z0, y0, x0;
        decode(g, min(pf, g.P - 8), n0, z0, y0, x0);
        const u32x4 av = (pin && co < g.Co) ? load8u(arow + pf) : zero;
#pragma unroll
        for (int nb = 0; nb < NB; ++nb) {
            const int zz = z0 + dz[nb], yy = y0 + dy[nb];
            const bool ok = pin && kk[nb] < K && zz >= 0 && zz < g.D && yy >= 0 && yy < g.H;
            u32x4 b = zero;
            if (ok) {
                const bf16_t *q = brow[nb] + pf + (long long)dz[nb] * HW + (long long)dy[nb] * g.W;
                const u32x4 v = load8u(q);
                if (dx[nb] == 0) {
                    b = v;
                } else if (dx[nb] < 0) {
                    // values x0-1 .. x0+6: the last of the group before, then v[0..6]
                    const unsigned prev = x0 > 0 ? load8u(q - 8)[3] : 0u;
                    b[0] = __builtin_amdgcn_alignbit(v[0], prev, 16);
                    b[1] = __builtin_amdgcn_alignbit(v[1], v[0], 16);
                    b[2] = __builtin_amdgcn_alignbit(v[2], v[1], 16);
                    b[3] = __builtin_amdgcn_alignbit(v[3], v[2], 16);
                } else {
                    // values x0+1 .. x0+8: v[1..7], then the first of the group after
                    const unsigned next = x0 + 8 < g.W ? load8u(q + 8)[0] : 0u;
                    b[0] = __builtin_amdgcn_alignbit(v[1], v[0], 16);
                    b[1] = __builtin_amdgcn_alignbit(v[2], v[1], 16);
                    b[2] = __builtin_amdgcn_alignbit(v[3], v[2], 16);
                    b[3] = __builtin_amdgcn_alignbit(next, v[3], 16);
                }
            }
            acc[nb] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, av),
                                                              __builtin_bit_cast(bf16x8, b), acc[nb], 0, 0, 0);
        }
    }
#pragma unroll
    for (int nb = 0; nb < NB; ++nb) {
        if (kk[nb] >= K) continue;
#pragma unroll
        for (int e = 0; e < 4; ++e) {
            const int c = ct * 16 + 4 * grp + e;
            if (c < g.Co) atomicAdd(dW + (long long)c * g.Kpad + kk[nb], acc[nb][e]);
        }
    }
}

// ---------------------------------------------------------------- weight gradient, LDS tiles

// dW[co][k] += sum_p dY[p][co] * X[p + off(tap)][ci] over tiles of 16 x 4 x
// TZ positions: a workgroup stages a tile's neighbourhood of X and its dY in
// LDS (channels last, as they lie in memory) and takes every tap of every
// channel from there.  The MFMA reduces over 32 positions (two rows of 16), so
// both operands run along positions, which channels-last data holds Ci apart:
// ds_read_b64_tr_b16 reads four positions x 16 channels and hands each lane
// one channel's four positions, and a tap is an address, not a shift.  (The
// channel-major kernel above, one load from L2 per operand, takes 1407 us
// for 48 -> 16 channels at 8 x 64^3.)
//
// Wave w of WAVES owns the column blocks w, w + WAVES, .. (16 weight columns
// k each) of 16*NC output channels and keeps their sums in registers over all
// of its workgroup's tiles; above 96 input channels, where the registers no
// longer hold all columns, workgroups share the columns out in ranges (8 x
// 16^3 104 -> 16 gathering 327 us, channel-major 132, now 31; 128 -> 128 856,
// 339, 164).  Every workgroup writes its partial dW to the
// workspace, and k_wgrad_reduce adds them up in a fixed order.
//
// Bound: LDS reads (two 8-byte reads per lane for each B operand, used for
// NC MFMAs).  With channel-major copies and now, 8 x 64^3: 48 -> 16 channels
// 1495 -> 302 us, 16 -> 16 498 -> 121; 8 x 32^3: 96 -> 32 688 -> 249.
constexpr int kWgWaves = 8;

typedef short s16x4 __attribute__((ext_vector_type(4)));

// 8 consecutive positions of one channel per lane: positions 0..3 of the
// lane group at `p`, 4..7 at `p + 4*S`; p is the lane's own place for the
// transposed read (position (lane & 15) / 4, channels 4*(lane & 3) ..)
__device__ __forceinline__ bf16x8 read_tr(const char *p, int S4)
{
    typedef __attribute__((address_space(3))) s16x4 L;
    const s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L *)(p));
    const s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((L *)(p + S4));
    typedef short s16x8 __attribute__((ext_vector_type(8)));
    const s16x8 v = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    return __builtin_bit_cast(bf16x8, v);
}

// NBW column blocks per wave (those below nkb exist) of the range of `cols`
// column blocks from cols*blockIdx.z, NC blocks of 16 output channels from
// c0 = 16*NC*blockIdx.y.  wide: dY can be read four channels at a time (Co a
// multiple of 4, 8-byte address).
template <int NC, int NBW, int TZ>
__global__ __launch_bounds__(64 * kWgWaves) void k_conv3_wgrad_tile(const bf16_t *__restrict__ X,
                                                                    const bf16_t *__restrict__ dY,
                                                                    float *__restrict__ part, TileGeom q, int ntiles, int cols,
                                                                    int wide)
{
    extern __shared__ __align__(16) char lds[];
    const ConvGeom &g = q.g;
    const int S = tile_stride(g.Ci);
    constexpr int SY = NC * 32 + (NC == 1 ? 0 : 16);  // dY position stride, bytes
    char *const ylds = lds + tile_positions(TZ) * S;
    const int lane = threadIdx.x & 63, w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int grp = lane >> 4, c0 = 16 * NC * (int)blockIdx.y;
    const int K = 27 * g.Ci, kb0 = cols * (int)blockIdx.z, nkb = min(kb0 + cols, (K + 15) / 16);
    const int wb = kb0 + w;  // the wave's first column block
    // the lane's place in a transposed read: positions 8*(grp & 1) + (lane & 15)/4
    // (+4) of row grp/2 of the step's two rows
    const int xr = 8 * (grp & 1) + ((lane & 15) >> 2);
    int boff[NBW];  // X: plus the tap and channel of the lane's four columns
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
        const int k = min((wb + i * kWgWaves) * 16 + 4 * (lane & 3), K - 4), tap = k / g.Ci;
        boff[i] = ((grp >> 1) * (kTx + 2) + xr) * S + tap_offset(tap, k - tap * g.Ci, S);
    }
    const int aoff = ((grp >> 1) * kTx + xr) * SY + 8 * (lane & 3);
    f32x4 acc[NBW][NC];
#pragma unroll
    for (int i = 0; i < NBW; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) acc[i][c] = f32x4{0.f, 0.f, 0.f, 0.f};

    for (int t = (int)blockIdx.x; t < ntiles; t += (int)gridDim.x) {
        int n, z0, y0, x0;
        tile_origin(q, t, TZ, n, z0, y0, x0);
        tile_stage<TZ, kWgWaves>(X, g, n, z0, y0, x0, lds, S);
        // dY of the tile: zero outside the sample and beyond Co
        const long long sample = (long long)n * g.D * g.H * g.W;
        for (int i = threadIdx.x; i < TZ * kTy * kTx * NC * 4; i += 64 * kWgWaves) {
            const int c4 = i % (NC * 4), p = i / (NC * 4), px = p % kTx, r = p / kTx;
            const int x = x0 + px, y = y0 + r % kTy, z = z0 + r / kTy, c = c0 + c4 * 4;
            uint2 v = make_uint2(0u, 0u);
            if (x < g.W && y < g.H && z < g.D && c < g.Co) {
                const bf16_t *src = dY + (sample + ((long long)z * g.H + y) * g.W + x) * g.Co + c;
                if (wide) v = *reinterpret_cast<const uint2 *>(src);
                else {
                    v.x = src[0] | (c + 1 < g.Co ? (unsigned)src[1] << 16 : 0u);
                    v.y = (c + 2 < g.Co ? (unsigned)src[2] : 0u) | (c + 3 < g.Co ? (unsigned)src[3] << 16 : 0u);
                }
            }
            *reinterpret_cast<uint2 *>(ylds + p * SY + c4 * 8) = v;
        }
        __syncthreads();
        const bool edge = x0 + kTx > g.W || y0 + kTy > g.H || z0 + TZ > g.D;
#pragma unroll 1
        for (int r = 0; r < TZ * kTy; r += 2) {
            const char *yp = ylds + r * kTx * SY + aoff;
            const char *xp = lds + (r / kTy * (kTy + 2) + r % kTy) * (kTx + 2) * S;
            bf16x8 a[NC];
#pragma unroll
            for (int c = 0; c < NC; ++c) a[c] = read_tr(yp + c * 32, 4 * SY);
            u32x4 keep = {~0u, ~0u, ~0u, ~0u};
            if (edge) {
                // positions outside the sample: X may hold infinities there
                // that a zero dY would turn into NaN
                const int rr = r + (grp >> 1);
                const bool in = y0 + rr % kTy < g.H && z0 + rr / kTy < g.D;
                const int left = in ? g.W - x0 - 8 * (grp & 1) : 0;  // positions of the lane inside
#pragma unroll
                for (int e = 0; e < 4; ++e)
                    keep[e] = (2 * e < left ? 0xffffu : 0u) | (2 * e + 1 < left ? 0xffff0000u : 0u);
            }
#pragma unroll
            for (int i = 0; i < NBW; ++i) {
                if (wb + i * kWgWaves >= nkb) break;
                bf16x8 b = read_tr(xp + boff[i], 4 * S);
                if (edge) b = __builtin_bit_cast(bf16x8, __builtin_bit_cast(u32x4, b) & keep);
#pragma unroll
                for (int c = 0; c < NC; ++c)
                    acc[i][c] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(a[c], b, acc[i][c], 0, 0, 0);
            }
        }
        __syncthreads();
    }
    // lane holds D[row co = 4*grp + e][column lane & 15] of each block
    float *const o = part + (long long)blockIdx.x * g.Co * g.Kpad;
#pragma unroll
    for (int i = 0; i < NBW; ++i) {
        const int k = (wb + i * kWgWaves) * 16 + (lane & 15);
        if (k >= min(16 * nkb, K)) continue;
#pragma unroll
        for (int c = 0; c < NC; ++c)
#pragma unroll
            for (int e = 0; e < 4; ++e) {
                const int co = c0 + c * 16 + 4 * grp + e;
                if (co < g.Co) o[(long long)co * g.Kpad + k] = acc[i][c][e];
            }
    }
}

// dW += the partial sums of all workgroups, in their order; padding columns
// (k >= 27*Ci) are not touched.  One atomic per weight, so that calls on other
// streams may add to the same gradient.
__global__ __launch_bounds__(256) void k_wgrad_reduce(const float *__restrict__ part, float *__restrict__ dW, int n,
                                                      int K, int Kpad, int parts)
{
    __shared__ float red[256];
    // four lanes' worth of partial sums per weight, 64 weights per workgroup
    const int e = (int)blockIdx.x * 64 + (threadIdx.x & 63), h = threadIdx.x >> 6;
    float s = 0.f;
    if (e < n && e % Kpad < K) {
        const int lo = parts * h / 4, hi = parts * (h + 1) / 4;
#pragma unroll 8
        for (int p = lo; p < hi; ++p) s += part[(long long)p * n + e];
    }
    red[threadIdx.x] = s;
    __syncthreads();
    if (h == 0 && e < n && e % Kpad < K)
        atomicAdd(dW + e, (red[threadIdx.x] + red[threadIdx.x + 64]) + (red[threadIdx.x + 128] + red[threadIdx.x + 192]));
}

// ---------------------------------------------------------------- small layers

// W[Co][Kpad] (k = tap*Ci + ci)  ->  Wt[Ci][KpadT] (k' = tap'*Co + co) with
// tap' = 26 - tap: the backward-data weights.
__global__ void k_wt_transpose(const bf16_t *__restrict__ w, bf16_t *__restrict__ wt, int Ci, int Co,
                               int Kpad, int KpadT)
{
    const long long n = (long long)Ci * KpadT;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x) {
        const int ci = (int)(t / KpadT);
        const int k2 = (int)(t % KpadT);
        bf16_t v = 0;
        if (k2 < 27 * Co) {
            const int tap2 = k2 / Co, co = k2 % Co;
            v = w[(long long)co * Kpad + (26 - tap2) * Ci + ci];
        }
        wt[t] = v;
    }
}

__global__ void k_f32_to_bf16(const float *__restrict__ a, bf16_t *__restrict__ b, long long n)
{
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x)
        b[t] = f2bf(a[t]);
}

__global__ void k_bf16_to_f32(const bf16_t *__restrict__ a, float *__restrict__ b, long long n)
{
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x)
        b[t] = bf2f(a[t]);
}

// The layers below move bytes and compute almost nothing: bound is memory, and
// one 2-byte channel per thread with 64-bit index divisions kept them at 1 to
// 2 TB/s.  They take V channels per thread (16-byte loads and stores; V = 1
// for channel counts or addresses that do not allow it) and count groups of
// V channels in 32 bits where those suffice.  Before and now, us: 8 samples of
// 64^3 with 16 channels k_relu_bwd 95 -> 46, k_bias_grad 48 -> 13, k_head_fwd
// 64 -> 14, k_head_bwd 97 -> 47; 8 samples of 32^3 (the smaller side)
// k_pool_fwd 16 channels 26 -> 13, 20 channels (V = 1) 32 -> 21, k_pool_bwd 16
// channels 103 -> 42, k_up_fwd 64 channels 509 -> 116, k_up_bwd stays at 31
// (16 channels) and 122 (64), bound by the strided gather of its eight
// children.  A workgroup laid out as groups by columns by rows of one plane
// instead: level on those, but 20 channels 51, 50000 planes of one position
// 34 where this takes 4.
template <typename T, int V> struct Pack { T v[V]; };

template <typename T, int V>
__device__ __forceinline__ Pack<T, V> load_pack(const T *p)
{
    if constexpr (V == 1) return {*p};
    else {
        static_assert(V * sizeof(T) == 16, "one 16-byte word");
        return __builtin_bit_cast(Pack<T, V>, *reinterpret_cast<const u32x4 *>(p));
    }
}

template <typename T, int V>
__device__ __forceinline__ void store_pack(T *p, const Pack<T, V> &a)
{
    if constexpr (V == 1) *p = a.v[0];
    else *reinterpret_cast<u32x4 *>(p) = __builtin_bit_cast(u32x4, a);
}

// f(plane, y, x, c) for every row y < H, column x < W and first channel c of
// a group (CV groups of V) of `planes` planes.
template <int V, typename I, typename F>
__device__ __forceinline__ void each_group_in(I n, int H, int W, int CV, F f)
{
    for (I t = (I)blockIdx.x * 256 + threadIdx.x; t < n; t += (I)gridDim.x * 256) {
        const I p = t / (I)CV, row = p / (I)W, pl = row / (I)H;
        f((long long)pl, (int)(row - pl * (I)H), (int)(p - row * (I)W), (int)(t - p * (I)CV) * V);
    }
}

template <int V, typename F>
__device__ __forceinline__ void each_group(long long planes, int H, int W, int CV, F f)
{
    const long long n = planes * H * W * CV;
    if (n < (1LL << 31)) each_group_in<V, unsigned>((unsigned)n, H, W, CV, f);
    else each_group_in<V, long long>(n, H, W, CV, f);
}

// g_out(bf16) = g(f32) * (y > 0)   (ReLU backward, y = the layer's BF16 output)
template <int V>
__global__ __launch_bounds__(256) void k_relu_bwd(const float *__restrict__ g, const bf16_t *__restrict__ y,
                                                  bf16_t *__restrict__ out, long long n)
{
    const long long nv = n / V, first = blockIdx.x * 256LL + threadIdx.x;
    for (long long t = first; t < nv; t += gridDim.x * 256LL) {
        const Pack<bf16_t, V> yv = load_pack<bf16_t, V>(y + t * V);
        Pack<bf16_t, V> o;
#pragma unroll
        for (int h = 0; h < V; h += 4) {
            const Pack<float, V == 1 ? 1 : 4> gv = load_pack<float, V == 1 ? 1 : 4>(g + t * V + h);
#pragma unroll
            for (int i = 0; i < (V == 1 ? 1 : 4); ++i) o.v[h + i] = bf2f(yv.v[h + i]) > 0.f ? f2bf(gv.v[i]) : (bf16_t)0;
        }
        store_pack<bf16_t, V>(out + t * V, o);
    }
    if (first < n - nv * V) out[nv * V + first] = bf2f(y[nv * V + first]) > 0.f ? f2bf(g[nv * V + first]) : (bf16_t)0;
}

// db[co] += sum_p g[p][co], C a power of two dividing 256, at least V: a
// thread sums the V channels of its group over a strided set of positions,
// the wave and then the block add up, and one atomic per channel and block
// goes out.  The atomics all fall on the same C words, about 13 ns each in
// turn, so the grid is one block of 8 waves per CU.
constexpr int kBgThreads = 512;

template <int V>
__global__ __launch_bounds__(kBgThreads) void k_bias_grad(const bf16_t *__restrict__ g, float *__restrict__ db,
                                                          long long P, int C)
{
    __shared__ float red[kBgThreads / 64 * 256];
    const int CV = C / V, lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    const long long n = P * CV, step = (long long)gridDim.x * kBgThreads;  // a multiple of CV
    float s[V];
#pragma unroll
    for (int i = 0; i < V; ++i) s[i] = 0.f;
    long long t = (long long)blockIdx.x * kBgThreads + threadIdx.x;
    for (; t + 3 * step < n; t += 4 * step) {
        Pack<bf16_t, V> a[4];
#pragma unroll
        for (int k = 0; k < 4; ++k) a[k] = load_pack<bf16_t, V>(g + (t + k * step) * V);
#pragma unroll
        for (int k = 0; k < 4; ++k)
#pragma unroll
            for (int i = 0; i < V; ++i) s[i] += bf2f(a[k].v[i]);
    }
    for (; t < n; t += step) {
        const Pack<bf16_t, V> a = load_pack<bf16_t, V>(g + t * V);
#pragma unroll
        for (int i = 0; i < V; ++i) s[i] += bf2f(a.v[i]);
    }
    // lanes and waves whose index is equal modulo CV hold the same channels
    for (int off = 32; off >= CV; off >>= 1)
#pragma unroll
        for (int i = 0; i < V; ++i) s[i] += __shfl_xor(s[i], off);
    const int per = CV < 64 ? CV : 64;  // groups a wave holds
    if (lane < per)
#pragma unroll
        for (int i = 0; i < V; ++i) red[wave * per * V + lane * V + i] = s[i];
    __syncthreads();
    // waves w, w + C / (per * V), ... hold the same channels
    if ((int)threadIdx.x < C) {
        float a = 0.f;
        for (int k = threadIdx.x; k < kBgThreads / 64 * per * V; k += C) a += red[k];
        atomicAdd(db + threadIdx.x, a);
    }
}

// 2x2x2 average pool, channels-last.  in [N][2D][2H][2W][C] -> out [N][D][H][W][C]
template <int V>
__global__ __launch_bounds__(256) void k_pool_fwd(const bf16_t *__restrict__ in, bf16_t *__restrict__ out, int N, int D,
                                                  int H, int W, int C)
{
    each_group<V>((long long)N * D, H, W, C / V, [&](long long zb, int y, int x, int c) {
        float s[V];
#pragma unroll
        for (int i = 0; i < V; ++i) s[i] = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const long long row = (2 * zb + (q >> 2)) * 2 * H + 2 * y + ((q >> 1) & 1);
            const Pack<bf16_t, V> a = load_pack<bf16_t, V>(in + (row * 2 * W + 2 * x + (q & 1)) * C + c);
#pragma unroll
            for (int i = 0; i < V; ++i) s[i] += bf2f(a.v[i]);
        }
        Pack<bf16_t, V> o;
#pragma unroll
        for (int i = 0; i < V; ++i) o.v[i] = f2bf(s[i] * 0.125f);
        store_pack<bf16_t, V>(out + ((zb * H + y) * W + x) * C + c, o);
    });
}

// backward of the pool: gin (f32, [N][2D][2H][2W][C]) = gout / 8 (accumulate)
template <int V>
__global__ __launch_bounds__(256) void k_pool_bwd(const float *__restrict__ gout, float *__restrict__ gin, int N, int D,
                                                  int H, int W, int C)
{
    each_group<V>((long long)N * 2 * D, 2 * H, 2 * W, C / V, [&](long long zb, int y, int x, int c) {
        const Pack<float, V> b = load_pack<float, V>(gout + (((zb >> 1) * H + y / 2) * W + x / 2) * C + c);
        float *p = gin + ((zb * 2 * H + y) * 2 * W + x) * C + c;
        Pack<float, V> a = load_pack<float, V>(p);
#pragma unroll
        for (int i = 0; i < V; ++i) a.v[i] += 0.125f * b.v[i];
        store_pack<float, V>(p, a);
    });
}

// nearest x2 upsample into channels [c0, c0+C) of a Ct-channel tensor:
// out[N][2D][2H][2W][Ct]; in [N][D][H][W][C]
template <int V>
__global__ __launch_bounds__(256) void k_up_fwd(const bf16_t *__restrict__ in, bf16_t *__restrict__ out, int N, int D,
                                                int H, int W, int C, int Ct, int c0)
{
    each_group<V>((long long)N * 2 * D, 2 * H, 2 * W, C / V, [&](long long zb, int y, int x, int c) {
        const Pack<bf16_t, V> a = load_pack<bf16_t, V>(in + (((zb >> 1) * H + y / 2) * W + x / 2) * C + c);
        store_pack<bf16_t, V>(out + ((zb * 2 * H + y) * 2 * W + x) * Ct + c0 + c, a);
    });
}

// backward of the upsample: gin[N][D][H][W][C] = sum of the 8 children of
// channel c0+c in gout[N][2D][2H][2W][Ct]
template <int V>
__global__ __launch_bounds__(256) void k_up_bwd(const float *__restrict__ gout, float *__restrict__ gin, int N, int D,
                                                int H, int W, int C, int Ct, int c0)
{
    each_group<V>((long long)N * D, H, W, C / V, [&](long long zb, int y, int x, int c) {
        Pack<float, V> s;
#pragma unroll
        for (int i = 0; i < V; ++i) s.v[i] = 0.f;
#pragma unroll
        for (int q = 0; q < 8; ++q) {
            const long long row = (2 * zb + (q >> 2)) * 2 * H + 2 * y + ((q >> 1) & 1);
            const Pack<float, V> a = load_pack<float, V>(gout + (row * 2 * W + 2 * x + (q & 1)) * Ct + c0 + c);
#pragma unroll
            for (int i = 0; i < V; ++i) s.v[i] += a.v[i];
        }
        store_pack<float, V>(gin + ((zb * H + y) * W + x) * C + c, s);
    });
}

// copy channels: dst[p][dc0 + c] = src[p][sc0 + c], c < C  (concat forward,
// gradient split backward); T is bf16_t or float
template <typename T, int V>
__global__ __launch_bounds__(256) void k_chan_copy(const T *__restrict__ src, T *__restrict__ dst, long long P, int C,
                                                   int Cs, int sc0, int Cd, int dc0, int accumulate)
{
    each_group<V>(P, 1, 1, C / V, [&](long long p, int, int, int c) {
        Pack<T, V> a = load_pack<T, V>(src + p * Cs + sc0 + c);
        T *d = dst + p * Cd + dc0 + c;
        if constexpr (sizeof(T) == 4) {
            if (accumulate) {
                const Pack<T, V> b = load_pack<T, V>(d);
#pragma unroll
                for (int i = 0; i < V; ++i) a.v[i] = b.v[i] + a.v[i];
            }
        }
        store_pack<T, V>(d, a);
    });
}

// 1x1 head: y[p] = b + sum_c w[c] * x[p][c]   (x BF16, w/b/y FP32)
template <int V>
__global__ __launch_bounds__(256) void k_head_fwd(const bf16_t *__restrict__ x, const float *__restrict__ w,
                                                  const float *__restrict__ b, float *__restrict__ y, long long P, int C)
{
    for (long long p = blockIdx.x * 256LL + threadIdx.x; p < P; p += gridDim.x * 256LL) {
        float s = b[0];
        for (int c = 0; c < C; c += V) {
            const Pack<bf16_t, V> a = load_pack<bf16_t, V>(x + p * C + c);
#pragma unroll
            for (int i = 0; i < V; ++i) s += w[c + i] * bf2f(a.v[i]);
        }
        y[p] = s;
    }
}

// head backward: gx[p][c] = g[p] * w[c] (f32); dw[c] += sum_p g[p] x[p][c];
// db += sum_p g[p].  A thread takes four channels of a position, so that a
// wave's loads and stores are whole lines; sums go through the wave, the
// block and one atomic per word and block (one block of 8 waves per CU: the
// atomics are serial, about 13 ns each).
constexpr int kHeadThreads = 512;

template <int C, bool ALIGNED>
__global__ __launch_bounds__(kHeadThreads) void k_head_bwd(const bf16_t *__restrict__ x, const float *__restrict__ w,
                                                           const float *__restrict__ g, float *__restrict__ gx,
                                                           float *__restrict__ dw, float *__restrict__ db, long long P)
{
    constexpr int G = C / 4;  // groups of four channels, a power of two up to 64
    __shared__ float red[kHeadThreads / 64][C + 1];
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6, c = (threadIdx.x & (G - 1)) * 4;
    float sdw[4] = {0.f, 0.f, 0.f, 0.f}, sdb = 0.f;
    float wc[4];
#pragma unroll
    for (int i = 0; i < 4; ++i) wc[i] = w[c + i];
    constexpr int kPos = kHeadThreads / G;
    for (long long p = (long long)blockIdx.x * kPos + threadIdx.x / G; p < P; p += (long long)gridDim.x * kPos) {
        const float gp = g[p];
        sdb += gp;
        uint16_t xv[4];
        if constexpr (ALIGNED) {
            const uint2 u = *reinterpret_cast<const uint2 *>(x + p * C + c);
            xv[0] = (uint16_t)u.x, xv[1] = (uint16_t)(u.x >> 16), xv[2] = (uint16_t)u.y, xv[3] = (uint16_t)(u.y >> 16);
            const f32x4 o = {gp * wc[0], gp * wc[1], gp * wc[2], gp * wc[3]};
            *reinterpret_cast<f32x4 *>(gx + p * C + c) = o;
        } else {
#pragma unroll
            for (int i = 0; i < 4; ++i) xv[i] = x[p * C + c + i], gx[p * C + c + i] = gp * wc[i];
        }
#pragma unroll
        for (int i = 0; i < 4; ++i) sdw[i] += gp * bf2f(xv[i]);
    }
    for (int off = 32; off >= G; off >>= 1) {
#pragma unroll
        for (int i = 0; i < 4; ++i) sdw[i] += __shfl_xor(sdw[i], off);
        sdb += __shfl_xor(sdb, off);
    }
    if (lane < G)
#pragma unroll
        for (int i = 0; i < 4; ++i) red[wave][c + i] = sdw[i];
    if (lane == 0) red[wave][C] = sdb;
    __syncthreads();
    if ((int)threadIdx.x <= C) {
        float a = 0.f;
#pragma unroll
        for (int k = 0; k < kHeadThreads / 64; ++k) a += red[k][threadIdx.x];
        atomicAdd((int)threadIdx.x < C ? dw + threadIdx.x : db, a);
    }
}

// prediction u = base + y on the interior of each n^3 sample, base elsewhere;
// loss += sum (u - target)^2 over the interior; g = 2 (u - target) / count
__global__ __launch_bounds__(256) void k_mse(const float *__restrict__ base,
                                             const float *__restrict__ y,
                                             const float *__restrict__ target,
                                             float *__restrict__ g, double *__restrict__ loss,
                                             float *__restrict__ pred, int N, int n, double scale)
{
    __shared__ double red[256];
    const long long P = (long long)N * n * n * n;
    double acc = 0.0;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < P;
         p += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(p % n), yy = (int)((p / n) % n), z = (int)((p / ((long long)n * n)) % n);
        const bool in = x > 0 && x < n - 1 && yy > 0 && yy < n - 1 && z > 0 && z < n - 1;
        const float u = in ? base[p] + y[p] : base[p];
        if (pred) pred[p] = u;
        float gg = 0.f;
        if (in && target) {
            const float d = u - target[p];
            acc += (double)d * d;
            gg = (float)(2.0 * scale) * d;
        }
        if (g) g[p] = gg;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0 && loss) atomicAdd(loss, red[0]);
}

// out = a*x + b*y (FP32)
__global__ void k_axpby(float *__restrict__ out, float a, const float *__restrict__ x, float b,
                        const float *__restrict__ y, long long n)
{
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x)
        out[t] = a * x[t] + b * y[t];
}

// loss += sum x^2 (FP64), g = 2*scale*x
__global__ __launch_bounds__(256) void k_sumsq(const float *__restrict__ x, float *__restrict__ g,
                                               double *__restrict__ loss, long long n, double scale)
{
    __shared__ double red[256];
    double acc = 0.0;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x) {
        const float v = x[t];
        acc += (double)v * v;
        if (g) g[t] = (float)(2.0 * scale) * v;
    }
    red[threadIdx.x] = acc;
    __syncthreads();
    for (int h = 128; h > 0; h >>= 1) {
        if ((int)threadIdx.x < h) red[threadIdx.x] += red[threadIdx.x + h];
        __syncthreads();
    }
    if (threadIdx.x == 0 && loss) atomicAdd(loss, red[0]);
}

// Adam (Kingma & Ba 2015) with bias correction; writes the BF16 copy of the
// weights for the MFMA kernels (zero columns of padded rows stay zero
// because their gradients are zero).
__global__ void k_adam(float *__restrict__ w, const float *__restrict__ g, float *__restrict__ m,
                       float *__restrict__ v, bf16_t *__restrict__ wbf, long long n, float lr,
                       float b1, float b2, float eps, float c1, float c2)
{
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x) {
        const float gt = g[t];
        const float mt = b1 * m[t] + (1.f - b1) * gt;
        const float vt = b2 * v[t] + (1.f - b2) * gt * gt;
        m[t] = mt;
        v[t] = vt;
        const float upd = lr * (mt / c1) / (sqrtf(vt / c2) + eps);
        const float wt = w[t] - upd;
        w[t] = wt;
        if (wbf) wbf[t] = f2bf(wt);
    }
}

// Input features of an n^3 sample from its field u (boundary shell filled):
// channel 0 = transfinite blend of the six faces
//   (1/3) sum over axes [(1-s) F_lo + s F_hi],  s = coordinate / (n-1),
// channel 1 = the boundary value on the shell (0 inside), channels 2..C-1 = 0.
// base[p] receives the blend inside and the boundary value on the shell.
__global__ void k_features(const float *__restrict__ u, bf16_t *__restrict__ feat,
                           float *__restrict__ base, int N, int n, int C)
{
    const long long P = (long long)N * n * n * n;
    const long long nn = (long long)n * n;
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < P;
         p += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(p % n), y = (int)((p / n) % n), z = (int)((p / nn) % n);
        const long long s0 = p - (long long)z * nn - (long long)y * n - x;  // sample origin
        const float inv = 1.0f / (float)(n - 1);
        const float sx = x * inv, sy = y * inv, sz = z * inv;
        const float fx = (1.f - sx) * u[s0 + (long long)z * nn + (long long)y * n] +
                         sx * u[s0 + (long long)z * nn + (long long)y * n + (n - 1)];
        const float fy = (1.f - sy) * u[s0 + (long long)z * nn + x] +
                         sy * u[s0 + (long long)z * nn + (long long)(n - 1) * n + x];
        const float fz = (1.f - sz) * u[s0 + (long long)y * n + x] +
                         sz * u[s0 + (long long)(n - 1) * nn + (long long)y * n + x];
        const float blend = (fx + fy + fz) * (1.0f / 3.0f);
        const bool shell = x == 0 || y == 0 || z == 0 || x == n - 1 || y == n - 1 || z == n - 1;
        const float bv = shell ? u[p] : 0.f;
        // channels: blend, shell value, the three coordinates, the distance
        // to the nearest face (scaled to [0, 1]), zeros
        const float dist =
            2.f * fminf(fminf(fminf(sx, 1.f - sx), fminf(sy, 1.f - sy)), fminf(sz, 1.f - sz));
        for (int c = 0; c < C; ++c) {
            const float v = c == 0 ? blend
                          : c == 1 ? bv
                          : c == 2 ? sx
                          : c == 3 ? sy
                          : c == 4 ? sz
                          : c == 5 ? dist
                          : 0.f;
            feat[p * C + c] = f2bf(v);
        }
        if (base) base[p] = shell ? u[p] : blend;
    }
}

// Trilinear interpolation of the interior of a node-centred m^3 field onto
// an M^3 field: fine node I maps to coarse coordinate I*(m-1)/(M-1).  The
// shell of `out` is left untouched (it holds the exact boundary).
__global__ void k_trilinear(const float *__restrict__ in, float *__restrict__ out, int m, int M)
{
    const long long n = (long long)M * M * M;
    const float sc = (float)(m - 1) / (float)(M - 1);
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n;
         t += (long long)gridDim.x * blockDim.x) {
        const int X = (int)(t % M), Y = (int)((t / M) % M), Z = (int)(t / ((long long)M * M));
        if (X == 0 || Y == 0 || Z == 0 || X == M - 1 || Y == M - 1 || Z == M - 1) continue;
        const float cx = X * sc, cy = Y * sc, cz = Z * sc;
        const int x0 = min((int)cx, m - 2), y0 = min((int)cy, m - 2), z0 = min((int)cz, m - 2);
        const float fx = cx - x0, fy = cy - y0, fz = cz - z0;
        auto at = [&](int a, int b, int c) { return in[((long long)c * m + b) * m + a]; };
        const float c00 = at(x0, y0, z0) * (1 - fx) + at(x0 + 1, y0, z0) * fx;
        const float c10 = at(x0, y0 + 1, z0) * (1 - fx) + at(x0 + 1, y0 + 1, z0) * fx;
        const float c01 = at(x0, y0, z0 + 1) * (1 - fx) + at(x0 + 1, y0, z0 + 1) * fx;
        const float c11 = at(x0, y0 + 1, z0 + 1) * (1 - fx) + at(x0 + 1, y0 + 1, z0 + 1) * fx;
        const float c0 = c00 * (1 - fy) + c10 * fy, c1 = c01 * (1 - fy) + c11 * fy;
        out[t] = c0 * (1 - fz) + c1 * fz;
    }
}

// Dirichlet faces from Fourier modes: face value sum_m a_m sin(pi kx s) sin(pi ky t)
// with (s, t) the face's two coordinates scaled to [0, 1]; modes[f*M*3 + m*3 + {0,1,2}]
// = (a, kx, ky) for the six faces x0, x1, y0, y1, z0, z1.  Writes the shell of
// the N samples' n^3 fields (the interior is untouched).
__global__ void k_fourier_faces(float *__restrict__ u, const float *__restrict__ modes, int N, int n,
                                int M)
{
    const long long nn = (long long)n * n;
    const long long P = (long long)N * nn * n;
    const float inv = 1.0f / (float)(n - 1);
    for (long long p = blockIdx.x * (long long)blockDim.x + threadIdx.x; p < P;
         p += (long long)gridDim.x * blockDim.x) {
        const int x = (int)(p % n), y = (int)((p / n) % n), z = (int)((p / nn) % n);
        const int b = (int)(p / (nn * n));
        int f = -1;
        float s = 0.f, t = 0.f;
        if (x == 0 || x == n - 1) { f = x == 0 ? 0 : 1; s = y * inv; t = z * inv; }
        else if (y == 0 || y == n - 1) { f = y == 0 ? 2 : 3; s = x * inv; t = z * inv; }
        else if (z == 0 || z == n - 1) { f = z == 0 ? 4 : 5; s = x * inv; t = y * inv; }
        if (f < 0) continue;
        const float *md = modes + ((long long)b * 6 + f) * M * 3;
        float v = 0.f;
        for (int m = 0; m < M; ++m)
            v += md[3 * m] * sinpif(md[3 * m + 1] * s) * sinpif(md[3 * m + 2] * t);
        u[p] = v;
    }
}

}  // namespace st

// ---------------------------------------------------------------- C ABI

using namespace st;

static dim3 gs_grid(long long n)
{
    long long b = (n + 255) / 256;
    if (b > 65536) b = 65536;
    if (b < 1) b = 1;
    return dim3((unsigned)b);
}

static bool on16(const void *a, const void *b = nullptr, const void *c = nullptr)
{
    return (((uintptr_t)a | (uintptr_t)b | (uintptr_t)c) & 15) == 0;
}

// Workgroups of each_group over n groups of channels.
static dim3 group_grid(long long n)
{
    return dim3((unsigned)std::max(1LL, std::min((n + 255) / 256, 65536LL)));
}

// Blocks of a sum over n values that ends in one atomic per block on one word,
// about 13 ns each in turn: 512 up to 2^22 values (2^21 53 us with 4096, 13
// with 512), then more for the memory's sake, up to 2048 (2^25 102 us with 512,
// 64 with 2048).
static long long loss_blocks(long long n) { return std::max(512LL, std::min(n >> 13, 2048LL)); }

static ConvGeom make_conv(int N, int D, int H, int W, int Ci, int Co, int Kpad)
{
    ConvGeom g;
    g.N = N; g.D = D; g.H = H; g.W = W; g.Ci = Ci; g.Co = Co; g.Kpad = Kpad;
    g.P = (int)((long long)N * D * H * W);
    return g;
}

// The tiled convolution of a layer (fn null: none).
struct ConvTilePlan {
    const void *fn = nullptr;
    TileGeom q;
    int nct, blocks, lds;
};

template <int NB>
static const void *conv_tile_fn(int mb)
{
    return mb == 4 ? reinterpret_cast<const void *>(&k_conv3_tile<NB, 4>)
                   : reinterpret_cast<const void *>(&k_conv3_tile<NB, 2>);
}

// blocks of 16 output channels of a wave of k_conv3
static int conv_flat_nb(int co) { return co >= 64 ? 4 : (co >= 32 ? 2 : 1); }

// Whether the tiles are ahead of k_conv3, by the time a chunk of 32 weight
// columns takes in each (us, fitted to 690 shapes of 8 to 262144 positions and
// 4 to 256 channels; there and on 417 random shapes the choice is within 0.3%
// of the better one on average, at worst 1.3 times).  Tiles: per round of workgroups, by channel blocks, depth
// and workgroups per CU.  k_conv3: a latency until the waves fill the card,
// then a rate; taps outside a sample of one plane, row or column cost it no
// load, which shows once there are waves enough.  64 -> 64 channels, tiles / k_conv3: 8 x 16^3 31 / 64, 1 x 40^3
// 83 / 69; 64 -> 80 (channel blocks in two halves, each staging the tile)
// 135 / 91; 1 x 300 x 300 x 3 (3 of 16 columns) 1136 / 232.
static bool conv_tile_ahead(const ConvGeom &g, int nb, int mb, bool two_per_cu, int blocks)
{
    static const double tile[4][2] = {{0.19, 0.36}, {0.29, 0.45}, {0.32, 0.70}, {0.43, 0.60}};
    const long long round = two_per_cu ? 512 : 256;
    double t = (double)((blocks + round - 1) / round) * tile[nb - 1][mb == 4 || (nb == 4 && two_per_cu)];
    if ((g.Co + 15) / 16 % nb) t *= 1.2;  // a last group of fewer blocks
    const int fb = conv_flat_nb(g.Co);
    // in 1024; of four channel blocks, those with fewer as their share
    const double groups = fb == 4 ? (g.Co + 15) / 16 / 4.0 : (g.Co + 16 * fb - 1) / (16 * fb);
    const double waves = (double)((g.P + 63) / 64) * groups / 1024;
    double f = fb == 1 ? std::max(0.95, 0.50 * waves) : fb == 2 ? std::max(0.85, 0.60 * waves) : std::max(1.15, 0.87 * waves);
    if (waves >= 0.25 && (g.D == 1 || g.H == 1 || g.W == 1)) f *= 0.7;
    return t <= f;
}

static ConvTilePlan conv_tile_plan(const ConvGeom &g, const void *out_bf, const void *out_f)
{
    ConvTilePlan t;
    // the kernel stores four channels at once
    if ((reinterpret_cast<uintptr_t>(out_bf) & 7) || (reinterpret_cast<uintptr_t>(out_f) & 15)) return t;
    int mb = 4;
    const int cb = (g.Co + 15) / 16;  // blocks of 16 output channels
    const int nb = cb <= 4 ? cb : cb % 4 == 0 ? 4 : cb % 3 == 0 ? 3 : 4;
    const int tab = (g.Kpad / 32 + 3) / 4 * 64 + 2 * conv_chunks(nb) * nb * 1024;
    t.lds = tile_positions(mb) * tile_stride(g.Ci) + tab;
    if (mb == 4 && t.lds > 80 * 1024) {
        mb = 2;
        t.lds = tile_positions(mb) * tile_stride(g.Ci) + tab;
    }
    if (t.lds > kMaxLds) return t;
    t.nct = (cb + nb - 1) / nb;
    t.q.g = g;
    t.q.tx = (g.W + kTx - 1) / kTx;
    t.q.ty = (g.H + kTy - 1) / kTy;
    t.q.tz = (g.D + mb - 1) / mb;
    const long long blocks = (long long)g.N * t.q.tx * t.q.ty * t.q.tz * t.nct;
    if (blocks >= (1LL << 31) || !conv_tile_ahead(g, nb, mb, t.lds <= kMaxLds / 2, (int)blocks)) return t;
    t.blocks = (int)blocks;
    t.fn = nb == 4 ? conv_tile_fn<4>(mb) : nb == 3 ? conv_tile_fn<3>(mb) : nb == 2 ? conv_tile_fn<2>(mb) : conv_tile_fn<1>(mb);
    return t;
}

// The tiled weight gradient of a layer (fn null: none).
struct WgradTilePlan {
    const void *fn = nullptr;
    TileGeom q;
    int ntiles, positions;   // tiles, positions of a tile
    int parts, groups;       // workgroups per group of 16*NC output channels
    int ranges, cols, lds;   // ranges of `cols` column blocks
};
constexpr int kWgMaxBlocks = 21;  // column blocks of a wave, the most its registers hold (Ci = 96)

template <int NC, int TZ>
static const void *wgrad_tile_fn(int nbw)
{
    if (nbw <= 2) return reinterpret_cast<const void *>(&k_conv3_wgrad_tile<NC, 2, TZ>);
    if (nbw <= 4) return reinterpret_cast<const void *>(&k_conv3_wgrad_tile<NC, 4, TZ>);
    if (nbw <= 7) return reinterpret_cast<const void *>(&k_conv3_wgrad_tile<NC, 7, TZ>);
    if (nbw <= 11) return reinterpret_cast<const void *>(&k_conv3_wgrad_tile<NC, 11, TZ>);
    if (nbw <= 14) return reinterpret_cast<const void *>(&k_conv3_wgrad_tile<NC, 14, TZ>);
    if (nbw <= 21) return reinterpret_cast<const void *>(&k_conv3_wgrad_tile<NC, 21, TZ>);
    return nullptr;
}

static WgradTilePlan wgrad_tile_plan(const ConvGeom &g)
{
    WgradTilePlan t;
    const int nc = g.Co > 16 ? 2 : 1;
    // ranges of weight columns of at most kWgMaxBlocks blocks per wave
    const int nkb = (27 * g.Ci + 15) / 16;
    t.ranges = (nkb + kWgMaxBlocks * kWgWaves - 1) / (kWgMaxBlocks * kWgWaves);
    t.cols = (nkb + t.ranges - 1) / t.ranges;
    const int nbw = (t.cols + kWgWaves - 1) / kWgWaves;
    // tiles of 4 planes while two workgroups fit a CU's LDS, else of 2
    auto lds = [&](int tz) { return tile_positions(tz) * tile_stride(g.Ci) + tz * kTy * kTx * (nc * 32 + (nc == 1 ? 0 : 16)); };
    const int tz = lds(4) <= 80 * 1024 ? 4 : 2;
    t.lds = lds(tz);
    if (t.lds > kMaxLds) return t;
    t.q.g = g;
    t.q.tx = (g.W + kTx - 1) / kTx;
    t.q.ty = (g.H + kTy - 1) / kTy;
    t.q.tz = (g.D + tz - 1) / tz;
    const long long tiles = (long long)g.N * t.q.tx * t.q.ty * t.q.tz;
    if (tiles >= (1LL << 31)) return t;
    t.ntiles = (int)tiles;
    t.positions = tz * kTy * kTx;
    t.groups = (g.Co + 16 * nc - 1) / (16 * nc);
    if (t.groups > 65535) return t;
    // one round of workgroups at most (one or two per CU, as their LDS lets
    // them) and 32 MiB of partial sums, which leaves 101 of 256 CUs at work for
    // 96 -> 32 channels and 150 for 64 -> 64
    const long long round = t.lds > kMaxLds / 2 ? 256 : 512;
    const long long want = std::min(round / (t.groups * t.ranges), (32LL << 20) / (4LL * g.Co * g.Kpad));
    t.parts = (int)std::max(1LL, std::min((long long)t.ntiles, want));
    if (nc == 1) t.fn = tz == 4 ? wgrad_tile_fn<1, 4>(nbw) : wgrad_tile_fn<1, 2>(nbw);
    else t.fn = tz == 4 ? wgrad_tile_fn<2, 4>(nbw) : wgrad_tile_fn<2, 2>(nbw);
    return t;
}

enum WgradForm { WG_TILE = 1, WG_CHANNEL_MAJOR, WG_GATHER };

// Where tiles are mostly padding and there are many of them, the kernels that
// flatten positions are ahead (us, tiles / channel-major rows / gathering:
// 1 x 1 x 1 x 100000 positions 64 -> 64 channels 570 / 185 / 527, 4000 x 2 x 2
// x 2 128 -> 128 1517 / - / 688, but 16 -> 16 few products and 1 x 1 x 1 x 1000
// 64 -> 64 few tiles: 20 / 66 / 151), and a handful of positions is one step
// of the gathering kernel (1 x 2 x 2 x 2 64 -> 64 16.5 / - / 8.1).
static WgradForm wgrad_form(const ConvGeom &g, const WgradTilePlan &t)
{
    const bool rows = g.W % 8 == 0 && g.Ci <= kTrMaxC && g.Co <= kTrMaxC;
    const WgradForm flat = rows ? WG_CHANNEL_MAJOR : WG_GATHER;
    if (!t.fn) return flat;
    // up to 256 positions: a step of the gathering kernel per 32, against the
    // columns of a wave and the reduction (us; within 3 of the measured times)
    if (g.P <= 256) {
        const double gather = 3.5 + 4.6 * ((g.P + 31) / 32);
        const double tile = 8 + 0.7 * ((t.cols + kWgWaves - 1) / kWgWaves) + t.parts * 2e-6 * g.Co * g.Kpad;
        if (gather < tile) return WG_GATHER;
    }
    const long long room = (long long)t.ntiles * t.positions, P = g.P;
    // rows of positions alone: 18 of 27 taps lie outside and cost no load
    const int least = rows || (g.D == 1 && g.H == 1) ? 8 : 16;
    if (t.ntiles >= 1024 && least * P <= room && (rows || g.Ci * g.Co >= 1536)) return flat;
    return WG_TILE;
}

extern "C" {

int st_nn_kpad(int ci) { return (27 * ci + 31) / 32 * 32; }

st_status st_nn_conv3(const void *act, const void *w, const float *bias, void *out_bf16, float *out_f32,
                      int N, int D, int H, int W, int Ci, int Co, int relu, int accumulate, void *stream)
{
    if (Ci % 8 || Ci < 8 || Co % 4 || Co < 4 || N < 1 || D < 1 || H < 1 || W < 1)
        return fail(ST_EINVAL, "conv3: Ci must be a multiple of 8 and Co of 4 (got %d, %d)", Ci, Co);
    if ((long long)N * D * H * W >= (1LL << 31)) return fail(ST_EINVAL, "conv3: too many positions");
    const ConvGeom g = make_conv(N, D, H, W, Ci, Co, st_nn_kpad(Ci));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16_t *a = static_cast<const bf16_t *>(act);
    const bf16_t *wt = static_cast<const bf16_t *>(w);
    bf16_t *ob = static_cast<bf16_t *>(out_bf16);
    const ConvTilePlan t = conv_tile_plan(g, out_bf16, out_f32);
    if (t.fn) {
        void *args[] = {&a, &wt, &bias, &ob, &out_f32, const_cast<TileGeom *>(&t.q), const_cast<int *>(&t.nct), &relu,
                        &accumulate};
        hipError_t e = hipFuncSetAttribute(t.fn, hipFuncAttributeMaxDynamicSharedMemorySize, t.lds);
        if (e != hipSuccess) return hip_check(e, "hipFuncSetAttribute(conv3 LDS)");
        return hip_check(hipLaunchKernel(t.fn, dim3(t.blocks), dim3(256), args, t.lds, s), "conv3 launch");
    }
    const int nb = conv_flat_nb(Co);
    const long long waves = ((g.P + 63) / 64) * ((Co + 16 * nb - 1) / (16 * nb));
    const dim3 grid((unsigned)((waves + 3) / 4)), block(256);
    if (nb == 4) hipLaunchKernelGGL((k_conv3<4, 4>), grid, block, 0, s, a, wt, bias, ob, out_f32, g, relu, accumulate);
    else if (nb == 2) hipLaunchKernelGGL((k_conv3<2, 4>), grid, block, 0, s, a, wt, bias, ob, out_f32, g, relu, accumulate);
    else hipLaunchKernelGGL((k_conv3<1, 4>), grid, block, 0, s, a, wt, bias, ob, out_f32, g, relu, accumulate);
    return hip_check(hipGetLastError(), "conv3 launch");
}

st_status st_nn_conv3_wgrad(const void *x, const void *dy, float *dw, int N, int D, int H, int W, int Ci,
                            int Co, void *stream)
{
    if (Ci % 8 || Ci < 8) return fail(ST_EINVAL, "conv3 wgrad: Ci must be a multiple of 8");
    if ((long long)N * D * H * W >= (1LL << 31)) return fail(ST_EINVAL, "conv3 wgrad: too many positions");
    const ConvGeom g = make_conv(N, D, H, W, Ci, Co, st_nn_kpad(Ci));
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16_t *xb = static_cast<const bf16_t *>(x), *yb = static_cast<const bf16_t *>(dy);
    StreamTurn turn(s);
    const WgradTilePlan t = wgrad_tile_plan(g);
    WgradForm form = wgrad_form(g, t);
    // partial sums, or channel-major copies of both operands (slot 0); the
    // gathering kernel where there is no room for them
    void *ws = nullptr;
    if (form != WG_GATHER) {
        const st_status st = workspace_slot(0, form == WG_TILE ? (size_t)t.parts * Co * g.Kpad * sizeof(float)
                                                               : ((size_t)g.P * Ci + (size_t)g.P * Co) * sizeof(bf16_t), s, &ws);
        if (st == ST_ENOMEM) {
            (void)hipGetLastError();
            form = WG_GATHER;
        } else if (st != ST_OK) {
            return st;
        }
    }
    if (form == WG_TILE) {
        float *part = static_cast<float *>(ws);
        int wide = Co % 4 == 0 && (reinterpret_cast<uintptr_t>(dy) & 7) == 0;
        void *args[] = {&xb, &yb, &part, const_cast<TileGeom *>(&t.q), const_cast<int *>(&t.ntiles), const_cast<int *>(&t.cols),
                        &wide};
        hipError_t e = hipFuncSetAttribute(t.fn, hipFuncAttributeMaxDynamicSharedMemorySize, t.lds);
        if (e != hipSuccess) return hip_check(e, "hipFuncSetAttribute(wgrad LDS)");
        e = hipLaunchKernel(t.fn, dim3(t.parts, t.groups, t.ranges), dim3(64 * kWgWaves), args, t.lds, s);
        if (e != hipSuccess) return hip_check(e, "conv3 wgrad launch");
        const int n = Co * g.Kpad;
        hipLaunchKernelGGL(k_wgrad_reduce, dim3((n + 63) / 64), dim3(256), 0, s, part, dw, n, 27 * Ci, g.Kpad, t.parts);
        return hip_check(hipGetLastError(), "conv3 wgrad reduce launch");
    }
    const int pchunk = 2048;
    const int K = 27 * Ci;
    const long long nkt = (K + 63) / 64, nct = (Co + 15) / 16, nch = (g.P + pchunk - 1) / pchunk;
    const long long waves = nkt * nct * nch;
    const dim3 grid((unsigned)((waves + 3) / 4));
    if (form == WG_CHANNEL_MAJOR) {
        bf16_t *xt = static_cast<bf16_t *>(ws), *dyt = xt + (size_t)g.P * Ci;
        const dim3 tg((unsigned)((g.P + 63) / 64));
        hipLaunchKernelGGL(k_pc_transpose, tg, dim3(256), 0, s, xb, xt, g.P, Ci);
        hipLaunchKernelGGL(k_pc_transpose, tg, dim3(256), 0, s, yb, dyt, g.P, Co);
        hipLaunchKernelGGL((k_conv3_wgrad_t<4>), grid, dim3(256), 0, s, xt, dyt, dw, g, pchunk);
        return hip_check(hipGetLastError(), "conv3 wgrad launch");
    }
    hipLaunchKernelGGL((k_conv3_wgrad<4>), grid, dim3(256), 0, s, xb, yb, dw, g, pchunk);
    return hip_check(hipGetLastError(), "conv3 wgrad launch");
}

st_status st_nn_wt_transpose(const void *w, void *wt, int Ci, int Co, void *stream)
{
    const int Kpad = st_nn_kpad(Ci), KpadT = st_nn_kpad(Co);
    hipLaunchKernelGGL(k_wt_transpose, gs_grid((long long)Ci * KpadT), dim3(256), 0,
                       static_cast<hipStream_t>(stream), static_cast<const bf16_t *>(w),
                       static_cast<bf16_t *>(wt), Ci, Co, Kpad, KpadT);
    return hip_check(hipGetLastError(), "wt transpose launch");
}

st_status st_nn_f32_to_bf16(const float *a, void *b, long long n, void *stream)
{
    hipLaunchKernelGGL(k_f32_to_bf16, gs_grid(n), dim3(256), 0, static_cast<hipStream_t>(stream), a,
                       static_cast<bf16_t *>(b), n);
    return hip_check(hipGetLastError(), "f32->bf16 launch");
}

st_status st_nn_bf16_to_f32(const void *a, float *b, long long n, void *stream)
{
    hipLaunchKernelGGL(k_bf16_to_f32, gs_grid(n), dim3(256), 0, static_cast<hipStream_t>(stream),
                       static_cast<const bf16_t *>(a), b, n);
    return hip_check(hipGetLastError(), "bf16->f32 launch");
}

st_status st_nn_relu_bwd(const float *g, const void *y, void *out, long long n, void *stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16_t *yb = static_cast<const bf16_t *>(y);
    bf16_t *ob = static_cast<bf16_t *>(out);
    if (on16(g, y, out)) hipLaunchKernelGGL(k_relu_bwd<8>, gs_grid((n + 7) / 8), dim3(256), 0, s, g, yb, ob, n);
    else hipLaunchKernelGGL(k_relu_bwd<1>, gs_grid(n), dim3(256), 0, s, g, yb, ob, n);
    return hip_check(hipGetLastError(), "relu bwd launch");
}

st_status st_nn_bias_grad(const void *g, float *db, long long P, int C, void *stream)
{
    if (C < 1 || 256 % C || (C & (C - 1))) return fail(ST_EINVAL, "bias grad: C must be a power of two dividing 256");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16_t *gb = static_cast<const bf16_t *>(g);
    const bool wide = C % 8 == 0 && on16(g);
    long long blocks = (P * (wide ? C / 8 : C) + kBgThreads - 1) / kBgThreads;
    if (blocks > 256) blocks = 256;
    if (wide) hipLaunchKernelGGL(k_bias_grad<8>, dim3((unsigned)blocks), dim3(kBgThreads), 0, s, gb, db, P, C);
    else hipLaunchKernelGGL(k_bias_grad<1>, dim3((unsigned)blocks), dim3(kBgThreads), 0, s, gb, db, P, C);
    return hip_check(hipGetLastError(), "bias grad launch");
}

st_status st_nn_pool_fwd(const void *in, void *out, int N, int D, int H, int W, int C, void *stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16_t *ib = static_cast<const bf16_t *>(in);
    bf16_t *ob = static_cast<bf16_t *>(out);
    const bool wide = C % 8 == 0 && on16(in, out);
    const dim3 grid = group_grid((long long)N * D * H * W * (wide ? C / 8 : C));
    if (wide) hipLaunchKernelGGL(k_pool_fwd<8>, grid, dim3(256), 0, s, ib, ob, N, D, H, W, C);
    else hipLaunchKernelGGL(k_pool_fwd<1>, grid, dim3(256), 0, s, ib, ob, N, D, H, W, C);
    return hip_check(hipGetLastError(), "pool launch");
}

st_status st_nn_pool_bwd(const float *gout, float *gin, int N, int D, int H, int W, int C, void *stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool wide = C % 4 == 0 && on16(gout, gin);
    const dim3 grid = group_grid(8LL * N * D * H * W * (wide ? C / 4 : C));
    if (wide) hipLaunchKernelGGL(k_pool_bwd<4>, grid, dim3(256), 0, s, gout, gin, N, D, H, W, C);
    else hipLaunchKernelGGL(k_pool_bwd<1>, grid, dim3(256), 0, s, gout, gin, N, D, H, W, C);
    return hip_check(hipGetLastError(), "pool bwd launch");
}

st_status st_nn_up_fwd(const void *in, void *out, int N, int D, int H, int W, int C, int Ct, int c0,
                       void *stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16_t *ib = static_cast<const bf16_t *>(in);
    bf16_t *ob = static_cast<bf16_t *>(out);
    const bool wide = (C | Ct | c0) % 8 == 0 && on16(in, out);
    const dim3 grid = group_grid(8LL * N * D * H * W * (wide ? C / 8 : C));
    if (wide) hipLaunchKernelGGL(k_up_fwd<8>, grid, dim3(256), 0, s, ib, ob, N, D, H, W, C, Ct, c0);
    else hipLaunchKernelGGL(k_up_fwd<1>, grid, dim3(256), 0, s, ib, ob, N, D, H, W, C, Ct, c0);
    return hip_check(hipGetLastError(), "upsample launch");
}

st_status st_nn_up_bwd(const float *gout, float *gin, int N, int D, int H, int W, int C, int Ct, int c0,
                       void *stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool wide = (C | Ct | c0) % 4 == 0 && on16(gout, gin);
    const dim3 grid = group_grid((long long)N * D * H * W * (wide ? C / 4 : C));
    if (wide) hipLaunchKernelGGL(k_up_bwd<4>, grid, dim3(256), 0, s, gout, gin, N, D, H, W, C, Ct, c0);
    else hipLaunchKernelGGL(k_up_bwd<1>, grid, dim3(256), 0, s, gout, gin, N, D, H, W, C, Ct, c0);
    return hip_check(hipGetLastError(), "upsample bwd launch");
}

extern "C++" {
template <typename T, int V>
static void chan_copy(const void *src, void *dst, long long P, int C, int Cs, int sc0, int Cd, int dc0, int accumulate,
                      hipStream_t s)
{
    hipLaunchKernelGGL((k_chan_copy<T, V>), group_grid(P * (C / V)), dim3(256), 0, s, static_cast<const T *>(src),
                       static_cast<T *>(dst), P, C, Cs, sc0, Cd, dc0, accumulate);
}
}

st_status st_nn_chan_copy(const void *src, void *dst, long long P, int C, int Cs, int sc0, int Cd, int dc0,
                          int is_f32, int accumulate, void *stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bool wide = (C | Cs | sc0 | Cd | dc0) % (is_f32 ? 4 : 8) == 0 && on16(src, dst);
    if (is_f32 && wide) chan_copy<float, 4>(src, dst, P, C, Cs, sc0, Cd, dc0, accumulate, s);
    else if (is_f32) chan_copy<float, 1>(src, dst, P, C, Cs, sc0, Cd, dc0, accumulate, s);
    else if (wide) chan_copy<bf16_t, 8>(src, dst, P, C, Cs, sc0, Cd, dc0, 0, s);
    else chan_copy<bf16_t, 1>(src, dst, P, C, Cs, sc0, Cd, dc0, 0, s);
    return hip_check(hipGetLastError(), "channel copy launch");
}

st_status st_nn_head_fwd(const void *x, const float *w, const float *b, float *y, long long P, int C,
                         void *stream)
{
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16_t *xb = static_cast<const bf16_t *>(x);
    if (C % 8 == 0 && on16(x)) hipLaunchKernelGGL(k_head_fwd<8>, gs_grid(P), dim3(256), 0, s, xb, w, b, y, P, C);
    else hipLaunchKernelGGL(k_head_fwd<1>, gs_grid(P), dim3(256), 0, s, xb, w, b, y, P, C);
    return hip_check(hipGetLastError(), "head launch");
}

st_status st_nn_head_bwd(const void *x, const float *w, const float *g, float *gx, float *dw, float *db,
                         long long P, int C, void *stream)
{
    if (C != 16) return fail(ST_EINVAL, "head: built for 16 channels");
    hipStream_t s = static_cast<hipStream_t>(stream);
    const bf16_t *xb = static_cast<const bf16_t *>(x);
    long long blocks = (P * 4 + kHeadThreads - 1) / kHeadThreads;
    if (blocks > 256) blocks = 256;
    if (on16(x, gx))
        hipLaunchKernelGGL((k_head_bwd<16, true>), dim3((unsigned)blocks), dim3(kHeadThreads), 0, s, xb, w, g, gx, dw, db, P);
    else
        hipLaunchKernelGGL((k_head_bwd<16, false>), dim3((unsigned)blocks), dim3(kHeadThreads), 0, s, xb, w, g, gx, dw, db, P);
    return hip_check(hipGetLastError(), "head bwd launch");
}

st_status st_nn_mse(const float *base, const float *y, const float *target, float *g, double *loss,
                    float *pred, int N, int n, double scale, void *stream)
{
    long long P = (long long)N * n * n * n;
    long long blocks = (P + 255) / 256;
    blocks = std::min(blocks, loss_blocks(P));
    hipLaunchKernelGGL(k_mse, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), base,
                       y, target, g, loss, pred, N, n, scale);
    return hip_check(hipGetLastError(), "mse launch");
}

st_status st_nn_adam(float *w, const float *g, float *m, float *v, void *wbf, long long n, float lr,
                     float b1, float b2, float eps, int step, void *stream)
{
    const float c1 = 1.f - powf(b1, (float)step), c2 = 1.f - powf(b2, (float)step);
    hipLaunchKernelGGL(k_adam, gs_grid(n), dim3(256), 0, static_cast<hipStream_t>(stream), w, g, m, v,
                       static_cast<bf16_t *>(wbf), n, lr, b1, b2, eps, c1, c2);
    return hip_check(hipGetLastError(), "adam launch");
}

st_status st_nn_axpby(float *out, float a, const float *x, float b, const float *y, long long n,
                      void *stream)
{
    hipLaunchKernelGGL(k_axpby, gs_grid(n), dim3(256), 0, static_cast<hipStream_t>(stream), out, a, x, b,
                       y, n);
    return hip_check(hipGetLastError(), "axpby launch");
}

st_status st_nn_sumsq(const float *x, float *g, double *loss, long long n, double scale, void *stream)
{
    long long blocks = (n + 255) / 256;
    blocks = std::min(blocks, loss_blocks(n));
    hipLaunchKernelGGL(k_sumsq, dim3((unsigned)blocks), dim3(256), 0, static_cast<hipStream_t>(stream), x,
                       g, loss, n, scale);
    return hip_check(hipGetLastError(), "sumsq launch");
}

st_status st_nn_features(const float *u, void *feat, float *base, int N, int n, int C, void *stream)
{
    hipLaunchKernelGGL(k_features, gs_grid((long long)N * n * n * n), dim3(256), 0,
                       static_cast<hipStream_t>(stream), u, static_cast<bf16_t *>(feat), base, N, n, C);
    return hip_check(hipGetLastError(), "features launch");
}

st_status st_nn_trilinear(const float *in, float *out, int m, int M, void *stream)
{
    hipLaunchKernelGGL(k_trilinear, gs_grid((long long)M * M * M), dim3(256), 0,
                       static_cast<hipStream_t>(stream), in, out, m, M);
    return hip_check(hipGetLastError(), "trilinear launch");
}

st_status st_nn_fourier_faces(float *u, const float *modes, int N, int n, int M, void *stream)
{
    hipLaunchKernelGGL(k_fourier_faces, gs_grid((long long)N * n * n * n), dim3(256), 0,
                       static_cast<hipStream_t>(stream), u, modes, N, n, M);
    return hip_check(hipGetLastError(), "fourier faces launch");
}

}  // extern "C"
