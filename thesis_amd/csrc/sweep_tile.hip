// SMEM_REGISTER family, tile form: one sweep, any row width and alignment,
// FP32 up to radius 16 and FP64 up to radius 10 (3D).
//
// The reference's smem_register kernels keep an xy tile in shared memory and
// each thread's z column in registers (src/stencil_kernel_smem_register.cu,
// src/prefetch_smem.cu:151-258).  Here a workgroup of 8 waves (16 where a
// lane owns two columns) owns a tile of 64 columns x 32*RY rows and marches
// it along z over a chunk of planes:
//   * per plane, the tile and its halo (R rows above and below, R columns
//     rounded up to whole quads left and right) go from registers, where the
//     plane was prefetched, to one of two LDS planes; one barrier per plane.
//     The loads are raw buffer loads: what lies outside the field reads 0,
//     what lies past a row's end reads the next row, and neither is ever
//     used by an interior cell, so no width or alignment is special;
//   * a lane owns CX = 4 consecutive columns in RY adjacent rows (16 lanes
//     along x, 4 along y), or 2 where the state of 4 does not fit its
//     registers: x neighbours come from the words beside its own, y
//     neighbours from the same word of the rows around it, which the RY rows
//     share;
//   * z: a ring of the R previous planes and R running partial sums per cell,
//     as in the row form (sweep_rows.hip): plane m starts P_m with its x, y
//     and z-previous terms in the reference's order and is added to P_{m-1} ..
//     P_{m-R}, the last of which it completes.
// The halo a tile loads is (64+2R)(32*RY+2R) cells for 64*32*RY; the row form
// reads 1 + 2R/rows rows per row, up to 2.3 where registers leave it few
// rows, and the register march 2R + rows (sweep_march.hip).
//
// Bound: VALU and the LDS reads for wide stars (512^3 R = 8: 188 us of VALU,
// 173 of the field's bytes at 6.2 TB/s; measured 286), memory for narrow ones.
// Before (row form, register march or plain kernel, whichever was faster) and
// now, us per sweep: FP32 333x251x207 R = 2 49 -> 24, R = 4 147 -> 34; 512^3
// R = 6 603 -> 233, R = 8 906 -> 288, R = 12 1151 -> 411, 384^3 R = 16 805 ->
// 301, 128^3 R = 4 22.7 -> 12.7, R = 8 20.1 -> 18.0; FP64 384^3 R = 4 263 -> 206,
// R = 8 871 -> 270, 192^3 R = 6 87 -> 34 (whole FP64 quads in LDS, with two-way
// bank conflicts: 384^3 R = 4 428).
#include <algorithm>
#include <utility>

#include "st_device.hpp"
#include "st_internal.hpp"

namespace st {

constexpr int kTileX = 64;
// waves of a workgroup whose lanes own CX columns
__host__ __device__ constexpr int tile_waves(int cx) { return 32 / cx; }

struct TileArgs {
    int nx, ny, nz;
    long long sz;            // nx*ny
    int tx, ty, zchunk;
    const int *eq;           // 1 when both buffers' shells are equal (whole
                             // rows are stored then, shell cells unchanged)
};

// columns of halo on each side: the radius rounded up to whole quads
__host__ __device__ constexpr int tile_ra(int r) { return (r + 3) / 4 * 4; }

// 16-byte words per row, rows and words per thread of a staged plane
template <int R, int RY, typename T> constexpr int tile_row_words() { return (kTileX + 2 * tile_ra(R)) * (int)sizeof(T) / 16; }
template <int R, int RY> constexpr int tile_rows() { return 32 * RY + 2 * R; }
template <int R, int RY, int CX, typename T> constexpr int tile_words()
{
    return (tile_row_words<R, RY, T>() * tile_rows<R, RY>() + 64 * tile_waves(CX) - 1) / (64 * tile_waves(CX));
}
template <int R, int RY, typename T> constexpr int tile_lds() { return 2 * tile_rows<R, RY>() * tile_row_words<R, RY, T>() * 16; }

template <int OP, int R, int RY, int CX, bool LIGHT, typename T>
__global__ __launch_bounds__(64 * tile_waves(CX)) void k_tile(const T *__restrict__ in, T *__restrict__ out, TileArgs a, T kc)
{
    constexpr int RA = tile_ra(R), RW = tile_row_words<R, RY, T>(), ROWS = tile_rows<R, RY>(), NW = tile_words<R, RY, CX, T>();
    constexpr int ES = (int)sizeof(T), NT = 64 * tile_waves(CX);
    constexpr int QN = RA / CX;                           // lanes' words of x halo per side
    constexpr bool HALVES = CX * ES == 32;                // a lane's cells are two 16-byte words
    typedef unsigned int W4 __attribute__((ext_vector_type(4)));
    typedef unsigned int W2 __attribute__((ext_vector_type(2)));
    // many registers of state: keep the LDS reads near their use
    constexpr bool tight = 2 * R * RY * CX * ES > (CX == 4 ? 384 : 192);
    extern __shared__ __align__(16) W4 lds[];
    const int tid = threadIdx.x, lane = tid & 63;
    const int w = __builtin_amdgcn_readfirstlane(tid >> 6);
    const unsigned id = xcd_remap(blockIdx.x, gridDim.x);
    const int tx = (int)(id % (unsigned)a.tx), ty = (int)(id / (unsigned)a.tx % (unsigned)a.ty),
              tz = (int)(id / (unsigned)(a.tx * a.ty));
    const int x0 = tx * kTileX, y0 = ty * 32 * RY;
    const int z0 = tz * a.zchunk, z1 = min(z0 + a.zchunk, a.nz);
    const int k_lo = max(z0, R), k_hi = min(z1, a.nz - R);
    if (k_lo >= k_hi) return;
    const bool eqs = a.eq != nullptr && *a.eq != 0;

    // the lane's cells: CX columns from x, rows y .. y + RY - 1
    constexpr int LX = kTileX / CX;  // lanes along x
    const int qx = lane % LX, x = x0 + CX * qx, ry = (w * (64 / LX) + lane / LX) * RY, y = y0 + ry;
    const bool whole = x >= R && x + CX <= a.nx - R, inrow = x < a.nx;
    const unsigned so = (unsigned)((y * a.nx + x) * ES);
    // LDS place of the lane's word QN words to the left, in the row R above y
    const int lw = ry * RW * 16 + qx * (HALVES ? 16 : CX * ES);

    // staging: word i of the plane is at row i / RW, 16-byte word i % RW
    unsigned go[NW];
    int to[NW];
#pragma unroll
    for (int i = 0; i < NW; ++i) {
        const int q = tid + i * NT, r = q / RW, c = q - r * RW;
        to[i] = !HALVES ? q : r * RW + (c & 1) * (RW / 2) + (c >> 1);
        // rows above and columns left of the field: negative offsets, out of
        // the buffer's range (words past the plane's last row: likewise)
        go[i] = r < ROWS ? (unsigned)(((y0 - R + r) * a.nx + x0 - RA) * ES + c * 16) : 0x80000000u;
    }
    W4 pf[NW];
    const long long plane = a.sz * ES;
    auto plane_of = [&](int k) {
        const char *p = reinterpret_cast<const char *>(in) + k * plane;
        return __builtin_amdgcn_make_buffer_rsrc(const_cast<char *>(p), 0, (int)min((a.nz - k) * plane, 0x7fffffffLL), 0x00020000);
    };
    auto load_plane = [&](int k) {
        const __amdgpu_buffer_rsrc_t rs = plane_of(k);
#pragma unroll
        for (int i = 0; i < NW; ++i) pf[i] = __builtin_amdgcn_raw_buffer_load_b128(rs, (int)go[i], 0, 0);
    };
    // the lane's own cells of plane k
    auto load_own = [&](int k, T (&v)[RY][CX]) {
        const __amdgpu_buffer_rsrc_t rs = plane_of(k);
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            const int o = (int)(so + (unsigned)(r * a.nx * ES));
            if constexpr (CX * ES == 8) {
                const W2 q = __builtin_amdgcn_raw_buffer_load_b64(rs, o, 0, 0);
                v[r][0] = __uint_as_float(q[0]), v[r][1] = __uint_as_float(q[1]);
            } else {
#pragma unroll
                for (int h = 0; h < CX * ES / 16; ++h) {
                    typedef T VW __attribute__((ext_vector_type(16 / ES)));
                    const VW q = __builtin_bit_cast(VW, __builtin_amdgcn_raw_buffer_load_b128(rs, o + 16 * h, 0, 0));
#pragma unroll
                    for (int e = 0; e < 16 / ES; ++e) v[r][h * (16 / ES) + e] = q[e];
                }
            }
        }
    };

    T ring[R][RY][CX], part[R][RY][CX];
#pragma unroll
    for (int i = 0; i < R; ++i)
#pragma unroll
        for (int r = 0; r < RY; ++r)
#pragma unroll
            for (int c = 0; c < CX; ++c) ring[i][r][c] = part[i][r][c] = (T)0;

    // An FP64 quad is kept as two 16-byte halves half a row apart, so that the
    // 16 lanes of a read are contiguous (whole 32-byte quads: two-way bank
    // conflicts).
    constexpr int QB = HALVES ? 16 : CX * ES;  // bytes from one lane's word to the next
    auto cells = [&](const char *p, T (&v)[CX]) {
        if constexpr (HALVES) {
            typedef double D2 __attribute__((ext_vector_type(2)));
            const D2 q0 = *reinterpret_cast<const D2 *>(p), q1 = *reinterpret_cast<const D2 *>(p + RW * 8);
            v[0] = q0[0]; v[1] = q0[1]; v[2] = q1[0]; v[3] = q1[1];
        } else {
            typedef T VX __attribute__((ext_vector_type(CX)));
            const VX q = *reinterpret_cast<const VX *>(p);
#pragma unroll
            for (int c = 0; c < CX; ++c) v[c] = q[c];
        }
    };

    // plane k from the ring slot and the sums rp, which it leaves complete
    auto emit = [&](auto phase, int k) {
        constexpr int rp = decltype(phase)::value;
        char *const po = reinterpret_cast<char *>(out) + k * plane;
#pragma unroll
        for (int r = 0; r < RY; ++r) {
            T res[CX];
            finish_sums<OP>(part[rp][r], ring[rp][r], kc, res);
            if (!interior1(y + r, a.ny, R) || !inrow) continue;
            T *const p = reinterpret_cast<T *>(po + (so + (unsigned)(r * a.nx * ES)));
            if (whole || (eqs && x + CX <= a.nx)) {
                typedef T VU __attribute__((ext_vector_type(CX), aligned(sizeof(T))));
                VU v;
#pragma unroll
                for (int c = 0; c < CX; ++c) {
                    const T mine = res[c], held = ring[rp][r][c];
                    v[c] = whole || interior1(x + c, a.nx, R) ? mine : held;
                }
                *reinterpret_cast<VU *>(p) = v;
            } else {
#pragma unroll
                for (int c = 0; c < CX; ++c)
                    if (x + c >= R && x + c < a.nx - R) p[c] = res[c];
            }
        }
    };

    // LIGHT: of the R planes before and after the chunk, which are z
    // neighbours only, a lane loads its own cells and nothing is staged
    const int m_lo = k_lo - R, m_hi = k_hi + R;
    T own[RY][CX];
    auto load = [&](int k) {
        if (!LIGHT || (k >= k_lo && k < k_hi)) load_plane(k);
        else load_own(k, own);
    };
    load(m_lo);
    // planes in phases of R, unrolled, so that the ring and the partial sums
    // rotate through their slots with no register moves
    for (int m0 = m_lo; m0 < m_hi; m0 += R) {
        each_phase(std::make_integer_sequence<int, R>{}, [&](auto phase) {
            constexpr int rp = decltype(phase)::value;
            const int m = m0 + rp;
            if (m >= m_hi) return false;
            __builtin_amdgcn_sched_barrier(0);
            T s[RY][CX], cur[RY][CX];
            if (LIGHT && (m < k_lo || m >= k_hi)) {
#pragma unroll
                for (int r = 0; r < RY; ++r)
#pragma unroll
                    for (int c = 0; c < CX; ++c) cur[r][c] = own[r][c], s[r][c] = (T)0;
                if (m + 1 < m_hi) load(m + 1);
            } else {
                W4 *const buf = lds + ((m - m_lo) & 1) * (ROWS * RW);
#pragma unroll
                for (int i = 0; i < NW; ++i) {
                    if ((i + 1) * NT <= ROWS * RW || tid + i * NT < ROWS * RW) buf[to[i]] = pf[i];
                }
                if (m + 1 < m_hi) load(m + 1);
                __syncthreads();
                const char *const at = reinterpret_cast<const char *>(buf) + lw;
                // x terms: own word and the QN words on each side
#pragma unroll
                for (int r = 0; r < RY; ++r) {
                    T v[CX * (2 * QN + 1)];
#pragma unroll
                    for (int q = 0; q < 2 * QN + 1; ++q) {
                        T t[CX];
                        cells(at + (R + r) * RW * 16 + q * QB, t);
#pragma unroll
                        for (int c = 0; c < CX; ++c) v[CX * q + c] = t[c];
                    }
#pragma unroll
                    for (int c = 0; c < CX; ++c) {
                        cur[r][c] = v[RA + c];
                        T u = v[RA + c - R];
#pragma unroll
                        for (int d = R - 1; d >= 1; --d) u += v[RA + c - d];
#pragma unroll
                        for (int d = 1; d <= R; ++d) u += v[RA + c + d];
                        s[r][c] = u;
                    }
                    if constexpr (tight) __builtin_amdgcn_sched_barrier(0);
                }
                // y terms: rows y-R .. y+RY-1+R in order, each for the rows it neighbours
#pragma unroll
                for (int t = -R; t < RY + R; ++t) {
                    T v[CX];
                    if (t >= 0 && t < RY) {
#pragma unroll
                        for (int c = 0; c < CX; ++c) v[c] = cur[t][c];
                    } else {
                        cells(at + (R + t) * RW * 16 + QN * QB, v);
                    }
#pragma unroll
                    for (int r = 0; r < RY; ++r)
                        if (t != r && t - r >= -R && t - r <= R)
#pragma unroll
                            for (int c = 0; c < CX; ++c) s[r][c] += v[c];
                    if constexpr (tight)
                        if ((t + R) % 3 == 2) __builtin_amdgcn_sched_barrier(0);
                }
                // z-previous terms: logical ring[i] = plane m-R+i, in slot (rp+i) % R
#pragma unroll
                for (int i = 0; i < R; ++i)
#pragma unroll
                    for (int r = 0; r < RY; ++r)
#pragma unroll
                        for (int c = 0; c < CX; ++c) s[r][c] += ring[(rp + i) % R][r][c];
            }
            // plane m is the next z-next term of P_{m-R} .. P_{m-1}
#pragma unroll
            for (int i = 0; i < R; ++i)
#pragma unroll
                for (int r = 0; r < RY; ++r)
#pragma unroll
                    for (int c = 0; c < CX; ++c) part[(rp + i) % R][r][c] += cur[r][c];
            // P_{m-R} (slot rp) is complete
            if (m - R >= k_lo) emit(phase, m - R);
#pragma unroll
            for (int r = 0; r < RY; ++r)
#pragma unroll
                for (int c = 0; c < CX; ++c) {
                    ring[rp][r][c] = cur[r][c];
                    part[rp][r][c] = s[r][c];
                }
            return true;
        });
    }
}

// ---------------------------------------------------------------- host side

struct TileKernel {
    const void *fn = nullptr;
    int lds = 0, words = 0;  // LDS bytes; 32-bit words of ring and partial sums per lane
};

template <int R, int RY, int CX, bool LIGHT, typename T>
static TileKernel tile_kernel(int op)
{
    constexpr int words = 2 * R * RY * CX * (int)sizeof(T) / 4;
    constexpr bool f64 = sizeof(T) == 8;
    // built where the kernel leaves no or few spills: quads while they do,
    // then pairs (FP64 R = 6 as pairs: 384^3 267 / 254, 128^3 18.5 / 17.5; R = 5
    // as quads: 128^3 17 / 23)
    constexpr bool quads = words <= (RY == 2 ? 112 : 96) && R <= (f64 ? 5 : 12);
    constexpr bool pairs = R > (f64 ? 5 : 12) && R <= (f64 ? 10 : 16);
    if constexpr (!(CX == 4 ? quads : pairs)) return {};
    else
        return {op == OP_THESIS ? reinterpret_cast<const void *>(&k_tile<OP_THESIS, R, RY, CX, LIGHT, T>)
                                : reinterpret_cast<const void *>(&k_tile<OP_JACOBI, R, RY, CX, LIGHT, T>),
                tile_lds<R, RY, T>(), words};
}

template <int RY, int CX, bool LIGHT, typename T>
static TileKernel tile_kernel_r(int op, int r)
{
    switch (r) {
#define TK(R) case R: return tile_kernel<R, RY, CX, LIGHT, T>(op);
    TK(1) TK(2) TK(3) TK(4) TK(5) TK(6) TK(7) TK(8)
    TK(9) TK(10) TK(11) TK(12) TK(13) TK(14) TK(15) TK(16)
#undef TK
    default: return {};
    }
}

template <typename T>
static TileKernel tile_kernel_t(const Cfg &c, int ry, int cx, bool light)
{
    if (cx == 2) return ry == 2 ? TileKernel{} : tile_kernel_r<1, 2, true, T>(c.op, c.r);
    if (light) return ry == 2 ? tile_kernel_r<2, 4, true, T>(c.op, c.r) : tile_kernel_r<1, 4, true, T>(c.op, c.r);
    return ry == 2 ? tile_kernel_r<2, 4, false, T>(c.op, c.r) : tile_kernel_r<1, 4, false, T>(c.op, c.r);
}

static TileKernel tile_kernel_for(const Cfg &c, int ry, int cx, bool light)
{
    return c.dtype == ST_F64 ? tile_kernel_t<double>(c, ry, cx, light) : tile_kernel_t<float>(c, ry, cx, light);
}

static int tile_cx(const Cfg &c) { return c.r > (c.dtype == ST_F64 ? 5 : 12) ? 2 : 4; }

// Planes' worth of work of a chunk of ch planes.  A plane of the halo that a
// LIGHT kernel does not stage costs it about 0.3 of a staged one, but the
// planes of the chunk 1.15 (128^3 FP32 R = 8 27 -> 18 us a sweep, 333x251x207
// R = 12 104 -> 84; the other way 512^3 R = 8 289 -> 453, 384^3 FP64 R = 4
// 207 -> 246).
static double tile_work(const Cfg &c, int ch, bool light)
{
    return light ? 1.15 * (ch + 0.3 * 2 * c.r) : ch + 2.0 * c.r;
}

static bool tile_light(const Cfg &c, int ch) { return tile_cx(c) == 2 || tile_work(c, ch, true) < tile_work(c, ch, false); }

// The library's choice among the SMEM_REGISTER forms (us per sweep, the
// other forms' best / this one):
//   * below 2^20 cells the plain kernel is AUTO's choice and the other forms
//     stay as they were (just above, 104^3 FP32 R = 1 8.5 / 8.1, R = 5 22 / 14,
//     R = 8 18.5 / 15.9, R = 12 25 / 22, FP64 R = 8 29 / 21); the few tiles of a
//     small grid march 2R planes each for a short chunk, so FP64 radii 9 and
//     10 wait for 2^21 cells (104^3 26 / 33, 128^3 44 / 35) and radius 16 for
//     2^22 (128^3 26 / 30, 192^3 82 / 51);
//   * rows of 256, 384 or 512 columns stay with the consecutive row layout,
//     which reads every row once per 8 to 16 rows and is level or ahead
//     (384^3 FP32 R = 4 92 / 100, 512^3 R = 2 203 / 218, 256^3 R = 4 29 / 29;
//     FP64 256^3 R = 4 50 / 53);
//   * rows over 512 columns of small 16-byte stars stay with the quad row
//     layout (640x320x200 FP32 R = 1 67 / 70, FP64 R = 2 121 / 140);
//   * else the tile is ahead: 320^3 FP32 R = 2 59 / 54, R = 4 75 / 61; widths
//     that are no multiple of 4, which only the register march took, 1.25x
//     (R = 1) to 4.3x (R = 4).
//   * a tile computes shell cells like any other and marches through 2R planes
//     of halo: FP32 radii 6 to 8 stay with the register march where little of
//     the grid is interior (1000x33x33 R = 8 11 / 16.5, R = 6 10.9 / 14), up to
//     a larger size where that is few planes beside the halo (40x4000x20
//     R = 8 10 / 12.6, 90x548x34 15 / 17.5, 1000x1000x20 R = 6 40 / 25.5), and radius 1 where 15/16 of
//     the tiles lie outside (9x9x100000 93 / 118).
static long long ceil_to(long long n, long long unit) { return (n + unit - 1) / unit * unit; }

// Interior cells, rows rounded up to the 64 lanes of a wave; cells of the
// tiles, a plane of z halo as 0.3.
static long long interior_rounded(const Cfg &c)
{
    return ceil_to(c.nx - 2 * c.r, 64) * (c.ny - 2 * c.r) * (c.nz - 2 * c.r);
}
static long long tiles_rounded(const Cfg &c) { return ceil_to(c.nx, kTileX) * ceil_to(c.ny, 32) * (c.nz - 2 * c.r + 6 * c.r / 10); }

bool tile_eligible(const Cfg &c)
{
    if (c.dims != 3 || (c.dtype != ST_F32 && c.dtype != ST_F64)) return false;
    const long long cells = (long long)c.nx * c.ny * c.nz, es = c.dtype == ST_F64 ? 8 : 4;
    const long long least = c.r == 16 ? 1LL << 22 : es == 8 && c.r > 8 ? 1LL << 21 : (1LL << 20) + 1;
    if (cells < least) return false;
    // 32-bit byte offsets within a plane and its halo
    if (((long long)c.nx * (c.ny + 2 * c.r + 64) + 128) * es >= (1LL << 30)) return false;
    if (c.r <= 4 && c.nx % 4 == 0 && (rows_consecutive(c) || (c.nx > 512 && c.r <= (es == 8 ? 2 : 1))))
        return false;
    if (c.r == 1 && 16 * cells < tiles_rounded(c)) return false;
    if (es == 4 && c.r >= 6 && c.r <= 8 && interior_rounded(c) < (c.nz < 5 * c.r ? 3LL << 20 : 1LL << 19)) return false;
    return tile_kernel_for(c, 1, tile_cx(c), true).fn != nullptr;
}

// AUTO's rule between the tile form and the plain kernel, which computes the
// interior alone (FP32 from radius 9, FP64 radius 3 and from 5; us per sweep,
// plain / tile): it is ahead while the interior is small (FP32 1000x33x33 R = 10
// 7 / 19, 104^3 R = 12 18 / 20, 128^3 R = 12 31 / 21; FP64 1000x33x33 R = 8 9.7 /
// 19.6, 4000x20x20 R = 6 12.6 / 14.3, 104^3 R = 8 29 / 21), and where the slower
// kernels of wide stars spend themselves on shell cells (33x33x2000 FP64 R = 10
// 48 / 93, FP32 R = 12 30 / 37; 2000x500x24 FP64 R = 10 148 / 121).  Between
// 3 << 17 and 7 << 17 interior cells FP32 goes either way (235x30x175 R = 10 20 /
// 15, 457x34x95 12 / 19).
bool tile_over_plain(const Cfg &c)
{
    const long long in = interior_rounded(c), all = tiles_rounded(c);
    if (c.dtype == ST_F32) return c.r < 9 || (in >= 7LL << 17 && 25 * in >= 4 * all);
    return c.r < 5 || (c.r < 9 ? in >= 5LL << 17 : 20 * in >= 7 * all);
}

st_status resolve_tile(Cfg &c)
{
    int dev = 0, cus = 256;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus < 1)
        cus = 256;
    // rows per lane and z chunk of the least busiest-CU work: rounds of
    // workgroups x planes marched x rows per lane (a plane costs a fixed part
    // beside its rows, hence the + 0.5)
    const int cx = tile_cx(c);
    double best = -1;
    for (int ry = 1; ry <= 2; ++ry) {
        const TileKernel t = tile_kernel_for(c, ry, cx, true);
        if (!t.fn) continue;
        const int per_cu = t.words <= 40 && t.lds <= kMaxLds / 2 ? 2 : 1;
        const long long xy = (long long)((c.nx + kTileX - 1) / kTileX) * ((c.ny + 32 * ry - 1) / (32 * ry));
        // For k rounds the most chunks that fit them are the best, and k
        // rounds take at least the planes of all chunks and their halo: the
        // search ends after some ten of them (every chunk count took 0.3 ms
        // of host time for 9 x 9 x 100000).
        const long long room = (long long)cus * per_cu;
        const int most = std::max(1, (c.nz - 1) / 2);  // chunks of 3 planes and more
        const double rows = (ry + 0.6) * (per_cu == 2 ? 1.6 : 1.0);
        for (long long k = (xy + room - 1) / room;; ++k) {
            const double least = ((double)xy * c.nz / room + 0.69 * c.r * k) * rows;
            if (best >= 0 && least > best * (1 + 1e-9)) break;
            const int nch = (int)std::min<long long>(most, room * k / xy), ch = (c.nz + nch - 1) / nch;
            const long long n = xy * ((c.nz + ch - 1) / ch);
            const double cost = (double)((n + room - 1) / room) * tile_work(c, ch, tile_light(c, ch)) * rows;
            if (best < 0 || cost < best) {
                best = cost;
                c.cy = ry;
                c.zchunk = ch;
                c.lds = t.lds;
                c.gx = (int)n;
            }
            if (nch == most) break;
        }
    }
    if (best < 0) return fail(ST_EUNSUPPORTED, "tile form: no kernel for radius %d", c.r);
    c.kind = 8;
    c.cx = cx;
    c.bx = kTileX;
    c.by = 32 * c.cy;
    c.bz = c.zchunk;
    c.gy = c.gz = 1;
    c.tsteps = 1;
    return ST_OK;
}

st_status launch_tile(const Cfg &c, const void *in, void *out, hipStream_t s)
{
    const TileKernel t = tile_kernel_for(c, c.cy, c.cx, tile_light(c, c.zchunk));
    if (!t.fn) return fail(ST_EUNSUPPORTED, "tile form: no kernel for radius %d", c.r);
    TileArgs a;
    a.nx = c.nx; a.ny = c.ny; a.nz = c.nz;
    a.sz = (long long)c.nx * c.ny;
    a.tx = (c.nx + kTileX - 1) / kTileX;
    a.ty = (c.ny + 32 * c.cy - 1) / (32 * c.cy);
    a.zchunk = c.zchunk;
    a.eq = c.shell_eq;
    double kd = c.op == OP_THESIS ? (double)(2 * c.dims * c.r) : c.weight;
    float kf = (float)kd;
    void *args[] = {&in, &out, &a, c.dtype == ST_F64 ? static_cast<void *>(&kd) : static_cast<void *>(&kf)};
    hipError_t e = hipFuncSetAttribute(t.fn, hipFuncAttributeMaxDynamicSharedMemorySize, t.lds);
    if (e != hipSuccess) return hip_check(e, "hipFuncSetAttribute(tile LDS)");
    return hip_check(hipLaunchKernel(t.fn, dim3(c.gx), dim3(64 * tile_waves(c.cx)), args, t.lds, s), "tile launch");
}

}  // namespace st
