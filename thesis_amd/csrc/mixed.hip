// 16-bit field storage (BF16 or FP16) with FP32 arithmetic and FP32 defect
// correction, for the JACOBI operator.  No reference counterpart; the
// arithmetic is restated bit for bit in oracle/stencil_oracle.c
// (or_mixed_run) and checked against it.
//
// The field is u = x + e: x an FP32 base field that carries the Dirichlet
// shell, e a 16-bit correction and d a 16-bit defect d = G(x) - x.  Because
// the sweep G is affine, G(x + e) = G(x) + G0(e), so one sweep of u is the
// correction sweep  e' = d + G0(e)  which moves 2 + 2 + 2 bytes per cell.
// Every `restart` sweeps the correction is folded into x in FP32 and the
// defect is recomputed in FP32 from the new x (the FP32-residual defect
// correction); 16-bit rounding then only ever applies to increments.
#include <algorithm>

#include "st_device.hpp"
#include "st_half.hpp"
#include "st_internal.hpp"

namespace st {

struct MixArgs {
    Geom g;
    int dims;
    float w;
};

// Decompose interior index t into (i, j, k).
__device__ __forceinline__ long long interior_idx(const MixArgs &a, long long t)
{
    const Geom &g = a.g;
    const int R = g.r;
    const int wx = g.nx - 2 * R, wy = g.ny - 2 * R;
    const long long wxy = (long long)wx * wy;
    const int kk = (int)(t / wxy);
    const long long rem = t - (long long)kk * wxy;
    const int j = R + (int)(rem / wx);
    const int i = R + (int)(rem - (long long)(j - R) * wx);
    const int k = a.dims == 3 ? R + kk : 0;
    return i + j * g.sy + k * g.sz;
}

__device__ __forceinline__ long long interior_count(const MixArgs &a)
{
    const Geom &g = a.g;
    const int R = g.r;
    return (long long)(g.nx - 2 * R) * (g.ny - 2 * R) * (a.dims == 3 ? g.nz - 2 * R : 1);
}

// d = round16(G(x) - x) on the interior; G is the FP32 JACOBI cell.
template <bool F16>
__global__ __launch_bounds__(256) void k_mx_defect(const float *__restrict__ x,
                                                   uint16_t *__restrict__ d, MixArgs a)
{
    const Geom &g = a.g;
    const int R = g.r;
    const long long n = interior_count(a), stride = (long long)gridDim.x * blockDim.x;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n; t += stride) {
        const long long idx = interior_idx(a, t);
        float u = 0.0f;
        for (int q = R; q >= 1; --q) u += x[idx - q];
        for (int q = 1; q <= R; ++q) u += x[idx + q];
        for (int q = R; q >= 1; --q) u += x[idx - q * g.sy];
        for (int q = 1; q <= R; ++q) u += x[idx + q * g.sy];
        if (a.dims == 3) {
            for (int q = R; q >= 1; --q) u += x[idx - q * g.sz];
            for (int q = 1; q <= R; ++q) u += x[idx + q * g.sz];
        }
        const float tcell = u * a.w;
        d[idx] = rnd16<F16>(tcell - x[idx]);
    }
}

// e' = round16(widen(d) + w * sum widen(e neighbours)).
template <bool F16>
__global__ __launch_bounds__(256) void k_mx_sweep(const uint16_t *__restrict__ e,
                                                  const uint16_t *__restrict__ d,
                                                  uint16_t *__restrict__ eo, MixArgs a)
{
    const Geom &g = a.g;
    const int R = g.r;
    const long long n = interior_count(a), stride = (long long)gridDim.x * blockDim.x;
    for (long long t = blockIdx.x * (long long)blockDim.x + threadIdx.x; t < n; t += stride) {
        const long long idx = interior_idx(a, t);
        float s = 0.0f;
        for (int q = R; q >= 1; --q) s += wid16<F16>(e[idx - q]);
        for (int q = 1; q <= R; ++q) s += wid16<F16>(e[idx + q]);
        for (int q = R; q >= 1; --q) s += wid16<F16>(e[idx - q * g.sy]);
        for (int q = 1; q <= R; ++q) s += wid16<F16>(e[idx + q * g.sy]);
        if (a.dims == 3) {
            for (int q = R; q >= 1; --q) s += wid16<F16>(e[idx - q * g.sz]);
            for (int q = 1; q <= R; ++q) s += wid16<F16>(e[idx + q * g.sz]);
        }
        const float sw = s * a.w;
        eo[idx] = rnd16<F16>(wid16<F16>(d[idx]) + sw);
    }
}

// The same with 64 columns x 4 rows of threads per workgroup, so that a cell is
// found without the divisions of a flat index, and the sums of radius 1 and 2
// unrolled (RS; 0: any radius).  Bound: the 2-byte loads of a cell's 4R or 6R
// neighbours, one instruction each.  f(index) for every interior cell.
template <typename F>
__device__ __forceinline__ void each_interior(const MixArgs &a, F f)
{
    const Geom &g = a.g;
    const int R = g.r, k0 = a.dims == 3 ? R : 0, k1 = a.dims == 3 ? g.nz - R : 1;
    for (int k = k0 + (int)blockIdx.z; k < k1; k += (int)gridDim.z)
        for (long long j = R + (long long)blockIdx.y * 4 + (threadIdx.x >> 6); j < g.ny - R; j += 4LL * gridDim.y)
            for (long long i = R + (long long)blockIdx.x * 64 + (threadIdx.x & 63); i < g.nx - R; i += 64LL * gridDim.x)
                f(i + j * g.sy + k * g.sz);
}

// Sum of the neighbours of p[0] in the reference's order, v(neighbour) each.
template <int RS, typename T, typename V>
__device__ __forceinline__ float neighbour_sum(const T *p, const MixArgs &a, V v)
{
    const int R = RS ? RS : a.g.r;
    float s = 0.0f;
    auto axis = [&](long long st) {
#pragma unroll
        for (int q = R; q >= 1; --q) s += v(p[-q * st]);
#pragma unroll
        for (int q = 1; q <= R; ++q) s += v(p[q * st]);
    };
    axis(1);
    axis(a.g.sy);
    if (a.dims == 3) axis(a.g.sz);
    return s;
}

template <bool F16, int RS>
__global__ __launch_bounds__(256) void k_mx_defect_rows(const float *__restrict__ x, uint16_t *__restrict__ d, MixArgs a)
{
    each_interior(a, [&](long long idx) {
        const float tcell = neighbour_sum<RS>(x + idx, a, [](float q) { return q; }) * a.w;
        d[idx] = rnd16<F16>(tcell - x[idx]);
    });
}

template <bool F16, int RS>
__global__ __launch_bounds__(256) void k_mx_sweep_rows(const uint16_t *__restrict__ e, const uint16_t *__restrict__ d,
                                                       uint16_t *__restrict__ eo, MixArgs a)
{
    each_interior(a, [&](long long idx) {
        const float sw = neighbour_sum<RS>(e + idx, a, [](uint16_t q) { return wid16<F16>(q); }) * a.w;
        eo[idx] = rnd16<F16>(wid16<F16>(d[idx]) + sw);
    });
}

// Whether the kernels with 64 x 4 threads per workgroup take the grid.  20
// sweeps with their passes, us, flat / 64 x 4:
// * a grid that is all in flight at once (2^18 lanes) has only its chain of
//   loads to wait for, and lanes without a cell cost nothing: 41^3 R = 5 161 /
//   129, R = 8 214 / 124, 99 x 270 R = 7 162 / 131, 59 x 202 R = 14 219 / 157.
//   Not for R = 3, nor for flat rows that are half empty with few loads to
//   save (41 x 3001 R = 5 123 / 137, R = 9 160 / 129);
// * beyond it the time is the loads' and an empty lane costs its share.  R = 1:
//   123 x 284 x 71 399 / 298, 67 columns (51 % filled) 298 / 330.  R = 2: 542 /
//   454, 70^3 (52 %) 150 / 180.  R = 3 to 7, whose sums are not unrolled in
//   eights: flat is ahead (333 x 251 x 207 R = 6 6481 / 8726, 123 x 284 x 71
//   R = 7 973 / 1192).  From 8: 256^3 R = 8 7805 / 3657, R = 12 10137 / 5959,
//   2048^2 R = 16 2579 / 1430, 114 x 99 x 104 R = 10 (73 %) 582 / 452; 97 x 50 x
//   351 R = 14 (54 %) 512 / 759, 100 x 5000 R = 15 (55 %) 331 / 381.  Whole
//   eights in 2D stay ahead down to a third: 88 x 2912 R = 8 197 / 137.  Odd
//   radii gain less: 123 x 284 x 71 R = 15 (73 %) 934 / 1099, 700^2 R = 11 259 /
//   304, 1031 x 1021 R = 11 506 / 370.
static bool mx_rows(const MixArgs &a, long long w, long long wy, long long wz)
{
    const int R = a.g.r;
    const long long lanes = (w + 63) / 64 * 64;
    const long long all = lanes * wy * wz;
    if (all <= 1 << 18 && R != 3 && (a.dims == 3 || R >= 8 || 2 * w >= lanes)) return true;
    if ((R > 2 && R < 8) || (R > 8 && R % 2 && a.dims == 2 && all < 1 << 19)) return false;
    return 100 * w >= (R == 1 ? 60 : R == 2 ? 80 : a.dims == 2 && R % 8 == 0 ? 35 : R % 2 ? 75 : 67) * lanes;
}

// The defect of x, or where x is null the sweep e -> eo.
template <bool F16>
static void mx_cells(const MixArgs &a, const float *x, const uint16_t *e, uint16_t *d, uint16_t *eo, hipStream_t s)
{
    auto blocks = [](long long n, long long per, long long most) { return (unsigned)std::max(1LL, std::min((n + per - 1) / per, most)); };
    const int R = a.g.r;
    const long long wx = a.g.nx - 2 * R, wy = a.g.ny - 2 * R, wz = a.dims == 3 ? a.g.nz - 2 * R : 1;
    if (!mx_rows(a, wx, wy, wz)) {
        const dim3 grid(blocks(wx * wy * wz, 256, 32768));
        if (x) hipLaunchKernelGGL(k_mx_defect<F16>, grid, dim3(256), 0, s, x, d, a);
        else hipLaunchKernelGGL(k_mx_sweep<F16>, grid, dim3(256), 0, s, e, d, eo, a);
        return;
    }
    const unsigned bx = blocks(wx, 64, 1024), by = blocks(wy, 4, 8192);
    const dim3 grid(bx, by, blocks(wz, 1, std::min(65535LL, (1LL << 23) / ((long long)bx * by))));   // 2^31 lanes in all
    auto launch = [&](auto rs) {
        constexpr int RS = decltype(rs)::value;
        if (x) hipLaunchKernelGGL((k_mx_defect_rows<F16, RS>), grid, dim3(256), 0, s, x, d, a);
        else hipLaunchKernelGGL((k_mx_sweep_rows<F16, RS>), grid, dim3(256), 0, s, e, d, eo, a);
    };
    if (R == 1) launch(std::integral_constant<int, 1>{});
    else if (R == 2) launch(std::integral_constant<int, 2>{});
    else launch(std::integral_constant<int, 0>{});
}

// u's shell <- x's (3D, fewer than 2^31 shell cells; the whole field took
// 103 us of 384^3)
__global__ __launch_bounds__(256) void k_mx_shell(const float *__restrict__ x, float *__restrict__ u, int nx, int ny, int nz,
                                                  int r)
{
    const unsigned n = (unsigned)shell_cells(nx, ny, nz, r), n1 = (unsigned)shell_full_cells(nx, ny, nz, r);
    for (unsigned i = blockIdx.x * 256 + threadIdx.x; i < n; i += gridDim.x * 256) {
        const long long p = shell_cell(i, n1, nx, ny, nz, r);
        u[p] = x[p];
    }
}

// v <- 0 over n 16-bit values (a kernel rather than a memset, so that the
// sequence can be captured in a graph and replayed)
__global__ void k_fill16(uint16_t *__restrict__ v, long long n)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += stride) v[i] = 0;
}

// x += widen(e); e <- 0 (whole grid, elementwise).
template <bool F16>
__global__ __launch_bounds__(256) void k_mx_fold(float *__restrict__ x, uint16_t *__restrict__ e,
                                                 long long n)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += stride) {
        x[i] = x[i] + wid16<F16>(e[i]);
        e[i] = 0;
    }
}

// u = x + widen(e).
template <bool F16>
__global__ __launch_bounds__(256) void k_mx_final(const float *__restrict__ x,
                                                  const uint16_t *__restrict__ e,
                                                  float *__restrict__ u, long long n)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += stride)
        u[i] = x[i] + wid16<F16>(e[i]);
}

// u += widen(e) (the final fold when the current field is already in u).
template <bool F16>
__global__ __launch_bounds__(256) void k_mx_final_inplace(float *__restrict__ u, const uint16_t *__restrict__ e,
                                                          long long n)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += stride)
        u[i] = u[i] + wid16<F16>(e[i]);
}

template <bool F16>
static st_status mixed_impl(const Cfg &c, float *x, uint16_t *e1, uint16_t *e2, uint16_t *d,
                            float *u, hipStream_t s)
{
    MixArgs a;
    a.g.nx = c.nx; a.g.ny = c.ny; a.g.nz = c.nz; a.g.r = c.r;
    a.g.sy = c.nx; a.g.sz = (long long)c.nx * c.ny;
    a.dims = c.dims;
    a.w = (float)c.weight;
    const long long n = (long long)c.nx * c.ny * c.nz;
    auto blocks = [](long long cnt) {
        long long b = (cnt + 255) / 256;
        if (b > 32768) b = 32768;
        return dim3((unsigned)(b < 1 ? 1 : b));
    };
    hipLaunchKernelGGL(k_fill16, blocks(n), dim3(256), 0, s, e1, n);
    hipLaunchKernelGGL(k_fill16, blocks(n), dim3(256), 0, s, e2, n);
    hipLaunchKernelGGL(k_fill16, blocks(n), dim3(256), 0, s, d, n);
    // 3D grids the row-streaming kernels take (FP32 arithmetic on 16-bit
    // loads, same operation order); the rest use the per-cell kernels
    const bool rows = c.dims == 3 && rows_mixed_eligible(c);
    st_status st = ST_OK;
    if (rows && c.iters > 0 && rows_mixed_fused_ok(c)) {
        // The same arithmetic with two passes fewer per restart: the defect
        // sweep also writes the first correction sweep of its cycle
        // (round16(widen(d) + w*0), which is what a sweep from a zero
        // correction computes), and the fold x += e of a restart is formed
        // on the fly by the next defect sweep, which writes x' to the other
        // FP32 buffer (u, given x's shell first) instead of updating x in
        // place.  Sweep it (1-based) is the first of its cycle when
        // (it - 1) % restart == 0.
        const long long ns = shell_cells(c.nx, c.ny, c.nz, c.r);
        if (ns >= (1LL << 31)) {
            if (hipMemcpyAsync(u, x, n * sizeof(float), hipMemcpyDeviceToDevice, s) != hipSuccess)
                return hip_check(hipGetLastError(), "mixed: copy of x");
        } else if (c.iters > c.restart) {
            hipLaunchKernelGGL(k_mx_shell, blocks(ns), dim3(256), 0, s, x, u, c.nx, c.ny, c.nz, c.r);
        }
        float *xa = x, *xb = u;
        uint16_t *ea = e1, *eb = e2;
        st = launch_rows_defect(c, F16, xa, nullptr, nullptr, d, ea, s);
        for (int it = 2; it <= c.iters && st == ST_OK; ++it) {
            if ((it - 1) % c.restart == 0) {
                st = launch_rows_defect(c, F16, xa, ea, xb, d, eb, s);
                float *t = xa; xa = xb; xb = t;
            } else {
                st = launch_rows_mixed(c, 0, F16, ea, eb, d, s);
            }
            uint16_t *t = ea; ea = eb; eb = t;
        }
        if (st != ST_OK) return st;
        if (xa == u) hipLaunchKernelGGL(k_mx_final_inplace<F16>, blocks(n), dim3(256), 0, s, u, ea, n);
        else hipLaunchKernelGGL(k_mx_final<F16>, blocks(n), dim3(256), 0, s, xa, ea, u, n);
        return hip_check(hipGetLastError(), "mixed launch");
    }
    auto defect = [&]() {
        if (rows) st = launch_rows_mixed(c, 1, F16, x, d, nullptr, s);
        else mx_cells<F16>(a, x, nullptr, d, nullptr, s);
    };
    auto sweep = [&](const uint16_t *ein, uint16_t *eout) {
        if (rows) st = launch_rows_mixed(c, 0, F16, ein, eout, d, s);
        else mx_cells<F16>(a, nullptr, ein, d, eout, s);
    };
    defect();
    uint16_t *ea = e1, *eb = e2;
    for (int it = 1; it <= c.iters && st == ST_OK; ++it) {
        sweep(ea, eb);
        uint16_t *t = ea; ea = eb; eb = t;
        if (it % c.restart == 0 && it < c.iters) {
            // eb's interior is overwritten by the next sweep and its shell is
            // still 0, so only the live correction needs clearing.
            hipLaunchKernelGGL(k_mx_fold<F16>, blocks(n), dim3(256), 0, s, x, ea, n);
            defect();
        }
    }
    if (st != ST_OK) return st;
    hipLaunchKernelGGL(k_mx_final<F16>, blocks(n), dim3(256), 0, s, x, ea, u, n);
    return hip_check(hipGetLastError(), "mixed launch");
}

st_status run_mixed(const Cfg &c, void *x, void *e1, void *e2, void *d, void *u, hipStream_t s)
{
    if (c.dtype == ST_F16)
        return mixed_impl<true>(c, static_cast<float *>(x), static_cast<uint16_t *>(e1),
                                static_cast<uint16_t *>(e2), static_cast<uint16_t *>(d),
                                static_cast<float *>(u), s);
    return mixed_impl<false>(c, static_cast<float *>(x), static_cast<uint16_t *>(e1),
                             static_cast<uint16_t *>(e2), static_cast<uint16_t *>(d),
                             static_cast<float *>(u), s);
}

}  // namespace st

namespace st {

template <bool F16>
__global__ void k_round16(const float *__restrict__ in, uint16_t *__restrict__ out, long long n)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = rnd16<F16>(in[i]);
}

template <bool F16>
__global__ void k_widen16(const uint16_t *__restrict__ in, float *__restrict__ out, long long n)
{
    const long long stride = (long long)gridDim.x * blockDim.x;
    for (long long i = blockIdx.x * (long long)blockDim.x + threadIdx.x; i < n; i += stride)
        out[i] = wid16<F16>(in[i]);
}

static dim3 conv_blocks(uint64_t n)
{
    uint64_t b = (n + 255) / 256;
    if (b > 65536) b = 65536;
    return dim3((unsigned)(b < 1 ? 1 : b));
}

}  // namespace st

extern "C" st_status stencil_round16(const float *d_in, uint16_t *d_out, uint64_t n, int dtype, void *stream)
{
    using namespace st;
    if (dtype != ST_BF16 && dtype != ST_F16) return fail(ST_EINVAL, "round16: dtype must be BF16 or F16");
    if (!d_in || !d_out) return fail(ST_EINVAL, "round16: null buffer");
    if (n == 0) return ST_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == ST_F16) hipLaunchKernelGGL(k_round16<true>, conv_blocks(n), dim3(256), 0, s, d_in, d_out, (long long)n);
    else hipLaunchKernelGGL(k_round16<false>, conv_blocks(n), dim3(256), 0, s, d_in, d_out, (long long)n);
    return hip_check(hipGetLastError(), "round16 launch");
}

extern "C" st_status stencil_widen16(const uint16_t *d_in, float *d_out, uint64_t n, int dtype, void *stream)
{
    using namespace st;
    if (dtype != ST_BF16 && dtype != ST_F16) return fail(ST_EINVAL, "widen16: dtype must be BF16 or F16");
    if (!d_in || !d_out) return fail(ST_EINVAL, "widen16: null buffer");
    if (n == 0) return ST_OK;
    hipStream_t s = static_cast<hipStream_t>(stream);
    if (dtype == ST_F16) hipLaunchKernelGGL(k_widen16<true>, conv_blocks(n), dim3(256), 0, s, d_in, d_out, (long long)n);
    else hipLaunchKernelGGL(k_widen16<false>, conv_blocks(n), dim3(256), 0, s, d_in, d_out, (long long)n);
    return hip_check(hipGetLastError(), "widen16 launch");
}
