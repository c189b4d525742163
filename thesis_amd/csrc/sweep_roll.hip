// Rolling form: 2D grids of wide stars, one or three sweeps per launch.  AUTO
// runs dispatches with it; it has no counterpart in the reference, whose
// kernels advance one sweep per launch (src/stencil_dispatch.cu:138-158).
//
// A wave owns a segment of 64 lanes x 16 bytes of columns and marches it
// along y over a chunk of rows.  When row m arrives, level l completes row
// m - l*R from the rows of level l-1: per level a lane holds the last R rows
// (the j-previous terms and the centres) and the R running sums that wait
// for their j-next terms, in the reference's order of terms
// (src/stencil_accumulators.cu:46-74).  x neighbours are the lane's own
// word and whole words of the next lanes (DPP rotates): no LDS, no barrier,
// and each row is read once instead of once per row offset.  Segments and
// chunks overlap by the levels' halo.
//
// Bound: memory for one sweep (8192^2 FP32 R = 4 132 us, 4.1 TB/s of one read
// and one write; register march before: 155), the VALU and the waves in
// flight for three (R = 2 60 us a sweep, R = 4 69, R = 6 88; before 151, 155,
// 407).  One sweep of 8192^2, before and now: FP32 R = 8 456 -> 148, R = 12
// 655 -> 162, R = 16 665 -> 181; FP64 R = 4 316 -> 166 (three), R = 8
// 950 -> 261, R = 16 1718 -> 363.
//
// Shell: as in the block form a pass advances an odd number of sweeps, so
// level l sees the shell of `in` for even l and of `out` for odd l; waves and
// rows that touch the shell load it from there, one row ahead.
#include <algorithm>
#include <type_traits>
#include <utility>

#include "st_device.hpp"
#include "st_internal.hpp"

namespace st {

struct RollArgs {
    int nx, ny;
    int nseg, nwaves;  // segments per chunk, waves
    int chunk;         // rows per chunk
    int bytes;         // of a field
};

// columns of a lane, and of halo on each side of a segment
template <typename T> constexpr int roll_cx() { return 16 / (int)sizeof(T); }
__host__ __device__ constexpr int roll_halo(int r, int steps, int cx) { return (r * steps + cx - 1) / cx * cx; }

template <int OP, int R, int STEPS, typename T>
__global__ __launch_bounds__(256) void k_roll(const T *__restrict__ in, T *out, RollArgs a, T kc)
{
    constexpr int CX = roll_cx<T>(), H = roll_halo(R, STEPS, CX), NL = (R + CX - 1) / CX, ES = (int)sizeof(T);
    constexpr int PH = R >= 4 ? R : R == 3 ? 6 : 4;         // phases of the march, a multiple of R
    constexpr int PF = PH <= 7 ? PH : PH % 4 == 0 ? 4 : PH % 5 == 0 ? 5 : PH % 3 == 0 ? 3 : PH;  // rows in flight
    typedef unsigned int W4 __attribute__((ext_vector_type(4)));
    typedef T VX __attribute__((ext_vector_type(CX)));
    const int lane = threadIdx.x & 63;
    const int id = (int)xcd_remap(blockIdx.x, gridDim.x) * 4 + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (id >= a.nwaves) return;
    const int seg = id % a.nseg, ch = id / a.nseg;
    const int base = seg * (64 * CX - 2 * H), c0 = base + lane * CX;
    const int y0 = ch * a.chunk, y1 = min(y0 + a.chunk, a.ny);
    const bool edge = base < R || base + 64 * CX > a.nx - R;  // the segment touches the x shell
    unsigned xin = 0;
#pragma unroll
    for (int c = 0; c < CX; ++c) xin |= interior1(c0 + c, a.nx, R) ? 1u << c : 0u;
    // exact columns: H away from the segment's ends, except at the field's
    const int s0 = seg == 0 ? 0 : base + H, s1 = seg == a.nseg - 1 ? a.nx : base + 64 * CX - H;
    const bool stores = c0 >= s0 && c0 < s1, whole = stores && c0 + CX <= s1;

    // row m (clamped to the field) of a buffer; words past its end read 0,
    // columns past the row's end what follows: no interior cell uses them
    const int pitch = a.nx * ES, at = c0 < a.nx ? c0 * ES : 0;
    const __amdgpu_buffer_rsrc_t rin = __builtin_amdgcn_make_buffer_rsrc(const_cast<T *>(in), 0, a.bytes, 0x00020000);
    const __amdgpu_buffer_rsrc_t rout = __builtin_amdgcn_make_buffer_rsrc(out, 0, a.bytes, 0x00020000);
    auto row_of = [&](const __amdgpu_buffer_rsrc_t &rs, int m) {
        m = min(max(m, 0), a.ny - 1);
        const W4 w = __builtin_amdgcn_raw_buffer_load_b128(rs, m * pitch + at, 0, 0);
        return __builtin_bit_cast(VX, w);
    };

    T ring[STEPS][R][CX], part[STEPS][R][CX];
    VX sh[STEPS], pre[PF];
#pragma unroll
    for (int l = 0; l < STEPS; ++l) {
        sh[l] = VX(0);
#pragma unroll
        for (int i = 0; i < R; ++i)
#pragma unroll
            for (int c = 0; c < CX; ++c) ring[l][i][c] = part[l][i][c] = (T)0;
    }
    const int m_lo = max(y0 - STEPS * R, 0), m_hi = min(y1, a.ny - R) + STEPS * R;
    if (m_lo >= m_hi) return;
    auto shell_rows = [&](int m) {  // the shell's values for step m
#pragma unroll
        for (int l = 0; l < STEPS; ++l) {
            const int y = m - (l + 1) * R;
            if (edge || !interior1(y, a.ny, R)) sh[l] = row_of(l & 1 ? rin : rout, y);
        }
    };
    shell_rows(m_lo);
#pragma unroll
    for (int i = 0; i < PF; ++i) pre[i] = row_of(rin, m_lo + i);

    for (int m0 = m_lo; m0 < m_hi; m0 += PH) {
        each_phase(std::make_integer_sequence<int, PH>{}, [&](auto phase) {
            constexpr int ph = decltype(phase)::value, rp = ph % R;
            const int m = m0 + ph;
            if (m >= m_hi) return false;
            __builtin_amdgcn_sched_barrier(0);
            T cur[CX];
#pragma unroll
            for (int c = 0; c < CX; ++c) cur[c] = pre[ph % PF][c];
            pre[ph % PF] = row_of(rin, m + PF);
            VX now[STEPS];
#pragma unroll
            for (int l = 0; l < STEPS; ++l) now[l] = sh[l];
            shell_rows(m + 1);
#pragma unroll
            for (int l = 0; l < STEPS; ++l) {
                // the words of NL lanes on each side
                T v[(2 * NL + 1) * CX];
#pragma unroll
                for (int c = 0; c < CX; ++c) v[NL * CX + c] = cur[c];
#pragma unroll
                for (int k = 1; k <= NL; ++k)
#pragma unroll
                    for (int c = 0; c < CX; ++c) {
                        v[(NL - k) * CX + c] = from_left(v[(NL - k + 1) * CX + c]);
                        v[(NL + k) * CX + c] = from_right(v[(NL + k - 1) * CX + c]);
                    }
                T s[CX], done[CX], old[CX], res[CX];
#pragma unroll
                for (int c = 0; c < CX; ++c) {
                    const int o = NL * CX + c;
                    T u = v[o - R];
#pragma unroll
                    for (int d = R - 1; d >= 1; --d) u += v[o - d];
#pragma unroll
                    for (int d = 1; d <= R; ++d) u += v[o + d];
                    // logical ring[i] = row q-R+i, in slot (rp+i) % R; row q is
                    // the next j-next term of the sums of rows q-R .. q-1
#pragma unroll
                    for (int i = 0; i < R; ++i) {
                        u += ring[l][(rp + i) % R][c];
                        part[l][(rp + i) % R][c] += cur[c];
                    }
                    s[c] = u;
                    done[c] = part[l][rp][c];
                    old[c] = ring[l][rp][c];
                }
                finish_sums<OP>(done, old, kc, res);
                const bool yin = interior1(m - (l + 1) * R, a.ny, R);
                if (edge || !yin) {
#pragma unroll
                    for (int c = 0; c < CX; ++c) {
                        const T mine = res[c], held = now[l][c];
                        res[c] = yin && ((xin >> c) & 1u) ? mine : held;
                    }
                }
#pragma unroll
                for (int c = 0; c < CX; ++c) {
                    ring[l][rp][c] = cur[c];
                    part[l][rp][c] = s[c];
                    cur[c] = res[c];
                }
            }
            const int y = m - STEPS * R;
            if (y >= y0 && y < y1 && interior1(y, a.ny, R) && stores) {
                T *const p = out + (long long)y * a.nx + c0;
                if (whole) {
                    typedef T VU __attribute__((ext_vector_type(CX), aligned(sizeof(T))));
                    VU o;
#pragma unroll
                    for (int c = 0; c < CX; ++c) o[c] = cur[c];
                    *reinterpret_cast<VU *>(p) = o;
                } else {
#pragma unroll
                    for (int c = 0; c < CX; ++c)
                        if (c0 + c < s1) p[c] = cur[c];
                }
            }
            return true;
        });
    }
}

// ---------------------------------------------------------------- host side

template <int OP, int STEPS, typename T, int... I>
static const void *roll_pick(int r, std::integer_sequence<int, I...>)
{
    const void *fn = nullptr;
    ((r == I + 2 ? void(fn = reinterpret_cast<const void *>(&k_roll<OP, I + 2, STEPS, T>)) : void()), ...);
    return fn;
}

// One sweep for radius 2 to 16; three while ring and sums leave two waves per
// SIMD (FP32 to radius 6, FP64 to 5: with one, radius 7 FP32 4096^2 takes 56 us
// a sweep against 32 singly).
constexpr int kRollSteps = 3;

template <int OP, typename T>
static const void *roll_fn(int r, int steps)
{
    if (steps == 1) return roll_pick<OP, 1, T>(r, std::make_integer_sequence<int, 15>{});
    return roll_pick<OP, kRollSteps, T>(r, std::make_integer_sequence<int, sizeof(T) == 4 ? 5 : 4>{});
}

static const void *roll_kernel(const Cfg &c, int steps)
{
    if (c.dtype == ST_F64) return c.op == OP_THESIS ? roll_fn<OP_THESIS, double>(c.r, steps) : roll_fn<OP_JACOBI, double>(c.r, steps);
    return c.op == OP_THESIS ? roll_fn<OP_THESIS, float>(c.r, steps) : roll_fn<OP_JACOBI, float>(c.r, steps);
}

// Segments along x and rows per chunk of a pass.
static RollArgs roll_args(const Cfg &c, int steps)
{
    const int es = c.dtype == ST_F64 ? 8 : 4, cx = 16 / es, len = 64 * cx, halo = roll_halo(c.r, steps, cx);
    RollArgs a;
    a.nx = c.nx;
    a.ny = c.ny;
    a.bytes = c.nx * c.ny * es;
    a.nseg = c.nx <= len ? 1 : (c.nx - len + (len - 2 * halo) - 1) / (len - 2 * halo) + 1;
    // Chunks: the rows a SIMD marches (halo included) times what a row costs
    // with k waves sharing the SIMD, as many as its registers hold: one wave
    // does not cover its latencies (8192^2 FP32 R = 4, three sweeps per pass,
    // 1 / 2 / 3 waves: 129 / 84 / 69 us a sweep).
    const int occ = std::min(8, 512 / (8 * c.r * steps + (es == 8 ? 84 : 72)));
    auto share = [](int k) { return k == 0 ? 0.0 : k == 1 ? 1.7 : k == 2 ? 2.26 : (double)k; };
    // For k rounds of 1024 waves the best is the most chunks that fit them (the
    // fewest rows each), so only those are looked at; k rounds cost at least
    // `least`, the rows of all waves and their halo at the cheapest share, so
    // the search ends after some ten of them (every chunk count took 20 ms of
    // host time for 5 x 20000000).
    const int most = std::max(1, (c.ny - 1) / 7);  // chunks of 8 rows and more
    const double cheap = share(occ) / occ;
    double best = -1;
    for (long long k = (a.nseg + 1023) / 1024;; ++k) {
        const double least = cheap * ((double)a.nseg * c.ny / 1024 + (double)k * 2 * steps * c.r);
        if (best >= 0 && least > best * (1 + 1e-9)) break;
        const int nch = (int)std::min<long long>(most, 1024 * k / a.nseg), rows = (c.ny + nch - 1) / nch;
        const long long waves = (long long)a.nseg * ((c.ny + rows - 1) / rows), per = (waves + 1023) / 1024;
        const double cost = ((double)(per / occ) * share(occ) + share((int)(per % occ))) * (rows + 2 * steps * c.r);
        if (best < 0 || cost < best) {
            best = cost;
            a.chunk = rows;
            a.nwaves = (int)waves;
        }
        if (nch == most) break;
    }
    return a;
}

// AUTO's rule for 2D grids of radius 2 to 16 (us per sweep of 16, JACOBI).
// Against the families named before, from 2^20 cells on: FP32 R = 2 1024^2
// 5.7 / 5.1, R = 5 11.0 / 8.6, FP64 R = 2 6.8 / 5.1, R = 16 28.9 / 24.3; below,
// the rows a wave marches one after the other take longer than a launch of
// the plain kernel (512^2 3.3 / 5 to 28).  The plain kernel's FP32 form is
// faster at radii that are multiples of 4 and at wide stars (1024^2 R = 4
// 5.8 / 7.2, R = 8 9.0 / 12.4, R = 14 16 / 24): the line is 2^22 there (2048^2
// R = 4 12.0 / 10.8, R = 8 25 / 16.5, R = 14 52 / 32, R = 16 40 / 37).
// Three sweeps per pass or one: three to radius 3 (R = 3 4096^2 18 / 28); from
// radius 4 on the halo pays from a field of 32 MiB (R = 4), 64 (R = 5) and
// 128 (R = 6): R = 4 2048^2 12.5 / 11.2, 4096^2 23.4 / 28.5, 8192^2 69 / 132;
// R = 6 4096^2 31 / 31, 8192^2 88 / 133.
void resolve_roll(Cfg &c)
{
    c.roll_steps = 0;
    if (c.dims != 2 || (c.dtype != ST_F32 && c.dtype != ST_F64) || c.nx < 2 * c.r + 1 || c.ny < 2 * c.r + 1) return;
    const long long es = c.dtype == ST_F64 ? 8 : 4, cells = (long long)c.nx * c.ny;
    if (cells * es >= (1LL << 31)) return;  // 32-bit byte offsets
    // a wave marches through the shell's rows too: not where they are over
    // three quarters (FP64 100000x40 R = 16, 8 rows of 40, 24 / 32; 300000x9
    // R = 4 5.8 / 6.4)
    if (4LL * (c.ny - 2 * c.r) < c.ny) return;
    const bool late = c.dtype == ST_F32 && (c.r % 4 == 0 || c.r > 8);
    if (cells < (late ? 1LL << 22 : 1LL << 20) || !roll_kernel(c, 1)) return;
    // Radius 2 on whole quads, the plain kernel's best case: up to 2^21 cells
    // (for FP32 not counting columns that a segment of 256 leaves empty) few
    // sweeps, and FP32 THESIS, stay with it (us, plain / this: 1024^2 3 sweeps
    // 14.9 / 16.8, FP64 19.1 / 20.6, 7 of THESIS 34.5 / 38.6, 16 of JACOBI 85 / 79;
    // 64x60000 7 of THESIS 74 / 86).
    if (c.r == 2 && c.nx % 4 == 0) {
        const bool f32 = c.dtype == ST_F32;
        const long long filled = f32 ? cells * std::min(c.nx, 256) / 256 : cells;
        if (filled < 1LL << 21 && (c.iters < 4 || (f32 && (c.op == OP_THESIS || c.iters < 8)))) return;
    }
    const bool deep = roll_kernel(c, kRollSteps) && (c.r <= 3 || cells * es >= 32LL << 20 << (c.r - 4));
    c.roll_steps = deep ? kRollSteps : 1;
}

// Passes of roll_steps sweeps while more than that are left, then single
// ones: odd passes, so their number has the parity of the sweeps', and a
// single last one, so both buffers end as single sweeps leave them.
static int roll_deep_passes(const Cfg &c)
{
    return c.roll_steps > 1 && c.iters > 0 ? (c.iters - 1) / c.roll_steps : 0;
}

int roll_launches(const Cfg &c)
{
    const int deep = roll_deep_passes(c);
    return deep + (c.iters - deep * c.roll_steps);
}

st_status run_roll(const Cfg &c, void *u1, void *u2, hipStream_t s, int *in_u2)
{
    *in_u2 = c.iters & 1;
    const double kd = c.op == OP_THESIS ? (double)(2 * c.dims * c.r) : c.weight;
    const float kf = (float)kd;
    const int deep = roll_deep_passes(c), n = roll_launches(c);
    RollArgs a;
    for (int i = 0; i < n; ++i) {
        const int steps = i < deep ? c.roll_steps : 1;
        if (i == 0 || i == deep) a = roll_args(c, steps);
        void *args[] = {&u1, &u2, &a, c.dtype == ST_F64 ? (void *)&kd : (void *)&kf};
        const hipError_t e = hipLaunchKernel(roll_kernel(c, steps), dim3((a.nwaves + 3) / 4), dim3(256), args, 0, s);
        if (e != hipSuccess) return hip_check(e, "rolling form launch");
        std::swap(u1, u2);
    }
    return ST_OK;
}

}  // namespace st
