// Block form: several sweeps of a register-resident block per launch, for 2D
// grids of radius 1.  AUTO runs dispatches of four sweeps and more with it;
// it has no counterpart in the reference, whose kernels advance one sweep
// per launch (src/stencil_dispatch.cu:138-158).
//
// A wave owns 64 columns x kRows2 rows, one column per lane (any nx, any
// alignment): it loads the block with a halo of `steps` cells, advances it
// `steps` sweeps in registers and stores the cells that are still exact.  x
// neighbours are one DPP rotate, y neighbours the lane's own registers;
// waves are independent (no LDS, no barrier).
//
// Shell: sweep s of a dispatch reads the shell of buffer s%2, so inside a
// pass the shell alternates between the two buffers' values.  `steps` is
// odd in every pass, which makes the buffer a pass reads (`in`) the one
// whose shell levels 0, 2, 4, .. see and the buffer it writes (`out`) the
// one of levels 1, 3, ..: the shell's two values are loaded once and change
// places at every level, and equal and different shells are one path with
// no comparison beforehand.  Where AUTO would name a per-sweep family the
// last pass is a single sweep, so both buffers end as single sweeps leave
// them; where it would name the streaming form, which leaves an earlier state
// in the other buffer, there is no such pass (24 sweeps of 8192^2 FP32
// JACOBI: streaming form 603 us, with it 695, without it 521).
//
// Bound: launches up to 512^2 (a launch per sweep costs 2.5 us, a pass of 9
// sweeps about 7), above that the VALU: a block computes every row at every
// level, 64*32 cells for (64-2*steps)*(32-2*steps) stored.  64 sweeps, FP32
// JACOBI, before (plain kernel below 2048^2, streaming form above) and now:
// 256^2 172 -> 59 us, 1024^2 322 -> 100, 2048^2 452 -> 178, 4096^2 696 ->
// 408, 16384^2 6.00 -> 5.26 ms; different shells, which the streaming form
// sweeps singly, 4096^2 THESIS 1946 -> 552 us.
#include <algorithm>

#include "st_device.hpp"
#include "st_internal.hpp"

namespace st {

struct BlockArgs {
    int nx, ny;
    int tx, ty;  // blocks per axis
    int steps;   // sweeps of this pass (odd)
};

// Rows of a block: 32 FP32 rows and their alternating shell values take 99
// VGPRs (four waves per SIMD).
constexpr int kRows2 = 32;

// One level.  EDGE: the block touches the shell; alt holds the shell cells'
// values of the next level's parity.
template <int OP, bool EDGE, typename T>
__device__ __forceinline__ void block2d_level(T (&cur)[kRows2], T (&alt)[kRows2], bool xsh, int rlo, int rhi, T kc)
{
    T prev = cur[0];
    constexpr int G = 4;
#pragma unroll
    for (int r0 = 0; r0 < kRows2; r0 += G) {
        T old[G], s[G], nw[G];
#pragma unroll
        for (int i = 0; i < G; ++i) old[i] = cur[r0 + i];
#pragma unroll
        for (int i = 0; i < G; ++i) {
            T u = from_left(old[i]);
            u += from_right(old[i]);
            u += i > 0 ? old[i - 1] : prev;
            s[i] = u + (r0 + i + 1 < kRows2 ? cur[r0 + i + 1] : old[i]);
        }
        finish_sums<OP>(s, old, kc, nw);
#pragma unroll
        for (int i = 0; i < G; ++i) {
            const int r = r0 + i;
            if constexpr (EDGE) {
                const bool sh = xsh || r <= rlo || r >= rhi;
                cur[r] = sh ? alt[r] : nw[i];
                alt[r] = old[i];
            } else {
                cur[r] = nw[i];
            }
        }
        prev = old[G - 1];
    }
}

template <int OP, typename T>
__global__ __launch_bounds__(256) void k_block2d(const T *__restrict__ in, T *__restrict__ out, BlockArgs a, T kc)
{
    const int lane = threadIdx.x & 63;
    const int id = (int)blockIdx.x * (int)(blockDim.x >> 6) + __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    if (id >= a.tx * a.ty) return;
    const int bx = id % a.tx, by = id / a.tx;
    const int x = bx * (64 - 2 * a.steps) + lane, y0 = by * (kRows2 - 2 * a.steps);
    const int xl = min(x, a.nx - 1);
    T cur[kRows2], alt[kRows2];
#pragma unroll
    for (int r = 0; r < kRows2; ++r) cur[r] = in[(long long)min(y0 + r, a.ny - 1) * a.nx + xl];
    const bool xsh = x == 0 || x >= a.nx - 1;
    // rows <= rlo or >= rhi of the block lie on the y shell (or beyond it)
    const int rlo = by == 0 ? 0 : -1, rhi = a.ny - 1 - y0;
    const bool edge = bx == 0 || x - lane + 64 >= a.nx || by == 0 || rhi < kRows2;
    if (edge) {
#pragma unroll
        for (int r = 0; r < kRows2; ++r) {
            const bool sh = xsh || r <= rlo || r >= rhi;
            alt[r] = sh ? out[(long long)min(y0 + r, a.ny - 1) * a.nx + xl] : (T)0;
        }
        for (int l = 0; l < a.steps; ++l) block2d_level<OP, true>(cur, alt, xsh, rlo, rhi, kc);
    } else {
        for (int l = 0; l < a.steps; ++l) block2d_level<OP, false>(cur, alt, false, -1, kRows2, kc);
    }
    // exact cells: `steps` away from the block's edges, except towards the shell
    const int r0 = by == 0 ? 1 : a.steps, r1 = rhi < kRows2 ? rhi : kRows2 - a.steps;
    const int l0 = bx == 0 ? 1 : a.steps, l1 = x - lane + 64 >= a.nx ? 64 : 64 - a.steps;
    if (lane < l0 || lane >= l1 || x >= a.nx - 1) return;
#pragma unroll
    for (int r = 0; r < kRows2; ++r)
        if (r >= r0 && r < r1) out[(long long)(y0 + r) * a.nx + x] = cur[r];
}

// ---------------------------------------------------------------- host side

// Blocks along an axis of n cells: block b covers [b*(len - 2*steps), +len),
// the last one reaches cell n-1.
static int blocks_along(int n, int len, int steps)
{
    const int stride = len - 2 * steps;
    return n <= len ? 1 : (n - len + stride - 1) / stride + 1;
}

// Passes of a dispatch: `n` passes of an odd number of sweeps each, at most
// c.block_steps, then `single` sweeps (0 or 1); their number has the parity
// of the sweeps'.  Pass i has 1 + 2*(q + (i < rem)) sweeps.
struct BlockPlan {
    int n, q, rem, single;
};
static BlockPlan block_plan(const Cfg &c)
{
    const int single = c.variant == ST_V_COOP ? 0 : 1, m = c.iters - single;
    int n = (m + c.block_steps - 1) / c.block_steps;
    if ((n ^ m) & 1) ++n;  // n odd numbers sum to m
    const int pairs = (m - n) / 2;
    return {n, n ? pairs / n : 0, n ? pairs % n : 0, single};
}

static BlockArgs block_args(const Cfg &c, int steps)
{
    BlockArgs a;
    a.nx = c.nx;
    a.ny = c.ny;
    a.tx = blocks_along(c.nx, 64, steps);
    a.ty = blocks_along(c.ny, kRows2, steps);
    a.steps = steps;
    return a;
}

// AUTO's rule.  Sweeps per pass, measured at 64 sweeps (us, 3 / 5 / 7 / 9):
// 256^2 118 / 85 / 69 / 61, 1024^2 138 / 110 / 107 / 103, 2048^2 242 / 203 /
// 178 / 184, 8192^2 2504 / 1646 / 1419 / 1777: deeper passes until the
// halo's extra work outweighs the launches and loads they save.  While the
// blocks are at most two waves per SIMD the launches decide (9); above that
// 7, and 5 for THESIS, whose quotient makes the halo dearer (4096^2 634 / 552
// / 605 / 751).  Planes of 2^29 cells and more stay with the streaming form,
// which is level there with equal shells (32768^2 23.6 against 22.1 ms;
// 16384^2 24 sweeps 2.03 against 2.10 here, 64 sweeps 6.00 against 5.26).
void resolve_block(Cfg &c)
{
    c.block_steps = 0;
    if (c.dims != 2 || c.r != 1 || (c.dtype != ST_F32 && c.dtype != ST_F64) || c.iters < 4 || c.nx < 8 || c.ny < 8 ||
        (long long)c.nx * c.ny >= (1LL << 29))
        return;
    auto waves = [&](int steps) {
        return (long long)blocks_along(c.nx, 64, steps) * blocks_along(c.ny, kRows2, steps);
    };
    c.block_steps = waves(9) <= 2048 ? 9 : (c.op == OP_THESIS && waves(7) > 8192 ? 5 : 7);
}

int block_launches(const Cfg &c)
{
    const BlockPlan p = block_plan(c);
    return p.n + p.single;
}

template <int OP, typename T>
static hipError_t block_launch(const void *in, void *out, const BlockArgs &a, double kc, hipStream_t s)
{
    hipLaunchKernelGGL((k_block2d<OP, T>), dim3((a.tx * a.ty + 3) / 4), dim3(256), 0, s, static_cast<const T *>(in),
                       static_cast<T *>(out), a, (T)kc);
    return hipGetLastError();
}

st_status run_block(const Cfg &c, void *u1, void *u2, hipStream_t s, int *in_u2)
{
    const BlockPlan p = block_plan(c);
    const double kc = c.op == OP_THESIS ? (double)(2 * c.dims) : c.weight;
    auto launch = c.dtype == ST_F64 ? (c.op == OP_THESIS ? &block_launch<OP_THESIS, double> : &block_launch<OP_JACOBI, double>)
                                    : (c.op == OP_THESIS ? &block_launch<OP_THESIS, float> : &block_launch<OP_JACOBI, float>);
    *in_u2 = c.iters & 1;
    for (int i = 0; i < p.n + p.single; ++i) {
        const hipError_t e = launch(u1, u2, block_args(c, i < p.n ? 1 + 2 * (p.q + (i < p.rem)) : 1), kc, s);
        if (e != hipSuccess) return hip_check(e, "block launch");
        std::swap(u1, u2);
    }
    return ST_OK;
}

}  // namespace st
