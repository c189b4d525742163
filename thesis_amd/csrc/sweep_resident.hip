// Resident form: every sweep of a dispatch in one cooperative launch, the
// field in registers, for 3D grids of radius 1 up to 256 columns that fit one
// workgroup per CU (128^3, 160^3, 256 x 128 x 128, and batches of such grids).
// AUTO runs dispatches with it; it has no counterpart in the reference, whose
// kernels read and write the field every sweep
// (src/stencil_dispatch.cu:138-158).
//
// A workgroup of ROWS waves (8 or 16) owns ROWS whole rows of NZ planes; a
// wave holds one row of each plane, CX consecutive columns per lane (nx <=
// 64*CX).  Per sweep a wave takes x neighbours from its own registers and one
// DPP rotate per side, y neighbours from LDS (ZS planes at a time, double
// buffered, one barrier per ZS planes), z neighbours from its own registers.
// The rows and planes at the edges of the workgroup's block go to the four
// neighbouring workgroups through memory, and nothing else does.
//
// Exchange: every 32-bit word travels as one 64-bit word with a 32-bit tag,
// the number of the sweep it belongs to, in relaxed agent-scope atomics.  A
// reader polls the word itself until the tag is the one it needs, so there
// is no flag, no fence and no grid barrier (a cooperative grid barrier costs
// 25 us here, a hop of this exchange about 0.4, a round trip 0.8).  Two slots alternate: a wave
// sends sweep n+2 only after it has its neighbour's words of sweep n+1, which
// the neighbour sends after reading those of sweep n.  Tags go on from launch
// to launch (ctl[0], advanced by the last workgroup to finish), so what an
// earlier launch left in a slot never matches.  All workgroups are
// co-resident (cooperative launch, at most one per CU); a poll that finds
// nothing for many seconds gives NaN and sets a word of host memory, so every
// wave ends and the next call that looks at the word says so.
//
// Shell: sweep n reads the shell of buffer n%2, so shell cells alternate
// between the two buffers' values: the x shell from an LDS table, shell rows
// and planes from the buffers themselves, fetched while the faces travel.
//
// Bound: the hops of the exchange and the instructions between them (64^3
// 1.5 us per sweep, about 3 hops; 128^3 3.4 us, of which the VALU's share is
// about 0.5).  Before and now, 200 sweeps FP32: 64^3 502 -> 321 us, 96^3
// 1165 -> 500, 128^3 1451 -> 693, 160^3 1920 -> 1416 (one launch per sweep
// of the plain and row kernels before).  Measured and dropped: polling every
// face before the first barrier (128^3 4.2 us), a pause before the first
// poll (no gain), blocks of 32 planes (spill).
#include <algorithm>
#include <type_traits>

#include "st_device.hpp"
#include "st_internal.hpp"

namespace st {

constexpr int kResProblems = 64;   // problems of one launch
constexpr int kResPolls = 1 << 25;  // about 0.4 us each

typedef unsigned long long ResWord;

struct ResArgs {
    unsigned *gave_up;   // host word, set by a wave whose poll found nothing
    int nx, ny, nz;
    long long sz;        // nx*ny
    int nyb, nzb;        // blocks along y and z, per problem
    int iters;
    ResWord *faces;
    unsigned *ctl;       // [0] tags used so far, [1] workgroups done
    void *u[kResProblems][2];
};

// A face row: CX values per lane, sizeof(T)/4 words each, word i of lane l
// at [i*64 + l].
__device__ __forceinline__ void word_put(ResWord *p, ResWord v)
{
    __hip_atomic_store(p, v, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ ResWord word_get(const ResWord *p)
{
    return __hip_atomic_load(p, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}

// an element at a wave-uniform base and a lane's byte offset
template <typename T>
__device__ __forceinline__ T *at(T *base, unsigned bytes)
{
    typedef typename std::conditional<std::is_const<T>::value, const char, char>::type C;
    return reinterpret_cast<T *>(reinterpret_cast<C *>(base) + bytes);
}

template <int CX, typename T>
struct Face {
    static constexpr int N = CX * (int)sizeof(T) / 4;
    ResWord w[N];
    __device__ __forceinline__ void load(const ResWord *row, int lane)
    {
#pragma unroll
        for (int i = 0; i < N; ++i) w[i] = word_get(at(row + i * 64, lane * 8u));
    }
    // whether every word of the wave carries `tag`
    __device__ __forceinline__ bool here(unsigned tag) const
    {
        bool ok = true;
#pragma unroll
        for (int i = 0; i < N; ++i) ok &= (unsigned)(w[i] >> 32) == tag;
        return __all(ok);
    }
    // the values; NaN when they never came
    __device__ __forceinline__ void get(T (&v)[CX], bool came) const
    {
#pragma unroll
        for (int c = 0; c < CX; ++c) {
            if constexpr (sizeof(T) == 4) v[c] = __uint_as_float((unsigned)w[c]);
            else v[c] = __longlong_as_double((long long)((w[2 * c] & 0xffffffffull) | (w[2 * c + 1] << 32)));
            if (!came) v[c] = (T)__builtin_nanf("");
        }
    }
    static __device__ __forceinline__ void send(ResWord *row, const T (&v)[CX], unsigned tag, int lane)
    {
#pragma unroll
        for (int i = 0; i < N; ++i) {
            unsigned bits;
            if constexpr (sizeof(T) == 4) bits = __float_as_uint(v[i]);
            else bits = (unsigned)((unsigned long long)__double_as_longlong(v[i / 2]) >> (32 * (i & 1)));
            word_put(at(row + i * 64, lane * 8u), ((ResWord)tag << 32) | bits);
        }
    }
};

// planes per LDS stage: two stages of 18 rows in about 147 KB at most
template <int CX, int NZ, typename T>
constexpr int res_stage()
{
    constexpr int b = CX * (int)sizeof(T), zs = b <= 16 ? 4 : b <= 32 ? 2 : 1;
    return NZ < zs ? NZ : zs;
}

// words of one block's incoming faces of one slot: rows [0, NZ) below,
// [NZ, 2*NZ) above in y; [2*NZ, +ROWS) below, [.., +ROWS) above in z
template <int ROWS, int CX, int NZ, typename T>
constexpr long long res_face_words() { return (2LL * NZ + 2 * ROWS) * 64 * CX * (sizeof(T) / 4); }

template <int OP, int ROWS, int CX, int NZ, typename T>
__global__ __launch_bounds__(64 * ROWS) void k_resident(ResArgs a, T kc)
{
    constexpr int ZS = res_stage<CX, NZ, T>(), NS = NZ / ZS;
    constexpr int RW = 64 * CX * (int)(sizeof(T) / 4);  // words of a face row
    typedef T V __attribute__((ext_vector_type(CX)));
    __shared__ __align__(16) T rows[2][ZS][ROWS + 2][64 * CX];  // row w at [w + 1]; [0], [ROWS + 1]: halo
    __shared__ T xsh[2][ROWS][NZ][2];                           // columns 0 and nx-1 of each buffer
    // Whether a poll of this workgroup gave up.  Where FP32 state fills the
    // registers a word of LDS holds it: `polls` outliving the sweeps would
    // spill (148x231x93 9% slower); elsewhere `polls` does, the LDS word
    // costing up to 26% (36x430x105 FP64).
    constexpr bool kWord = sizeof(T) == 4 && CX * NZ >= (ROWS == 16 ? 32 : 64);
    __shared__ int gave_up;
    if constexpr (kWord) {
        if (threadIdx.x == 0) gave_up = 0;
        __syncthreads();
    }
    const int lane = threadIdx.x & 63;
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int per = a.nyb * a.nzb;
    // neighbouring blocks on one XCD as far as they go
    const int id = (int)xcd_remap(blockIdx.x, gridDim.x);
    const int prob = id / per, blk = id - prob * per;
    const int bz = blk / a.nyb, by = blk - bz * a.nyb;
    T *const u0 = static_cast<T *>(a.u[prob][0]);
    T *const u1 = static_cast<T *>(a.u[prob][1]);
    const int y = by * ROWS + w, z0 = bz * NZ;
    const bool yshell = y == 0 || y >= a.ny - 1;       // never computed (shell, or past the grid)
    const bool zlo = bz == 0;
    const int zs = a.nz - 1 - z0;                       // plane nz-1 (>= NZ: above the block)
    const int x = lane * CX;
    const long long row0 = (long long)min(y, a.ny - 1) * a.nx;
    const unsigned epoch = __hip_atomic_load(a.ctl, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) + 1u;
    const bool nyl = by > 0, nyh = by < a.nyb - 1, nzl = bz > 0, nzh = bz < a.nzb - 1;

    // faces (word offsets): this block's incoming ones, and the neighbours'
    // that it fills
    constexpr int FW = (int)res_face_words<ROWS, CX, NZ, T>();
    const unsigned mine = (unsigned)id * 2u * FW;
    const unsigned to_yl = mine - 2 * FW + NZ * RW;  // upper y face of block by-1
    const unsigned to_yh = mine + 2 * FW;            // lower y face of block by+1
    const unsigned to_zl = mine - 2u * FW * a.nyb + (2 * NZ + ROWS + w) * RW;
    const unsigned to_zh = mine + 2u * FW * a.nyb + (2 * NZ + w) * RW;
    const unsigned from_zl = mine + (2 * NZ + w) * RW, from_zh = from_zl + ROWS * RW;

    unsigned xb[CX];  // byte offsets of the lane's columns (past the grid: column nx-1)
#pragma unroll
    for (int c = 0; c < CX; ++c) xb[c] = (unsigned)min(x + c, a.nx - 1) * (unsigned)sizeof(T);
    // a row of plane z0 + z from buffer u
    auto load_row = [&](const T *u, int z, T (&d)[CX]) {
        const T *p = u + (long long)min(z0 + z, a.nz - 1) * a.sz + row0;
#pragma unroll
        for (int c = 0; c < CX; ++c) d[c] = *at(p, xb[c]);
    };
    T cur[NZ][CX];
#pragma unroll
    for (int z = 0; z < NZ; ++z) load_row(u0, z, cur[z]);
    for (int i = lane; i < 4 * NZ; i += 64) {
        const int z = i >> 2, b = (i >> 1) & 1, e = i & 1;
        xsh[b][w][z][e] = (b ? u1 : u0)[(long long)min(z0 + z, a.nz - 1) * a.sz + row0 + (e ? a.nx - 1 : 0)];
    }
    bool xm[CX];  // this lane's column c is on the x shell
#pragma unroll
    for (int c = 0; c < CX; ++c) xm[c] = x + c == 0 || x + c == a.nx - 1;
    const int xe = lane == 0 ? 0 : 1;

    typedef Face<CX, T> F;
    auto send = [&](ResWord *faces, int z, int slot, unsigned tag) {
        const unsigned so = slot * FW;
        if (z == 0 && nzl) F::send(faces + to_zl + so, cur[z], tag, lane);
        if (z == NZ - 1 && nzh) F::send(faces + to_zh + so, cur[z], tag, lane);
        if (w == 0 && nyl) F::send(faces + to_yl + so + z * RW, cur[z], tag, lane);
        if (w == ROWS - 1 && nyh) F::send(faces + to_yh + so + z * RW, cur[z], tag, lane);
    };
    auto store_all = [&](T *u) {
        if (yshell) return;
#pragma unroll
        for (int z = 0; z < NZ; ++z) {
            if ((z == 0 && zlo) || z >= zs) continue;
            T *p = u + (long long)(z0 + z) * a.sz + row0;
#pragma unroll
            for (int c = 0; c < CX; ++c)
                if (x + c > 0 && x + c < a.nx - 1) *at(p, xb[c]) = cur[z][c];
        }
    };
#pragma unroll
    for (int z = 0; z < NZ; ++z) send(a.faces, z, 0, epoch);

    int st = 0;             // parity of the stage
    int polls = kResPolls;  // 0 once a poll has given up
    for (int n = 0; n < a.iters; ++n) {
        const int slot = n & 1;
        const unsigned so = slot * FW;
        const unsigned tag = epoch + (unsigned)n;
        // a zero the compiler does not know: keeps the addresses formed from
        // it from being held in registers across sweeps
        unsigned opaque = 0;
        asm volatile("" : "+s"(opaque));
        ResWord *const faces = a.faces + opaque;
        const T *const other = (slot ? u0 : u1) + opaque;  // the buffer of state n + 1
        if (n == a.iters - 1) {
            store_all((slot ? u1 : u0) + opaque);
        }
        T prev[CX];
#pragma unroll
        for (int c = 0; c < CX; ++c) prev[c] = (T)0;
#pragma unroll
        for (int s = 0; s < NS; ++s) {
            T(*const buf)[ROWS + 2][64 * CX] = rows[st];
            st ^= 1;
#pragma unroll
            for (int q = 0; q < ZS; ++q) {
                V v;
#pragma unroll
                for (int c = 0; c < CX; ++c) v[c] = cur[s * ZS + q][c];
                *reinterpret_cast<V *>(&buf[q][w + 1][x]) = v;
            }
            // shell rows and the stage's shell plane turn to the other
            // buffer's values, fetched while the faces travel
            const int zq = s == 0 && zlo ? 0 : zs;
            const bool zsh = !yshell && zq >= s * ZS && zq < s * ZS + ZS;
            T shell[CX];
#pragma unroll
            for (int c = 0; c < CX; ++c) shell[c] = (T)0;
            if (zsh) load_row(other, zq, shell);
            if (yshell) {
#pragma unroll
                for (int q = 0; q < ZS; ++q) load_row(other, s * ZS + q, cur[s * ZS + q]);
            }
            const bool wl = s == 0 && nzl, wh = s == NS - 1 && nzh;
            F fl, fh;
            if (wl) fl.load(faces + from_zl + so, lane);
            if (wh) fh.load(faces + from_zh + so, lane);
            // wave q < 2*ZS fetches one of the stage's y halo rows
            if (w < 2 * ZS && (w < ZS ? nyl : nyh)) {
                const bool low = w < ZS;
                const int q = low ? w : w - ZS;
                const ResWord *row = faces + mine + so + ((low ? 0 : NZ) + s * ZS + q) * RW;
                F fy;
                fy.load(row, lane);
                for (int left = polls; !fy.here(tag); fy.load(row, lane))
                    if (--left < 0) {
                        polls = 0;
                        if constexpr (kWord) gave_up = 1;
                        break;
                    }
                T h[CX];
                fy.get(h, polls > 0);
                V v;
#pragma unroll
                for (int c = 0; c < CX; ++c) v[c] = h[c];
                *reinterpret_cast<V *>(&buf[q][low ? 0 : ROWS + 1][x]) = v;
            }
            __syncthreads();
            for (int left = polls;;) {
                bool all = true;
                if (wl && !fl.here(tag)) {
                    all = false;
                    fl.load(faces + from_zl + so, lane);
                }
                if (wh && !fh.here(tag)) {
                    all = false;
                    fh.load(faces + from_zh + so, lane);
                }
                if (all) break;
                if (--left < 0) {
                    polls = 0;
                    if constexpr (kWord) gave_up = 1;
                    break;
                }
            }
            T up[CX];  // plane above the block
#pragma unroll
            for (int c = 0; c < CX; ++c) up[c] = (T)0;
            if (wl) fl.get(prev, polls > 0);
            if (wh) fh.get(up, polls > 0);
#pragma unroll
            for (int q = 0; q < ZS; ++q) {
                __builtin_amdgcn_sched_barrier(0);
                const int z = s * ZS + q;
                T old[CX];
#pragma unroll
                for (int c = 0; c < CX; ++c) old[c] = cur[z][c];
                if (!yshell && z == zq) {
#pragma unroll
                    for (int c = 0; c < CX; ++c) cur[z][c] = shell[c];
                } else if (!yshell && z < zs) {
                    const V m = *reinterpret_cast<const V *>(&buf[q][w][x]);
                    const V p = *reinterpret_cast<const V *>(&buf[q][w + 2][x]);
                    const T xv = xsh[slot ^ 1][w][z][xe];
                    const T xl = from_left(old[CX - 1]), xr = from_right(old[0]);
                    T sum[CX], res[CX];
#pragma unroll
                    for (int c = 0; c < CX; ++c) {
                        T t = c > 0 ? old[c - 1] : xl;
                        t += c + 1 < CX ? old[c + 1] : xr;
                        t += m[c];
                        t += p[c];
                        t += prev[c];
                        sum[c] = t + (z + 1 < NZ ? cur[z + 1][c] : up[c]);
                    }
                    finish_sums<OP>(sum, old, kc, res);
#pragma unroll
                    for (int c = 0; c < CX; ++c) cur[z][c] = xm[c] ? xv : res[c];
                }
                if (n + 1 < a.iters) send(faces, z, slot ^ 1, tag + 1u);
#pragma unroll
                for (int c = 0; c < CX; ++c) prev[c] = old[c];
            }
        }
    }
    store_all((a.iters & 1) ? u1 : u0);
    if constexpr (!kWord) {
        if (polls == 0 && lane == 0) __hip_atomic_store(a.gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
    }
    // the last workgroup to finish moves the tags on
    __syncthreads();
    if (threadIdx.x == 0) {
        if constexpr (kWord) {
            if (gave_up) __hip_atomic_store(a.gave_up, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
        }
        const unsigned d = __hip_atomic_fetch_add(a.ctl + 1, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (d == gridDim.x - 1) {
            __hip_atomic_store(a.ctl + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(a.ctl, epoch + (unsigned)a.iters, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
}

__global__ __launch_bounds__(256) void k_resident_clear(ResWord *p, long long n)
{
    for (long long i = blockIdx.x * 256LL + threadIdx.x; i < n; i += 256LL * gridDim.x) p[i] = 0;
}

// ---------------------------------------------------------------- host side

struct ResKernel {
    const void *fn = nullptr;
    int rows = 0, cx = 0, nz = 0;
    long long words = 0;  // face words of one block, one slot
    int blocks = 0;
};

template <int ROWS, int CX, int NZ, typename T>
static ResKernel res_kernel(int op)
{
    // cells per lane (32-bit words) that leave the kernel without spills
    if constexpr (CX * NZ * (int)sizeof(T) / 4 > (ROWS == 16 ? 32 : 64)) return {};
    else
        return {op == OP_THESIS ? reinterpret_cast<const void *>(&k_resident<OP_THESIS, ROWS, CX, NZ, T>)
                                : reinterpret_cast<const void *>(&k_resident<OP_JACOBI, ROWS, CX, NZ, T>),
                ROWS, CX, NZ, res_face_words<ROWS, CX, NZ, T>(), 0};
}

template <int ROWS, int CX, typename T>
static ResKernel res_kernel_nz(int op, int nz)
{
    switch (nz) {
    case 2: return res_kernel<ROWS, CX, 2, T>(op);
    case 4: return res_kernel<ROWS, CX, 4, T>(op);
    case 8: return res_kernel<ROWS, CX, 8, T>(op);
    default: return res_kernel<ROWS, CX, 16, T>(op);
    }
}

template <int ROWS, typename T>
static ResKernel res_kernel_for(int op, int nx, int nz)
{
    if (nx <= 64) return res_kernel_nz<ROWS, 1, T>(op, nz);
    if (nx <= 128) return res_kernel_nz<ROWS, 2, T>(op, nz);
    if (nx <= 256) return res_kernel_nz<ROWS, 4, T>(op, nz);
    return {};
}

static int device_cus()
{
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess)
        return 0;
    return cus;
}

// The kernel of `rows` rows per block with the fewest planes whose blocks
// (of all problems) fit one workgroup per CU.
static ResKernel res_fit(const Cfg &c, int problems, int cus, int rows)
{
    for (int nz : {2, 4, 8, 16}) {
        ResKernel k;
        if (rows == 8)
            k = c.dtype == ST_F64 ? res_kernel_for<8, double>(c.op, c.nx, nz) : res_kernel_for<8, float>(c.op, c.nx, nz);
        else
            k = c.dtype == ST_F64 ? res_kernel_for<16, double>(c.op, c.nx, nz) : res_kernel_for<16, float>(c.op, c.nx, nz);
        const long long blocks = (long long)problems * ((c.ny + rows - 1) / rows) * ((c.nz + nz - 1) / nz);
        if (!k.fn || blocks > cus) continue;
        k.blocks = (int)blocks;
        return k;
    }
    return {};
}

// 8 or 16 rows per block (us per sweep, FP32, 8 rows / 16 rows, with the
// planes each gets): wide flat blocks send less (128x128x64 2.43 with 4
// planes / 3.37 with 2; 256x128x128 5.09 with 8 / 7.58 with 4), tall narrow
// ones step through their planes with more waves (64x128x128 2.42 with 8 /
// 2.08 with 4; 96^3, 144 blocks either way, 3.4 with 8 / 2.4 with 4; 8
// problems of 64^3 4.7 with 16 / 2.9 with 8).
static ResKernel res_pick(const Cfg &c, int problems, int cus)
{
    const ResKernel a = res_fit(c, problems, cus, 8), b = res_fit(c, problems, cus, 16);
    if (!a.fn || !b.fn) return a.fn ? a : b;
    return a.nz <= 4 || (a.nz <= 8 && a.cx >= 2 && a.blocks >= 192) ? a : b;
}

// AUTO's rule: the launch costs about 20 us more than a plain one, a sweep
// less than the launch or the cache traffic it replaces (us per sweep, FP32:
// 64^3 1.5 against 2.5, 96^3 2.4 against 5.8, 128^3 3.4 against 7.2, 160^3
// 6.6 against 9.6).
bool resident_eligible(const Cfg &c, int problems)
{
    if (c.dims != 3 || c.r != 1 || (c.dtype != ST_F32 && c.dtype != ST_F64) || problems < 1 || problems > kResProblems ||
        c.nz < 6)
        return false;
    if (c.iters < ((long long)c.nx * c.ny * c.nz * problems < (1 << 19) ? 24 : 12)) return false;
    return res_pick(c, problems, device_cus()).fn != nullptr;
}

st_status resident_outcome(hipStream_t s)
{
    unsigned *word = nullptr;
    if (workspace_host_word(s, false, &word) != ST_OK || !word) return ST_OK;
    if (__atomic_exchange_n(word, 0u, __ATOMIC_RELAXED) == 0) return ST_OK;
    return fail(ST_ELAUNCH, "an earlier dispatch on this stream waited in vain for a neighbouring workgroup: its field holds NaN");
}

st_status run_resident(const Cfg &c, int problems, void *const (*u)[2], hipStream_t s, bool *done)
{
    *done = false;
    const int cus = device_cus();
    const ResKernel k = res_pick(c, problems, cus);
    if (!k.fn) return ST_OK;
    hipStreamCaptureStatus cap = hipStreamCaptureStatusNone;
    if (hipStreamIsCapturing(s, &cap) != hipSuccess || cap != hipStreamCaptureStatusNone || workspace_is_fixed()) {
        (void)hipGetLastError();
        return ST_OK;
    }
    st_status st = resident_outcome(s);
    if (st != ST_OK) return st;
    ResArgs a;
    if (workspace_host_word(s, true, &a.gave_up) != ST_OK) {
        (void)hipGetLastError();
        return ST_OK;
    }
    a.nx = c.nx; a.ny = c.ny; a.nz = c.nz;
    a.sz = (long long)c.nx * c.ny;
    a.nyb = (c.ny + k.rows - 1) / k.rows;
    a.nzb = (c.nz + k.nz - 1) / k.nz;
    a.iters = c.iters;
    const int blocks = k.blocks;
    if ((unsigned long long)blocks * 2 * k.words >= (1ull << 31)) return ST_OK;
    const size_t head = 256;
    const size_t bytes = head + (size_t)blocks * 2 * k.words * sizeof(ResWord);
    void *ws = nullptr;
    size_t fresh = 0;
    st = workspace_slot(kSlotResident, bytes, s, &ws, &fresh);
    if (st == ST_ENOMEM) {
        // no room for the faces: the caller's other form, which needs none
        (void)hipGetLastError();
        return ST_OK;
    }
    if (st != ST_OK) return st;
    if (fresh) {
        // tags start at 1
        hipLaunchKernelGGL(k_resident_clear, dim3(1024), dim3(256), 0, s, static_cast<ResWord *>(ws),
                           (long long)(fresh / sizeof(ResWord)));
        if ((st = hip_check(hipGetLastError(), "resident clear launch")) != ST_OK) return st;
    }
    a.ctl = static_cast<unsigned *>(ws);
    a.faces = static_cast<ResWord *>(ws) + head / sizeof(ResWord);
    for (int i = 0; i < kResProblems; ++i) {
        a.u[i][0] = i < problems ? u[i][0] : nullptr;
        a.u[i][1] = i < problems ? u[i][1] : nullptr;
    }
    double kd = c.op == OP_THESIS ? 6.0 : c.weight;
    float kf = (float)kd;
    void *args[] = {&a, c.dtype == ST_F64 ? static_cast<void *>(&kd) : static_cast<void *>(&kf)};
    const hipError_t e = hipLaunchCooperativeKernel(k.fn, dim3(blocks), dim3(64 * k.rows), args, 0, s);
    if (e != hipSuccess) {
        // no cooperative launch from this process now: the caller's other form
        (void)hipGetLastError();
        return ST_OK;
    }
    *done = true;
    return ST_OK;
}

}  // namespace st
