// FDTD pressure update for gfx950: 7-point leapfrog stencil (FP64 arithmetic on FP32
// storage) fused with the first-order absorbing boundary, or the split-field PML.
//
// Reference behaviour: FDTD::step (src/algorithm/fdtd.h:73-87), fdtd_inner_kernel and
// laplacian (src/algorithm/fdtd.cu:7-33), ab_condition_solve / Solve4x4Linear
// (fdtd.cu:36-137), fdtd_boundary_kernel (fdtd.cu:139-150), pml_step_kernel (fdtd.cu:162-232).
//
// The first blocks stream the interior (indices 2..N-3 in every dimension, z contiguous so a
// wave reads 256 B rows), the remaining blocks solve the 4x4 ABC system for the index-1 / N-2
// shell. Interior and shell write disjoint cells of level t+1; the shell also writes the ghost
// layer of level t, which no thread of the launch reads except the writing thread itself (masked
// terms of its own system), so the fusion is race-free. Without a mesh, or with phases timed, these
// blocks are a launch (k_fdtd_abc); in a step with a mesh they run beside the far-field sums
// (k_step_head). From an interior edge of 128 cells (kMarchMin) the interior is instead marched along
// x by its own launch before that (k_fdtd_march). t is read from device memory, so the launches
// can be replayed from a graph: a step in three launches hands it on (k_dirichlet, k_near),
// otherwise a one-thread kernel advances it.
#include "fdtd_device.hpp"
#include "scene_device.hpp"

#include <algorithm>

namespace pppm_amd
{

namespace
{

// Interior edge (N - 4) from which the interior is marched along x instead of one thread per cell.
// The line dates from FDTD steps of their own. The march is a launch more in a step with a mesh and
// has few blocks in the middle of the range; a step of 80 triangles marched / per cell: 132^3 46 / 25,
// 141^3 47 / 28, 200^3 57 / 45, 256^3 64 / 70, 324^3 223 / 149, 400^3 291 / 254 us, so a line further
// up would serve such steps better.
constexpr int kMarchMin = 128;

// Interior of a large grid: a block owns MTY x MTZ (y, z) columns of one chunk of x planes and
// marches them along x, so the x-neighbours come from registers and the y/z neighbours of the
// current plane from cache: each level-t value is fetched from HBM about once instead of once
// per plane that reads it. A thread holds MCPT columns 64 apart, so a wave covers MTZ z-values
// of one row from a 256-byte boundary (cells outside 2..N-3 idle, reading a live cell); the 16
// rows of a block are marched by its 16 waves together, so only the two rows past the tile and
// the two cache lines past its ends come from other blocks. Distinct noalias parameters let the compiler issue the loads of the next planes ahead
// of this plane's store.
//
// STREAM: the previous level is read and the next one written past the caches, which leaves them
// to the level-t rows that several waves read. It pays where two of the three levels no longer fit
// the Infinity Cache (256 MB), so that the next step would not find them there: a step at 512^3
// 384 -> 367 us (1.61 GB, 4.4 TB/s; a copy reaches 4.8), with the shell 448^3 365 -> 344 and
// 352^3 214 -> 195 us, but 284^3 140 -> 175 and 141^3 29 -> 37 us; at 316^3 it gives nothing. The
// division by h^2 takes the reciprocal from scalar registers (141^3: 30 -> 29 us).
constexpr long long kStreamBytes = 384LL << 20;  // of three levels
constexpr int MTY = 16;
constexpr int MBLK = 64 * MTY;
constexpr int MCPT = 4;            // z columns per thread, 64 apart: a tile is 16 rows x 256 z
constexpr int MTZ = 64 * MCPT;
template <bool STREAM>
__device__ __forceinline__ void march_columns(const float *__restrict__ g, const float *__restrict__ gm,
                                              float *__restrict__ gp, int N, int x0, int x1, int y, int z0,
                                              const FdtdParams &p)
{
    const int NN2 = N * N;
    const double rhh = uniform_rcp(p.hh);
    bool on[MCPT];
    float gxm[MCPT], gc[MCPT], gxp[MCPT];
    int me = lin3(x0, y, 0, N);
#pragma unroll
    for (int c = 0; c < MCPT; c++)
    {
        const int z = z0 + 64 * c;
        on[c] = z >= 2 && z <= N - 3;
        const int zz = on[c] ? z : 2;
        gxm[c] = g[me + zz - NN2];
        gc[c] = g[me + zz];
        gxp[c] = g[me + zz + NN2];
    }
#pragma unroll 2
    for (int x = x0; x < x1; x++)
    {
#pragma unroll
        for (int c = 0; c < MCPT; c++)
        {
            const int z = on[c] ? z0 + 64 * c : 2;
            const int q = me + z;
            const float gym = g[q - N], gyp = g[q + N], gzm = g[q - 1], gzp = g[q + 1];
            const float gnx = g[q + 2 * NN2];  // x + 2 <= N - 1
            const float gmv = STREAM ? __builtin_nontemporal_load(gm + q) : gm[q];
            const float v = leapfrog(gxm[c], gxp[c], gym, gyp, gzm, gzp, gc[c], gmv, p, rhh);
            if (on[c])
            {
                if constexpr (STREAM)
                    __builtin_nontemporal_store(v, gp + q);
                else
                    gp[q] = v;
            }
            gxm[c] = gc[c];
            gc[c] = gxp[c];
            gxp[c] = gnx;
        }
        me += NN2;
    }
}

// Marched-interior layout: tiles of MTY x MTZ columns times chunks of xch planes, tile index z
// fastest, then y, then the x chunk; n_tiles of them, launched as n_blocks (a multiple of 8).
struct MarchShape
{
    int ntz, nty, xch, n_tiles, n_blocks;
};

template <bool STREAM>
__global__ __launch_bounds__(MBLK) void k_fdtd_march(float *__restrict__ grid3, FdtdParams p,
                                                     const StepState *__restrict__ st, MarchShape ms,
                                                     const int *__restrict__ skip)
{
    if (skip && *skip)
        return;
    const int N = p.N;
    const size_t nn = (size_t)N * N * N;
    const int t = st->t;
    // blocks go to the 8 XCDs in turn; give each XCD a contiguous run of tiles so that
    // neighbouring tiles (and their shared halo rows) meet in one L2
    const int b = blockIdx.x, per = ms.n_blocks >> 3;
    const int tile = (b & 7) * per + (b >> 3);
    if (tile >= ms.n_tiles)
        return;
    const int tz = tile % ms.ntz, r = tile / ms.ntz;
    const int ty = r % ms.nty, xc = r / ms.nty;
    const int z0 = tz * MTZ + (int)(threadIdx.x & 63);
    const int y = 2 + ty * MTY + (int)(threadIdx.x >> 6);
    if (y > N - 3 || z0 > N - 3)
        return;
    const int x0 = 2 + xc * ms.xch;
    const int x1 = min(x0 + ms.xch, N - 2);
    march_columns<STREAM>(level(grid3, t, 0, nn), level(grid3, t, -1, nn), level(grid3, t, 1, nn), N, x0, x1, y, z0, p);
}

// The FDTD of one scene alone: the interior blocks, then the ABC shell
__global__ __launch_bounds__(BLK) void k_fdtd_abc(float *__restrict__ grid3, FdtdParams p, const StepState *__restrict__ st,
                                                  int nb_inner, const int *__restrict__ skip, StatusOut f)
{
    copy_status(f);
    if (skip && *skip)
        return;
    fdtd_block(grid3, p, st->t, (int)blockIdx.x, nb_inner);
}

// Interior of a small grid as LDS-staged 2.5D tiles: a block of TY x TZ threads owns TY x TZ
// (y, z) columns of one chunk of x planes and marches them along x. Per plane the block stages
// the level-t values of its tile plus a one-cell halo in y and z in LDS (double buffered), so
// each level-t value comes from memory about once ((TY+2)(TZ+2) / (TY TZ) with the halo); the
// x-neighbours stay in registers. Threads outside 2..N-3 only help with the staging. The
// update is the same leapfrog on the same seven values, so the results equal the one thread
// per cell kernel's bit for bit.
template <int TY, int TZ>
__device__ __forceinline__ void tile_march(float *__restrict__ grid3, const FdtdParams &p, int t, int tile, int xch,
                                           float *__restrict__ lds)
{
    constexpr int LY = TY + 2, LZ = TZ + 2, LN = LY * LZ, NT = TY * TZ;
    const int N = p.N, M = N - 4;
    const double rhh = uniform_rcp(p.hh);
    const size_t nn = (size_t)N * N * N;
    const float *__restrict__ g = level(grid3, t, 0, nn);
    const float *__restrict__ gm = level(grid3, t, -1, nn);
    float *__restrict__ gp = level(grid3, t, 1, nn);
    const int ntz = (M + TZ - 1) / TZ, nty = (M + TY - 1) / TY;
    const int tz = tile % ntz, r = tile / ntz;
    const int ty = r % nty, xc = r / nty;
    const int y0 = 2 + ty * TY, z0 = 2 + tz * TZ;
    const int x0 = 2 + xc * xch, x1 = min(x0 + xch, N - 2);
    const int tid = threadIdx.x;
    const int ly = tid / TZ, lz = tid % TZ;
    const int y = y0 + ly, z = z0 + lz;
    const bool on = y <= N - 3 && z <= N - 3;
    const int me_l = (ly + 1) * LZ + lz + 1;
    // stage plane x (tile plus halo, clamped into the grid) into buf
    auto stage = [&](int x, float *buf) {
        const float *pl = g + (size_t)x * N * N;
        for (int i = tid; i < LN; i += NT)
        {
            const int gy = min(max(y0 - 1 + i / LZ, 0), N - 1), gz = min(max(z0 - 1 + i % LZ, 0), N - 1);
            buf[i] = pl[gy * N + gz];
        }
    };
    float *cur = lds, *nxt = lds + LN;
    stage(x0, cur);
    const int yy = on ? y : 2, zz = on ? z : 2;
    float gxm = g[lin3(x0 - 1, yy, zz, N)];
    __syncthreads();
    float gc = cur[me_l];
    for (int x = x0; x < x1; x++)
    {
        stage(x + 1, nxt);  // x + 1 <= N - 2: inside the grid
        const int q = lin3(x, yy, zz, N);
        const float gmv = gm[q];
        __syncthreads();
        const float gxp = nxt[me_l];
        const float v = leapfrog(gxm, gxp, cur[me_l - LZ], cur[me_l + LZ], cur[me_l - 1], cur[me_l + 1], gc, gmv, p, rhh);
        if (on)
            gp[q] = v;
        gxm = gc;
        gc = gxp;
        __syncthreads();  // every thread is done with cur before it is staged again
        float *tmp = cur;
        cur = nxt;
        nxt = tmp;
    }
}

template <int TY, int TZ>
__global__ __launch_bounds__(TY *TZ) void k_batch_tile(const FdtdScene *__restrict__ ds, BatchMap m)
{
    __shared__ float lds[2 * (TY + 2) * (TZ + 2)];
    int sc, lb;
    if (!map_block(m, (int)blockIdx.x, sc, lb))
        return;
    const FdtdScene d = scene_desc(ds, sc);
    tile_march<TY, TZ>(d.grid3, d.p, d.st->t, lb, d.xch, lds);
}

// the ABC shell of every scene, plus the interior of the scenes stepped one thread per cell
__global__ __launch_bounds__(BLK) void k_batch_fdtd(const FdtdScene *__restrict__ ds, BatchMap m)
{
    int sc, lb;
    if (!map_block(m, (int)blockIdx.x, sc, lb))
        return;
    const FdtdScene d = scene_desc(ds, sc);
    fdtd_block(d.grid3, d.p, d.st->t, lb, d.nb_inner);
}

// get_damp (fdtd.cu:162-169)
__device__ inline float pml_damp(const FdtdParams &p, int x, int y, int z)
{
    const int N = p.N, w = p.pml;
    if (x < w || x >= N - w || y < w || y >= N - w || z < w || z >= N - w)
        return p.damp;
    return 0.0f;
}

// pml_step_kernel (fdtd.cu:179-232); PML state: 6 floats per cell (v1[3], v2[3]) per level
__global__ __launch_bounds__(BLK) void k_fdtd_pml(float *__restrict__ grid3, float *__restrict__ pml3, FdtdParams p,
                                                  const StepState *__restrict__ st, const int *__restrict__ skip)
{
    if (skip && *skip)
        return;
    const int N = p.N;
    const size_t nn = (size_t)N * N * N;
    const int t = st->t;
    const float *g = level(grid3, t, 0, nn);
    const float *gm = level(grid3, t, -1, nn);
    float *gp = level(grid3, t, 1, nn);
    const int l0 = ((t % 3) + 3) % 3, l1 = (((t + 1) % 3) + 3) % 3;
    const float *P = pml3 + (size_t)l0 * nn * 6;
    float *Pn = pml3 + (size_t)l1 * nn * 6;
    const int S = N - 2;
    const long long idx = (long long)blockIdx.x * BLK + threadIdx.x;
    if (idx < (long long)S * S * S)
    {
        const int x = 1 + (int)(idx / (S * S));
        const int rem = (int)(idx % (S * S));
        const int y = 1 + rem / S, z = 1 + rem % S;
        const int co[3] = {x, y, z};
        const int strd[3] = {N * N, N, 1};
        int sg[3];
#pragma unroll
        for (int i = 0; i < 3; i++)
            sg[i] = co[i] > N / 2 ? 1 : -1;
        const float cd = pml_damp(p, x, y, z);
        const int me = lin3(x, y, z, N);
        const float c = p.c, h = p.h, dt = p.dt;
        auto dmp = [&](int i, int d) {
            int q[3] = {x, y, z};
            q[i] += d;
            return pml_damp(p, q[0], q[1], q[2]);
        };
        float rhs = 0;
#pragma unroll
        for (int i = 0; i < 3; i++)
        {
            rhs += 1 / (h * h) * (g[me + strd[i]] - 2 * g[me] + g[me - strd[i]]);
            rhs += 1 / h *
                   (cd * P[(size_t)(me + sg[i] * strd[i]) * 6 + 3 + i] -
                    dmp(i, -sg[i]) * P[(size_t)(me - sg[i] * strd[i]) * 6 + i]);
        }
        gp[me] = g[me] * 2 - gm[me] + c * c * dt * dt * rhs;
        if (cd != 0)
        {
#pragma unroll
            for (int i = 0; i < 3; i++)
            {
                float r = 0;
                r += -1.0f / 2.0f * (dmp(i, -sg[i]) * P[(size_t)(me - sg[i] * strd[i]) * 6 + i] + cd * P[(size_t)me * 6 + i]);
                r += -1.0f / (h * 2.0f) * (g[me + sg[i] * strd[i]] - g[me - sg[i] * strd[i]]);
                Pn[(size_t)me * 6 + i] = P[(size_t)me * 6 + i] + c * dt * r;
            }
#pragma unroll
            for (int i = 0; i < 3; i++)
            {
                float r = 0;
                r += -1.0f / 2.0f *
                     (dmp(i, -sg[i]) * P[(size_t)me * 6 + 3 + i] + cd * P[(size_t)(me + sg[i] * strd[i]) * 6 + 3 + i]);
                r += -1.0f / (h * 2.0f) * (g[me + sg[i] * strd[i]] - g[me - sg[i] * strd[i]]);
                Pn[(size_t)me * 6 + 3 + i] = P[(size_t)me * 6 + 3 + i] + c * dt * r;
            }
        }
    }
}

}  // namespace

// (TY, TZ) of the tile variants (FdtdVariant::Tile*)
static void tile_shape(int variant, int &ty, int &tz)
{
    switch (variant)
    {
    case 1: ty = 8, tz = 64; break;
    case 2: ty = 16, tz = 32; break;
    case 3: ty = 4, tz = 64; break;
    default: ty = 8, tz = 32; break;
    }
}

int fdtd_shell_blocks(int N)
{
    const long long S = N - 2;
    const long long zt = (S - 2 + 15) / 16;
    const long long fxy = 2 * S * S + 2 * (S - 2) * S, fz = 2 * zt * zt * 256;
    return (int)((fxy + BLK - 1) / BLK) + 8 * (int)((fz + 8LL * BLK - 1) / (8LL * BLK));
}

int fdtd_inner_blocks(int N)
{
    const long long M = N - 4;
    return (int)(((M + XC - 1) / XC) * ((M * M + BLK - 1) / BLK));
}

int fdtd_tile_blocks(int N, int variant, int &xch)
{
    int ty, tz;
    tile_shape(variant, ty, tz);
    const int M = N - 4;
    const long long cols = (long long)((M + ty - 1) / ty) * ((M + tz - 1) / tz);
    // chunks of at least 8 planes, enough tiles that a scene alone spreads over the CUs
    const long long nxc = std::max<long long>(1, std::min<long long>((M + 7) / 8, (512 + cols - 1) / cols));
    xch = (int)((M + nxc - 1) / nxc);
    return (int)(cols * ((M + xch - 1) / xch));
}

hipError_t launch_batch_fdtd(const FdtdScene *ds, const BatchMap &m, hipStream_t s)
{
    k_batch_fdtd<<<8 * m.per, BLK, 0, s>>>(ds, m);
    return hipGetLastError();
}

hipError_t launch_batch_tile(int variant, const FdtdScene *ds, const BatchMap &m, hipStream_t s)
{
    switch (variant)
    {
    case 1: k_batch_tile<8, 64><<<8 * m.per, 8 * 64, 0, s>>>(ds, m); break;
    case 2: k_batch_tile<16, 32><<<8 * m.per, 16 * 32, 0, s>>>(ds, m); break;
    case 3: k_batch_tile<4, 64><<<8 * m.per, 4 * 64, 0, s>>>(ds, m); break;
    default: k_batch_tile<8, 32><<<8 * m.per, 8 * 32, 0, s>>>(ds, m); break;
    }
    return hipGetLastError();
}

hipError_t launch_fdtd_march(float *grid3, const FdtdParams &p, const StepState *st, const int *skip, hipStream_t s,
                             int &nb_inner)
{
    const int N = p.N;
    const long long M = N - 4;
    nb_inner = fdtd_inner_blocks(N);
    if (M < kMarchMin)
        return hipSuccess;
    // about 2048 tiles or more; chunks of at least 16 planes (each chunk re-reads 2 planes)
    MarchShape ms{};
    ms.ntz = (N - 3) / MTZ + 1;  // z tiles [MTZ tz, MTZ tz + MTZ) up to z = N - 3
    ms.nty = (int)((M + MTY - 1) / MTY);
    const long long cols = (long long)ms.ntz * ms.nty;
    const long long nxc = std::max<long long>(1, (2048 + cols - 1) / cols);
    ms.xch = (int)std::max<long long>(16, (M + nxc - 1) / nxc);
    ms.n_tiles = (int)(cols * ((M + ms.xch - 1) / ms.xch));
    ms.n_blocks = (ms.n_tiles + 7) / 8 * 8;
    if (12LL * N * N * N > kStreamBytes)
        k_fdtd_march<true><<<ms.n_blocks, MBLK, 0, s>>>(grid3, p, st, ms, skip);
    else
        k_fdtd_march<false><<<ms.n_blocks, MBLK, 0, s>>>(grid3, p, st, ms, skip);
    nb_inner = 0;
    return hipGetLastError();
}

hipError_t launch_fdtd(float *grid3, float *pml3, const FdtdParams &p, const StepState *st, hipStream_t s,
                       const int *skip, const StatusOut *status)
{
    const int N = p.N;
    if (p.pml > 0)
    {
        long long cells = (long long)(N - 2) * (N - 2) * (N - 2);
        int nb = (int)((cells + BLK - 1) / BLK);
        k_fdtd_pml<<<nb, BLK, 0, s>>>(grid3, pml3, p, st, skip);
        return hipGetLastError();
    }
    int nb_inner = 0;
    const hipError_t e = launch_fdtd_march(grid3, p, st, skip, s, nb_inner);
    if (e != hipSuccess)
        return e;
    k_fdtd_abc<<<nb_inner + fdtd_shell_blocks(N), BLK, 0, s>>>(grid3, p, st, nb_inner, skip,
                                                              status ? *status : StatusOut{});
    return hipGetLastError();
}

}  // namespace pppm_amd
