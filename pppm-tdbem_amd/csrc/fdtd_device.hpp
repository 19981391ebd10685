// Device code of the FDTD shared by the launches that step it (fdtd.hip: alone or marched;
// step.hip: beside the far-field gather): the leapfrog update of the interior and the first-order
// absorbing boundary.
#pragma once
#include "divide.hpp"
#include "internal.hpp"

namespace pppm_amd
{

constexpr int BLK = 256;  // threads of an FDTD block

// the launch's last block writes the mesh update's status block to the host, whether or not the
// launch then steps: an update that raised an error is reported too
__device__ inline void copy_status(const StatusOut &f)
{
    if (f.host && blockIdx.x == gridDim.x - 1 && (int)threadIdx.x < f.n)
        f.host[threadIdx.x] = f.status[threadIdx.x];
}

__device__ inline float *level(float *g3, int t, int rel, size_t nn)
{
    int l = ((t + rel) % 3 + 3) % 3;
    return g3 + (size_t)l * nn;
}

// Solve4x4Linear (fdtd.cu:36-86): cofactor inverse in FP32, FP64 reciprocal of the determinant.
__device__ inline void solve4(const float a[4][4], const float b[4], float res[4])
{
    float s0 = a[0][0] * a[1][1] - a[1][0] * a[0][1];
    float s1 = a[0][0] * a[1][2] - a[1][0] * a[0][2];
    float s2 = a[0][0] * a[1][3] - a[1][0] * a[0][3];
    float s3 = a[0][1] * a[1][2] - a[1][1] * a[0][2];
    float s4 = a[0][1] * a[1][3] - a[1][1] * a[0][3];
    float s5 = a[0][2] * a[1][3] - a[1][2] * a[0][3];
    float c5 = a[2][2] * a[3][3] - a[3][2] * a[2][3];
    float c4 = a[2][1] * a[3][3] - a[3][1] * a[2][3];
    float c3 = a[2][1] * a[3][2] - a[3][1] * a[2][2];
    float c2 = a[2][0] * a[3][3] - a[3][0] * a[2][3];
    float c1 = a[2][0] * a[3][2] - a[3][0] * a[2][2];
    float c0 = a[2][0] * a[3][1] - a[3][0] * a[2][1];
    float invdet = (float)(1.0 / (double)(s0 * c5 - s1 * c4 + s2 * c3 + s3 * c2 - s4 * c1 + s5 * c0));
    float inv[4][4];
    inv[0][0] = (a[1][1] * c5 - a[1][2] * c4 + a[1][3] * c3) * invdet;
    inv[0][1] = (-a[0][1] * c5 + a[0][2] * c4 - a[0][3] * c3) * invdet;
    inv[0][2] = (a[3][1] * s5 - a[3][2] * s4 + a[3][3] * s3) * invdet;
    inv[0][3] = (-a[2][1] * s5 + a[2][2] * s4 - a[2][3] * s3) * invdet;
    inv[1][0] = (-a[1][0] * c5 + a[1][2] * c2 - a[1][3] * c1) * invdet;
    inv[1][1] = (a[0][0] * c5 - a[0][2] * c2 + a[0][3] * c1) * invdet;
    inv[1][2] = (-a[3][0] * s5 + a[3][2] * s2 - a[3][3] * s1) * invdet;
    inv[1][3] = (a[2][0] * s5 - a[2][2] * s2 + a[2][3] * s1) * invdet;
    inv[2][0] = (a[1][0] * c4 - a[1][1] * c2 + a[1][3] * c0) * invdet;
    inv[2][1] = (-a[0][0] * c4 + a[0][1] * c2 - a[0][3] * c0) * invdet;
    inv[2][2] = (a[3][0] * s4 - a[3][1] * s2 + a[3][3] * s0) * invdet;
    inv[2][3] = (-a[2][0] * s4 + a[2][1] * s2 - a[2][3] * s0) * invdet;
    inv[3][0] = (-a[1][0] * c3 + a[1][1] * c1 - a[1][2] * c0) * invdet;
    inv[3][1] = (a[0][0] * c3 - a[0][1] * c1 + a[0][2] * c0) * invdet;
    inv[3][2] = (-a[3][0] * s3 + a[3][1] * s1 - a[3][2] * s0) * invdet;
    inv[3][3] = (a[2][0] * s3 - a[2][1] * s1 + a[2][2] * s0) * invdet;
#pragma unroll
    for (int i = 0; i < 4; i++)
    {
        float r = 0;
#pragma unroll
        for (int j = 0; j < 4; j++)
            r += inv[i][j] * b[j];
        res[i] = r;
    }
}

// ab_condition_solve (fdtd.cu:88-137) for one shell cell
__device__ inline void abc_cell(float *g, const float *gm, float *gp, int N, int i, int j, int k, const FdtdParams &p)
{
    const int co[3] = {i, j, k};
    int judge[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
        judge[d] = -((int)(co[d] == 1)) + ((int)(co[d] == N - 2));
    const int strd[3] = {N * N, N, 1};
    const int me = lin3(i, j, k, N);
    const float dt = p.dt, h = p.h, c = p.c;
    float a[4][4], b[4];
    float coef = c * c * dt * dt / (h * h);
    a[3][3] = 1;
#pragma unroll
    for (int d = 0; d < 3; d++)
        a[3][d] = -coef * (float)(judge[d] != 0);
    const float gc = g[me], gmc = gm[me];
    b[3] = -gmc + 2 * gc - coef * (6 * gc);
#pragma unroll
    for (int d = 0; d < 3; d++)
        b[3] += coef * g[me + strd[d]] * (float)(judge[d] <= 0) + coef * g[me - strd[d]] * (float)(judge[d] >= 0);
    float coef1 = 1 / (dt * dt), coef2 = c / (2 * h * dt), coef3 = -(c * c) / (2 * h * h);
#pragma unroll
    for (int idx = 0; idx < 3; idx++)
    {
        const int x = idx, y = (idx + 1) % 3, z = (idx + 2) % 3;
        a[idx][3] = coef1;
        a[idx][x] = coef2;
        a[idx][y] = coef3 * (float)(judge[y] != 0);
        a[idx][z] = coef3 * (float)(judge[z] != 0);
        b[idx] = -coef1 * (gmc - 2 * gc) +
                 -coef2 * (g[me + strd[x]] * (float)(-(int)(judge[x] < 0)) +
                           g[me - strd[x]] * (float)(-(int)(judge[x] > 0)) + gm[me + strd[x]] * (float)(-judge[x]) +
                           gm[me - strd[x]] * (float)judge[x]) +
                 -coef3 * (g[me + strd[y]] * (float)(judge[y] <= 0) + g[me - strd[y]] * (float)(judge[y] >= 0) +
                           g[me + strd[z]] * (float)(judge[z] <= 0) + g[me - strd[z]] * (float)(judge[z] >= 0) -
                           4 * gc);
    }
    float r[4];
    solve4(a, b, r);
    gp[me] = r[3];
#pragma unroll
    for (int d = 0; d < 3; d++)
        if (judge[d] != 0)
            g[me + judge[d] * strd[d]] = r[d];
}

// Leapfrog update of one interior cell from its six neighbours, in the reference's FP64
// operation order: sum x-, x+, y-, y+, z-, z+, then -6 * centre; / h^2; 2 p + coef lap - p_prev.
// rhh = uniform_rcp(p.hh), formed once per thread: an FP32-range sum over the square of an FP32
// value stays far from FP64's exponent limits.
__device__ __forceinline__ float leapfrog(float xm, float xp, float ym, float yp, float zm, float zp, float gc,
                                          float gmv, const FdtdParams &p, double rhh)
{
    double sum = 0;
    sum += xm;
    sum += xp;
    sum += ym;
    sum += yp;
    sum += zm;
    sum += zp;
    sum -= 6 * gc;
    const double lap = shared_div(sum, p.hh, rhh);
    double v = 2 * gc;
    v += p.coef * lap;
    v += -gmv;
    return (float)v;
}

// Interior cells per thread of the thread-per-column path: XC consecutive x planes
constexpr int XC = 4;

// Interior columns (blocks [0, nb_inner)) and the ABC shell (the remaining blocks); nb_inner = 0
// when the interior is marched by another kernel. blk: the block's index within this scene's
// launch (or its share of a batched launch). An interior block covers 256 consecutive (y, z)
// cells of one chunk of XC x planes (a chunk takes ceil((N-4)^2 / 256) blocks; every index is
// 32-bit); each thread loads the XC + 2 values of its column, the y / z neighbours and the
// previous level of its XC cells before it writes any of them, so the loads of XC cells are in
// flight together.
__device__ __forceinline__ void fdtd_block(float *__restrict__ grid3, const FdtdParams &p, int t, int blk,
                                           int nb_inner)
{
    const int N = p.N;
    const size_t nn = (size_t)N * N * N;
    float *g = level(grid3, t, 0, nn);
    const float *gm = level(grid3, t, -1, nn);
    float *gp = level(grid3, t, 1, nn);
    if (blk < nb_inner)
    {
        const unsigned M = N - 4, MM = M * M;
        const unsigned bpp = (MM + BLK - 1) / BLK;
        const unsigned xb = (unsigned)blk / bpp;
        const unsigned q = ((unsigned)blk - xb * bpp) * BLK + threadIdx.x;
        if (q < MM)
        {
            const unsigned yq = q / M;
            const int y = 2 + (int)yq, z = 2 + (int)(q - yq * M), x0 = 2 + (int)xb * XC;
            const int NN2 = N * N;
            const double rhh = uniform_rcp(p.hh);
            const int c0 = lin3(x0, y, z, N);
            float col[XC + 2], ym[XC], yp[XC], zm[XC], zp[XC], pm[XC];
#pragma unroll
            for (int i = 0; i < XC + 2; i++)
                col[i] = g[c0 + (min(x0 - 1 + i, N - 2) - x0) * NN2];  // planes past N - 2 are not used
#pragma unroll
            for (int i = 0; i < XC; i++)
            {
                const int me = c0 + (min(x0 + i, N - 3) - x0) * NN2;
                ym[i] = g[me - N];
                yp[i] = g[me + N];
                zm[i] = g[me - 1];
                zp[i] = g[me + 1];
                pm[i] = gm[me];
            }
#pragma unroll
            for (int i = 0; i < XC; i++)
                if (x0 + i <= N - 3)
                    // laplacian + update in FP64, sum order x-, x+, y-, y+, z-, z+, -6*centre (fdtd.cu:7-33)
                    gp[c0 + i * NN2] = leapfrog(col[i], col[i + 2], ym[i], yp[i], zm[i], zp[i], col[i + 1], pm[i], p, rhh);
        }
    }
    else
    {
        const int S = N - 2;
        // z faces in 16 x 16 tiles of (x, y), padded: a block's cells share their neighbour rows
        const int zt = (S - 2 + 15) / 16;
        const int fx = 2 * S * S, fy = 2 * (S - 2) * S, fz = 2 * zt * zt * 256;
        // blocks [nb_inner, nb_inner + nb_fxy): the x and y faces (rows along z, coalesced);
        // the rest: the z faces, one cell per row, so their blocks are handed to the XCDs in
        // contiguous runs of x planes and a plane's rows meet its neighbours' in one L2
        const int b = blk - nb_inner;
        const int nb_fxy = (fx + fy + BLK - 1) / BLK;
        int idx;
        if (b < nb_fxy)
        {
            idx = b * BLK + (int)threadIdx.x;
            if (idx >= fx + fy)
                idx = -1;
        }
        else
        {
            const int bz = b - nb_fxy, per = (fz + 8 * BLK - 1) / (8 * BLK);
            idx = fx + fy + ((bz & 7) * per + (bz >> 3)) * BLK + (int)threadIdx.x;
        }
        int i = -1, j = 0, k = 0;
        if (idx >= fx + fy + fz)
            idx = -1;
        if (idx < 0)
            ;
        else if (idx < fx)
        {
            const int side = idx / (S * S);
            const int r = idx - side * (S * S);
            i = side ? N - 2 : 1;
            j = 1 + r / S;
            k = 1 + r % S;
        }
        else if ((idx -= fx) < fy)
        {
            const int side = idx / ((S - 2) * S);
            const int r = idx - side * ((S - 2) * S);
            j = side ? N - 2 : 1;
            i = 2 + r / S;
            k = 1 + r % S;
        }
        else if ((idx -= fy) < fz)
        {
            const int side = idx / (zt * zt * 256);
            const int r = idx - side * (zt * zt * 256);
            const int tile = r >> 8, w = r & 255;
            k = side ? N - 2 : 1;
            i = 2 + (tile / zt) * 16 + (w >> 4);
            j = 2 + (tile % zt) * 16 + (w & 15);
            if (i > N - 3 || j > N - 3)
                i = -1;
        }
        if (i >= 0)
            abc_cell(g, gm, gp, N, i, j, k, p);
    }
}

}  // namespace pppm_amd
