// Modal sound source of a rigid body on the GPU (the C ABI's pppm_modal_*).
//
// Reference behaviour: ModalInfo::SetCoeffs (src/utils/RigidBody.cu:11-27), MatrixVertToTri
// (RigidBody.cu:206-230), the IIR recursion of CalculateIIR_ (RigidBody.cu:282-291) and
// update_surf_acc_kernel (RigidBody.cu:240-250). The reference steps the oscillators on the
// host one sample at a time and launches one surface-acceleration kernel per sample; here a
// call covers a block of samples: one thread per mode runs its oscillator recursion through the
// block, one thread per (mode, sample) forms the modal accelerations Q from the displacements,
// then the matrix cores form the surface accelerations of tiles of 128 triangles by 64 or 128
// samples, one mode at a time. Every value keeps the reference's FP32 operations and order
// (host-side arithmetic of the oscillators uncontracted, the device sum as fused multiply-adds).
//
// Layout: the surface matrix is stored mode-major, Mt[i][t], so the accelerations stream it with
// coalesced loads; Q (modal accelerations) is mode-major too, Q[i][s] with a padded row stride,
// so a wave reads the values of its samples as one contiguous run.
#include "internal.hpp"

#include <cmath>
#include <string>
#include <vector>

#include "pppm_hip.h"

namespace pppm_amd
{

namespace
{
constexpr int MB = 256;
constexpr int SPT = 128;  // most samples a block of the acceleration kernel takes; q's rows are padded to it

// MatrixVertToTri: M(t, i) = dot((u(v0) + u(v1) + u(v2)) / 3, n_t), u(v) = rows 3v..3v+2 of
// column i of the eigenvector matrix; written mode-major
__global__ __launch_bounds__(MB) void k_modal_surface(const float *__restrict__ eig, int nmodes,
                                                      const int *__restrict__ tris, const float *__restrict__ normals,
                                                      int nt, int ldm, float *__restrict__ mt)
{
    const long long e = (long long)blockIdx.x * MB + threadIdx.x;
    if (e >= (long long)ldm * nmodes)
        return;
    const int t = (int)(e % ldm), i = (int)(e / ldm);
    if (t >= nt)
    {
        mt[e] = 0.0f;
        return;
    }
    const int v[3] = {tris[3 * t], tris[3 * t + 1], tris[3 * t + 2]};
    float sx = eig[(size_t)(3 * v[0]) * nmodes + i] + eig[(size_t)(3 * v[1]) * nmodes + i];
    float sy = eig[(size_t)(3 * v[0] + 1) * nmodes + i] + eig[(size_t)(3 * v[1] + 1) * nmodes + i];
    float sz = eig[(size_t)(3 * v[0] + 2) * nmodes + i] + eig[(size_t)(3 * v[1] + 2) * nmodes + i];
    sx = (sx + eig[(size_t)(3 * v[2]) * nmodes + i]) / 3.0f;
    sy = (sy + eig[(size_t)(3 * v[2] + 1) * nmodes + i]) / 3.0f;
    sz = (sz + eig[(size_t)(3 * v[2] + 2) * nmodes + i]) / 3.0f;
    mt[e] = sx * normals[3 * t] + sy * normals[3 * t + 1] + sz * normals[3 * t + 2];
}

// Barrier for what the waves hand on in LDS: global loads and stores stay in flight over it
__device__ __forceinline__ void lds_barrier()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "workgroup", "local");
    __builtin_amdgcn_s_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "workgroup", "local");
}

// One thread per mode: q0 = c1 q1 + c2 q2 + c3 f; (q3, q2, q1) <- (q2, q1, q0), for each sample
// of the block in order. Only the recursion is sequential, so one wave keeps to it: a block holds
// 64 modes, and while the stepping wave runs window w of FD samples from LDS into LDS, the
// loading waves have the forces of windows w + 1 .. w + NL in flight and the storing wave writes
// the displacements of window w - 1, whole lines of the modes' rows. The barrier leaves those loads
// and stores in flight. 200 modes and 1024 samples: 39 us with one loading wave and a barrier that
// drains memory, 33 us so. Row layout (stride ldp, a
// multiple of 4): [2] = q2 and [3] = q1 of the state at the start of the call, [4 + s] = q0 of
// sample s; the last four entries' part past ns is written 0.
constexpr int FD = 32;
constexpr int NL = 6;

template <bool GUARD>
__device__ __forceinline__ void iir_window(const float (*__restrict__ sf)[64], float (*__restrict__ so)[65], int lane,
                                           int n, float c1, float c2, float c3, float &q1, float &q2, float &q3)
{
#pragma unroll
    for (int k = 0; k < FD; k++)
    {
        float out = 0.0f;
        if (!GUARD || k < n)
        {
            const float q0 = c1 * q1 + c2 * q2 + c3 * sf[k][lane];
            q3 = q2;
            q2 = q1;
            q1 = q0;
            out = q0;
        }
        so[k][lane] = out;
    }
}

__global__ __launch_bounds__(64 * (2 + NL)) void k_modal_iir(const float *__restrict__ coeff, float *__restrict__ state,
                                                             int nmodes, const float *__restrict__ forces, int ns,
                                                             float *__restrict__ qp, int ldp)
{
    __shared__ float sf[2][FD][64];
    __shared__ float so[2][FD][65];
    const int lane = threadIdx.x & 63;
    const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
    const int loader = wave - 2;  // -2: the stepping wave, -1: the storing wave
    const int i0 = blockIdx.x * 64, i = i0 + lane;
    const bool live = i < nmodes;
    const int nw = (ns + FD - 1) / FD;
    float v[FD];
    const float *col = forces + min(i, nmodes - 1);
    auto load = [&](int w) {  // entries past the last sample or mode load the last one (not used)
#pragma unroll
        for (int k = 0; k < FD; k++)
            v[k] = col[(size_t)min(w * FD + k, ns - 1) * nmodes];
    };
    // window w into its LDS buffer (loaded NL windows ago), then the loads of window w + NL
    auto pass_on = [&](int w) {
#pragma unroll
        for (int k = 0; k < FD; k++)
            sf[w & 1][k][lane] = v[k];
        if (w + NL < nw)
            load(w + NL);
    };
    float c1 = 0, c2 = 0, c3 = 0, q1 = 0, q2 = 0, q3 = 0;
    if (loader >= 0)
    {
        if (loader < nw)
            load(loader);
        if (loader == 0)
            pass_on(0);
    }
    else if (loader == -2 && live)
    {
        c1 = coeff[3 * i], c2 = coeff[3 * i + 1], c3 = coeff[3 * i + 2];
        q1 = state[3 * i], q2 = state[3 * i + 1], q3 = state[3 * i + 2];
        qp[(size_t)i * ldp + 2] = q2;
        qp[(size_t)i * ldp + 3] = q1;
    }
    lds_barrier();
    for (int w = 0; w <= nw; w++)
    {
        if (loader >= 0)
        {
            if (w + 1 < nw && loader == (w + 1) % NL)
                pass_on(w + 1);
        }
        else if (loader == -2)
        {
            if ((w + 1) * FD <= ns)
                iir_window<false>(sf[w & 1], so[w & 1], lane, FD, c1, c2, c3, q1, q2, q3);
            else if (w < nw)
                iir_window<true>(sf[w & 1], so[w & 1], lane, ns - w * FD, c1, c2, c3, q1, q2, q3);
        }
        else if (w > 0)
        {
            const int k = 4 * (lane & 7), s = (w - 1) * FD + k;
#pragma unroll
            for (int r = 0; r < 64; r += 8)
            {
                const int m = r + (lane >> 3);
                const float(*o)[65] = so[(w - 1) & 1];
                if (i0 + m < nmodes && s < ns)
                    *(float4 *)(qp + (size_t)(i0 + m) * ldp + 4 + s) = make_float4(o[k][m], o[k + 1][m], o[k + 2][m], o[k + 3][m]);
            }
        }
        lds_barrier();
    }
    if (loader == -2 && live)
    {
        state[3 * i] = q1;
        state[3 * i + 1] = q2;
        state[3 * i + 2] = q3;
    }
}

// Modal accelerations Q = (q1 + q3 - 2 q2) / (dt dt) after each sample's shift, i.e. from the
// displacements of samples s, s - 2 and s - 1: thread per (mode, sample), Q stored mode-major
// (row stride ldq, a multiple of SPT; entries of the last sample block past ns are written 0).
__global__ __launch_bounds__(MB) void k_modal_q(const float *__restrict__ qp, int ldp, int nmodes, int ns,
                                                int ns_pad, float dt, float *__restrict__ q, int ldq)
{
    const long long e = (long long)blockIdx.x * MB + threadIdx.x;
    if (e >= (long long)nmodes * ns_pad)
        return;
    const int i = (int)(e / ns_pad), s = (int)(e % ns_pad);
    const float *row = qp + (size_t)i * ldp + 2 + s;  // row[0] = q3, row[1] = q2, row[2] = q1
    const float dt2 = dt * dt;
    q[(size_t)i * ldq + s] = s < ns ? (row[2] + row[0] - 2 * row[1]) / dt2 : 0.0f;
}

// acc[s][t] = sum_i Mt[i][t] Q[i][s] in mode order, each term added with one fused multiply-add
// (the reference's device loop `acc += M(t, i) * Q[i]` as its compiler contracts it), on the matrix
// cores: the FP32 32 x 32 x 1 product adds a single term to every element, so a chain of them over
// the modes is the sequential sum, with the same bits.
//
// A block takes 128 triangles by 64 * NS samples, a wave 64 triangles (two blocks of 32 columns) by
// 32 * NS samples (rows; NS products share the triangles' operand, the samples' operand is broadcast
// to both column blocks). Both operands are staged through LDS, KC modes at a time, the next
// modes' 16-byte loads in flight meanwhile; rows are padded (ldm, ldq), so no load needs a guard.
// Samples run fastest over the blocks and each XCD takes a contiguous run of triangles, whose
// matrix stays in its L2. Bound by the matrix cores (55 us at the rate of a large FP32 product)
// and the write of the result. 20480 triangles, 200 modes and 1024 samples (8.4 GFLOP): 151 us as
// vector FMAs with 32 samples a thread, 123 us on the matrix cores with operands straight from
// memory, 100 to 104 us so.
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef float f32x32 __attribute__((ext_vector_type(32)));
constexpr int KC = 16, TT = 128;
template <int NS>
__global__ __launch_bounds__(MB, 4) void k_modal_accs(const float *__restrict__ mt, int ldm, int nt, int nmodes,
                                                   const float *__restrict__ q, int ldq, int ns, int t_tiles, int s_tiles,
                                                   int per, float *__restrict__ accs)
{
    constexpr int TS = 64 * NS;
    __shared__ __align__(16) float sm[2][KC][TT];
    __shared__ __align__(16) float sq[2][KC][TS];
    const int tile = (int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3);
    const int tt = tile / s_tiles, st = tile - tt * s_tiles;
    if (tt >= t_tiles)
        return;
    const int tid = threadIdx.x, lane = tid & 63;
    const int wid = __builtin_amdgcn_readfirstlane(tid >> 6), wt = 64 * (wid & 1), ws = 32 * NS * (wid >> 1);
    const int la = ws + (NS == 2 ? lane : lane & 31), lb = wt + lane;
    f32x4 rm[2], rq[NS];
    auto load = [&](int i0) {  // modes past the last load the last one (not used)
#pragma unroll
        for (int j = 0; j < 2; j++)
        {
            const int e = tid + MB * j, row = min(i0 + e / (TT / 4), nmodes - 1);
            rm[j] = *reinterpret_cast<const f32x4 *>(mt + (size_t)row * ldm + TT * tt + 4 * (e % (TT / 4)));
        }
#pragma unroll
        for (int j = 0; j < NS; j++)
        {
            const int e = tid + MB * j, row = min(i0 + e / (TS / 4), nmodes - 1);
            rq[j] = *reinterpret_cast<const f32x4 *>(q + (size_t)row * ldq + TS * st + 4 * (e % (TS / 4)));
        }
    };
    auto stage = [&](int buf) {
#pragma unroll
        for (int j = 0; j < 2; j++)
        {
            const int e = tid + MB * j;
            *reinterpret_cast<f32x4 *>(&sm[buf][e / (TT / 4)][4 * (e % (TT / 4))]) = rm[j];
        }
#pragma unroll
        for (int j = 0; j < NS; j++)
        {
            const int e = tid + MB * j;
            *reinterpret_cast<f32x4 *>(&sq[buf][e / (TS / 4)][4 * (e % (TS / 4))]) = rq[j];
        }
    };
    f32x32 acc[NS];
#pragma unroll
    for (int n = 0; n < NS; n++)
#pragma unroll
        for (int k = 0; k < 32; k++)
            acc[n][k] = 0.0f;
    auto add = [&](int buf, int k) {
        const float a = sq[buf][k][la], b = sm[buf][k][lb];
        if constexpr (NS == 2)
        {
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, acc[0], 1, 0, 0);
            acc[1] = __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, acc[1], 1, 1, 0);
        }
        else
            acc[0] = __builtin_amdgcn_mfma_f32_32x32x1f32(a, b, acc[0], 0, 0, 0);
    };
    load(0);
    stage(0);
    __syncthreads();
    int i = 0, buf = 0;
    for (; i + KC <= nmodes; i += KC, buf ^= 1)
    {
        load(i + KC);
        __builtin_amdgcn_sched_barrier(0);  // the compiler would issue the loads where they are stored
#pragma unroll
        for (int k = 0; k < KC; k++)
            add(buf, k);
        __builtin_amdgcn_sched_barrier(0);
        stage(buf ^ 1);
        __syncthreads();
    }
    for (int k = 0; k < nmodes - i; k++)
        add(buf, k);
    // lane l holds column l % 32 of each block, rows 8 (v / 4) + 4 (l / 32) + v % 4
#pragma unroll
    for (int n = 0; n < NS; n++)
#pragma unroll
        for (int v = 0; v < 32; v++)
        {
            const int t = TT * tt + wt + 32 * (v >> 4) + (lane & 31);
            const int s = TS * st + ws + 32 * n + 8 * ((v & 15) >> 2) + 4 * (lane >> 5) + (v & 3);
            if (t < nt && s < ns)
                accs[(size_t)s * nt + t] = acc[n][v];
        }
}

template <int NS>
void launch_accs(const float *mt, int ldm, int nt, int nmodes, const float *q, int ldq, int ns, float *accs,
                 hipStream_t stream)
{
    const int t_tiles = (nt + TT - 1) / TT, s_tiles = (ns + 64 * NS - 1) / (64 * NS);
    const int per = (int)(((long long)t_tiles * s_tiles + 7) / 8);
    k_modal_accs<NS><<<8 * per, MB, 0, stream>>>(mt, ldm, nt, nmodes, q, ldq, ns, t_tiles, s_tiles, per, accs);
}

inline unsigned nblocks(long long n) { return (unsigned)(n > 0 ? (n + MB - 1) / MB : 1); }

}  // namespace

// ModalInfo::SetCoeffs in FP32 with the host's libm, as the reference computes it on the host
void modal_coeffs(float eigval, float timestep, float alpha, float beta, float *c123)
{
    const float lambda = eigval;
    const float omega = std::sqrt(lambda);
    const float ksi = (alpha + beta * lambda) / (2 * omega);
    const float omega_prime = omega * std::sqrt(1 - ksi * ksi);
    const float epsilon = std::exp(-ksi * omega * timestep);
    const float sqr_epsilon = epsilon * epsilon;
    const float theta = omega_prime * timestep;
    const float gamma = std::asin(ksi);
    c123[0] = 2 * epsilon * std::cos(theta);
    c123[1] = -sqr_epsilon;
    const float item1 = epsilon * std::cos(theta + gamma);
    const float item2 = sqr_epsilon * std::cos(2 * theta + gamma);
    c123[2] = 2 * (item1 - item2) / (3 * omega * omega_prime);
}

}  // namespace pppm_amd

using namespace pppm_amd;

struct pppm_modal
{
    int nt = 0, nmodes = 0;
    float dt = 0;
    hipStream_t stream = nullptr;
    float *mt = nullptr;      // nmodes rows of ldm (nt rounded up to the acceleration kernel's tiles, 0 past nt)
    int ldm = 0;
    float *coeff = nullptr;   // nmodes x 3
    float *state = nullptr;   // nmodes x 3 (q1, q2, q3)
    float *q = nullptr;       // nmodes x cap_samples (mode-major, row stride cap_samples)
    float *qp = nullptr;      // nmodes x (cap_samples + 4): displacements, two of them from before the call
    float *forces = nullptr;  // staging for host forces, cap_samples x nmodes
    int cap_samples = 0;      // a multiple of SPT
    std::vector<float> coeff_h;
};

namespace
{
int modal_release(pppm_modal *m)
{
    for (float *p : {m->mt, m->coeff, m->state, m->q, m->qp, m->forces})
        if (p)
            (void)hipFree(p);
    m->mt = m->coeff = m->state = m->q = m->qp = m->forces = nullptr;
    return PPPM_OK;
}

#define MCK(x)                                \
    do                                        \
    {                                         \
        if ((x) != hipSuccess)                \
            return PPPM_ERR_HIP;              \
    } while (0)
}  // namespace

extern "C" {

int pppm_modal_create(pppm_modal **out, const float *eigvecs, int nv, int nmodes, const float *eigvals,
                      const int *tris, int nt, const float *normals, float alpha, float beta, float sample_rate,
                      void *hip_stream)
{
    if (!out || !eigvecs || !eigvals || !tris || !normals || nv < 3 || nmodes < 1 || nt < 1 || !(sample_rate > 0) ||
        nt > 65535 * MB)
        return PPPM_ERR_ARG;
    for (int t = 0; t < 3 * nt; t++)
        if (tris[t] < 0 || tris[t] >= nv)
            return PPPM_ERR_ARG;
    *out = nullptr;
    pppm_modal *m = new pppm_modal();
    m->nt = nt;
    m->nmodes = nmodes;
    m->ldm = (nt + TT - 1) / TT * TT;
    m->dt = 1.0f / sample_rate;  // RigidBody::InitIIR_ (RigidBody.cu:192)
    m->stream = (hipStream_t)hip_stream;
    m->coeff_h.resize((size_t)nmodes * 3);
    for (int i = 0; i < nmodes; i++)
        modal_coeffs(eigvals[i], m->dt, alpha, beta, &m->coeff_h[3 * (size_t)i]);
    float *eig = nullptr, *nrm = nullptr;
    int *tri = nullptr;
    auto fail = [&](int rc) {
        for (void *p : {(void *)eig, (void *)nrm, (void *)tri})
            if (p)
                (void)hipFree(p);
        modal_release(m);
        delete m;
        return rc;
    };
    const size_t neig = (size_t)3 * nv * nmodes;
    if (hipMalloc((void **)&m->mt, sizeof(float) * (size_t)m->ldm * nmodes) != hipSuccess ||
        hipMalloc((void **)&m->coeff, sizeof(float) * 3 * (size_t)nmodes) != hipSuccess ||
        hipMalloc((void **)&m->state, sizeof(float) * 3 * (size_t)nmodes) != hipSuccess ||
        hipMalloc((void **)&eig, sizeof(float) * neig) != hipSuccess ||
        hipMalloc((void **)&nrm, sizeof(float) * 3 * (size_t)nt) != hipSuccess ||
        hipMalloc((void **)&tri, sizeof(int) * 3 * (size_t)nt) != hipSuccess)
        return fail(PPPM_ERR_HIP);
    if (hipMemcpyAsync(m->coeff, m->coeff_h.data(), sizeof(float) * 3 * nmodes, hipMemcpyHostToDevice, m->stream) ||
        hipMemsetAsync(m->state, 0, sizeof(float) * 3 * nmodes, m->stream) ||
        hipMemcpyAsync(eig, eigvecs, sizeof(float) * neig, hipMemcpyHostToDevice, m->stream) ||
        hipMemcpyAsync(nrm, normals, sizeof(float) * 3 * nt, hipMemcpyHostToDevice, m->stream) ||
        hipMemcpyAsync(tri, tris, sizeof(int) * 3 * nt, hipMemcpyHostToDevice, m->stream))
        return fail(PPPM_ERR_HIP);
    k_modal_surface<<<nblocks((long long)m->ldm * nmodes), MB, 0, m->stream>>>(eig, nmodes, tri, nrm, nt, m->ldm, m->mt);
    if (hipGetLastError() != hipSuccess || hipStreamSynchronize(m->stream) != hipSuccess)
        return fail(PPPM_ERR_HIP);
    (void)hipFree(eig);
    (void)hipFree(nrm);
    (void)hipFree(tri);
    *out = m;
    return PPPM_OK;
}

int pppm_modal_destroy(pppm_modal *m)
{
    if (!m)
        return PPPM_ERR_ARG;
    if (m->stream)
        (void)hipStreamSynchronize(m->stream);
    modal_release(m);
    delete m;
    return PPPM_OK;
}

int pppm_modal_run(pppm_modal *m, const float *forces, int nsamples, float *accs, int on_device)
{
    if (!m || !forces || !accs || nsamples < 0 || nsamples > (1 << 30))
        return PPPM_ERR_ARG;
    if (nsamples == 0)
        return PPPM_OK;
    if (nsamples > m->cap_samples)
    {
        MCK(hipStreamSynchronize(m->stream));
        for (float **p : {&m->q, &m->qp, &m->forces})
            if (*p)
            {
                (void)hipFree(*p);
                *p = nullptr;
            }
        m->cap_samples = 0;
        const int cap = (int)(((long long)nsamples + SPT - 1) / SPT * SPT);
        MCK(hipMalloc((void **)&m->q, sizeof(float) * (size_t)cap * m->nmodes));
        MCK(hipMalloc((void **)&m->qp, sizeof(float) * (size_t)(cap + 4) * m->nmodes));
        MCK(hipMalloc((void **)&m->forces, sizeof(float) * (size_t)cap * m->nmodes));
        m->cap_samples = cap;
    }
    const float *f = forces;
    if (!on_device)
    {
        MCK(hipMemcpyAsync(m->forces, forces, sizeof(float) * (size_t)nsamples * m->nmodes, hipMemcpyHostToDevice,
                           m->stream));
        f = m->forces;
    }
    const int ldp = m->cap_samples + 4;
    const int ns_pad = (nsamples + SPT - 1) / SPT * SPT;
    k_modal_iir<<<(m->nmodes + 63) / 64, 64 * (2 + NL), 0, m->stream>>>(m->coeff, m->state, m->nmodes, f, nsamples, m->qp, ldp);
    k_modal_q<<<nblocks((long long)m->nmodes * ns_pad), MB, 0, m->stream>>>(m->qp, ldp, m->nmodes, nsamples, ns_pad,
                                                                             m->dt, m->q, m->cap_samples);
    // 128 x 128 tiles where every CU gets two, else 128 x 64: fewer reads of the triangles' operand
    // against twice the blocks to spread. The whole call at 200 modes, smaller / larger tiles: 128
    // tiles (of 128 x 128) 35.7 / 42.1 us, 320 55.7 / 62.6, 448 70.9 / 71.0, 512 75.6 / 75.1, 1024
    // 141 / 137, 2048 265 / 260; beyond the line either can be ahead by how full the last round of
    // blocks is (640 90 / 97, 768 106 / 106, 1280 127 / 130, 1536 200 / 208, 2560 234 / 234)
    const long long tiles = (long long)((m->nt + TT - 1) / TT) * ((nsamples + 127) / 128);
    if (tiles >= 512)
        launch_accs<2>(m->mt, m->ldm, m->nt, m->nmodes, m->q, m->cap_samples, nsamples, accs, m->stream);
    else
        launch_accs<1>(m->mt, m->ldm, m->nt, m->nmodes, m->q, m->cap_samples, nsamples, accs, m->stream);
    MCK(hipGetLastError());
    if (!on_device)
        MCK(hipStreamSynchronize(m->stream));  // the host forces must outlive the copy
    return PPPM_OK;
}

int pppm_modal_state(pppm_modal *m, float *q3)
{
    if (!m || !q3)
        return PPPM_ERR_ARG;
    MCK(hipMemcpyAsync(q3, m->state, sizeof(float) * 3 * m->nmodes, hipMemcpyDeviceToHost, m->stream));
    MCK(hipStreamSynchronize(m->stream));
    return PPPM_OK;
}

int pppm_modal_set_state(pppm_modal *m, const float *q3)
{
    if (!m || !q3)
        return PPPM_ERR_ARG;
    MCK(hipMemcpyAsync(m->state, q3, sizeof(float) * 3 * m->nmodes, hipMemcpyHostToDevice, m->stream));
    MCK(hipStreamSynchronize(m->stream));
    return PPPM_OK;
}

int pppm_modal_surface_matrix(pppm_modal *m, float *host_out)
{
    if (!m || !host_out)
        return PPPM_ERR_ARG;
    std::vector<float> mt((size_t)m->ldm * m->nmodes);
    MCK(hipMemcpyAsync(mt.data(), m->mt, sizeof(float) * mt.size(), hipMemcpyDeviceToHost, m->stream));
    MCK(hipStreamSynchronize(m->stream));
    for (int i = 0; i < m->nmodes; i++)
        for (int t = 0; t < m->nt; t++)
            host_out[(size_t)t * m->nmodes + i] = mt[(size_t)i * m->ldm + t];
    return PPPM_OK;
}

int pppm_modal_coeffs(pppm_modal *m, float *host_out)
{
    if (!m || !host_out)
        return PPPM_ERR_ARG;
    for (size_t k = 0; k < m->coeff_h.size(); k++)
        host_out[k] = m->coeff_h[k];
    return PPPM_OK;
}

}  // extern "C"
