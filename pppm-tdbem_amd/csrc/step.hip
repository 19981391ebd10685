// Per-step near-field kernels: far-field extraction, Dirichlet update, near-field
// correction. Sparse and HBM-bound: no MFMA.
//
// Reference behaviour: solve_fdtd_far_kernel (src/algorithm/pppm.cu:8-51),
// set_neumann_condition_kernel (pppm.cu:206-225), solve_face_far_kernel,
// solve_face_near_kernel and update_dirichlet_kernel (pppm.cu:116-204),
// solve_fdtd_near_kernel (pppm.cu:53-114), LayerWeightHalf::convolution (bem.h:203-213).
//
// Segmented gather with a fixed summation order. A "segment" is a C3 cell (far / near)
// or a triangle (Dirichlet); its pairs are contiguous in a CSR list. Entry w of the wave map
// built with the lists holds the segments whose first pair lies in [64w, 64w+64) and the first
// pair of that range; a wave takes one, two or four entries (gather_gran) and walks their pairs
// in rounds of 64. Four lanes fetch a pair's record and windows and form its 16 terms, the pair's
// lane adds them sequentially (k = 0..15, as the reference's loop) and parks the value in LDS;
// after a chunk of 256 pairs each lane adds the values of its own segment in list order
// (gather_wave). Every sum therefore has the order of a sequential loop, whatever the segment
// lengths, and lanes stay busy across segment boundaries.
//
// What bounds it: the records' HBM stream (without it the far and near gathers of 64 scenes take
// half the time), then the waves' serial start and end. One lane fetching its pair's 64 B rows
// and every lane sweeping all 64 values of a round for its sums issued 620 vector instructions
// and 500 cache accesses per round; now about 230 and 190. 64 scenes together (7.45M face, 2.68M
// cell pairs): Dirichlet 181 -> 166 us, near 99 -> 72 us, far 87 -> 73 us. Fetching a round's
// records one round ahead, or all of a round's loads at once, costs two waves per SIMD and was
// slower (187, 175 us Dirichlet).
//
// Weights: 64 B record per pair (16 x half2 {S_k, D_k}) + float2 scales. History: the
// reference's 32-slot rings (slot = t mod 32), one 128 B line per triangle and field, plus
// per-step windows of the 16 latest values in tap order (one 64 B row per triangle and field)
// from which the gathers read.
//
// Time index: all kernels read t from device memory (StepState), so one captured HIP
// graph replays any step.
#include "fdtd_device.hpp"
#include "internal.hpp"
#include "scene_device.hpp"

#include <algorithm>

namespace pppm_amd
{

namespace
{
constexpr int WPB = 4;            // waves per block
constexpr int TB = WPB * WAVE;    // threads per block

// Workgroups are dealt to the 8 XCDs in turn (block b to XCD b % 8). A gather launch covers
// 8 * per blocks and block b takes virtual block (b % 8) * per + b / 8, so each XCD works on
// one contiguous eighth of the wave range: neighbouring triangles and cells share history
// windows and grid values in that XCD's L2. Waves past a kernel's work do nothing.
__device__ inline int xcd_wave(int per, int wid)
{
    return ((int)(blockIdx.x & 7) * per + (int)(blockIdx.x >> 3)) * WPB + wid;
}

__device__ inline int wave_in_block() { return __builtin_amdgcn_readfirstlane((int)(threadIdx.x >> 6)); }

__device__ inline void wave_sync()
{
    __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
    __builtin_amdgcn_wave_barrier();
    __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// Pairs a wave convolves and parks in LDS before its lanes add them up: enough that the segments
// of a chunk are many and most rounds of 64 full.
constexpr int CH = 4 * WAVE;

// LDS of one wave of a gather: the terms of a round, the values of a chunk
template <class V>
struct GatherLds
{
    float4 term[4 * WAVE];
    V vals[CH];
};

// acc plus vals[0], ..., vals[n - 1], added one at a time in that order (V: float, or float2
// for two sums side by side). Each lane reads its own range: sixteen at a time, then the rest
// by halves, so the wave issues about as many additions as its longest segment has values.
template <int K, class V>
__device__ __forceinline__ void add_run(V &acc, const V *&vals)
{
    V v[K];
#pragma unroll
    for (int i = 0; i < K; i++)
        v[i] = vals[i];
#pragma unroll
    for (int i = 0; i < K; i++)
        acc += v[i];
    vals += K;
}
template <class V>
__device__ __forceinline__ V segment_sum(V acc, const V *vals, int n)
{
    for (; n >= 16; n -= 16)
        add_run<16>(acc, vals);
    if (n & 8)
        add_run<8>(acc, vals);
    if (n & 4)
        add_run<4>(acc, vals);
    if (n & 2)
        add_run<2>(acc, vals);
    if (n & 1)
        add_run<1>(acc, vals);
    return acc;
}

__device__ inline float read_lane(float v, int l) { return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), l)); }
__device__ inline float2 read_lane(float2 v, int l) { return make_float2(read_lane(v.x, l), read_lane(v.y, l)); }

// The segmented gather of one wave over the segments [w0.x, w1.x) and their pairs [w0.y, w1.y):
// chunks of CH pairs are convolved 64 at a time into LDS (g.load: a pair's indices; g.conv: a round); then lane l adds the
// part of segment cs + l that lies in the chunk, in list order, and finished segments are handed
// to g.done. At most one segment is open at a chunk's end; its sum is carried to the next chunk.
// g.early / g.late load what done needs, behind the first and the last round of a chunk.
template <class V, class G>
__device__ __forceinline__ void gather_wave(G &g, const int *__restrict__ start, int2 w0, int2 w1, int lane,
                                            GatherLds<V> &lds)
{
    V *__restrict__ vals = lds.vals;
    int cs = w0.x;
    const int c1 = w1.x, q0 = w0.y, q1 = w1.y;
    V carry{};
    typename G::Index idx = g.load(min(q0 + lane, q1 - 1));
    for (int base = q0; base < q1; base += CH)
    {
        const int end = min(base + CH, q1);
        int s = cs + lane;
        int m0 = s < c1 ? start[s] : q1, m1 = s < c1 ? start[s + 1] : q1 + 1;
        for (int b = base; b < end; b += WAVE)
        {
            // the next round's indices are loaded beside this round's records
            const typename G::Index next = g.load(min(b + WAVE + lane, q1 - 1));
            g.conv(idx, end - b, lane, lds.term, vals + (b - base));
            idx = next;
            if (b == base)
                g.early(s, s < c1 && (m0 < end || end == q1));
        }
        g.late();
        wave_sync();
        for (;;)
        {
            const bool in = s < c1 && (m0 < end || end == q1), fin = in && m1 <= end;
            V acc{};
            if (lane == 0)
                acc = carry;
            if (in)
            {
                const int lo = max(m0, base);
                acc = segment_sum(acc, vals + (lo - base), min(m1, end) - lo);
            }
            if (fin)
                g.done(s, acc);
            const unsigned long long done = __ballot(fin);
            const int nd = (int)__popcll(done);
            carry = V{};
            if (__ballot(in) != done)
                carry = read_lane(acc, nd);  // finished segments are lanes 0 .. nd - 1
            cs += nd;
            if (nd < WAVE || cs >= c1)
                break;
            s = cs + lane;
            m0 = s < c1 ? start[s] : q1;
            m1 = s < c1 ? start[s + 1] : q1 + 1;
            g.early(s, s < c1 && (m0 < end || end == q1));
            g.late();
        }
        wave_sync();
    }
}

// map entries [gran * wave, gran * (wave + 1)) of a gather's wave map: its first segment and pair
__device__ __forceinline__ void wave_range(const int *__restrict__ map, int waves, int gran, int wave, int2 &w0, int2 &w1)
{
    w0 = const_load(reinterpret_cast<const int2 *>(map) + gran * wave);
    w1 = const_load(reinterpret_cast<const int2 *>(map) + min(gran * (wave + 1), waves));
}
__host__ __device__ inline int gran_waves(int waves, int gran) { return (waves + gran - 1) / gran; }

// LayerWeightHalf::convolution (bem.h:203-213) of a round of up to 64 pairs, taps in order, from the
// pair triangles' history windows (row k of a window: the value at t - k, tap k). rec / tri: this
// lane's pair's record and triangle (any valid ones past the round's n pairs). K0: first tap that
// counts. DZERO0: the Dirichlet value of step t is read as 0 (pppm.cu:143). fac (may be null):
// receives D_0 times its scale for pair i at fac[2 * i].
//
// Four lanes share a pair: lane 4 h + q fetches quarter q of the 64 B record and of both windows
// of pairs h, 16 + h, 32 + h and 48 + h, so a load instruction covers whole cache lines (1 KB of
// consecutive records) instead of 16 B of each of 64 rows, and forms the terms of its four taps.
// They pass through LDS to the lane of the pair, which adds all sixteen in order; quarters are
// stored at q ^ (pair / 4 mod 4), which keeps both sides free of bank conflicts.
template <int K0, bool DZERO0>
__device__ __forceinline__ float conv_round(const uint32_t *__restrict__ w16, const float2 *__restrict__ scale, int rec,
                                            int tri, int n, const float *__restrict__ wn, const float *__restrict__ wd,
                                            int lane, float4 *__restrict__ term, float *__restrict__ fac)
{
    const int h = lane >> 2, q = lane & 3;
    const int col = q ^ ((h >> 2) & 3);
    wave_sync();  // the reads of the round before
#pragma unroll
    for (int half = 0; half < 2; half++)
    {
        if (32 * half >= n)
            break;
        uint4 w[2];
        float4 hn[2], hd[2];
        float2 sc[2];
#pragma unroll
        for (int i = 0; i < 2; i++)
        {
            const int src = 32 * half + 16 * i + h;
            const int r = __shfl(rec, src), t = __shfl(tri, src);
            w[i] = reinterpret_cast<const uint4 *>(w16)[4 * (size_t)r + q];
            sc[i] = scale[r];
            hn[i] = reinterpret_cast<const float4 *>(wn)[4 * (size_t)t + q];
            hd[i] = reinterpret_cast<const float4 *>(wd)[4 * (size_t)t + q];
        }
#pragma unroll
        for (int i = 0; i < 2; i++)
        {
            const int pair = 32 * half + 16 * i + h;
            if (DZERO0 && q == 0)
                hd[i].x = 0.0f;
            const uint32_t ww[4] = {w[i].x, w[i].y, w[i].z, w[i].w};
            const float nn[4] = {hn[i].x, hn[i].y, hn[i].z, hn[i].w}, dd[4] = {hd[i].x, hd[i].y, hd[i].z, hd[i].w};
            float v[4];
#pragma unroll
            for (int c = 0; c < 4; c++)
            {
                const float a = -f16_bits_to_f32(ww[c]) * sc[i].x * nn[c];
                const float b = f16_bits_to_f32(ww[c] >> 16) * sc[i].y * dd[c];
                v[c] = a + b;
            }
            term[4 * pair + col] = make_float4(v[0], v[1], v[2], v[3]);
            if (fac && q == 0)
                fac[2 * pair] = f16_bits_to_f32(ww[0] >> 16) * sc[i].y;
        }
    }
    wave_sync();
    float r = 0.0f;
#pragma unroll
    for (int qq = 0; qq < 4; qq++)
    {
        const float4 v = term[4 * lane + (qq ^ ((lane >> 2) & 3))];
        if (qq > 0 || K0 == 0)
            r += v.x;
        r += v.y;
        r += v.z;
        r += v.w;
    }
    return r;
}

// History windows for the gathers of step t: row k of triangle i holds the ring value at t - k, the
// value of tap k. back = 0 when launched before t is advanced (the time step: the values at t do
// not exist yet; the far-field launch writes the Neumann value and the Dirichlet update the
// Dirichlet value into row 0 as into the ring), 1 after it (the phase entry points: the ring
// holds them).
// windows of step t in their half of wn / wd
__device__ __forceinline__ size_t window_base(const SceneStep &d, int t)
{
    return d.win2 && (t & 1) ? (size_t)d.a.nt * STEPS : 0;
}
__device__ __forceinline__ void windows_item(const SceneStep &d, int tn, int i)
{
    if (i >= d.a.nt * STEPS || (d.err && *d.err))
        return;
    const int tri = i / STEPS, k = i % STEPS;
    const int slot = (tn - k) & (RING - 1);
    const size_t o = window_base(d, tn) + i;
    d.wn[o] = d.hn[tri * RING + slot];
    d.wd[o] = d.hd[tri * RING + slot];
}

// far(c) = p(c) - sum_pairs W^fdtd (*) (N, D). W^fdtd has tap 0 == 0 (pppm_cache.cu:111),
// so taps 1..15 only (adding the zero tap leaves the sum bit-identical); the Neumann slot
// of step t is therefore free to be written by the extra waves of this launch.
struct FarGather
{
    struct Index
    {
        int p, rec;
    };
    const SceneStep &d;
    const float *wn, *wd;
    const float *g;
    size_t nn;
    unsigned cell;
    float gv;
    __device__ __forceinline__ Index load(int p) const { return Index{p, d.c3_pairs[p]}; }
    __device__ __forceinline__ void conv(Index i, int n, int lane, float4 *term, float *vals) const
    {
        vals[lane] = conv_round<1, false>(d.owf ? d.owf : d.wf, d.owf ? d.osf : d.sf, d.owf ? i.p : i.rec, i.rec / GC, n, wn,
                                          wd, lane, term, nullptr);
    }
    __device__ __forceinline__ void early(int s, bool in) { cell = in && !d.fused ? (unsigned)d.c3_cells[s] : ~0u; }
    __device__ __forceinline__ void late() { gv = cell < nn ? g[cell] : 0.0f; }
    __device__ __forceinline__ void done(int s, float acc) const
    {
        d.far[s] = d.fused ? acc : cell < nn ? gv - acc : 0.0f;
    }
};
__device__ __forceinline__ void far_wave(const SceneStep &d, int wave, int lane, GatherLds<float> &lds)
{
    // the wave map is read before the error word is waited on (in bounds either way), so the
    // two loads take one memory round trip
    const int nw = gran_waves(d.c3_waves, d.gran3);
    int2 w0 = {0, 0}, w1 = {0, 0};
    if (wave < nw)
        wave_range(d.c3_wave, d.c3_waves, d.gran3, wave, w0, w1);
    if (d.err && *d.err)  // behind a mesh update that failed: the step is run again after the update is
        return;
    const int t = d.st->t + d.fused;
    const size_t wb = window_base(d, t);
    if (wave < nw)
    {
        if (w0.x >= w1.x)
            return;
        const size_t nn = (size_t)d.a.N * d.a.N * d.a.N;
        FarGather g{d, d.wn + wb, d.wd + wb, d.grid3 + (size_t)(((t % 3) + 3) % 3) * nn, nn, ~0u, 0.0f};
        gather_wave(g, d.c3_start, w0, w1, lane, lds);
    }
    else
    {
        // Neumann input of step t into the ring (set_neumann_condition_kernel)
        const int i = (wave - nw) * WAVE + lane;
        if (d.neumann && i < d.a.nt)
        {
            const float v = d.neumann[(size_t)(t - d.a.t0) * d.a.stride + i];
            d.hn[i * RING + (t & (RING - 1))] = v;
            d.wn[wb + i * STEPS] = v;  // tap 0 of the Dirichlet update and the near field
        }
    }
}

// One of the eight corners a triangle's far field is interpolated from (pppm.cu:116-144): its C3
// cell, the triangle's base cell and the interpolation weight
struct Corner
{
    int ci, base;
    float iw;
    __device__ __forceinline__ void load(const SceneStep &d, int i)  // i = 8 * triangle + corner
    {
        ci = d.corner[i];  // corners of a base cell are C3 cells (>= 0)
        iw = d.interp[i];
        base = d.geom[i >> 3].base;
    }
    // g: the pressure level of the step
    __device__ __forceinline__ float term(const SceneStep &d, const float *__restrict__ g, int w) const
    {
        float fv = 0.0f;
        if (ci >= 0)
        {
            fv = d.far[ci];
            if (d.fused)
                fv = g[base + ((w >> 2) * d.a.N + (w >> 1 & 1)) * d.a.N + (w & 1)] - fv;
        }
        return iw * fv;
    }
};

// The face far field of every triangle by a launch of its own, thread 8 * triangle + corner; the
// eight terms are added in corner order
__device__ __forceinline__ void face_far_item(const SceneStep &d, int i)
{
    if (i >= 8 * d.a.nt || *d.err)
        return;  // whole groups of eight
    const int t = d.st->t + d.fused;
    Corner k;
    k.load(d, i);
    const float v = k.term(d, d.grid3 + (size_t)(((t % 3) + 3) % 3) * d.a.N * d.a.N * d.a.N, i & 7);
    float sum = 0.0f;
#pragma unroll
    for (int w = 0; w < 8; w++)
        sum += __shfl(v, w, 8);
    if ((i & 7) == 0)
        d.ffar[i >> 3] = sum;
}

// Face far field (8-corner interpolation, pppm.cu:116-144), face near field against the
// 4x4x4 list with D[t] = 0 and its tap-0 factors (pppm.cu:146-170), then
// D_c[t] = (far*rc + near) / (0.5*area - sum_j D_0(c, j)) (pppm.cu:172-193).
// The two sums of a pair are parked side by side: x the convolution, y the tap-0 factor.
template <bool PASS>
struct FaceGather
{
    struct Index
    {
        int j, rec;
    };
    const SceneStep &d;
    const float *wn;
    float *wd;
    const float *g;  // pressure level of step t
    int t;
    int lane;
    int s0, n;        // the group's segments s0 .. s0 + n - 1 (lane l's is s0 + l)
    Corner k;         // corner lane & 7 of segment s0 + lane / 8
    float ff, area;   // this lane's segment
    __device__ __forceinline__ Index load(int p) const { return Index{d.face_nbr[p], d.ofw ? p : d.face_slot[p]}; }
    __device__ __forceinline__ void conv(Index i, int n, int lane, float4 *term, float2 *vals) const
    {
        vals[lane].x = conv_round<0, true>(d.ofw ? d.ofw : d.fw, d.ofw ? d.ofsc : d.fsc, i.rec, i.j, n, wn, wd, lane, term,
                                           &vals[0].y);  // face_factor = (float)D_0 * scale_D
    }
    // The face far field of the group's segments. PASS: k_face_far has left it. Else a lane per
    // (segment, corner), eight segments at a time (a chunk of 256 pairs rarely holds more), then
    // each segment's lane adds its eight terms in corner order.
    __device__ __forceinline__ void early(int s, bool in)
    {
        s0 = __builtin_amdgcn_readfirstlane(s - lane);
        n = (int)__popcll(__ballot(in));
        if (!PASS && (lane >> 3) < n)
            k.load(d, 8 * s0 + lane);
        if (PASS && in)
        {
            ff = d.ffar[s];
            area = d.geom[s].area;
        }
    }
    __device__ __forceinline__ void late()
    {
        if (PASS)
            return;
        ff = 0.0f;
        area = 0.0f;
        if (lane < n)
            area = d.geom[s0 + lane].area;
        for (int g0 = 0; g0 < n; g0 += 8)
        {
            float term = 0.0f;
            if (g0 + (lane >> 3) < n)
            {
                if (g0 > 0)
                    k.load(d, 8 * (s0 + g0) + lane);
                term = k.term(d, g, lane & 7);
            }
            const int at = (lane - g0) & 7;
            float sum = 0.0f;
#pragma unroll
            for (int w = 0; w < 8; w++)
                sum += __shfl(term, 8 * at + w);
            if (lane >= g0 && lane < g0 + 8)
                ff = sum;
        }
    }
    __device__ __forceinline__ void done(int s, float2 acc) const
    {
        const float num = ff * d.a.rc + acc.x;
        const double den = 0.5 * (double)area - (double)acc.y;
        const float dv = (float)((double)num / den);
        d.hd[s * RING + (t & (RING - 1))] = dv;
        wd[s * STEPS] = dv;  // tap 0 of the near field
    }
};
template <bool PASS>
__device__ __forceinline__ void dirichlet_wave(const SceneStep &d, int wave, int lane, GatherLds<float2> &lds)
{
    const int t = d.st->t + d.fused;
    if (wave >= gran_waves(d.face_waves, d.gran4))
        return;
    // the wave map is read before the error word is waited on (one memory round trip)
    int2 w0, w1;
    wave_range(d.face_wave, d.face_waves, d.gran4, wave, w0, w1);
    // after a flagged mesh update the face lists may be incomplete: leave D[t] untouched
    if (*d.err != 0)
        return;
    if (d.fused && wave == 0 && lane == 0)
        d.st->next = t;
    if (w0.x >= w1.x)
        return;
    const size_t wb = window_base(d, t), nn = (size_t)d.a.N * d.a.N * d.a.N;
    FaceGather<PASS> g{d, d.wn + wb, d.wd + wb, d.grid3 + (size_t)(((t % 3) + 3) % 3) * nn, t, lane, 0, 0, {}, 0.0f, 0.0f};
    gather_wave(g, d.face_start, w0, w1, lane, lds);
}

// p(c) = far + 0.98 * sum W^bem (*) (N, D) over all 16 taps; records listener samples.
struct NearGather
{
    struct Index
    {
        int p, rec;
    };
    const SceneStep &d;
    const float *wn, *wd;
    float *g;
    size_t nn;
    int t, lc;
    unsigned cell;
    float fv;
    __device__ __forceinline__ Index load(int p) const { return Index{p, d.c3_pairs[p]}; }
    __device__ __forceinline__ void conv(Index i, int n, int lane, float4 *term, float *vals) const
    {
        vals[lane] = conv_round<0, false>(d.owb ? d.owb : d.wb, d.owb ? d.osb : d.sb, d.owb ? i.p : i.rec, i.rec / GC, n, wn,
                                          wd, lane, term, nullptr);
    }
    __device__ __forceinline__ void early(int s, bool in)
    {
        cell = in ? (unsigned)d.c3_cells[s] : ~0u;
        fv = in ? d.far[s] : 0.0f;
    }
    __device__ __forceinline__ void late()
    {
        if (d.fused)
            fv = cell < nn ? g[cell] - fv : 0.0f;
    }
    __device__ __forceinline__ void done(int s, float acc) const
    {
        if (d.keep_far)
            d.far[s] = fv;  // (no other wave of the launch reads it)
        const float v = (float)((double)fv + (double)acc * 0.98);
        if (cell < nn)
            g[cell] = v;
        if (d.out)
            for (int l = 0; l < d.a.n_listen; l++)
                if (__builtin_amdgcn_readlane(lc, l) == s)
                    d.out[(size_t)(t - d.a.t0) * d.out_stride + l] = v;
    }
};
__device__ __forceinline__ void near_wave(const SceneStep &d, int wave, int lane, GatherLds<float> &lds)
{
    // the wave map is read before the error word is waited on (in bounds either way), and lane l
    // reads listener l's C3 index: the table set with the listeners, or, for lists that move with
    // the mesh (lc3 null), this update's map of the listener's cell
    const int nw = gran_waves(d.c3_waves, d.gran3);
    int2 w0 = {0, 0}, w1 = {0, 0};
    if (wave < nw)
        wave_range(d.c3_wave, d.c3_waves, d.gran3, wave, w0, w1);
    int lc = -1;
    if (d.out && lane < d.a.n_listen)
        lc = d.lc3 ? d.lc3[lane] : d.c3_index[d.lcell[lane]];
    if (d.err && *d.err)
        return;
    const int t = d.fused ? d.st->next : d.st->t;
    if (d.fused && wave == 0 && lane == 0)
        d.st->t = t;
    const size_t nn = (size_t)d.a.N * d.a.N * d.a.N;
    float *g = d.grid3 + (size_t)(((t % 3) + 3) % 3) * nn;
    if (wave < nw)
    {
        if (w0.x >= w1.x)
            return;
        const size_t wb = window_base(d, t);
        NearGather ng{d, d.wn + wb, d.wd + wb, g, nn, t, lc, ~0u, 0.0f};
        gather_wave(ng, d.c3_start, w0, w1, lane, lds);
    }
    else if (d.out && wave == nw)
    {
        // listeners outside the corrected region read the grid directly (no wave writes them)
        if (lane < d.a.n_listen && lc < 0)
            d.out[(size_t)(t - d.a.t0) * d.out_stride + lane] = g[d.lcell[lane]];
    }
}

// ---------------------------------------------------------------- single-scene kernels
__global__ __launch_bounds__(256) void k_windows(SceneStep d, int back)
{
    windows_item(d, d.st->t - back + 1, blockIdx.x * 256 + threadIdx.x);
}

// The FDTD and the far-field sums of one step in one launch: the sums read only the histories, so
// neither waits for the other. The gather's blocks come first (they run longest). A step is this
// launch, the Dirichlet update and the near field; with the FDTD, the time advance and the far
// field as launches of their own and the windows rebuilt in between it was five, and each costs a
// small scene about 5 us. One pass of 64 steps alone, with the same gathers in five and in three
// launches: 32^3 1.33 -> 1.00 ms, 64^3 1.89 -> 1.56 ms.
__global__ __launch_bounds__(TB) void k_step_head(SceneStep d, FdtdParams p, int far_blocks, int nb_inner, StatusOut f)
{
    static_assert(TB == BLK, "gather and FDTD blocks share the launch");
    __shared__ GatherLds<float> lds[WPB];
    copy_status(f);
    if ((int)blockIdx.x < far_blocks)
    {
        const int wid = wave_in_block();
        far_wave(d, xcd_wave(far_blocks >> 3, wid), threadIdx.x & 63, lds[wid]);
        return;
    }
    if (*d.err)
        return;
    fdtd_block(d.grid3, p, d.st->t, (int)blockIdx.x - far_blocks, nb_inner);
}

__global__ __launch_bounds__(TB) void k_far(SceneStep d, int xper)
{
    __shared__ GatherLds<float> lds[WPB];
    const int wid = wave_in_block();
    far_wave(d, xcd_wave(xper, wid), threadIdx.x & 63, lds[wid]);
}

__global__ __launch_bounds__(256) void k_face_far(SceneStep d) { face_far_item(d, blockIdx.x * 256 + threadIdx.x); }

template <bool PASS>
__global__ __launch_bounds__(TB) void k_dirichlet(SceneStep d)
{
    __shared__ GatherLds<float2> lds[WPB];
    const int wid = wave_in_block();
    dirichlet_wave<PASS>(d, blockIdx.x * WPB + wid, threadIdx.x & 63, lds[wid]);
}

// near_blocks gather blocks, then (win2) the windows of the next step, whose ring values are all
// written by now; they go to the half the gather does not read
__global__ __launch_bounds__(TB) void k_near(SceneStep d, int xper, int near_blocks)
{
    __shared__ GatherLds<float> lds[WPB];
    if ((int)blockIdx.x >= near_blocks)
    {
        windows_item(d, d.st->next + 1, ((int)blockIdx.x - near_blocks) * TB + (int)threadIdx.x);
        return;
    }
    const int wid = wave_in_block();
    near_wave(d, xcd_wave(xper, wid), threadIdx.x & 63, lds[wid]);
}

__global__ void k_listen_direct(SceneStep d)
{
    const int t = d.st->t;
    const int l = threadIdx.x;
    if (l >= d.a.n_listen || (d.err && *d.err))
        return;
    const size_t nn = (size_t)d.a.N * d.a.N * d.a.N;
    const float *g = d.grid3 + (size_t)(((t % 3) + 3) % 3) * nn;
    d.out[(size_t)(t - d.a.t0) * d.out_stride + l] = g[d.lcell[l]];
}

__global__ __launch_bounds__(256) void k_order_records(const int *__restrict__ c3_pairs, int n3,
                                                       const uint4 *__restrict__ wf, const float2 *__restrict__ sf,
                                                       const uint4 *__restrict__ wb, const float2 *__restrict__ sb,
                                                       uint4 *__restrict__ owf, float2 *__restrict__ osf,
                                                       uint4 *__restrict__ owb, float2 *__restrict__ osb,
                                                       const int *__restrict__ face_slot, int n4, int pool_cap,
                                                       const uint4 *__restrict__ fw, const float2 *__restrict__ fsc,
                                                       uint4 *__restrict__ ofw, float2 *__restrict__ ofsc)
{
    // one thread per 16-byte quarter of a record: consecutive threads write consecutive bytes
    long long i = (long long)blockIdx.x * 256 + threadIdx.x;
    if (i < 4LL * n3)
    {
        const int pr = (int)(i >> 2), q = (int)(i & 3);
        const int r = c3_pairs[pr];
        const bool ok = (unsigned)r < (unsigned)n3;  // the C3 pairs are a permutation of [0, n3)
        owf[4 * (size_t)pr + q] = ok ? wf[4 * (size_t)r + q] : make_uint4(0, 0, 0, 0);
        owb[4 * (size_t)pr + q] = ok ? wb[4 * (size_t)r + q] : make_uint4(0, 0, 0, 0);
        if (q == 0)
        {
            osf[pr] = ok ? sf[r] : make_float2(0, 0);
            osb[pr] = ok ? sb[r] : make_float2(0, 0);
        }
        return;
    }
    i -= 4LL * n3;
    if (i < 4LL * n4)
    {
        const int pr = (int)(i >> 2), q = (int)(i & 3);
        const int sl = face_slot[pr];
        const bool ok = (unsigned)sl < (unsigned)pool_cap;
        ofw[4 * (size_t)pr + q] = ok ? fw[4 * (size_t)sl + q] : make_uint4(0, 0, 0, 0);
        if (q == 0)
            ofsc[pr] = ok ? fsc[sl] : make_float2(0, 0);
    }
}

__global__ void k_listen_setup(ListenTable lt, int N, const int *__restrict__ c3_index, int *__restrict__ cell,
                               int *__restrict__ c3)
{
    const int l = threadIdx.x;
    if (l >= lt.n)
        return;
    const int q = lin3(lt.xyz[3 * l], lt.xyz[3 * l + 1], lt.xyz[3 * l + 2], N);
    cell[l] = q;
    c3[l] = c3_index[q];
}

__global__ void k_set_neumann(SceneStep d)
{
    const int t = d.st->t;
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < d.a.nt)
        d.hn[i * RING + (t & (RING - 1))] = d.neumann[(size_t)(t - d.a.t0) * d.a.stride + i];
}

// ---------------------------------------------------------------- batched kernels
// (map_block and scene_desc: scene_device.hpp)
__global__ __launch_bounds__(256) void k_batch_windows(const SceneStep *__restrict__ ds, BatchMap m)
{
    int sc, lb;
    if (map_block(m, (int)blockIdx.x, sc, lb))
        {
        const SceneStep d = scene_desc(ds, sc);
        windows_item(d, d.st->t + 1, lb * 256 + threadIdx.x);
    }
}

__global__ __launch_bounds__(TB) void k_batch_head(const SceneStep *__restrict__ ds, BatchMap mf,
                                                   const FdtdScene *__restrict__ fd, BatchMap mb)
{
    __shared__ GatherLds<float> lds[WPB];
    int sc, lb;
    if ((int)blockIdx.x < 8 * mf.per)
    {
        if (!map_block(mf, (int)blockIdx.x, sc, lb))
            return;
        const int wid = wave_in_block();
        far_wave(scene_desc(ds, sc), lb * WPB + wid, threadIdx.x & 63, lds[wid]);
        return;
    }
    if (!map_block(mb, (int)blockIdx.x - 8 * mf.per, sc, lb))
        return;
    const FdtdScene d = scene_desc(fd, sc);
    fdtd_block(d.grid3, d.p, d.st->t, lb, d.nb_inner);
}

__global__ __launch_bounds__(TB) void k_batch_far(const SceneStep *__restrict__ ds, BatchMap m)
{
    __shared__ GatherLds<float> lds[WPB];
    int sc, lb;
    if (!map_block(m, (int)blockIdx.x, sc, lb))
        return;
    const int wid = wave_in_block();
    far_wave(scene_desc(ds, sc), lb * WPB + wid, threadIdx.x & 63, lds[wid]);
}

__global__ __launch_bounds__(256) void k_batch_face_far(const SceneStep *__restrict__ ds, BatchMap m)
{
    int sc, lb;
    if (map_block(m, (int)blockIdx.x, sc, lb))
        face_far_item(scene_desc(ds, sc), lb * 256 + threadIdx.x);
}

template <bool PASS>
__global__ __launch_bounds__(TB) void k_batch_dirichlet(const SceneStep *__restrict__ ds, BatchMap m)
{
    __shared__ GatherLds<float2> lds[WPB];
    int sc, lb;
    if (!map_block(m, (int)blockIdx.x, sc, lb))
        return;
    const int wid = wave_in_block();
    dirichlet_wave<PASS>(scene_desc(ds, sc), lb * WPB + wid, threadIdx.x & 63, lds[wid]);
}

__global__ __launch_bounds__(TB) void k_batch_near(const SceneStep *__restrict__ ds, BatchMap m, BatchMap mw)
{
    __shared__ GatherLds<float> lds[WPB];
    int sc, lb;
    if ((int)blockIdx.x >= 8 * m.per)
    {
        if (map_block(mw, (int)blockIdx.x - 8 * m.per, sc, lb))
        {
            const SceneStep d = scene_desc(ds, sc);
            windows_item(d, d.st->next + 1, lb * TB + (int)threadIdx.x);
        }
        return;
    }
    if (!map_block(m, (int)blockIdx.x, sc, lb))
        return;
    const int wid = wave_in_block();
    near_wave(scene_desc(ds, sc), lb * WPB + wid, threadIdx.x & 63, lds[wid]);
}

__global__ void k_batch_advance(const SceneStep *__restrict__ ds, int n)
{
    const int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n)
        ds[i].st->t = ds[i].st->t + 1;
}

inline int blocks_for_waves(long long waves) { return waves > 0 ? (int)((waves + WPB - 1) / WPB) : 1; }

// blocks per XCD of a gather launch over `waves` waves (the launch has 8 times as many)
inline int xcd_per(long long waves) { return (blocks_for_waves(waves) + 7) / 8; }

long long far_waves(const SceneStep &d)
{
    return (long long)gran_waves(d.c3_waves, d.gran3) + (d.neumann ? (d.a.nt + WAVE - 1) / WAVE : 0);
}
long long near_waves(const SceneStep &d) { return (long long)gran_waves(d.c3_waves, d.gran3) + (d.out ? 1 : 0); }
}  // namespace

int batch_blocks(const SceneStep &d, BatchKernel k)
{
    switch (k)
    {
    case BatchKernel::Windows:
    {
        const long long n = (long long)d.a.nt * STEPS;
        return n > 0 ? (int)((n + 255) / 256) : 1;
    }
    case BatchKernel::Far:
        return blocks_for_waves(far_waves(d));
    case BatchKernel::FaceFar:
        return std::max(1, (int)((8LL * d.a.nt + 255) / 256));
    case BatchKernel::DirichletOnly:
    case BatchKernel::Dirichlet:
        return blocks_for_waves(gran_waves(d.face_waves, d.gran4));
    case BatchKernel::Near:
        return blocks_for_waves(near_waves(d));
    }
    return 1;
}

hipError_t launch_windows(const SceneStep &d, int back, hipStream_t s)
{
    const long long n = (long long)d.a.nt * STEPS;
    k_windows<<<n > 0 ? (int)((n + 255) / 256) : 1, 256, 0, s>>>(d, back);
    return hipGetLastError();
}

hipError_t launch_far(const SceneStep &d, hipStream_t s)
{
    const int per = xcd_per(far_waves(d));
    k_far<<<8 * per, TB, 0, s>>>(d, per);
    return hipGetLastError();
}

hipError_t launch_dirichlet(const SceneStep &d, hipStream_t s)
{
    // plain block order: the heavy face lists of finely meshed objects sit together in the wave
    // range, and round-robin spreads them over the XCDs (the contiguous mapping of the C3 gathers
    // cut this kernel's HBM traffic from 47.6 to 39.7 MB but raised its time from 19.1 to 21.6 us)
    const int blocks = blocks_for_waves(gran_waves(d.face_waves, d.gran4));
    if (d.ffar)
    {
        k_face_far<<<(8 * d.a.nt + 255) / 256, 256, 0, s>>>(d);
        k_dirichlet<true><<<blocks, TB, 0, s>>>(d);
    }
    else
        k_dirichlet<false><<<blocks, TB, 0, s>>>(d);
    return hipGetLastError();
}

hipError_t launch_near(const SceneStep &d, hipStream_t s)
{
    const int per = xcd_per(near_waves(d));
    const int nwin = d.win2 ? (int)(((long long)d.a.nt * STEPS + TB - 1) / TB) : 0;
    k_near<<<8 * per + nwin, TB, 0, s>>>(d, per, 8 * per);
    return hipGetLastError();
}

hipError_t launch_step_head(const SceneStep &d, const FdtdParams &p, const StatusOut &status, hipStream_t s)
{
    int nb_inner = 0;
    const hipError_t e = launch_fdtd_march(d.grid3, p, d.st, d.err, s, nb_inner);
    if (e != hipSuccess)
        return e;
    const int far_blocks = 8 * xcd_per(far_waves(d));
    k_step_head<<<far_blocks + nb_inner + fdtd_shell_blocks(p.N), TB, 0, s>>>(d, p, far_blocks, nb_inner, status);
    return hipGetLastError();
}

hipError_t launch_batch_head(const SceneStep *descs, const BatchMap &mf, const FdtdScene *fd, const BatchMap &mb,
                             hipStream_t s)
{
    k_batch_head<<<8 * mf.per + 8 * mb.per, TB, 0, s>>>(descs, mf, fd, mb);
    return hipGetLastError();
}

hipError_t launch_batch_near(const SceneStep *descs, const BatchMap &mn, const BatchMap &mw, hipStream_t s)
{
    k_batch_near<<<8 * mn.per + 8 * mw.per, TB, 0, s>>>(descs, mn, mw);
    return hipGetLastError();
}

hipError_t launch_listen_direct(const SceneStep &d, hipStream_t s)
{
    k_listen_direct<<<1, 64, 0, s>>>(d);
    return hipGetLastError();
}

hipError_t launch_listen_setup(const ListenTable &lt, int N, const int *c3_index, int *cell, int *c3,
                               hipStream_t s)
{
    k_listen_setup<<<1, 64, 0, s>>>(lt, N, c3_index, cell, c3);
    return hipGetLastError();
}

hipError_t launch_order_records(const int *c3_pairs, int n3, const uint32_t *wf, const float2 *sf, const uint32_t *wb,
                                const float2 *sb, uint32_t *owf, float2 *osf, uint32_t *owb, float2 *osb,
                                const int *face_slot, int n4, int pool_cap, const uint32_t *fw, const float2 *fsc,
                                uint32_t *ofw, float2 *ofsc, hipStream_t s)
{
    const long long n = 4LL * n3 + 4LL * n4;
    if (n <= 0)
        return hipSuccess;
    k_order_records<<<(unsigned)((n + 255) / 256), 256, 0, s>>>(
        c3_pairs, n3, (const uint4 *)wf, sf, (const uint4 *)wb, sb, (uint4 *)owf, osf, (uint4 *)owb, osb, face_slot, n4,
        pool_cap, (const uint4 *)fw, fsc, (uint4 *)ofw, ofsc);
    return hipGetLastError();
}

hipError_t launch_set_neumann(const SceneStep &d, hipStream_t s)
{
    k_set_neumann<<<(d.a.nt + 255) / 256 > 0 ? (d.a.nt + 255) / 256 : 1, 256, 0, s>>>(d);
    return hipGetLastError();
}

hipError_t launch_batch(BatchKernel k, const SceneStep *descs, const BatchMap &m, hipStream_t s)
{
    const int grid = 8 * m.per;
    switch (k)
    {
    case BatchKernel::Windows:
        k_batch_windows<<<grid, 256, 0, s>>>(descs, m);
        break;
    case BatchKernel::Far:
        k_batch_far<<<grid, TB, 0, s>>>(descs, m);
        break;
    case BatchKernel::FaceFar:
        k_batch_face_far<<<grid, 256, 0, s>>>(descs, m);
        break;
    case BatchKernel::DirichletOnly:
        k_batch_dirichlet<true><<<grid, TB, 0, s>>>(descs, m);
        break;
    case BatchKernel::Dirichlet:
        k_batch_dirichlet<false><<<grid, TB, 0, s>>>(descs, m);
        break;
    case BatchKernel::Near:
        k_batch_near<<<grid, TB, 0, s>>>(descs, m, BatchMap{});
        break;
    }
    return hipGetLastError();
}

hipError_t launch_batch_advance(const SceneStep *descs, int n, hipStream_t s)
{
    k_batch_advance<<<(n + 255) / 256, 256, 0, s>>>(descs, n);
    return hipGetLastError();
}

}  // namespace pppm_amd
