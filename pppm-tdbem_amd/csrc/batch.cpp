// Batched scenes: many independent PPPM scenes (solver handles with their meshes set) stepped
// together. Each kernel of the time step is one launch over every scene's blocks (a scene
// table in device memory gives each block its scene); longer runs replay a captured HIP graph of 32
// such batch steps. The FDTD interior of each scene uses the kernel variant picked
// for its size class by the autotuner (one thread per cell, or LDS-staged 2.5D tiles); every
// variant gives the same bits, so the batch equals the scenes' single-scene runs bit for bit.
//
// Reference behaviour per scene: PPPMSolver::update_grid_and_face (src/algorithm/pppm.h:137-145)
// as in pppm_run; the reference steps one scene at a time.
#include "pppm_hip.h"

#include <algorithm>
#include <cstring>
#include <string>
#include <vector>

#include "solver_state.hpp"

using namespace pppm_amd;

namespace
{

// size classes of the autotuner table, by grid edge N: [lo, next lo)
constexpr int kClassLo[] = {0, 40, 56, 72, 88, 112, 160};
constexpr int kClasses = sizeof(kClassLo) / sizeof(kClassLo[0]);
int size_class(int N)
{
    int c = 0;
    while (c + 1 < kClasses && N >= kClassLo[c + 1])
        c++;
    return c;
}
// FDTD interior variant per size class before any tuning (0: one thread per cell)
constexpr int kDefaultVariant[kClasses] = {0, 0, 0, 0, 0, 0, 0};

constexpr int kGraphSteps = 32;  // steps of a captured graph; runs of fewer than two are launched step by step

struct Map
{
    DBuf<int> scene_of, first;
    int total = 0, per = 0;
    BatchMap view() const { return BatchMap{scene_of.p, first.p, total, per}; }
};

}  // namespace

struct pppm_batch
{
    std::vector<pppm_solver *> sc;
    hipStream_t stream = nullptr;
    bool own_stream = false;
    std::string err;
    std::vector<int> variant;  // FDTD interior variant per scene
    DBuf<SceneStep> descs;
    DBuf<FdtdScene> fdescs;
    DBuf<int> firsts;  // first virtual blocks of the maps being built
    Map m_fdtd, m_tile[kFdtdVariants], m_win, m_far, m_ffar, m_dir, m_near;
    bool face_far = false;  // the face far field takes a launch of its own (face_far_pass)
    // batched adjoint: scene table and one block map per reverse-step kernel
    DBuf<AdjScene> adescs;
    Map m_adj[kAdjKernels];
    // per-phase HIP event timing of eager batch steps: 0 FDTD (shell and interiors), 1 history
    // windows and time advance, 2 far field, 3 Dirichlet update, 4 near field
    bool timing = false;
    std::vector<std::pair<int, std::pair<hipEvent_t, hipEvent_t>>> spans;
    std::vector<hipEvent_t> pool;
    double phase_ms[8] = {0};
    long long phase_n[8] = {0};
};

namespace
{

int bfail(pppm_batch *b, int code, const std::string &msg)
{
    if (b)
        b->err = msg;
    return code;
}

#define BCK(expr)                                                                                \
    do                                                                                           \
    {                                                                                            \
        hipError_t e_ = (expr);                                                                  \
        if (e_ != hipSuccess)                                                                    \
            return bfail(b, PPPM_ERR_HIP, std::string(#expr) + ": " + hipGetErrorString(e_));    \
    } while (0)

#define BRC(expr)         \
    do                    \
    {                     \
        int rc_ = (expr); \
        if (rc_)          \
            return rc_;   \
    } while (0)

// The maps of several launches (blocks[i]: scene i's blocks): the first virtual block of every
// scene goes up in one copy and the device spreads the scene numbers over the blocks, so a run
// waits for its set-up once (a map each with two copies and a wait: eleven waits a run)
struct MapJob
{
    Map *m;
    const std::vector<int> *blocks;
};
int build_maps(pppm_batch *b, const std::vector<MapJob> &jobs)
{
    const size_t n = b->sc.size();
    std::vector<int> first(jobs.size() * n);
    for (size_t k = 0; k < jobs.size(); k++)
    {
        int total = 0;
        for (size_t i = 0; i < n; i++)
        {
            first[k * n + i] = total;
            total += (*jobs[k].blocks)[i];
        }
        jobs[k].m->total = total;
        jobs[k].m->per = (total + 7) / 8;
        BCK(jobs[k].m->first.ensure(n));
        BCK(jobs[k].m->scene_of.ensure(std::max(total, 1)));
    }
    BCK(b->firsts.ensure(first.size()));
    BCK(hipMemcpyAsync(b->firsts.p, first.data(), first.size() * sizeof(int), hipMemcpyHostToDevice, b->stream));
    for (size_t k = 0; k < jobs.size(); k++)
        BCK(launch_scene_map(b->firsts.p + k * n, (int)n, jobs[k].m->total, jobs[k].m->first.p, jobs[k].m->scene_of.p,
                             b->stream));
    BCK(hipStreamSynchronize(b->stream));  // the host vector, and the caller's descriptors, go out of scope
    return PPPM_OK;
}

// FDTD scene table and maps for the current variants
int build_fdtd(pppm_batch *b)
{
    const int n = (int)b->sc.size();
    std::vector<FdtdScene> fd(n);
    std::vector<int> shell(n);
    std::vector<std::vector<int>> tiles(kFdtdVariants, std::vector<int>(n, 0));
    for (int i = 0; i < n; i++)
    {
        const pppm_solver *s = b->sc[i];
        FdtdScene &f = fd[i];
        f.p = solver_fdtd_params(s);
        f.grid3 = s->grid.p;
        f.st = s->state.p;
        f.xch = 0;
        const int v = b->variant[i];
        f.nb_inner = v == 0 ? fdtd_inner_blocks(s->N) : 0;
        shell[i] = fdtd_shell_blocks(s->N) + f.nb_inner;
        if (v > 0)
            tiles[v][i] = fdtd_tile_blocks(s->N, v, f.xch);
    }
    BCK(b->fdescs.ensure(n));
    BCK(hipMemcpyAsync(b->fdescs.p, fd.data(), n * sizeof(FdtdScene), hipMemcpyHostToDevice, b->stream));
    std::vector<MapJob> jobs{{&b->m_fdtd, &shell}};
    for (int v = 1; v < kFdtdVariants; v++)
        jobs.push_back({&b->m_tile[v], &tiles[v]});
    return build_maps(b, jobs);
}

// FDTD of every scene (no advance) in launches of its own, as a timed step takes it
int enqueue_fdtd(pppm_batch *b)
{
    BCK(launch_batch_fdtd(b->fdescs.p, b->m_fdtd.view(), b->stream));
    for (int v = 1; v < kFdtdVariants; v++)
        if (b->m_tile[v].total > 0)
            BCK(launch_batch_tile(v, b->fdescs.p, b->m_tile[v].view(), b->stream));
    return PPPM_OK;
}

hipEvent_t take_event(pppm_batch *b)
{
    if (!b->pool.empty())
    {
        hipEvent_t e = b->pool.back();
        b->pool.pop_back();
        return e;
    }
    hipEvent_t e = nullptr;
    return hipEventCreate(&e) == hipSuccess ? e : nullptr;
}

int span_begin(pppm_batch *b, int phase)
{
    if (!b->timing)
        return -1;
    hipEvent_t a = take_event(b), c = take_event(b);
    if (!a || !c || hipEventRecord(a, b->stream) != hipSuccess)
        return -1;
    b->spans.push_back({phase, {a, c}});
    return (int)b->spans.size() - 1;
}

void span_end(pppm_batch *b, int i)
{
    if (i >= 0)
        (void)hipEventRecord(b->spans[i].second.second, b->stream);
}

int collect_spans(pppm_batch *b)
{
    if (b->spans.empty())
        return PPPM_OK;
    BCK(hipStreamSynchronize(b->stream));
    for (auto &sp : b->spans)
    {
        float ms = 0;
        if (hipEventElapsedTime(&ms, sp.second.first, sp.second.second) == hipSuccess)
        {
            b->phase_ms[sp.first] += ms;
            b->phase_n[sp.first]++;
        }
        b->pool.push_back(sp.second.first);
        b->pool.push_back(sp.second.second);
    }
    b->spans.clear();
    return PPPM_OK;
}

// windows of the next step from the rings (a fused step leaves the next one's behind)
int enqueue_batch_windows(pppm_batch *b)
{
    BCK(launch_batch(BatchKernel::Windows, b->descs.p, b->m_win.view(), b->stream));
    return PPPM_OK;
}

// the tiled interiors, then the FDTD beside the far-field sums. No advance: idempotent, the autotuner
// times it repeatedly
int enqueue_batch_head(pppm_batch *b)
{
    for (int v = 1; v < kFdtdVariants; v++)
        if (b->m_tile[v].total > 0)
            BCK(launch_batch_tile(v, b->fdescs.p, b->m_tile[v].view(), b->stream));
    BCK(launch_batch_head(b->descs.p, b->m_far.view(), b->fdescs.p, b->m_fdtd.view(), b->stream));
    return PPPM_OK;
}

int enqueue_batch_dirichlet(pppm_batch *b)
{
    if (b->face_far)
        BCK(launch_batch(BatchKernel::FaceFar, b->descs.p, b->m_ffar.view(), b->stream));
    BCK(launch_batch(b->face_far ? BatchKernel::DirichletOnly : BatchKernel::Dirichlet, b->descs.p, b->m_dir.view(),
                     b->stream));
    return PPPM_OK;
}

// last: of the run, or of a graph: its near field takes the second table, whose scenes keep their far
// field
int enqueue_batch_step(pppm_batch *b, bool last)
{
    if (!b->timing)
    {
        // three launches, as a single scene's step: the FDTD beside the far-field sums (tiled
        // interiors before it), the Dirichlet update, the near field with the next windows
        BRC(enqueue_batch_head(b));
        BRC(enqueue_batch_dirichlet(b));
        BCK(launch_batch_near(b->descs.p + (last ? b->sc.size() : 0), b->m_near.view(), b->m_win.view(), b->stream));
        return PPPM_OK;
    }
    // a span per phase: a launch each
    int sp = span_begin(b, 0);
    BRC(enqueue_fdtd(b));
    span_end(b, sp);
    const int n = (int)b->sc.size();
    sp = span_begin(b, 1);
    BRC(enqueue_batch_windows(b));
    BCK(launch_batch_advance(b->descs.p, n, b->stream));
    span_end(b, sp);
    sp = span_begin(b, 2);
    BCK(launch_batch(BatchKernel::Far, b->descs.p, b->m_far.view(), b->stream));
    span_end(b, sp);
    sp = span_begin(b, 3);
    BRC(enqueue_batch_dirichlet(b));
    span_end(b, sp);
    sp = span_begin(b, 4);
    BCK(launch_batch(BatchKernel::Near, b->descs.p, b->m_near.view(), b->stream));
    span_end(b, sp);
    if (b->spans.size() > 4096)
        return collect_spans(b);
    return PPPM_OK;
}

int check_scenes(pppm_batch *b)
{
    for (pppm_solver *s : b->sc)
    {
        const int rc = solver_check_ready(s, "batch");
        if (rc)
            return bfail(b, rc, s->err);
        if (s->use_pml)
            return bfail(b, PPPM_ERR_ARG, "batch: scenes with the PML are not batched (use pppm_run)");
    }
    return PPPM_OK;
}

}  // namespace

extern "C" {

int pppm_batch_create(pppm_batch **out, pppm_solver *const *scenes, int n_scenes)
{
    if (!out)
        return PPPM_ERR_ARG;
    *out = nullptr;
    if (!scenes || n_scenes < 1)
        return PPPM_ERR_ARG;
    for (int i = 0; i < n_scenes; i++)
        if (!scenes[i])
            return PPPM_ERR_ARG;
    pppm_batch *b = new pppm_batch();
    b->sc.assign(scenes, scenes + n_scenes);
    if (hipStreamCreate(&b->stream) != hipSuccess)
    {
        delete b;
        return PPPM_ERR_HIP;
    }
    b->own_stream = true;
    b->variant.resize(n_scenes);
    for (int i = 0; i < n_scenes; i++)
        b->variant[i] = kDefaultVariant[size_class(scenes[i]->N)];
    *out = b;
    return PPPM_OK;
}

int pppm_batch_destroy(pppm_batch *b)
{
    if (!b)
        return PPPM_ERR_ARG;
    if (b->stream)
        (void)hipStreamSynchronize(b->stream);
    for (auto &sp : b->spans)
    {
        (void)hipEventDestroy(sp.second.first);
        (void)hipEventDestroy(sp.second.second);
    }
    for (hipEvent_t e : b->pool)
        (void)hipEventDestroy(e);
    if (b->own_stream && b->stream)
        (void)hipStreamDestroy(b->stream);
    delete b;
    return PPPM_OK;
}

const char *pppm_batch_last_error(const pppm_batch *b) { return b ? b->err.c_str() : "null handle"; }

int pppm_batch_set_stream(pppm_batch *b, void *hip_stream)
{
    if (!b)
        return PPPM_ERR_ARG;
    BCK(hipStreamSynchronize(b->stream));
    if (b->own_stream)
        BCK(hipStreamDestroy(b->stream));
    b->own_stream = false;
    b->stream = (hipStream_t)hip_stream;
    return PPPM_OK;
}

int pppm_batch_run(pppm_batch *b, const float *const *neumann_series, const long long *strides, int steps,
                   int n_listen, const int *listen_xyz, float *out_dev, int use_graph)
{
    if (!b)
        return PPPM_ERR_ARG;
    const int n = (int)b->sc.size();
    if (steps < 0 || !neumann_series || !strides || !listen_xyz || !out_dev || n_listen < 1 || n_listen > 64)
        return bfail(b, PPPM_ERR_ARG, "batch_run: bad arguments (1 to 64 listeners per scene)");
    BRC(check_scenes(b));
    for (int i = 0; i < n; i++)
        if (!neumann_series[i] || strides[i] < b->sc[i]->nt)
            return bfail(b, PPPM_ERR_ARG, "batch_run: scene " + std::to_string(i) + ": Neumann series missing or stride < nt");
    if (steps == 0)
        return PPPM_OK;
    // per-scene set-up: list-ordered weight records, listener tables, pending work of the
    // scenes' own streams
    std::vector<SceneStep> hd(n);
    for (int i = 0; i < n; i++)
    {
        pppm_solver *s = b->sc[i];
        if (solver_ensure_ordered(s))
            return bfail(b, PPPM_ERR_HIP, "batch_run: scene " + std::to_string(i) + ": " + s->err);
        const int rc = solver_set_listeners(s, listen_xyz + 3 * (size_t)i * n_listen, n_listen);
        if (rc)
            return bfail(b, rc, "batch_run: scene " + std::to_string(i) + ": " + s->err);
        BCK(hipStreamSynchronize(s->stream));
        hd[i] = solver_scene_step(s, neumann_series[i], s->t_host + 1, strides[i], n_listen,
                                  out_dev + (size_t)i * n_listen);
        hd[i].out_stride = (long long)n * n_listen;
    }
    // the waves of a launch are those of all scenes together
    long long w3 = 0, w4 = 0;
    for (const SceneStep &d : hd)
    {
        w3 += d.c3_waves;
        w4 += d.face_waves;
    }
    b->face_far = face_far_pass(w4);
    for (int i = 0; i < n; i++)
    {
        const pppm_solver *s = b->sc[i];
        SceneStep &d = hd[i];
        d.gran3 = gather_gran(w3);
        d.gran4 = gather_gran(w4);
        d.fused = d.win2 = b->timing ? 0 : 1;
        d.ffar = b->face_far ? s->ffar.p : nullptr;
    }
    hd.resize(2 * (size_t)n);  // the second table, for a last step's near field
    std::copy(hd.begin(), hd.begin() + n, hd.begin() + n);
    for (int i = n; i < 2 * n; i++)
        hd[i].keep_far = hd[i].fused;
    BCK(b->descs.ensure(2 * (size_t)n));
    BCK(hipMemcpyAsync(b->descs.p, hd.data(), 2 * (size_t)n * sizeof(SceneStep), hipMemcpyHostToDevice, b->stream));
    std::vector<int> nw(n), nf(n), nff(n), nd(n), nn(n);
    for (int i = 0; i < n; i++)
    {
        nw[i] = batch_blocks(hd[i], BatchKernel::Windows);
        nf[i] = batch_blocks(hd[i], BatchKernel::Far);
        nff[i] = batch_blocks(hd[i], BatchKernel::FaceFar);
        nd[i] = batch_blocks(hd[i], BatchKernel::Dirichlet);
        nn[i] = batch_blocks(hd[i], BatchKernel::Near);
    }
    BRC(build_maps(b, {{&b->m_win, &nw}, {&b->m_far, &nf}, {&b->m_ffar, &nff}, {&b->m_dir, &nd}, {&b->m_near, &nn}}));
    BRC(build_fdtd(b));
    if (!b->timing)
        BRC(enqueue_batch_windows(b));

    int done = 0;
    // A graph costs its capture and instantiation on each call, with the device idle, which one replay
    // never makes good, not for the smallest batches either (one scene of 24^3, 63 steps: launched
    // 1.06 ms, with a graph 1.44; eight of 32^3 1.26 and 1.44; reversed 2.1 and 3.0). More replays
    // share it (eight of 32^3, 64 steps 1.24 and 1.41, 256 steps 4.24 and 4.37 ms), and spare a busy host
    // three launches a step.
    if (use_graph && !b->timing && steps >= 2 * kGraphSteps)
    {
        const int chunk = kGraphSteps;
        hipGraph_t g = nullptr;
        hipGraphExec_t ge = nullptr;
        BCK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        int rc = PPPM_OK;
        for (int i = 0; i < chunk && rc == PPPM_OK; i++)
            rc = enqueue_batch_step(b, i == chunk - 1);
        const hipError_t ee = hipStreamEndCapture(b->stream, &g);
        if (rc || ee != hipSuccess)
        {
            if (g)
                (void)hipGraphDestroy(g);
            return rc ? rc : bfail(b, PPPM_ERR_HIP, std::string("batch graph capture: ") + hipGetErrorString(ee));
        }
        if (hipGraphInstantiate(&ge, g, nullptr, nullptr, 0) != hipSuccess)
        {
            (void)hipGraphDestroy(g);
            return bfail(b, PPPM_ERR_HIP, "batch graph instantiate failed");
        }
        hipError_t le = hipSuccess;
        for (; done + chunk <= steps && le == hipSuccess; done += chunk)
            le = hipGraphLaunch(ge, b->stream);
        const hipError_t se = hipStreamSynchronize(b->stream);
        (void)hipGraphExecDestroy(ge);
        (void)hipGraphDestroy(g);
        BCK(le);
        BCK(se);
    }
    for (; done < steps; done++)
        BRC(enqueue_batch_step(b, done == steps - 1));
    BCK(hipStreamSynchronize(b->stream));
    for (pppm_solver *s : b->sc)
        s->t_host += steps;
    return PPPM_OK;
}

int pppm_batch_adjoint_reset(pppm_batch *b, int t_last)
{
    if (!b)
        return PPPM_ERR_ARG;
    BRC(check_scenes(b));
    for (size_t i = 0; i < b->sc.size(); i++)
    {
        const int rc = pppm_adjoint_reset(b->sc[i], t_last);
        if (rc)
            return bfail(b, rc, "batch_adjoint_reset: scene " + std::to_string(i) + ": " + b->sc[i]->err);
    }
    return PPPM_OK;
}

int pppm_batch_adjoint_run(pppm_batch *b, const float *gout_dev, int steps, int n_listen, const int *listen_xyz,
                           float *const *grad_dev, const long long *grad_strides, int use_graph)
{
    if (!b)
        return PPPM_ERR_ARG;
    const int n = (int)b->sc.size();
    if (steps < 0 || !grad_dev || !grad_strides || n_listen < 0 || n_listen > 64 ||
        (n_listen > 0 && (!listen_xyz || !gout_dev)))
        return bfail(b, PPPM_ERR_ARG, "batch_adjoint_run: bad arguments (at most 64 listeners per scene)");
    BRC(check_scenes(b));
    const int t_last = b->sc[0]->adj_t;
    for (int i = 0; i < n; i++)
    {
        pppm_solver *s = b->sc[i];
        const std::string sn = "batch_adjoint_run: scene " + std::to_string(i) + ": ";
        if (!grad_dev[i] || grad_strides[i] < s->nt)
            return bfail(b, PPPM_ERR_ARG, sn + "gradient missing or stride < nt");
        if (s->adj_version != s->mesh_version)
            return bfail(b, PPPM_ERR_STATE, sn + "no adjoint_reset since the mesh changed");
        if (s->adj_t != t_last)
            return bfail(b, PPPM_ERR_STATE, sn + "its reverse time differs from scene 0's (reset them together)");
    }
    if (steps > t_last + 1)
        return bfail(b, PPPM_ERR_ARG, "batch_adjoint_run: more steps than remain before t = 0");
    if (steps == 0)
        return PPPM_OK;
    // per-scene set-up: listener tables, pending work of the scenes' own streams
    const int t_first = t_last - steps + 1;
    std::vector<AdjScene> hd(n);
    for (int i = 0; i < n; i++)
    {
        pppm_solver *s = b->sc[i];
        const int rc = solver_set_listeners(s, n_listen > 0 ? listen_xyz + 3 * (size_t)i * n_listen : nullptr, n_listen);
        if (rc)
            return bfail(b, rc, "batch_adjoint_run: scene " + std::to_string(i) + ": " + s->err);
        BCK(hipStreamSynchronize(s->stream));
        // cotangent rows: (steps, n_scenes, n_listen), scene i at column block i
        hd[i] = solver_adj_scene(s, n_listen > 0 ? gout_dev + (size_t)i * n_listen : nullptr, (long long)n * n_listen,
                                 n_listen, grad_dev[i], grad_strides[i], t_first);
    }
    BCK(b->adescs.ensure(n));
    BCK(hipMemcpyAsync(b->adescs.p, hd.data(), n * sizeof(AdjScene), hipMemcpyHostToDevice, b->stream));
    BatchMap maps[kAdjKernels];
    std::vector<std::vector<int>> nb(kAdjKernels, std::vector<int>(n));
    std::vector<MapJob> jobs;
    for (int k = 0; k < kAdjKernels; k++)
    {
        for (int i = 0; i < n; i++)
            nb[k][i] = adj_blocks(hd[i], k);
        jobs.push_back({&b->m_adj[k], &nb[k]});
    }
    BRC(build_maps(b, jobs));
    for (int k = 0; k < kAdjKernels; k++)
        maps[k] = b->m_adj[k].view();
    int done = 0;
    if (use_graph && steps >= 2 * kGraphSteps)
    {
        const int chunk = kGraphSteps;
        hipGraph_t g = nullptr;
        hipGraphExec_t ge = nullptr;
        BCK(hipStreamBeginCapture(b->stream, hipStreamCaptureModeThreadLocal));
        hipError_t e = hipSuccess;
        for (int i = 0; i < chunk && e == hipSuccess; i++)
            e = enqueue_batch_adjoint_step(b->adescs.p, maps, n, b->stream);
        const hipError_t ee = hipStreamEndCapture(b->stream, &g);
        if (e != hipSuccess || ee != hipSuccess)
        {
            if (g)
                (void)hipGraphDestroy(g);
            return bfail(b, PPPM_ERR_HIP, "batch adjoint graph capture failed");
        }
        if (hipGraphInstantiate(&ge, g, nullptr, nullptr, 0) != hipSuccess)
        {
            (void)hipGraphDestroy(g);
            return bfail(b, PPPM_ERR_HIP, "batch adjoint graph instantiate failed");
        }
        hipError_t le = hipSuccess;
        for (; done + chunk <= steps && le == hipSuccess; done += chunk)
            le = hipGraphLaunch(ge, b->stream);
        const hipError_t se = hipStreamSynchronize(b->stream);
        (void)hipGraphExecDestroy(ge);
        (void)hipGraphDestroy(g);
        BCK(le);
        BCK(se);
    }
    for (; done < steps; done++)
        BCK(enqueue_batch_adjoint_step(b->adescs.p, maps, n, b->stream));
    BCK(hipStreamSynchronize(b->stream));
    for (pppm_solver *s : b->sc)
        s->adj_t -= steps;
    return PPPM_OK;
}

int pppm_batch_set_timing(pppm_batch *b, int enable)
{
    if (!b)
        return PPPM_ERR_ARG;
    BRC(collect_spans(b));
    b->timing = enable != 0;
    return PPPM_OK;
}

int pppm_batch_get_timing(pppm_batch *b, double *ms8, long long *count8)
{
    if (!b)
        return PPPM_ERR_ARG;
    BRC(collect_spans(b));
    for (int i = 0; i < 8; i++)
    {
        if (ms8)
            ms8[i] = b->phase_ms[i];
        if (count8)
            count8[i] = b->phase_n[i];
        b->phase_ms[i] = 0;
        b->phase_n[i] = 0;
    }
    return PPPM_OK;
}

int pppm_batch_variants(pppm_batch *b, int *variants)
{
    if (!b || !variants)
        return PPPM_ERR_ARG;
    std::memcpy(variants, b->variant.data(), b->variant.size() * sizeof(int));
    return PPPM_OK;
}

int pppm_batch_set_variants(pppm_batch *b, const int *variants)
{
    if (!b || !variants)
        return PPPM_ERR_ARG;
    for (size_t i = 0; i < b->sc.size(); i++)
        if (variants[i] < 0 || variants[i] >= kFdtdVariants)
            return bfail(b, PPPM_ERR_ARG, "batch_set_variants: variant out of range");
    b->variant.assign(variants, variants + b->sc.size());
    return PPPM_OK;
}

int pppm_batch_autotune(pppm_batch *b, int reps, float *ms_out)
{
    if (!b || reps < 1)
        return PPPM_ERR_ARG;
    BRC(check_scenes(b));
    const int n = (int)b->sc.size();
    // What a step launches, so that an interior in a launch of its own is charged for the far-field
    // sums it no longer runs beside (16 scenes of 64^3 and 1280 triangles: 12 us here and in the
    // step, 8 us where the FDTD is timed alone).
    // The sums read the windows as they are and go to scratch: a scene's own far field stays.
    std::vector<SceneStep> hd(n);
    std::vector<int> nf(n);
    size_t n_far = 0;
    long long w3 = 0;
    for (int i = 0; i < n; i++)
    {
        pppm_solver *s = b->sc[i];
        if (solver_ensure_ordered(s))
            return bfail(b, PPPM_ERR_HIP, "autotune: scene " + std::to_string(i) + ": " + s->err);
        BCK(hipStreamSynchronize(s->stream));
        hd[i] = solver_scene_step(s, nullptr, s->t_host + 1, 0, 0, nullptr);
        w3 += hd[i].c3_waves;
        n_far += (size_t)s->cap_c3;
    }
    DBuf<float> far;
    BCK(far.ensure(n_far));
    n_far = 0;
    for (int i = 0; i < n; i++)
    {
        hd[i].gran3 = gather_gran(w3);
        hd[i].fused = hd[i].win2 = 1;
        hd[i].far = far.p + n_far;
        n_far += (size_t)b->sc[i]->cap_c3;
        nf[i] = batch_blocks(hd[i], BatchKernel::Far);
    }
    BCK(b->descs.ensure(n));
    BCK(hipMemcpyAsync(b->descs.p, hd.data(), n * sizeof(SceneStep), hipMemcpyHostToDevice, b->stream));
    BRC(build_maps(b, {{&b->m_far, &nf}}));
    hipEvent_t e0, e1;
    BCK(hipEventCreate(&e0));
    BCK(hipEventCreate(&e1));
    int rc = PPPM_OK;
    for (int c = 0; c < kClasses && rc == PPPM_OK; c++)
    {
        std::vector<int> members;
        for (int i = 0; i < n; i++)
            if (size_class(b->sc[i]->N) == c)
                members.push_back(i);
        if (members.empty())
            continue;
        float best = 1e30f;
        int best_v = b->variant[members[0]];
        for (int v = 0; v < kFdtdVariants && rc == PPPM_OK; v++)
        {
            for (int i : members)
                b->variant[i] = v;
            if ((rc = build_fdtd(b)) != PPPM_OK)
                break;
            // these launches do not advance t: repeating them rewrites the same values
            for (int w = 0; w < 2 && rc == PPPM_OK; w++)
                rc = enqueue_batch_head(b);
            if (hipEventRecord(e0, b->stream) != hipSuccess)
                rc = bfail(b, PPPM_ERR_HIP, "autotune: event record");
            for (int r = 0; r < reps && rc == PPPM_OK; r++)
                rc = enqueue_batch_head(b);
            if (rc == PPPM_OK && (hipEventRecord(e1, b->stream) != hipSuccess ||
                                  hipEventSynchronize(e1) != hipSuccess))
                rc = bfail(b, PPPM_ERR_HIP, "autotune: event wait");
            float ms = 0;
            if (rc == PPPM_OK && hipEventElapsedTime(&ms, e0, e1) == hipSuccess)
            {
                if (ms_out)
                    ms_out[c * kFdtdVariants + v] = ms / reps;
                if (ms < best)
                {
                    best = ms;
                    best_v = v;
                }
            }
        }
        for (int i : members)
            b->variant[i] = best_v;
    }
    (void)hipEventDestroy(e0);
    (void)hipEventDestroy(e1);
    (void)hipStreamSynchronize(b->stream);  // the scratch goes out of scope
    return rc;
}

}  // extern "C"
