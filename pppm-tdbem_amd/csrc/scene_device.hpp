// Scene descriptors of the batched launches, as a block reads them.
//
// A descriptor lives in device memory, so without help its pointers are generic: every access
// through them is a FLAT instruction (an LDS aperture check, both wait counters, a 64-bit address per
// lane), and each word of it a vector register. Here a block reads it through the scalar cache (no
// kernel writes descriptors) and its pointers are declared global.
#pragma once
#include "internal.hpp"

namespace pppm_amd
{

// a T that no thread writes while the kernel runs, through the scalar cache
template <class T>
__device__ __forceinline__ T const_load(const T *p)
{
    static_assert(sizeof(T) % 4 == 0, "copied by words");
    typedef const __attribute__((address_space(4))) unsigned *Src;
    const Src src = (Src)(unsigned long long)p;
    unsigned w[sizeof(T) / 4];
#pragma unroll
    for (unsigned i = 0; i < sizeof(T) / 4; i++)
        w[i] = src[i];
    T out;
    __builtin_memcpy(&out, w, sizeof(T));
    return out;
}

template <class T>
__device__ __forceinline__ void as_global(T *&p)
{
    // by way of an integer: a cast to global and back would be folded away
    p = (T *)(__attribute__((address_space(1))) T *)(unsigned long long)p;
}
template <class... P>
__device__ __forceinline__ void all_global(P &...p)
{
    (as_global(p), ...);
}

__device__ __forceinline__ SceneStep scene_desc(const SceneStep *ds, int i)
{
    SceneStep d = const_load(ds + i);
    all_global(d.st, d.grid3, d.c3_cells, d.c3_start, d.c3_wave, d.c3_pairs, d.face_start, d.face_wave, d.face_nbr,
               d.face_slot, d.wf, d.wb, d.fw, d.sf, d.sb, d.fsc, d.owf, d.owb, d.ofw, d.osf, d.osb, d.ofsc, d.interp,
               d.corner, d.geom, d.err, d.hn, d.hd, d.wn, d.wd, d.far, d.ffar, d.neumann, d.lcell, d.lc3, d.c3_index, d.out);
    return d;
}
__device__ __forceinline__ FdtdScene scene_desc(const FdtdScene *ds, int i)
{
    FdtdScene d = const_load(ds + i);
    all_global(d.grid3, d.st);
    return d;
}
__device__ __forceinline__ AdjScene scene_desc(const AdjScene *ds, int i)
{
    AdjScene d = const_load(ds + i);
    all_global(d.ast, d.lam3, d.bb, d.ln, d.ld, d.unear, d.lfar, d.v, d.c3_cells, d.tc3, d.wf, d.wb, d.fw, d.sf, d.sb,
               d.fsc, d.ft_start, d.ft_c, d.ft_slot, d.tfw, d.tfsc, d.ct_start, d.ct_c, d.ct_w, d.den, d.lcell, d.lc3,
               d.gout, d.grad);
    return d;
}

// Scene and local block of block b of a launch that covers the blocks of every scene: virtual
// block v belongs to scene m.scene_of[v] as its local block v - m.first[scene]. Blocks go to the 8
// XCDs in turn and block b takes virtual block (b % 8) * m.per + b / 8, so each XCD works through
// one contiguous run of scenes (their lists, windows and grids stay in that XCD's L2).
__device__ __forceinline__ bool map_block(const BatchMap &m, int b, int &scene, int &local)
{
    const int v = (b & 7) * m.per + (b >> 3);
    if (v >= m.total)
        return false;
    scene = const_load(m.scene_of + v);
    local = v - const_load(m.first + scene);
    return true;
}

}  // namespace pppm_amd
