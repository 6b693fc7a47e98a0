// dvg_memory.h -- address spaces of the kernels' tables.
//
// A pointer that a kernel loads from memory (a job table, its own argument block) is generic
// to the compiler: accesses through it become flat instructions, and even a load whose
// address is the same for the whole wave goes to the vector memory unit.  The scene's tables
// live in global memory and no render kernel writes them, so pointers to them are marked
// constant: uniform loads then go through the scalar cache, the others are global loads.
// Pointers to what kernels write are marked global.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "dvg_scene.h"

namespace dvg {

template <class T>
__device__ __forceinline__ void mark_constant(const T *&p) {
    p = (const T *)(const __attribute__((address_space(4))) T *)(uint64_t)p;
}
template <class T>
__device__ __forceinline__ void mark_global(T *&p) {
    p = (T *)(__attribute__((address_space(1))) T *)(uint64_t)p;
}

// Copy of a trivially copyable object in memory that is constant while the kernel runs; the
// members that are used are read by scalar loads.
template <class T>
__device__ __forceinline__ T load_constant_raw(uint64_t at) {
    static_assert(sizeof(T) % 8 == 0 && alignof(T) <= 8, "read as 64-bit words");
    const __attribute__((address_space(4))) uint64_t *src =
        (const __attribute__((address_space(4))) uint64_t *)at;
    uint64_t words[sizeof(T) / 8];
#pragma unroll
    for (size_t i = 0; i < sizeof(T) / 8; i++) words[i] = src[i];
    T out;
    __builtin_memcpy(&out, words, sizeof(T));
    return out;
}

__device__ __forceinline__ void mark(DevScene &S) {
    mark_constant(S.shape_type), mark_constant(S.stroke_width), mark_constant(S.param_off), mark_constant(S.params);
    mark_constant(S.seg_begin), mark_constant(S.nsegs), mark_constant(S.pt_off), mark_constant(S.npt);
    mark_constant(S.has_thick), mark_constant(S.closed), mark_constant(S.approx), mark_constant(S.shape_box);
    mark_constant(S.seg_idx), mark_constant(S.seg_kind), mark_constant(S.seg_pid), mark_constant(S.seg_box);
    mark_constant(S.seg_maxr), mark_constant(S.seg_wf), mark_constant(S.seg_dfs), mark_constant(S.seg_cdf);
    mark_constant(S.seg_pmf), mark_constant(S.points), mark_constant(S.thickness);
    mark_constant(S.g_off), mark_constant(S.g_n), mark_constant(S.g_ids);
    mark_constant(S.fill_type), mark_constant(S.fill_off), mark_constant(S.fill_ns);
    mark_constant(S.stroke_type), mark_constant(S.stroke_off), mark_constant(S.stroke_ns);
    mark_constant(S.color), mark_constant(S.even_odd), mark_constant(S.s2c), mark_constant(S.c2s);
    mark_constant(S.g_lbox), mark_constant(S.g_box), mark_constant(S.g_maxr), mark_constant(S.g_sdf);
    mark_constant(S.top);
    mark_constant(S.shape_length), mark_constant(S.shapes_cdf), mark_constant(S.shapes_pmf);
    mark_constant(S.sample_shape_id), mark_constant(S.sample_group_id);
    mark_global(S.d_params), mark_global(S.d_points), mark_global(S.d_thickness), mark_global(S.d_stroke_width);
    mark_global(S.d_color), mark_global(S.d_xform), mark_global(S.d_filter_radius);
}

template <class T>
__device__ __forceinline__ T load_constant(uint64_t at) {
    T out = load_constant_raw<T>(at);
    mark(out);
    return out;
}

}  // namespace dvg
