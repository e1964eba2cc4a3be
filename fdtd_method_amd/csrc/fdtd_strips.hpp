// The strip passes of one storage type: kernel selection and launches of
// single grids and batches.  Included by one translation unit per type
// (fdtd_strips_fp64/fp32/fp16.hip), which compile side by side.
#pragma once

#include <hip/hip_runtime.h>

#include "fdtd_internal.hpp"

namespace fdtd::rt {

// The strip kernel of a launch (STAGE: planes through LDS; FIRST: with the
// run's first half step).  FP16: the pass
// after an in-run rescaling decision scales its reads; passes of a run with
// probes record them.
template <typename S, int V, int R, int L, bool FINAL, bool STAGE, int LN, bool FIRST>
auto strip_kernel(bool rescale, bool probe) {
    using C = typename fdtd::ComputeOf<S>::type;
    auto kern = probe ? fdtd::strip_sweep<S, C, V, R, L, FINAL, STAGE, LN, FIRST, true>
                      : fdtd::strip_sweep<S, C, V, R, L, FINAL, STAGE, LN, FIRST, false>;
    if constexpr (sizeof(S) == 2 && !FIRST)
        if (rescale)
            kern = probe ? fdtd::strip_rescale_sweep<S, C, V, R, L, FINAL, STAGE, true>
                         : fdtd::strip_rescale_sweep<S, C, V, R, L, FINAL, STAGE, false>;
    return kern;
}

template <typename S, int V, int R, int L, bool FINAL>
int launch_strip_v(fdtd_grid* g, bool first, int slot, int in, int out, void* const* in_b,
                   void* const* ahead) {
    using C = typename fdtd::ComputeOf<S>::type;
    if constexpr (!strip_built(sizeof(C), V, R)) {
        return fail(FDTD_ERR_UNSUPPORTED, "strip variant V=%d R=%d not built", V, R);
    } else {
        const BlockTuning& t = g->btune;
        fdtd::StripArgs<S, C> a;
        a.in = fields_of<S>(g, in);
        if (in_b)
            for (int d = 0; d < 3; ++d) a.in.b[d] = static_cast<S*>(in_b[d]);
        a.out = fields_of<S>(g, out);
        for (int d = 0; d < 3; ++d) a.ahead[d] = ahead ? static_cast<S*>(ahead[d]) : nullptr;
        a.src = g->d_src;
        a.kstart = g->d_kstart;
        a.vals = g->d_vals ? g->d_vals + (size_t)slot * g->nsrc : nullptr;
        a.nsrc = g->nsrc;
        a.vstride = g->nsrc;
        a.c = make_coefs<C>(g);
        a.g = make_strip_geom(g, t);
        for (int c = 0; c < 6; ++c) a.iscale[c] = g->pass_iscale[c];
        a.probe = probe_args(g);
        if (first && a.g.depth != 2)  // (it reads E of the next plane from the stage)
            return fail(FDTD_ERR_UNSUPPORTED, "a first pass stages two planes, this one %d", a.g.depth);
        constexpr int SL = fdtd::strip_stage_lanes(sizeof(C));
        auto kern = strip_kernel<S, V, R, L, FINAL, false, 64, false>(g->pass_rescale, probing(g));
        if constexpr (sizeof(C) == 8)
            if (strip_lanes(t, g->precision, a.g.depth) == 32)
                kern = strip_kernel<S, V, R, L, FINAL, false, 32, false>(false, probing(g));
        if constexpr (fdtd::strip_stage_built(V, R, L))
            if (a.g.depth > 0)
                kern = first ? strip_kernel<S, V, R, L, FINAL, true, SL, true>(false, probing(g))
                             : strip_kernel<S, V, R, L, FINAL, true, SL, false>(g->pass_rescale, probing(g));
        const size_t lds = fdtd::strip_lds_bytes(L, a.g.W, V, R, sizeof(C), sizeof(S), a.g.depth);
        if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds)) return rc;
        hipLaunchKernelGGL(kern, dim3(8 * a.g.per_xcd), dim3(64 * a.g.W), lds, g->stream, a);
        HIP_TRY(hipGetLastError());
        if (a.probe.n > 0) g->probe_rows += L;
        return FDTD_OK;
    }
}

// Workgroups of a strip variant resident per CU (0 if it cannot launch).
template <typename S, int V, int R, int L>
int strip_occupancy_v(int W, int depth, int lanes) {
    using C = typename fdtd::ComputeOf<S>::type;
    if constexpr (!strip_built(sizeof(C), V, R)) {
        return 0;
    } else {
        auto kern = fdtd::strip_sweep<S, C, V, R, L, false, false, 64, false>;
        if constexpr (sizeof(C) == 8)
            if (lanes == 32) kern = fdtd::strip_sweep<S, C, V, R, L, false, false, 32, false>;
        if constexpr (fdtd::strip_stage_built(V, R, L))
            if (depth > 0)
                kern = fdtd::strip_sweep<S, C, V, R, L, false, true, fdtd::strip_stage_lanes(sizeof(C)), false>;
        const size_t lds = fdtd::strip_lds_bytes(L, W, V, R, sizeof(C), sizeof(S), depth);
        if (allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds) != FDTD_OK) return 0;
        int n = 0;
        if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&n, kern, 64 * W, lds) != hipSuccess) {
            (void)hipGetLastError();
            return 0;
        }
        return n;
    }
}

template <typename S, int V, int R>
int strip_occupancy_l(int L, int W, int depth, int lanes) {
    switch (L) {
        case 1: return strip_occupancy_v<S, V, R, 1>(W, depth, lanes);
        case 2: return strip_occupancy_v<S, V, R, 2>(W, depth, lanes);
        case 3: return strip_occupancy_v<S, V, R, 3>(W, depth, lanes);
        default: return strip_occupancy_v<S, V, R, 4>(W, depth, lanes);
    }
}

template <typename S>
int strip_occupancy_s(const BlockTuning& t, int depth) {
    const int W = t.TYg / t.R, lanes = t.row_lanes[t.L];
    if (t.V == 1 && t.R == 2) return strip_occupancy_l<S, 1, 2>(t.L, W, depth, lanes);
    if (t.V == 1 && t.R == 4) return strip_occupancy_l<S, 1, 4>(t.L, W, depth, lanes);
    if (t.V == 2 && t.R == 2) return strip_occupancy_l<S, 2, 2>(t.L, W, depth, lanes);
    return 0;
}

template <typename S, int V, int R, bool FINAL>
int launch_strip_l(fdtd_grid* g, bool first, int slot, int in, int out, void* const* in_b,
                   void* const* ahead) {
    switch (g->btune.L) {
        case 1: return launch_strip_v<S, V, R, 1, FINAL>(g, first, slot, in, out, in_b, ahead);
        case 2: return launch_strip_v<S, V, R, 2, FINAL>(g, first, slot, in, out, in_b, ahead);
        case 3: return launch_strip_v<S, V, R, 3, FINAL>(g, first, slot, in, out, in_b, ahead);
        case 4: return launch_strip_v<S, V, R, 4, FINAL>(g, first, slot, in, out, in_b, ahead);
        default: return fail(FDTD_ERR_UNSUPPORTED, "unsupported blocking depth %d", g->btune.L);
    }
}

template <typename S, bool FINAL>
int launch_strip_f(fdtd_grid* g, bool first, int slot, int in, int out, void* const* in_b,
                   void* const* ahead) {
    const int V = g->btune.V, R = g->btune.R;
    if (V == 1 && R == 2) return launch_strip_l<S, 1, 2, FINAL>(g, first, slot, in, out, in_b, ahead);
    if (V == 1 && R == 4) return launch_strip_l<S, 1, 4, FINAL>(g, first, slot, in, out, in_b, ahead);
    if (V == 2 && R == 2) return launch_strip_l<S, 2, 2, FINAL>(g, first, slot, in, out, in_b, ahead);
    return fail(FDTD_ERR_UNSUPPORTED, "unsupported strip shape V=%d R=%d", V, R);
}

// The batched strip kernel of a shape (null: not built).
template <typename S, int V, int R, int L, bool FINAL>
const void* batch_strip_kernel_v(int lanes, bool stage, bool first) {
    using C = typename fdtd::ComputeOf<S>::type;
    if constexpr (!strip_built(sizeof(C), V, R)) {
        return nullptr;
    } else {
        if constexpr (fdtd::strip_stage_built(V, R, L)) {
            constexpr int SL = fdtd::strip_stage_lanes(sizeof(C));
            if (stage)
                return first ? reinterpret_cast<const void*>(fdtd::batch_strip_sweep<S, C, V, R, L, FINAL, true, SL, true>)
                             : reinterpret_cast<const void*>(fdtd::batch_strip_sweep<S, C, V, R, L, FINAL, true, SL, false>);
        }
        if constexpr (sizeof(C) == 8)
            if (lanes == 32)
                return reinterpret_cast<const void*>(fdtd::batch_strip_sweep<S, C, V, R, L, FINAL, false, 32, false>);
        return reinterpret_cast<const void*>(fdtd::batch_strip_sweep<S, C, V, R, L, FINAL, false, 64, false>);
    }
}

template <typename S, int V, int R, bool FINAL>
const void* batch_strip_kernel_l(int L, int lanes, bool stage, bool first) {
    switch (L) {
        case 1: return batch_strip_kernel_v<S, V, R, 1, FINAL>(lanes, stage, first);
        case 2: return batch_strip_kernel_v<S, V, R, 2, FINAL>(lanes, stage, first);
        case 3: return batch_strip_kernel_v<S, V, R, 3, FINAL>(lanes, stage, first);
        default: return batch_strip_kernel_v<S, V, R, 4, FINAL>(lanes, stage, first);
    }
}

template <typename S, bool FINAL>
const void* batch_strip_kernel_s(int V, int R, int L, int lanes, bool stage, bool first) {
    if (V == 1 && R == 2) return batch_strip_kernel_l<S, 1, 2, FINAL>(L, lanes, stage, first);
    if (V == 1 && R == 4) return batch_strip_kernel_l<S, 1, 4, FINAL>(L, lanes, stage, first);
    if (V == 2 && R == 2) return batch_strip_kernel_l<S, 2, 2, FINAL>(L, lanes, stage, first);
    return nullptr;
}

template <typename S>
int launch_strip(fdtd_grid* g, bool final, bool first, int slot, int in, int out, void* const* in_b,
                 void* const* ahead) {
    return final ? launch_strip_f<S, true>(g, first, slot, in, out, in_b, ahead)
                 : launch_strip_f<S, false>(g, first, slot, in, out, in_b, ahead);
}

template <typename S>
const void* batch_strip_kernel(int V, int R, int L, int lanes, bool final, int depth, bool first) {
    if (first && depth != 2) return nullptr;
    const bool stage = depth > 0;
    return final ? batch_strip_kernel_s<S, true>(V, R, L, lanes, stage, first)
                 : batch_strip_kernel_s<S, false>(V, R, L, lanes, stage, first);
}

}  // namespace fdtd::rt
