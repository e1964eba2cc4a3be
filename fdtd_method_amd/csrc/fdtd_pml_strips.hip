// PML strip passes of FP64 and FP32 grids: the launch.
#include "fdtd_pml_strips.hpp"

namespace fdtd::rt {

template <typename S>
int launch_pml_strip_s(fdtd_grid* g, bool final, int slot) {
    using C = S;
    const int in = g->cur, out = 1 - g->cur, bin = g->bs_cur, bout = 1 - g->bs_cur;
    fdtd::PmlStripArgs<S, C> a;
    a.in = fields_of<S>(g, in);
    a.out = fields_of<S>(g, out);
    a.es_in = static_cast<const S*>(g->ES[in][0]);
    a.es_out = static_cast<S*>(g->ES[out][0]);
    a.bs_in = static_cast<const S*>(g->BS[bin][0]);
    a.bs_out = static_cast<S*>(g->BS[bout][0]);
    a.stride = g->split_stride / sizeof(S);
    a.tx = static_cast<const C*>(g->pml_tab);
    a.ty = a.tx + 5 * g->Ni;
    a.tz = a.tx + 5 * (g->Ni + g->Nj);
    a.pi = g->pml_p[0];
    a.pj = g->pml_p[1];
    a.pk = g->pml_p[2];
    a.packs = g->Ni * sizeof(S) % 16 == 0;
    a.nsrc = g->nsrc;
    a.pad = 0;
    a.src = g->d_src;
    a.kstart = g->d_kstart;
    a.vals = g->d_vals ? g->d_vals + (size_t)slot * g->nsrc : nullptr;
    a.c = make_coefs<C>(g);
    a.g = make_pml_strip_geom(g, g->pml_strip_kchunk);
    auto kern = final ? fdtd::pml_strip_sweep<S, C, true> : fdtd::pml_strip_sweep<S, C, false>;
    const size_t lds = fdtd::pml_strip_lds_bytes(sizeof(C), a.g.kchunk);
    if (int rc = allow_dynamic_lds(reinterpret_cast<const void*>(kern), lds)) return rc;
    hipLaunchKernelGGL(kern, dim3(8 * a.g.per_xcd), dim3(64 * a.g.W), lds, g->stream, a);
    HIP_TRY(hipGetLastError());
    g->cur = out;
    g->bs_cur = bout;
    return FDTD_OK;
}

int launch_pml_strip(fdtd_grid* g, bool final, int slot) {
    switch (g->precision) {
        case FDTD_FP64: return launch_pml_strip_s<double>(g, final, slot);
        case FDTD_FP32: return launch_pml_strip_s<float>(g, final, slot);
        default: return fail(FDTD_ERR_UNSUPPORTED, "PML strip passes hold FP64 or FP32");
    }
}

}  // namespace fdtd::rt
