// PML strip passes: two steps of a PML grid per read and write of its state.
#pragma once

#include <hip/hip_runtime.h>

#include "fdtd_internal.hpp"

namespace fdtd {

// A pass maps the state between two steps of a PML run, (E_n, B after step
// n+1's first B update), to the state two steps later; the lanes and level
// pipeline are the strip passes' (strip_tile, L = 2).  Level l
// at iteration kk computes E_l at plane kk-l and B_l at plane kk-l-1, main
// cells with the strip passes' expressions, layer cells by their splits with
// the fused PML sweep's, so a pass is bit-identical to two of its sweeps.
//
// A layer cell is its twelve splits: the totals are their sums (rounded as
// stored) and are neither read nor written, except that the last pass of a
// run writes every total.  Neighbouring tiles recompute ghost cells from the
// pass's input, so the B splits are ping-ponged like the others.
//
// Split fields through a pass, per row of a lane: E splits of plane kk go
// from level 0 to level 1 one iteration later (esh); the B splits of plane
// kk wait one iteration for E of plane kk+1 (bs0), and level 0's results
// another one for level 1 (bs1).
//
// Planes come in through LDS (a layer cell's splits or, in the same places, a
// main cell's E and B): they are on their way while the previous plane is
// worked on, and hold no registers.  The wait for a plane leaves the stores
// issued after its loads under way.
//
// What bounds it: memory.  512^3 FP32 with a 0.2 layer: 3.32 ms per pass, where
// two fused sweeps take 6.4; 18.6 GB of traffic (a cell's words once would be
// 11.5; neighbouring tiles read their ghost cells again, and 52 columns touch
// three 128-byte lines a row), 5.6 TB/s where a plain copy reaches 4.7; the
// arithmetic alone takes 1.7 ms.  Registers and LDS hold no larger
// tile: 42 words of state a cell.  FP32 tiles of 128 x 16 cells, one workgroup a
// CU, took 3.73 ms, of 64 x 32 3.92.  FP64: 256^3 0.95 ms (two sweeps 1.59),
// 128^3 0.168 (0.200).
constexpr int kPmlStripL = 2;

template <typename S, typename C>
struct PmlStripArgs {
    Fields<S> in;
    Fields<S> out;
    const S* es_in;           // six E splits, `stride` cells apart, and so on
    const S* bs_in;
    S* es_out;
    S* bs_out;
    size_t stride;
    const C* tx;              // per-axis tables, see Pml
    const C* ty;
    const C* tz;
    int pi, pj, pk;
    int packs;                // rows are whole 16-byte packs
    int nsrc;
    int pad;
    const PointSource* src;   // sorted by plane
    const int* kstart;
    const double* vals;       // values of the pass's first step; step l at vals + l*nsrc
    Coefs<C> c;
    StripGeom g;
};

// Tiles: W wavefronts of 64 lanes, a column and R rows of cells a lane.  Two
// FP32 workgroups share a CU (128 registers a lane, 66 KB of LDS each), one FP64
// workgroup fills it.
constexpr int kPmlStripW = 8, kPmlStripR = 2;
__host__ __device__ constexpr int pml_strip_wgs(int csize) { return csize == 8 ? 1 : 2; }
// ghost and stored columns: ghosts of at least L, stored rows of whole 64-byte
// granules (FP32 48 of 64 columns, FP64 56)
__host__ __device__ constexpr int pml_strip_ghost(int csize) { return 32 / csize; }
__host__ __device__ constexpr int pml_strip_columns(int csize) { return 64 - 2 * pml_strip_ghost(csize); }
// LDS: the row exchange, one input plane of twelve components, and the tables
// of the tile's columns, rows and planes.
__host__ __device__ constexpr size_t pml_strip_lds_bytes(int csize, int kchunk) {
    const int RW = 64, rows = kPmlStripW * kPmlStripR;
    return (static_cast<size_t>(4) * strip_exchange_bufs(kPmlStripL) * kPmlStripW * RW +
            static_cast<size_t>(12) * rows * RW +
            static_cast<size_t>(5) * (RW + rows + kchunk + 2 * kPmlStripL + 1)) * csize;
}

template <typename S, typename C, bool FINAL>
__global__ void __launch_bounds__(64 * kPmlStripW)
__attribute__((amdgpu_waves_per_eu(2 * pml_strip_wgs(sizeof(C)), 2 * pml_strip_wgs(sizeof(C)))))
pml_strip_sweep(PmlStripArgs<S, C> a) {
    static_assert(sizeof(S) == sizeof(C), "loads in units of 4 bytes");
    extern __shared__ __align__(16) unsigned char lds_raw[];
    const int blk = blockIdx.x;
    const int tile = (blk & 7) * a.g.per_xcd + (blk >> 3);
    if (tile >= a.g.ntiles) return;  // whole workgroup
    constexpr int L = kPmlStripL, R = kPmlStripR, W = kPmlStripW;
    constexpr int RW = 64;             // tile columns
    constexpr int RB = RW * static_cast<int>(sizeof(S));
    constexpr int CB = R * RB;         // one component's rows of a wavefront
    constexpr int NP = 1024 / CB;      // components of a 16-byte load of a wavefront
    static_assert(NP == 1 || NP == 2, "whole components per load");
    const StripGeom& G = a.g;
    const int txy = G.ntx * G.nty;
    const int chunk = tile / txy;
    const int rem = tile - chunk * txy;
    const int ty = rem / G.ntx, tx = rem - ty * G.ntx;
    const int Ni = G.Ni, Nj = G.Nj, Nk = G.Nk;
    const int px0 = tx * G.TX, py0 = ty * G.TY;
    const int k0 = chunk * G.kchunk, k1 = min(k0 + G.kchunk, Nk);
    const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), lane = threadIdx.x & 63;
    const int wm = w > 0 ? w - 1 : w, wp = w + 1 < W ? w + 1 : w;
    const int cx = lane;               // tile column
    const size_t plane = static_cast<size_t>(Ni) * Nj;
    const Coefs<C> c = a.c;

    // this lane's cells
    const int gi = wrap_mod(px0 - G.Gx + cx, Ni);
    const bool col_out = cx >= G.Gx && cx < G.Gx + G.TX && px0 + cx - G.Gx < Ni;
    const bool xmain = in_main(gi, Ni, a.pi);
    unsigned off[R];
    bool row_out[R], xym[R];           // xym: main box in x and y
    bool some_main[R], all_main[R];    // of this wavefront's row
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int tr = w * R + r, gj = wrap_mod(py0 - L + tr, Nj);
        row_out[r] = tr >= L && tr < L + G.TY && py0 + tr - L < Nj;
        off[r] = static_cast<unsigned>(gj * Ni + gi) * static_cast<unsigned>(sizeof(S));
        xym[r] = xmain && in_main(gj, Nj, a.pj);
        const unsigned long long m = __ballot(xym[r]);
        some_main[r] = m != 0;
        all_main[r] = m == ~0ull;
    }

    bool wave_main = false;
#pragma unroll
    for (int r = 0; r < R; ++r) wave_main = wave_main || some_main[r];

    using lds_c = __attribute__((address_space(3))) C*;
    using lds_b = __attribute__((address_space(3))) char*;
    using lds_s = const __attribute__((address_space(3))) S*;
    constexpr int NXB = strip_exchange_bufs(L);
    constexpr int XB = 4 * NXB * RW;
    const lds_c xch = (lds_c)reinterpret_cast<C*>(lds_raw);
    auto sB = [&](int l, int q, int ww) { return xch + ww * XB + ((l % NXB) * 4 + q) * RW + cx; };
    auto sE = [&](int l, int q, int ww) { return xch + ww * XB + ((l % NXB) * 4 + 2 + q) * RW + cx; };
    // [wavefront][component][row][RW]
    const lds_b my_stage = (lds_b)(xch + W * XB) + w * (12 * CB);
    const lds_s in_own = (lds_s)my_stage + cx;
    const lds_c sTx = xch + W * XB + 12 * W * R * RW;        // [5][RW]
    const lds_c sTy = sTx + 5 * RW;                          // [5][W * R]
    for (int q = threadIdx.x; q < 5 * RW; q += 64 * W)
        sTx[q] = a.tx[q / RW * Ni + wrap_mod(px0 - G.Gx + q % RW, Ni)];
    for (int q = threadIdx.x; q < 5 * W * R; q += 64 * W)
        sTy[q] = a.ty[q / (W * R) * Nj + wrap_mod(py0 - L + q % (W * R), Nj)];
    const int nz = G.kchunk + 2 * L + 1;
    const lds_c sTz = sTy + 5 * W * R;                       // [5][nz], planes kfirst-2 to klast
    for (int q = threadIdx.x; q < 5 * nz; q += 64 * W)
        sTz[q] = a.tz[q / nz * Nk + wrap_mod(k0 - L - 1 + q % nz, Nk)];

    // E and B pointers are read from the kernel's arguments, and the multiples
    // of the splits' distance formed, where they are used: kept in scalar
    // registers, they would be spilled.
    auto split_stride = [&]() {
        size_t st = a.stride;
        asm volatile("" : "+s"(st));
        return st;
    };
    auto kernel_args = [&]() {
        auto ka = (cptr<PmlStripArgs<S, C>>)__builtin_amdgcn_kernarg_segment_ptr();
        asm volatile("" : "+s"(ka));
        return ka;
    };
    // Plane loads.  Where rows are whole 16-byte packs (a.packs), 16 bytes per
    // lane: one load for the wavefront's rows of a component (FP64) or of two
    // split fields (FP32, the upper lanes one stride further on).  Packs that
    // hold both kinds of cells, and other rows, take 4 bytes per lane, lane l
    // dwords l and 64 + l of a row.
    constexpr int PK = 16 / static_cast<int>(sizeof(S)), ES = static_cast<int>(sizeof(S));
    // of the pack that starts at column i: does it hold main cells, layer cells
    auto pack_main = [&](int i) { return i + PK > a.pi && i < Ni - a.pi; };
    auto pack_layer = [&](int i) { return i < a.pi || i + PK > Ni - a.pi; };
    const int pcol = lane * 16 % RB / ES;
    const int pgi = wrap_mod(px0 - G.Gx + pcol, Ni);
    const int pgj = wrap_mod(py0 - L + w * R + lane * 16 % CB / RB, Nj);
    const unsigned p_off = static_cast<unsigned>(pgj * Ni + pgi) * static_cast<unsigned>(ES);
    const unsigned p_off2 = p_off + (lane * 16 / CB) * static_cast<unsigned>(a.stride * ES);
    const bool p_need = a.packs && pcol + PK > G.Gx - L && pcol < G.Gx + G.TX + L;
    const bool p_row = in_main(pgj, Nj, a.pj);
    const bool p_main = p_need && p_row && !pack_layer(pgi);       // main box, where the plane is
    const bool p_mixed = p_need && p_row && pack_main(pgi) && pack_layer(pgi);
    constexpr int ND = RB / 256;
    unsigned l_off[ND];                // of a row
    bool l_need[ND], l_xmain[ND];
    bool some_mixed = false;
#pragma unroll
    for (int h = 0; h < ND; ++h) {
        const int lb = (h * 64 + lane) * 4, lc = lb / ES, lgi = wrap_mod(px0 - G.Gx + lc, Ni);
        const int lp = lgi / PK * PK;
        l_off[h] = static_cast<unsigned>(lgi * ES + lb % ES);
        l_need[h] = lc >= G.Gx - L && lc < G.Gx + G.TX + L &&
                    (!a.packs || (pack_main(lp) && pack_layer(lp)));
        l_xmain[h] = in_main(lgi, Ni, a.pi);
        some_mixed = some_mixed || __ballot(l_need[h]) != 0;
    }
    const unsigned stage_addr = __builtin_amdgcn_readfirstlane(
        static_cast<unsigned>(reinterpret_cast<unsigned long long>(my_stage)));
    auto stage_load = [&](int kw) {
        auto ka = kernel_args();
        const size_t st = split_stride();
        const bool km = in_main(kw, Nk, a.pk);
        const size_t po = kw * plane;
        const S* const es_p = a.es_in + po;
        const S* const bs_p = a.bs_in + po;
        if (a.packs) {
            if (p_need && !(km && (p_main || p_mixed))) {
#pragma unroll
                for (int q = 0; q < 6; q += NP) {
                    load_to_lds<16>(uniform_gptr<const S>(es_p + q * st), p_off2, stage_addr + q * CB);
                    load_to_lds<16>(uniform_gptr<const S>(bs_p + q * st), p_off2, stage_addr + (6 + q) * CB);
                }
            }
            if (km && p_main && lane * 16 < CB) {
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    load_to_lds<16>(uniform_gptr<const S>(ka->in.e[d] + po), p_off, stage_addr + d * CB);
                    load_to_lds<16>(uniform_gptr<const S>(ka->in.b[d] + po), p_off, stage_addr + (6 + d) * CB);
                }
            }
        }
        if (some_mixed && (km || !a.packs)) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int gj = wrap_mod(py0 - L + w * R + r, Nj);
                const bool rowm = km && in_main(gj, Nj, a.pj);
                if (a.packs && !rowm) continue;
                const size_t ro = static_cast<size_t>(gj) * Ni;
#pragma unroll
                for (int h = 0; h < ND; ++h) {
                    const unsigned dst = stage_addr + r * RB + h * 256;
                    if (l_need[h] && !(rowm && l_xmain[h])) {
#pragma unroll
                        for (int q = 0; q < 6; ++q) {
                            load_to_lds<4>(uniform_gptr<const S>(es_p + (q * st + ro)), l_off[h], dst + q * CB);
                            load_to_lds<4>(uniform_gptr<const S>(bs_p + (q * st + ro)), l_off[h], dst + (6 + q) * CB);
                        }
                    }
                    if (rowm && l_need[h] && l_xmain[h]) {
#pragma unroll
                        for (int d = 0; d < 3; ++d) {
                            load_to_lds<4>(uniform_gptr<const S>(ka->in.e[d] + (po + ro)), l_off[h], dst + d * CB);
                            load_to_lds<4>(uniform_gptr<const S>(ka->in.b[d] + (po + ro)), l_off[h], dst + (6 + d) * CB);
                        }
                    }
                }
            }
        }
    };

    // Whether a point source lies in this tile's columns and rows.
    bool tile_src = a.nsrc > kTileSrcScan;
    if (a.nsrc > 0 && !tile_src) {
        const cptr<PointSource> src = as_const(a.src);
        for (int q = 0; q < a.nsrc; ++q) {
            const int di = wrap_mod(src[q].i - px0 + G.Gx, Ni), dj = wrap_mod(src[q].j - py0 + L, Nj);
            tile_src = tile_src || (di < RW && dj < W * R);
        }
    }
    const cptr<int> kst = as_const(a.kstart);
    auto add_sources = [&](C (&t)[R][3], int q0, int q1, const double* vals_g) {
        const cptr<PointSource> src = as_const(a.src);
        const cptr<double> vals = as_const(vals_g);
        for (int q = q0; q < q1; ++q) {
            const int comp = src[q].comp;
            const C x = (comp == 0 ? c.jx : (comp == 1 ? c.jy : c.jz)) * C(vals[q]);
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const bool row = wrap_mod(py0 - L + w * R + r, Nj) == src[q].j;
                const bool hit = row && src[q].i == gi;
#pragma unroll
                for (int d = 0; d < 3; ++d)
                    if (comp == d) t[r][d] = hit ? x + t[r][d] : t[r][d];
            }
        }
    };

    const int kfirst = k0 - L + 1, klast = k1 + L - 1;

    C eP[L][R][3], bP[L][R][3];  // as in strip_tile
    C esh[R][6], bs0[R][6], bs1[R][6];
#pragma unroll
    for (int r = 0; r < R; ++r) {
#pragma unroll
        for (int q = 0; q < 6; ++q) esh[r][q] = bs0[r][q] = bs1[r][q] = C(0);
#pragma unroll
        for (int l = 0; l < L; ++l)
#pragma unroll
            for (int d = 0; d < 3; ++d) eP[l][r][d] = bP[l][r][d] = C(0);
    }
    int kp[L + 1];                     // planes kk, kk-1, kk-2
#pragma unroll
    for (int l = 0; l <= L; ++l) kp[l] = wrap_mod(kfirst - l, Nk);
    stage_load(kp[0]);
    {
        // Bx and By of plane kfirst-1
        const bool km = in_main(kp[1], Nk, a.pk);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const size_t at0 = kp[1] * plane + off[r] / sizeof(S);
            if (km && xym[r]) {
                bP[0][r][0] = a.in.b[0][at0];
                bP[0][r][1] = a.in.b[1][at0];
            } else {
                bP[0][r][0] = as_stored<S>(a.bs_in[kBxy * a.stride + at0] + a.bs_in[kBxz * a.stride + at0]);
                bP[0][r][1] = as_stored<S>(a.bs_in[kByz * a.stride + at0] + a.bs_in[kByx * a.stride + at0]);
            }
        }
    }
    // level 0's E rows (read for ghost-plane results only)
    sE(0, 0, w)[0] = C(0);
    sE(0, 1, w)[0] = C(0);

    // Plane k's x[0..n) to o(0)..o(n-1), the cells of this tile whose kind is
    // `main` or, with all, every one.
    auto store = [&](auto o, auto ncomp, const auto& x, int k, bool kmain, bool main, bool all) {
        constexpr int n = decltype(ncomp)::value;
        const size_t po = static_cast<size_t>(k) * plane;
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (row_out[r] && col_out && (all || (kmain && xym[r]) == main)) {
#pragma unroll
                for (int q = 0; q < n; ++q)
                    __builtin_nontemporal_store(static_cast<S>(x[r][q]),
                                                generic(at(uniform_gptr<S>(o(q) + po), off[r])));
            }
    };
    const std::integral_constant<int, 6> splits{};
    const std::integral_constant<int, 3> fields{};
    int nst = 0;                       // stores certainly issued after the staged plane's loads
    for (int kk = kfirst; kk <= klast; ++kk) {
        // main box in z at those planes
        const bool km[L + 1] = {in_main(kp[0], Nk, a.pk), in_main(kp[1], Nk, a.pk), in_main(kp[2], Nk, a.pk)};
        const int kn = kp[0] + 1 == Nk ? 0 : kp[0] + 1;
        // whether E of plane kk-L+1 and B of plane kk-L are stored
        const bool e_here = kk - L + 1 >= k0 && kk - L + 1 < k1, b_here = kk - L >= k0 && kk - L < k1;
        C es[R][6], bsn[R][6], bin[R][3], ein[R][3];
        // plane kk has arrived; stores issued after its loads may be under way
        if (nst >= 24)
            __builtin_amdgcn_s_waitcnt(0x4F78);  // vmcnt(24)
        else if (nst >= 12)
            __builtin_amdgcn_s_waitcnt(0x0F7C);  // vmcnt(12)
        else
            wait_vmem_all();
        asm volatile("" ::: "memory");  // the plane's reads stay behind the wait for it
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                es[r][q] = in_own[(q * R + r) * RW];
                bsn[r][q] = in_own[((6 + q) * R + r) * RW];
            }
        // these reads end before the next plane's loads write there
        asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
        if (kk < klast) stage_load(kn);
        nst = 0;
#pragma unroll
        for (int r = 0; r < R; ++r)
            if (row_out[r])
                nst += (e_here && !(km[L - 1] && some_main[r]) ? 6 : 0) + (b_here && !(km[L] && some_main[r]) ? 6 : 0);
#pragma unroll
        for (int r = 0; r < R; ++r) {
            const bool m = km[0] && xym[r];
            C (&s)[6] = bsn[r];
            bin[r][0] = m ? s[0] : as_stored<S>(s[kBxy] + s[kBxz]);
            bin[r][1] = m ? s[1] : as_stored<S>(s[kByz] + s[kByx]);
            bin[r][2] = m ? s[2] : as_stored<S>(s[kBzx] + s[kBzy]);
#pragma unroll
            for (int d = 0; d < 3; ++d) ein[r][d] = es[r][d];
        }
        sB(0, 0, w)[0] = bin[R - 1][0];
        sB(0, 1, w)[0] = bin[R - 1][2];
        __syncthreads();

#pragma unroll
        for (int l = 0; l < L; ++l) {
            C (&se)[R][6] = l == 0 ? es : esh;    // E splits of plane kk-l
            C (&sb)[R][6] = l == 0 ? bs0 : bs1;   // B splits of plane kk-l-1
            C bx_jm[R], bz_jm[R], by_im[R], bz_im[R], enew[R][3], bnew[R][3];
#pragma unroll
            for (int r = 0; r < R; ++r) {
                bx_jm[r] = r > 0 ? bin[r > 0 ? r - 1 : 0][0] : sB(l, 0, wm)[0];
                bz_jm[r] = r > 0 ? bin[r > 0 ? r - 1 : 0][2] : sB(l, 1, wm)[0];
                by_im[r] = lane_prev(bin[r][1]);
                bz_im[r] = lane_prev(bin[r][2]);
#pragma unroll
                for (int d = 0; d < 3; ++d) enew[r][d] = C(0);
            }
            if (km[l] && wave_main) {
                C t[R][3];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    t[r][0] = c.ex_bz * (bin[r][2] - bz_jm[r]);
                    t[r][1] = c.ey_bx * (bin[r][0] - bP[l][r][0]);
                    t[r][2] = c.ez_by * (bin[r][1] - by_im[r]);
                }
                if (tile_src) {
                    const int q0 = kst[kp[l]], q1 = kst[kp[l] + 1];
                    if (q1 > q0) add_sources(t, q0, q1, a.vals + static_cast<size_t>(l) * a.nsrc);
                }
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    enew[r][0] = ein[r][0] + sub_mul(t[r][0], c.ex_by, bin[r][1] - bP[l][r][1]);
                    enew[r][1] = ein[r][1] + sub_mul(t[r][1], c.ey_bz, bin[r][2] - bz_im[r]);
                    enew[r][2] = ein[r][2] + sub_mul(t[r][2], c.ez_bx, bin[r][0] - bx_jm[r]);
                }
            }
            {
                const lds_c z = sTz + (kk - l - (k0 - L - 1));
                const C az = z[0], cz_xz = z[nz], cz_yz = z[2 * nz];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    if (km[l] && all_main[r]) continue;
                    const int tr = w * R + r;
                    const C ay = sTy[tr], cy_xy = sTy[W * R + tr], cy_zy = sTy[2 * W * R + tr];
                    C (&s)[6] = se[r];
                    const C ax = sTx[cx], cx_yx = sTx[RW + cx], cx_zx = sTx[2 * RW + cx];
                    s[kExy] = stored<S, C>(s[kExy] * ay + cy_xy * (bin[r][2] - bz_jm[r]));
                    s[kEzy] = stored<S, C>(s[kEzy] * ay - cy_zy * (bin[r][0] - bx_jm[r]));
                    s[kExz] = stored<S, C>(s[kExz] * az - cz_xz * (bin[r][1] - bP[l][r][1]));
                    s[kEyz] = stored<S, C>(s[kEyz] * az + cz_yz * (bin[r][0] - bP[l][r][0]));
                    s[kEyx] = stored<S, C>(s[kEyx] * ax - cx_yx * (bin[r][2] - bz_im[r]));
                    s[kEzx] = stored<S, C>(s[kEzx] * ax + cx_zx * (bin[r][1] - by_im[r]));
                    const bool m = km[l] && xym[r];
                    enew[r][0] = m ? enew[r][0] : s[kExz] + s[kExy];
                    enew[r][1] = m ? enew[r][1] : s[kEyx] + s[kEyz];
                    enew[r][2] = m ? enew[r][2] : s[kEzy] + s[kEzx];
                }
            }
            if (l == L - 1 && e_here) {
                auto ka = kernel_args();
                const size_t st = split_stride();
                store([&](int q) { return a.es_out + q * st; }, splits, esh, kk - L + 1, km[L - 1], false, false);
                if (FINAL || (km[L - 1] && wave_main))
                    store([&](int q) { return ka->out.e[q]; }, fields, enew, kk - L + 1, km[L - 1], true, FINAL);
            }
            // B of plane kk-l-1
            {
                const lds_c z = sTz + (kk - l - 1 - (k0 - L - 1));
                const C az = z[0], cz_xz = z[3 * nz], cz_yz = z[4 * nz];
#pragma unroll
                for (int r = 0; r < R; ++r) {
                    const bool some = km[l + 1] && some_main[r], all = km[l + 1] && all_main[r];
                    const int tr = w * R + r;
                    const C ey_ip = lane_next(eP[l][r][1]), ez_ip = lane_next(eP[l][r][2]);
                    const C ex_jp = r < R - 1 ? eP[l][r < R - 1 ? r + 1 : r][0] : sE(l, 0, wp)[0];
                    const C ez_jp = r < R - 1 ? eP[l][r < R - 1 ? r + 1 : r][2] : sE(l, 1, wp)[0];
                    const C ex = eP[l][r][0], ey = eP[l][r][1], ez = eP[l][r][2];
                    C b[3] = {bP[l][r][0], bP[l][r][1], bP[l][r][2]};
                    if (some) {
                        const C dbx = sub_mul(c.bx_ey * (enew[r][1] - ey), c.bx_ez, ez_jp - ez);
                        const C dby = sub_mul(c.by_ez * (ez_ip - ez), c.by_ex, enew[r][0] - ex);
                        const C dbz = sub_mul(c.bz_ex * (ex_jp - ex), c.bz_ey, ey_ip - ey);
                        b[0] = b[0] + dbx;
                        b[1] = b[1] + dby;
                        b[2] = b[2] + dbz;
                        if (!(FINAL && l == L - 1)) {
                            b[0] = b[0] + dbx;
                            b[1] = b[1] + dby;
                            b[2] = b[2] + dbz;
                        }
                    }
                    if (!all) {
                        const bool m = km[l + 1] && xym[r];
                        C x[3] = {bP[l][r][0], bP[l][r][1], bP[l][r][2]};
                        // (a run's last B update leaves the layer as it is)
                        if (!(FINAL && l == L - 1)) {
                            const C ax = sTx[cx], ay = sTy[tr];
                            C (&s)[6] = sb[r];
                            s[kByx] = stored<S, C>(s[kByx] * ax + sTx[3 * RW + cx] * (ez_ip - ez));
                            s[kBzx] = stored<S, C>(s[kBzx] * ax - sTx[4 * RW + cx] * (ey_ip - ey));
                            s[kBxy] = stored<S, C>(s[kBxy] * ay - sTy[3 * W * R + tr] * (ez_jp - ez));
                            s[kBzy] = stored<S, C>(s[kBzy] * ay + sTy[4 * W * R + tr] * (ex_jp - ex));
                            s[kBxz] = stored<S, C>(s[kBxz] * az + cz_xz * (enew[r][1] - ey));
                            s[kByz] = stored<S, C>(s[kByz] * az - cz_yz * (enew[r][0] - ex));
                            x[0] = s[kBxy] + s[kBxz];
                            x[1] = s[kByz] + s[kByx];
                            x[2] = s[kBzx] + s[kBzy];
                        }
#pragma unroll
                        for (int d = 0; d < 3; ++d) b[d] = m ? b[d] : x[d];
                    }
#pragma unroll
                    for (int d = 0; d < 3; ++d) bnew[r][d] = as_stored<S>(b[d]);
                }
            }
#pragma unroll
            for (int r = 0; r < R; ++r)
#pragma unroll
                for (int d = 0; d < 3; ++d) {
                    ein[r][d] = as_stored<S>(eP[l][r][d]);
                    eP[l][r][d] = enew[r][d];
                    bP[l][r][d] = bin[r][d];
                    bin[r][d] = bnew[r][d];
                }
            if (l < L - 1) {
                sB(l + 1, 0, w)[0] = bin[R - 1][0];
                sB(l + 1, 1, w)[0] = bin[R - 1][2];
                sE(l + 1, 0, w)[0] = eP[l + 1][0][0];
                sE(l + 1, 1, w)[0] = eP[l + 1][0][2];
                __syncthreads();
            }
        }
        if (b_here) {
            auto ka = kernel_args();
            const size_t st = split_stride();
            store([&](int q) { return a.bs_out + q * st; }, splits, bs1, kk - L, km[L], false, false);
            if (FINAL || (km[L] && wave_main))
                store([&](int q) { return ka->out.b[q]; }, fields, bin, kk - L, km[L], true, FINAL);
        }
#pragma unroll
        for (int r = 0; r < R; ++r)
#pragma unroll
            for (int q = 0; q < 6; ++q) {
                esh[r][q] = es[r][q];
                bs1[r][q] = bs0[r][q];
                bs0[r][q] = bsn[r][q];
            }
        sE(0, 0, w)[0] = eP[0][0][0];
        sE(0, 1, w)[0] = eP[0][0][2];
        kp[2] = kp[1];
        kp[1] = kp[0];
        kp[0] = kn;
    }
}

}  // namespace fdtd
